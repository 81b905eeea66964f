"""A small system's finest level by plain block rows for few columns, on the GPU: every column is bit for
bit the single-column V-cycle and solve, in each form, where the columns fill a wavefront's chains and
where they leave some idle."""
import threading

import numpy as np
import pytest

import refcpu
import solidfem_amd as sf
from workloads import FINGERPRINT_PLATE, block_config, loaded

pytestmark = pytest.mark.gpu

ROWS_BATCH_FORM = 112


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


# block rows per wavefront; 16: the form with a lane per scalar row (also on larger systems); -16: the
# restrictions with four wavefronts per row
@pytest.mark.parametrize("rows", [2, 4, 16, -16])
@pytest.mark.parametrize("precision", [0, 1, 2], ids=["double", "single-storage", "single"])
def test_few_columns_by_rows_keep_each_columns_bits(ctx, forced_variant, rows, precision):
    ref = refcpu.Problem(loaded(*FINGERPRINT_PLATE[:2]))
    csr = sf.CsrMatrix.new(ctx, *ref.csr())
    setup = sf.MultigridSetup.new(ctx, csr, ref.rigid_modes(), ref.free_positions(),
                                  sf.MultigridOptions(coarse_dofs=100, precision=precision, coarse_solve=1))
    while not setup.step(2 ** 62):
        pass
    mg = setup.finish()
    opts = sf.PcgOptions(tolerance=1e-8, dot_order=sf.DotOrder.TREE)
    forced_variant(ROWS_BATCH_FORM + rows)
    rng = np.random.default_rng(rows + 16)
    # every count the forms are compiled for (six rows' buffers fit the LDS up to six or seven columns), and
    # 9: past the forms and past the final sums formed by their consumers
    for columns in (1, 2, 3, 4, 5, 6, 7, 8, 9):
        r = rng.standard_normal((columns, ref.free_dofs))
        z = mg.apply_batch(r)
        for m in range(columns):
            assert np.array_equal(bits(z[m]), bits(mg.apply(r[m]))), f"{columns} columns: column {m}"
        if precision == 1 or columns not in (3, 6, 8, 9):
            continue
        batch = sf.PcgBatch.new(ctx, csr, mg, r, opts)
        assert batch.step(100000)[0] == 0
        x = batch.estimate()
        for m in range(columns):
            single = sf.Pcg.new(ctx, csr, mg, r[m], opts)
            single.step(100000)
            assert np.array_equal(bits(single.estimate()), bits(x[m])), f"{columns} columns: column {m}"


def test_a_staged_group_takes_odd_counts_past_a_workgroup_in_another_form(ctx, forced_variant):
    # rows of six and 64 columns, two a thread, are 192 threads' sums, 45 columns, one a thread, 270
    ref = refcpu.Problem(loaded(*FINGERPRINT_PLATE[:2]))
    csr = sf.CsrMatrix.new(ctx, *ref.csr())
    setup = sf.MultigridSetup.new(ctx, csr, ref.rigid_modes(), ref.free_positions(), sf.MultigridOptions(coarse_dofs=100, precision=2, coarse_solve=1))
    while not setup.step(2 ** 62):
        pass
    mg = setup.finish()
    forced_variant(80)
    for columns in (64, 45, 43, 42):
        r = np.random.default_rng(columns).standard_normal((columns, ref.free_dofs))
        z = mg.apply_batch(r)
        for m in range(columns):
            assert np.array_equal(bits(z[m]), bits(mg.apply(r[m]))), f"{columns} columns: column {m}"


def test_a_large_batchs_columns_arrive_and_return_in_pieces(ctx):
    # 48 columns of 11,970 unknowns are 4.4 MiB: one whole pinned piece of 4 MiB and the rest
    ref = refcpu.Problem(block_config(0, divisions=(9, 7, 7)))
    columns = 48
    assert 4 << 20 < columns * ref.free_dofs * 8 < 8 << 20
    csr = sf.CsrMatrix.new(ctx, *ref.csr())
    setup = sf.MultigridSetup.new(ctx, csr, ref.rigid_modes(), ref.free_positions(), sf.MultigridOptions(coarse_dofs=100, precision=2, coarse_solve=1))
    while not setup.step(2 ** 62):
        pass
    mg = setup.finish()
    opts = sf.PcgOptions(tolerance=1e-8, dot_order=sf.DotOrder.TREE)
    r = np.random.default_rng(5).standard_normal((columns, ref.free_dofs))
    batch = sf.PcgBatch.new(ctx, csr, mg, r, opts)
    assert batch.step(100000)[0] == 0
    x = batch.estimate()
    for m in (0, 41, 42, 43, columns - 1):  # the pieces meet in column 43
        single = sf.Pcg.new(ctx, csr, mg, r[m], opts)
        single.step(100000)
        assert np.array_equal(bits(single.estimate()), bits(x[m])), f"column {m}"


def test_two_threads_batches_of_one_context_pass_their_columns_at_once(ctx):
    # one thread's copy at a time holds the context's pinned buffers; the other's is a plain one
    columns, cases = 48, (block_config(0, divisions=(9, 7, 7)), block_config(1, divisions=(9, 8, 7)))
    opts = sf.PcgOptions(tolerance=1e-8, dot_order=sf.DotOrder.TREE)
    batches = []
    for w in cases:
        b = sf.StudyBuilder.new(ctx, sf.Model.from_workload(w), opts, sf.MultigridOptions(coarse_dofs=100, precision=2, coarse_solve=1))
        b.step(2 ** 62)
        study = b.finish()
        rhs = study.rhs() * np.random.default_rng(3).uniform(0.5, 2.0, (columns, 1))
        assert rhs.nbytes > 4 << 20
        batch = sf.PcgBatch.new(ctx, study.system(), study.multigrid(), rhs, opts)
        batch.step(100000)
        batches.append((study, batch, rhs, bits(batch.estimate())))
    wrong = []

    def repeat(batch, rhs, expected):
        for _ in range(10):
            batch.restart(rhs)
            batch.step(100000)
            if not np.array_equal(bits(batch.estimate()), expected):
                wrong.append(rhs.shape)

    threads = [threading.Thread(target=repeat, args=b[1:]) for b in batches]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
