"""The coarsest level's two solves and the restriction's four-wavefronts-per-row form, on the GPU, at
the sizes where their panels, chunks and last rows are cut: every sum is a fixed serial order, so
each is compared bit for bit."""
import numpy as np
import pytest

import refcpu
import solidfem_amd as sf
from workloads import block_config, loaded, plate_config

pytestmark = pytest.mark.gpu

WIDE_ROWS = 96


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def multigrid(ctx, ref, precision, coarse, coarse_solve=0):
    csr = sf.CsrMatrix.new(ctx, *ref.csr())
    setup = sf.MultigridSetup.new(ctx, csr, ref.rigid_modes(), ref.free_positions(),
                                  sf.MultigridOptions(coarse_dofs=coarse, precision=precision, coarse_solve=coarse_solve))
    while not setup.step(2 ** 62):
        pass
    return setup.finish()


def serial(first, terms):
    """first + terms[0] + terms[1] + ..., one rounding each, in order."""
    return np.add.accumulate(np.concatenate([[first], terms]))[-1]


# 54 and 108 unknowns: one panel; 162, the first past it: two; 600: panels of 9 columns; 1260: of 4, and two chunks of 1024;
# 3000, the most that a level is factored for: panels of one column, three chunks, 158 KB of LDS;
# 64 columns of the inverse's product are past the form of eight sums a workgroup from 600 on, 3 columns within it
@pytest.mark.parametrize("divisions", [(1, 1, 1), (2, 1, 1), (3, 1, 1), (4, 2, 2), (6, 3, 2), (4, 2, 12)])
def test_coarse_solves_follow_their_serial_orders(ctx, divisions):
    ref = refcpu.Problem(loaded([float(d) for d in divisions], list(divisions)))
    mg_ref = refcpu.Multigrid(ref, refcpu.options(precision=0, coarse_dofs=100000))
    L = np.tril(mg_ref.coarse_factor())
    n = L.shape[0]
    b = np.random.default_rng(n).standard_normal((3, n))
    mg = multigrid(ctx, ref, 0, 100000)
    want = []
    for column in b:  # block.rs:357-373
        x = column.copy()
        for k in range(n):
            x[k] = x[k] / L[k, k]
            x[k + 1:] -= L[k + 1:, k] * x[k]
        for i in range(n - 1, -1, -1):
            x[i] = serial(x[i], -(L[i + 1:, i] * x[i + 1:])) / L[i, i]
        want.append(x)
    assert np.array_equal(bits(mg.apply(b[0])), bits(want[0]))
    assert np.array_equal(bits(mg.solve_coarsest(b[1])), bits(want[1]))
    assert np.array_equal(bits(mg.apply_batch(b)), bits(np.array(want)))
    fast = mg.with_precision(sf.Precision.DOUBLE, coarse_solve=1)
    inverse = fast.apply_batch(np.eye(n)[:64])  # columns of the inverse, exactly
    for first in range(64, n, 64):
        inverse = np.vstack([inverse, fast.apply_batch(np.eye(n)[first:first + 64])])
    assert np.array_equal(bits(inverse), bits(inverse.T))
    got = fast.apply(b[2])
    assert np.array_equal(bits(fast.apply_batch(b)[2]), bits(got))
    assert np.array_equal(bits(got), bits([serial(0.0, inverse[:, i] * b[2]) for i in range(n)]))


@pytest.mark.parametrize("precision", [0, 1, 2], ids=["double", "single-storage", "single"])
@pytest.mark.parametrize("w", [block_config(0, divisions=(7, 5, 5)), plate_config(divisions=(12, 12, 2))], ids=["block", "plate"])
def test_wide_restriction_rows_keep_the_cycles_bits(ctx, forced_variant, w, precision):
    ref = refcpu.Problem(w)
    r = np.random.default_rng(3).standard_normal(ref.free_dofs)
    expected = multigrid(ctx, ref, precision, 100).apply(r)
    forced_variant(WIDE_ROWS)
    mg = multigrid(ctx, ref, precision, 100)
    assert mg.stats().levels >= 2
    assert np.array_equal(bits(mg.apply(r)), bits(expected))


ROWS_FORCED = 1024


# block rows per wavefront + 256 (blocks a lane loads at once - 1)
@pytest.mark.parametrize("form", [1, 2, 4, 256 + 4])
@pytest.mark.parametrize("precision", [0, 1, 2], ids=["double", "single-storage", "single"])
@pytest.mark.parametrize("w", [block_config(0, divisions=(7, 5, 5)), plate_config(divisions=(5, 7, 2))], ids=["block", "plate"])
def test_row_forms_keep_the_cycles_and_the_solves_bits(ctx, forced_variant, w, precision, form):
    ref = refcpu.Problem(w)
    r = np.random.default_rng(form).standard_normal(ref.free_dofs)

    def results(code):
        forced_variant(ROWS_FORCED + code)  # 0: the sliced forms
        csr = sf.CsrMatrix.new(ctx, *ref.csr())
        mg = multigrid(ctx, ref, precision, 100)
        z = mg.apply(r)
        solve = sf.Pcg.new(ctx, csr, mg, r, sf.PcgOptions(tolerance=1e-8, dot_order=sf.DotOrder.TREE))
        solve.step(100000)
        return bits(z), bits(solve.estimate())

    for got, expected in zip(results(form), results(0)):
        assert np.array_equal(got, expected)
