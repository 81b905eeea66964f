"""Properties of the compiled device code that no result shows reliably, read from the assembly of small
kernels compiled here for gfx950 (no GPU takes part)."""
import re
import shutil
import subprocess

import pytest

from solidfem_amd import build

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None, reason="needs hipcc")


def assembly(tmp_path, source):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(source)
    subprocess.run([build.HIPCC, "-x", "hip", "-S", "--offload-device-only", str(src), "-o", str(out), "-I" + str(build.CSRC)]
                   + [f for f in build.COMMON if f != "-fPIC"], check=True, capture_output=True, timeout=300)
    return out.read_text()


def test_lane_sums_keep_their_registers_apart_from_their_terms(tmp_path):
    # A sum that starts with the value of one of its terms: the instructions after the first still read
    # that term, so the sum must not share its register, nor that of the factor one.
    text = assembly(tmp_path, """
#include "sf_kernels.hpp"
using namespace sf::dev;
__global__ void f64_term(double *out, const double *in) {
    const double x = in[threadIdx.x], y = in[64 + threadIdx.x];
    double acc = x;
    add_from_lanes<0>(acc, x, y);
    out[threadIdx.x] = acc;
}
__global__ void f64_one(double *out, const double *in) {
    double acc = 1.0;
    add_from_lanes<4>(acc, in[threadIdx.x], in[64 + threadIdx.x]);
    out[threadIdx.x] = acc;
}
__global__ void f32_term(float *out, const float *in) {
    const float x = in[threadIdx.x];
    float acc = x;
    add_from_lanes<8>(acc, x, in[64 + threadIdx.x], in[128 + threadIdx.x], in[192 + threadIdx.x]);
    out[threadIdx.x] = acc;
}
__global__ void f64_three(double *out, const double *in) {
    double t[3][3], acc[3];
    for (int p = 0; p < 3; ++p) {
        for (int q = 0; q < 3; ++q) t[p][q] = in[(p * 3 + q) * 64 + threadIdx.x];
        acc[p] = t[p][2];
    }
    add_three_from_lanes<12>(acc, t);
    for (int p = 0; p < 3; ++p) out[p * 64 + threadIdx.x] = acc[p];
}
""")
    adds = re.findall(r"(v_fmac_f64_dpp|v_add_f32_dpp) (\S+), (\S+), (\S+) row_newbcast", text)
    assert len(adds) == 8 + 8 + 16 + 36
    for op, total, term, other in adds:
        assert total != term, (op, total, term, other)
        assert op == "v_add_f32_dpp" or total != other, (op, total, term, other)


def test_batched_rows_of_six_stay_within_64_kb_of_lds(tmp_path):
    # what a launch asks for (the chains' terms: rows_batch_fits) and what the kernels declare besides
    def asked(columns, size):
        return 6 * columns * (32 * 6 * size + 16)

    cases = [(v, size, m) for v, size in (("float", 4), ("double", 8)) for m in range(1, 9) if asked(m, size) <= 65536]
    assert ("double", 8, 7) in cases and asked(7, 8) > 65536 - 512
    text = assembly(tmp_path, "#include \"sf_batch_kernels.hpp\"\nnamespace sf::dev {\n" + "\n".join(
        f"template __global__ void rows_batch_kernel<6, 6, {m}, 1, {v}, {v}>(Bsr<{v}>, int, const {v} *, {v} *, const {v} *, Start<{v}, {v}>);\n"
        f"template __global__ void cheb_rows_batch_kernel<6, {m}, 1, {v}, {v}>(Bsr<{v}>, const {v} *, const {v} *, const {v} *, {v}, {v}, {v} *, {v} *,"
        f" {v} *, {v} *, double *);" for v, _, m in cases) + "\n}\n")
    declared = re.findall(r"\.group_segment_fixed_size: (\d+).*?\.name: +(\S+)", text, re.S)
    found = 0
    for static, name in declared:
        kernel = re.search(r"(?:cheb_rows_batch_kernelILi6E|rows_batch_kernelILi6ELi6E)Li(\d)ELi1E([fd])", name)
        if kernel:
            found += 1
            assert int(static) + asked(int(kernel[1]), 8 if kernel[2] == "d" else 4) <= 65536, (name, static)
    assert found == 2 * len(cases)
