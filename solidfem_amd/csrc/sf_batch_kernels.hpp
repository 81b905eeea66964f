// Device kernels for several right-hand sides at once (load cases sharing one matrix and one
// multigrid hierarchy).
//
// Vectors of M columns are stored row-interleaved: entry (row i, column m) at v[i * M + m], so
// the M values of a row are contiguous. The matrices are the sliced block matrices of the
// single-column kernels, read with another lane mapping: a group of G lanes (G a power of two,
// G >= M) takes one block row, lane m of the group its column m, and every lane forms the RB
// row sums of its block row for its column. In the sliced layout the RB x CB values of the block
// in slot k of slice row j are contiguous at vals[((start + k) * 64 + j * RB) * CB], so a group
// reads each block once (one broadcast) and each column of x as G consecutive values.
//
// Each row sum runs over the row's blocks in stored order and over a block's columns in order,
// from zero, exactly as the single-column kernels and the reference's block product
// (crates/solidfem-solve/src/multigrid/block.rs:136-154) do: column m of a batched product is
// bit for bit the single-column product of column m. The same holds for every kernel below, so a
// column's solve does not depend on the columns batched with it.
#pragma once

#include "sf_kernels.hpp"

namespace sf {
namespace dev {

// A group's place: the node position (slice * NPW + j) it works on and its column.
struct GroupLane {
    uint32_t pos;  // node position in slice order
    int m;         // column of this lane
};

// With ORDER_GROUP_RUNS in the matrix view's order, each XCD takes one contiguous run of the
// workgroups (as xcd_runs_block): the rows an XCD works on at a time are then neighbours, and so
// are the rows of x they gather, which its L2 can hold for all their columns. Which workgroup
// takes which rows changes no bit.
__device__ __forceinline__ uint32_t group_block(uint32_t order) {
    if (order & ORDER_GROUP_RUNS) return xcd_runs_block();
    if (order & ORDER_GROUP_CHUNKS) return xcd_chunks_block(order >> ORDER_CHUNK_SHIFT);
    return blockIdx.x;
}

__device__ __forceinline__ GroupLane group_lane(int log2g, uint32_t order) {
    const uint32_t t = group_block(order) * blockDim.x + threadIdx.x;
    return {t >> log2g, (int)(t & ((1u << log2g) - 1u))};
}

// CPL consecutive columns of one row-interleaved vector at p (p aligned to CPL values).
template <int CPL, typename V>
__device__ __forceinline__ void load_columns(const V *__restrict__ p, V (&out)[CPL]) {
    if constexpr (CPL == 1) {
        out[0] = p[0];
    } else if constexpr (CPL == 2) {
        using T = typename std::conditional<std::is_same<V, float>::value, float2, double2>::type;
        const T t = *reinterpret_cast<const T *>(p);
        out[0] = t.x;
        out[1] = t.y;
    } else if constexpr (std::is_same<V, float>::value) {
        static_assert(CPL % 4 == 0, "two, four or eight columns per lane");
#pragma unroll
        for (int h = 0; h < CPL / 4; ++h) {
            const float4 t = reinterpret_cast<const float4 *>(p)[h];
            out[4 * h] = t.x;
            out[4 * h + 1] = t.y;
            out[4 * h + 2] = t.z;
            out[4 * h + 3] = t.w;
        }
    } else {
        static_assert(CPL % 4 == 0, "two, four or eight columns per lane");
#pragma unroll
        for (int h = 0; h < CPL / 2; ++h) {
            const double2 t = reinterpret_cast<const double2 *>(p)[h];
            out[2 * h] = t.x;
            out[2 * h + 1] = t.y;
        }
    }
}

// Stores CPL consecutive columns at p (aligned as for load_columns).
template <int CPL, typename V>
__device__ __forceinline__ void store_columns(V *__restrict__ p, const V (&in)[CPL]) {
    if constexpr (CPL == 1) {
        p[0] = in[0];
    } else if constexpr (CPL == 2) {
        using T = typename std::conditional<std::is_same<V, float>::value, float2, double2>::type;
        *reinterpret_cast<T *>(p) = T{in[0], in[1]};
    } else if constexpr (std::is_same<V, float>::value) {
#pragma unroll
        for (int h = 0; h < CPL / 4; ++h) reinterpret_cast<float4 *>(p)[h] = float4{in[4 * h], in[4 * h + 1], in[4 * h + 2], in[4 * h + 3]};
    } else {
#pragma unroll
        for (int h = 0; h < CPL / 2; ++h) reinterpret_cast<double2 *>(p)[h] = double2{in[2 * h], in[2 * h + 1]};
    }
}

// Row sums of one block row for the CPL columns m0 .. m0 + CPL - 1: sum[p][c] = sum over stored
// blocks k and block columns q of A[p][q] x[(col * CB + q) * M + m0 + c], each from zero in the
// reference order. A lane reads a block once for all its columns.
template <int RB, int CB, int BATCH, typename S, typename V, int CPL>
__device__ __forceinline__ void rows_product_columns(const Sliced<S> &a, uint32_t slot0, uint32_t len, int j, int m0, uint32_t M,
                                                     const V *__restrict__ x, V (&sum)[RB][CPL]) {
    constexpr int NPW = Shape<RB>::NPW;
#pragma unroll
    for (int p = 0; p < RB; ++p)
#pragma unroll
        for (int c = 0; c < CPL; ++c) sum[p][c] = (V)0;
    const uint32_t *cp = a.cols + (size_t)slot0 * NPW + j;
    const S *vp = a.vals + ((size_t)slot0 * WAVE + (size_t)j * RB) * CB;
    const uint32_t full = len - len % BATCH;
    // the next batch's block columns are loaded with this batch's values and x entries, so a
    // batch costs one dependent memory round trip instead of two
    uint32_t col[BATCH];
    if (full) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) col[b] = cp[(size_t)b * NPW];
    }
    for (uint32_t k = 0; k < full; k += BATCH) {
        uint32_t next[BATCH];
        if (k + BATCH < full) {
#pragma unroll
            for (int b = 0; b < BATCH; ++b) next[b] = cp[(size_t)(k + BATCH + b) * NPW];
        }
        V xv[BATCH][CB][CPL];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) load_columns<CPL, V>(x + ((size_t)col[b] * CB + q) * M + m0, xv[b][q]);
        S v[BATCH][RB * CB];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int e = 0; e < RB * CB; ++e) v[b][e] = vp[(size_t)(k + b) * WAVE * CB + e];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int p = 0; p < RB; ++p)
#pragma unroll
                for (int q = 0; q < CB; ++q)
#pragma unroll
                    for (int c = 0; c < CPL; ++c) sum[p][c] = sum[p][c] + widen<V>(v[b][p * CB + q]) * xv[b][q][c];
#pragma unroll
        for (int b = 0; b < BATCH; ++b) col[b] = next[b];
    }
    for (uint32_t k = full; k < len; ++k) {
        const uint32_t cl = cp[(size_t)k * NPW];
        V xv[CB][CPL];
#pragma unroll
        for (int q = 0; q < CB; ++q) load_columns<CPL, V>(x + ((size_t)cl * CB + q) * M + m0, xv[q]);
        const S *blk = vp + (size_t)k * WAVE * CB;
#pragma unroll
        for (int p = 0; p < RB; ++p)
#pragma unroll
            for (int q = 0; q < CB; ++q)
#pragma unroll
                for (int c = 0; c < CPL; ++c) sum[p][c] = sum[p][c] + widen<V>(blk[p * CB + q]) * xv[q][c];
    }
}

// The same for one column m.
template <int RB, int CB, int BATCH, typename S, typename V>
__device__ __forceinline__ void rows_product(const Sliced<S> &a, uint32_t slot0, uint32_t len, int j, int m, uint32_t M,
                                             const V *__restrict__ x, V (&sum)[RB]) {
    V s[RB][1];
    rows_product_columns<RB, CB, BATCH, S, V, 1>(a, slot0, len, j, m, M, x, s);
#pragma unroll
    for (int p = 0; p < RB; ++p) sum[p] = s[p][0];
}

// The Chebyshev start on CPL columns of block row `row`, whose values y a lane holds (Start,
// cheb_start_batch_kernel): z = D^-1 y summed over the block row in order from zero, d = z / theta, x = d.
template <int RB, int CPL, typename S, typename V>
__device__ __forceinline__ void start_columns(const Start<S, V> &st, uint32_t row, uint32_t m0, uint32_t M, const V (&y)[RB][CPL]) {
    const S *dr = st.dinv + (size_t)row * RB * RB;
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        V d[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            V z = (V)0;
#pragma unroll
            for (int q = 0; q < RB; ++q) z = z + widen<V>(dr[p * RB + q]) * y[q][c];
            d[c] = z / st.theta;
        }
        const size_t at = ((size_t)row * RB + p) * M + m0;
        store_columns<CPL, V>(st.d + at, d);
        store_columns<CPL, V>(st.x + at, d);
    }
}

// Y = A X (STORE), Y = B - A X (RESIDUAL) or Y = Y + A X (ADD) for M columns: the batched form
// of spmv_kernel (products, residuals, restriction over the stored transpose, prolongation),
// optionally followed by the Chebyshev start on Y.
template <int RB, int CB, int BATCH, typename S, typename V, int CPL>
__global__ __launch_bounds__(256) void spmm_kernel(Sliced<S> a, int log2g, uint32_t M, int epi, const V *__restrict__ x,
                                                   V *__restrict__ y, const V *__restrict__ b, Start<S, V> then) {
    // CPL > 1: lane m of the group takes the CPL columns from m * CPL (M a multiple of CPL)
    constexpr int NPW = Shape<RB>::NPW;
    const GroupLane g = group_lane(log2g, a.order);
    const uint32_t m0 = (uint32_t)g.m * CPL;
    if (g.pos >= a.slices * (uint32_t)NPW || m0 >= M) return;
    const uint32_t row = a.perm[g.pos];
    if (row == NONE) return;
    const uint32_t slice = g.pos / NPW;
    const int j = (int)(g.pos - slice * NPW);
    V sum[RB][CPL];
    rows_product_columns<RB, CB, BATCH, S, V, CPL>(a, a.slice_start[slice], a.row_len[g.pos], j, (int)m0, M, x, sum);
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const size_t out = ((size_t)row * RB + p) * M + m0;
        V v[CPL];
        if (epi == EPI_STORE) {
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[c] = sum[p][c];
        } else {
            load_columns<CPL, V>((epi == EPI_RESIDUAL ? b : y) + out, v);
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[c] = epi == EPI_RESIDUAL ? v[c] - sum[p][c] : v[c] + sum[p][c];
        }
        store_columns<CPL, V>(y + out, v);
#pragma unroll
        for (int c = 0; c < CPL; ++c) sum[p][c] = v[c];
    }
    if (then.dinv) start_columns<RB, CPL, S, V>(then, row, m0, M, sum);
}

// ---- few columns: a lane per scalar row ----

// The columns of a scalar row, read or written: a vector where the count is one's, else one by one. The
// count is a compile-time one: with a test of each column against a count known only at run time the
// loads waited on one another (62 us a step for 5 columns of 6480 rows).
template <int MM, typename V>
__device__ __forceinline__ void load_few(const V *p, V (&out)[MM]) {
    if constexpr (MM == 2 || MM % 4 == 0) {
        load_columns<MM, V>(p, out);
    } else {
#pragma unroll
        for (int m = 0; m < MM; ++m) out[m] = p[m];
    }
}
template <int MM, typename V>
__device__ __forceinline__ void store_few(V *p, const V (&in)[MM]) {
    if constexpr (MM == 2 || MM % 4 == 0) {
        store_columns<MM, V>(p, in);
    } else {
#pragma unroll
        for (int m = 0; m < MM; ++m) p[m] = in[m];
    }
}

// MM columns of row_product (the single-column kernels' lane mapping): a lane reads its row's values of
// a block once and the columns of the x entries they meet, which the RB lanes of a block row share in
// cache.
template <int RB, int CB, int BATCH, int MM, typename S, typename V>
__device__ __forceinline__ void row_product_few(const Sliced<S> &a, uint32_t slot0, uint32_t len, int j, int lane,
                                                const V *__restrict__ x, V (&sum)[MM]) {
    constexpr int NPW = Shape<RB>::NPW;
#pragma unroll
    for (int m = 0; m < MM; ++m) sum[m] = (V)0;
    const uint32_t *cp = a.cols + (size_t)slot0 * NPW + j;
    const S *vp = a.vals + ((size_t)slot0 * WAVE + lane) * CB;
    auto columns = [&](uint32_t col, V(&xv)[CB][MM]) {
#pragma unroll
        for (int q = 0; q < CB; ++q) load_few<MM, V>(x + ((size_t)col * CB + q) * MM, xv[q]);
    };
    auto add = [&](const S(&v)[CB], const V(&xv)[CB][MM]) {
#pragma unroll
        for (int q = 0; q < CB; ++q)
#pragma unroll
            for (int m = 0; m < MM; ++m)
                sum[m] = sum[m] + widen<V>(v[q]) * xv[q][m];
    };
    const uint32_t full = len - len % BATCH;
    uint32_t c[BATCH];
    if (full) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) c[b] = cp[(size_t)b * NPW];
    }
    for (uint32_t k = 0; k < full; k += BATCH) {
        S v[BATCH][CB];
        V xv[BATCH][CB][MM];
        uint32_t cn[BATCH];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) v[b][q] = vp[(size_t)(k + b) * WAVE * CB + q];
#pragma unroll
        for (int b = 0; b < BATCH; ++b) columns(c[b], xv[b]);
        if (k + BATCH < full) {
#pragma unroll
            for (int b = 0; b < BATCH; ++b) cn[b] = cp[(size_t)(k + BATCH + b) * NPW];
        }
#pragma unroll
        for (int b = 0; b < BATCH; ++b) add(v[b], xv[b]);
#pragma unroll
        for (int b = 0; b < BATCH; ++b) c[b] = cn[b];
    }
    for (uint32_t k = full; k < len; ++k) {
        S v[CB];
        V xv[CB][MM];
#pragma unroll
        for (int q = 0; q < CB; ++q) v[q] = vp[(size_t)k * WAVE * CB + q];
        columns(cp[(size_t)k * NPW], xv);
        add(v, xv);
    }
}
// Blocks in flight per lane: what the columns of x leave of its registers.
template <int MM>
constexpr int FEW_DEPTH = MM <= 4 ? 4 : 2;

// z[m] = sum over q in order from zero of drow[q] times the value of lane j RB + q (the block row's row q).
template <int RB, int MM, typename S, typename V>
__device__ __forceinline__ void block_times_few(const S *drow, int first_lane, bool live, const V (&mine)[MM], V (&z)[MM]) {
#pragma unroll
    for (int m = 0; m < MM; ++m) z[m] = (V)0;
#pragma unroll
    for (int q = 0; q < RB; ++q)
#pragma unroll
        for (int m = 0; m < MM; ++m) {
            const V other = __shfl(mine[m], first_lane + q, WAVE);
            if (live) z[m] = z[m] + widen<V>(drow[q]) * other;
        }
}

// spmv_kernel and cheb_step_kernel for MM columns. The lane-group kernels read a block by lanes that
// each walk whole block rows and hold few blocks in flight: on the 603k-unknown plate a batch of one
// column took 2.4 times the single solve.
template <int RB, int CB, int MM, typename S, typename V>
__global__ __launch_bounds__(256) void spmm_few_kernel(Sliced<S> a, int epi, const V *__restrict__ x, V *__restrict__ y,
                                                       const V *__restrict__ b, Start<S, V> then) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t slice = slice_of(a.order);
    if (slice >= a.slices) return;  // whole wave leaves together
    const int lane = threadIdx.x % WAVE;
    const int j = lane / RB, p = lane - j * RB;
    const bool in_wave = j < NPW;
    const uint32_t pos = slice * NPW + (in_wave ? j : 0);
    const uint32_t row = in_wave ? a.perm[pos] : NONE;
    const bool live = row != NONE;
    const size_t out = live ? ((size_t)row * RB + p) * MM : 0;
    V value[MM] = {};
    if (live) {
        V sum[MM];
        row_product_few<RB, CB, FEW_DEPTH<MM>, MM, S, V>(a, a.slice_start[slice], a.row_len[pos], j, lane, x, sum);
        if (epi != EPI_STORE) load_few<MM, V>((epi == EPI_RESIDUAL ? b : y) + out, value);
#pragma unroll
        for (int m = 0; m < MM; ++m) value[m] = epi == EPI_STORE ? sum[m] : epi == EPI_RESIDUAL ? value[m] - sum[m] : value[m] + sum[m];
        store_few<MM, V>(y + out, value);
    }
    if (!then.dinv) return;  // uniform: every lane takes part in the shuffles
    V z[MM];
    block_times_few<RB, MM, S, V>(then.dinv + (live ? (size_t)row * RB * RB + (size_t)p * RB : 0), in_wave ? j * RB : 0, live, value, z);
    if (!live) return;
#pragma unroll
    for (int m = 0; m < MM; ++m) z[m] = z[m] / then.theta;
    store_few<MM, V>(then.d + out, z);
    store_few<MM, V>(then.x + out, z);
}

template <int RB, int MM, typename S, typename V>
__global__ __launch_bounds__(256) void cheb_step_few_kernel(Sliced<S> a, const S *__restrict__ dinv, const V *__restrict__ d_in,
                                                            const V *__restrict__ r_in, V keep, V step, V *__restrict__ d_out,
                                                            V *__restrict__ r_out, V *__restrict__ x, V *__restrict__ sum_into,
                                                            double *__restrict__ widen_into) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t slice = slice_of(a.order);
    if (slice >= a.slices) return;  // whole wave leaves together
    const int lane = threadIdx.x % WAVE;
    const int j = lane / RB, p = lane - j * RB;
    const bool in_wave = j < NPW;
    const uint32_t pos = slice * NPW + (in_wave ? j : 0);
    const uint32_t row = in_wave ? a.perm[pos] : NONE;
    const bool live = row != NONE;
    const size_t i = live ? ((size_t)row * RB + p) * MM : 0;
    V r_new[MM] = {};
    if (live) {
        V ad[MM];
        row_product_few<RB, RB, FEW_DEPTH<MM>, MM, S, V>(a, a.slice_start[slice], a.row_len[pos], j, lane, d_in, ad);
        load_few<MM, V>(r_in + i, r_new);
#pragma unroll
        for (int m = 0; m < MM; ++m) r_new[m] = r_new[m] - ad[m];
    }
    V z[MM];
    block_times_few<RB, MM, S, V>(dinv + (live ? (size_t)row * RB * RB + (size_t)p * RB : 0), in_wave ? j * RB : 0, live, r_new, z);
    if (!live) return;
    V dn[MM], xn[MM];
    load_few<MM, V>(d_in + i, dn);
    load_few<MM, V>(x + i, xn);
#pragma unroll
    for (int m = 0; m < MM; ++m) {
        dn[m] = keep * dn[m] + step * z[m];
        xn[m] = xn[m] + dn[m];
    }
    store_few<MM, V>(d_out + i, dn);
    store_few<MM, V>(r_out + i, r_new);
    store_few<MM, V>(x + i, xn);
    if (!sum_into) return;
    V total[MM];
    load_few<MM, V>(sum_into + i, total);
#pragma unroll
    for (int m = 0; m < MM; ++m) total[m] = total[m] + xn[m];
    store_few<MM, V>(sum_into + i, total);
    if (!widen_into) return;
    double wide[MM];
#pragma unroll
    for (int m = 0; m < MM; ++m) wide[m] = (double)total[m];
    store_few<MM, double>(widen_into + i, wide);
}

// The same product with one wavefront per block row: the row's position, block columns and block
// values are the same for every lane, so they are read through the scalar unit into registers
// every lane uses, and only the M columns of x are vector loads. Lane m takes column m (lanes
// from M up idle). Row sums in the same order as rows_product.
template <int RB, int CB, int BATCH, typename S, typename V>
__device__ __forceinline__ void node_product(const Sliced<S> &a, uint32_t pos, int m, uint32_t M, const V *__restrict__ x,
                                             uint32_t &row_out, V (&sum)[RB]) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t slice = pos / NPW;
    const int j = (int)(pos - slice * NPW);
    const uint32_t row = a.perm[pos];
    row_out = row;
#pragma unroll
    for (int p = 0; p < RB; ++p) sum[p] = (V)0;
    if (row == NONE) return;
    const uint32_t slot0 = a.slice_start[slice], len = a.row_len[pos];
    const uint32_t *__restrict__ cp = a.cols + (size_t)slot0 * NPW + j;
    const S *__restrict__ vp = a.vals + ((size_t)slot0 * WAVE + (size_t)j * RB) * CB;
    const uint32_t full = len - len % BATCH;
    for (uint32_t k = 0; k < full; k += BATCH) {
        uint32_t c[BATCH];
#pragma unroll
        for (int b = 0; b < BATCH; ++b) c[b] = __builtin_amdgcn_readfirstlane(cp[(size_t)(k + b) * NPW]);
        V xv[BATCH][CB];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) xv[b][q] = (uint32_t)m < M ? x[((size_t)c[b] * CB + q) * M + m] : (V)0;
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int p = 0; p < RB; ++p)
#pragma unroll
                for (int q = 0; q < CB; ++q) sum[p] = sum[p] + widen<V>(vp[(size_t)(k + b) * WAVE * CB + p * CB + q]) * xv[b][q];
    }
    for (uint32_t k = full; k < len; ++k) {
        const uint32_t col = __builtin_amdgcn_readfirstlane(cp[(size_t)k * NPW]);
        V xv[CB];
#pragma unroll
        for (int q = 0; q < CB; ++q) xv[q] = (uint32_t)m < M ? x[((size_t)col * CB + q) * M + m] : (V)0;
#pragma unroll
        for (int p = 0; p < RB; ++p)
#pragma unroll
            for (int q = 0; q < CB; ++q) sum[p] = sum[p] + widen<V>(vp[(size_t)k * WAVE * CB + p * CB + q]) * xv[q];
    }
}

// Position of this wavefront's block row, made uniform for the compiler.
__device__ __forceinline__ uint32_t node_of_wave(uint32_t order) {
    return __builtin_amdgcn_readfirstlane(group_block(order) * (blockDim.x / WAVE) + threadIdx.x / WAVE);
}

// The same product with one workgroup per block row, for matrices of few, long rows (the stored
// transposes of the coarse levels): the workgroup stages a chunk of the row's blocks and the x entries
// they gather in LDS, all loads in flight at once, then thread (p, CPL columns from m) adds the chunk's
// terms of row entry p in the stored order. The next chunk's values and x entries are on their way to
// registers meanwhile, and the block columns of the one after it: a chunk costs its additions, not a
// round trip, and one barrier (two LDS buffers). Every sum is the lane-group form's: from zero, blocks
// in order, block columns in order. x moves in units of UNIT: 16 bytes where a block's CB * M entries
// are whole units, else single entries.
// A chunk holds at most STAGE_BLOCKS blocks (9 KB of values a buffer) and what x a thread's registers
// carry: few columns take long chunks, so that a row of some hundred blocks is two or three (355 blocks
// and 5 columns: 18.5 us a launch, 25.8 by 32). From 16 columns on 32 blocks: longer ones cost more of a CU's
// workgroups than they save.
template <int LEN, typename S>
constexpr int STAGE_BLOCKS = 9216 / (LEN * (int)sizeof(S)) < 32 ? 32 : 9216 / (LEN * (int)sizeof(S)) > 128 ? 128 : 9216 / (LEN * (int)sizeof(S));
template <typename UNIT, typename V>
constexpr int STAGE_UNITS = sizeof(UNIT) == 16 && sizeof(V) < 16 ? 4 : 8;  // x units a thread holds
// Blocks per chunk for `units` units of x per block.
__host__ __device__ inline uint32_t stage_chunk(uint32_t units, uint32_t held, uint32_t M, uint32_t most) {
    const uint32_t c = 256u * held / units, cap = M < 16 || most < 32 ? most : 32;
    return c < cap ? c : cap;
}
template <int RB, int CB, typename S, typename V, typename UNIT, int CPL>
__global__ __launch_bounds__(256) void spmm_staged_kernel(Sliced<S> a, uint32_t M, int epi, const V *__restrict__ x,
                                                          V *__restrict__ y, const V *__restrict__ b, Start<S, V> then) {
    constexpr int NPW = Shape<RB>::NPW, LEN = RB * CB, UX = STAGE_UNITS<UNIT, V>, BLOCKS = STAGE_BLOCKS<LEN, S>,
                  UV = (BLOCKS * LEN + 255) / 256;
    const uint32_t pos = blockIdx.x;
    if (pos >= a.slices * (uint32_t)NPW) return;  // the whole workgroup leaves together
    const uint32_t row = a.perm[pos];
    if (row == NONE) return;
    const uint32_t slice = pos / NPW;
    const int j = (int)(pos - slice * NPW);
    const uint32_t slot0 = a.slice_start[slice], len = a.row_len[pos];
    const uint32_t *__restrict__ cp = a.cols + (size_t)slot0 * NPW + j;
    const S *__restrict__ vp = a.vals + ((size_t)slot0 * WAVE + (size_t)j * RB) * CB;
    __shared__ uint32_t columns[2][BLOCKS];
    extern __shared__ __align__(16) unsigned char staged_x[];  // two buffers of chunk * CB * M entries of x, two of the values
    const uint32_t units = (uint32_t)(CB * M * sizeof(V) / sizeof(UNIT)), chunk = stage_chunk(units, UX, M, BLOCKS);
    // offsets and not an array of pointers, which would make every access a flat one
    UNIT *const staged_units = reinterpret_cast<UNIT *>(staged_x);
    S *const staged_values = reinterpret_cast<S *>(staged_x + (size_t)2 * chunk * units * sizeof(UNIT));
    const uint32_t t = threadIdx.x, across = M / CPL;
    const bool computes = t < (uint32_t)RB * across;
    const uint32_t p = computes ? t / across : 0, m = computes ? t % across * CPL : 0;
    // this thread's units of a chunk: block k and unit r of its x
    uint32_t uk[UX], ur[UX];
#pragma unroll
    for (int u = 0; u < UX; ++u) {
        uk[u] = (t + 256u * u) / units;
        ur[u] = (t + 256u * u) - uk[u] * units;
        if (uk[u] >= chunk) uk[u] = NONE;
    }
    UNIT xv[UX];
    S vv[UV];
    auto fetch = [&](uint32_t k0, const uint32_t *cols) {
        const uint32_t n = k0 < len ? min(chunk, len - k0) : 0u;
#pragma unroll
        for (int u = 0; u < UX; ++u)
            if (uk[u] < n) xv[u] = reinterpret_cast<const UNIT *>(x + (size_t)cols[uk[u]] * CB * M)[ur[u]];
#pragma unroll
        for (int u = 0; u < UV; ++u) {
            const uint32_t e = t + 256u * u, k = e / LEN;
            if (k < n) vv[u] = vp[(size_t)(k0 + k) * WAVE * CB + (e - k * LEN)];
        }
    };
    V sum[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) sum[c] = (V)0;
    if (t < chunk && t < len) columns[0][t] = cp[(size_t)t * NPW];
    uint32_t column = t < chunk && chunk + t < len ? cp[(size_t)(chunk + t) * NPW] : 0;
    __syncthreads();
    fetch(0, columns[0]);
    uint32_t buf = 0;
    for (uint32_t k0 = 0; k0 < len; k0 += chunk, buf ^= 1) {
        const uint32_t n = min(chunk, len - k0);
#pragma unroll
        for (int u = 0; u < UX; ++u)
            if (uk[u] < n) staged_units[buf * chunk * units + t + 256u * u] = xv[u];
#pragma unroll
        for (int u = 0; u < UV; ++u)
            if (t + 256u * u < n * LEN) staged_values[buf * chunk * LEN + t + 256u * u] = vv[u];
        if (t < chunk) columns[buf ^ 1][t] = column;
        // one barrier per chunk: a buffer is written again two chunks on, which a wavefront reaches
        // only after the barrier between, and so after the others have read it
        __syncthreads();
        const uint32_t k2 = k0 + 2 * chunk;
        if (t < chunk && k2 + t < len) column = cp[(size_t)(k2 + t) * NPW];
        fetch(k0 + chunk, columns[buf ^ 1]);
        if (computes) {
            const V *xb = reinterpret_cast<const V *>(staged_units + buf * chunk * units) + m;
            const S *vb = staged_values + buf * chunk * LEN + p * CB;
#pragma unroll 4
            for (uint32_t k = 0; k < n; ++k)
#pragma unroll
                for (int q = 0; q < CB; ++q) {
                    V xe[CPL];
                    load_columns<CPL, V>(xb + (k * CB + q) * M, xe);
                    const V v = widen<V>(vb[k * LEN + q]);
#pragma unroll
                    for (int c = 0; c < CPL; ++c) sum[c] = sum[c] + v * xe[c];
                }
        }
    }
    const size_t out = ((size_t)row * RB + p) * M + m;
    if (computes) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (epi == EPI_RESIDUAL) sum[c] = b[out + c] - sum[c];
            else if (epi == EPI_ADD) sum[c] = y[out + c] + sum[c];
            y[out + c] = sum[c];
        }
    }
    if (!then.dinv) return;  // uniform
    // the start: the block row's entries meet in LDS (RB * M entries: within the two x buffers of at
    // least one block of CB >= 3 each), which every thread has done with after the barrier
    V *row_values = reinterpret_cast<V *>(staged_x);
    __syncthreads();
    if (computes) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) row_values[p * M + m + c] = sum[c];
    }
    __syncthreads();
    if (computes) {
        const S *drow = then.dinv + (size_t)row * RB * RB + (size_t)p * RB;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            V z = (V)0;
#pragma unroll
            for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * row_values[q * M + m + c];
            const V dv = z / then.theta;
            then.d[out + c] = dv;
            then.x[out + c] = dv;
        }
    }
}

template <int RB, int CB, int BATCH, typename S, typename V>
__global__ __launch_bounds__(256) void spmm_node_kernel(Sliced<S> a, uint32_t M, int epi, const V *__restrict__ x,
                                                        V *__restrict__ y, const V *__restrict__ b, Start<S, V> then) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t pos = node_of_wave(a.order);
    if (pos >= a.slices * (uint32_t)NPW) return;
    const int m = threadIdx.x % WAVE;
    uint32_t row;
    V sum[RB];
    node_product<RB, CB, BATCH, S, V>(a, pos, m, M, x, row, sum);
    if (row == NONE || (uint32_t)m >= M) return;
    V v[RB][1];
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const size_t out = ((size_t)row * RB + p) * M + m;
        v[p][0] = epi == EPI_STORE ? sum[p] : epi == EPI_RESIDUAL ? b[out] - sum[p] : y[out] + sum[p];
        y[out] = v[p][0];
    }
    if (then.dinv) start_columns<RB, 1, S, V>(then, row, (uint32_t)m, M, v);
}

template <int RB, int BATCH, typename S, typename V>
__global__ __launch_bounds__(256) void cheb_step_node_kernel(Sliced<S> a, uint32_t M, const S *__restrict__ dinv,
                                                             const V *__restrict__ d_in, const V *__restrict__ r_in, V keep,
                                                             V step, V *__restrict__ d_out, V *__restrict__ r_out,
                                                             V *__restrict__ x, V *__restrict__ sum_into,
                                                             double *__restrict__ widen_into) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t pos = node_of_wave(a.order);
    if (pos >= a.slices * (uint32_t)NPW) return;
    const int m = threadIdx.x % WAVE;
    uint32_t row;
    V ad[RB];
    node_product<RB, RB, BATCH, S, V>(a, pos, m, M, d_in, row, ad);
    if (row == NONE || (uint32_t)m >= M) return;
    V r_new[RB];
#pragma unroll
    for (int p = 0; p < RB; ++p) r_new[p] = r_in[((size_t)row * RB + p) * M + m] - ad[p];
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const S *drow = dinv + (size_t)row * RB * RB + (size_t)p * RB;
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * r_new[q];
        const size_t i = ((size_t)row * RB + p) * M + m;
        const V dn = keep * d_in[i] + step * z;
        const V xn = x[i] + dn;
        d_out[i] = dn;
        r_out[i] = r_new[p];
        x[i] = xn;
        if (sum_into) {
            const V total = sum_into[i] + xn;
            sum_into[i] = total;
            if (widen_into) widen_into[i] = (double)total;
        }
    }
}

// The rounding bound terms of CsrMatrix::multiply_rounding_bound (crates/solidfem-solve/src/csr.rs:142-154)
// for M columns: per row and column, ((terms * eps) * sum |a x|)^2.
template <int RB, int CB>
__global__ __launch_bounds__(256) void rounding_bound_batch_kernel(Sliced<double> a, int log2g, uint32_t M,
                                                                   const double *__restrict__ x, double *__restrict__ out) {
    constexpr int NPW = Shape<RB>::NPW;
    const GroupLane g = group_lane(log2g, a.order);
    if (g.pos >= a.slices * (uint32_t)NPW || (uint32_t)g.m >= M) return;
    const uint32_t row = a.perm[g.pos];
    if (row == NONE) return;
    const uint32_t slice = g.pos / NPW;
    const int j = (int)(g.pos - slice * NPW);
    const uint32_t len = a.row_len[g.pos], slot0 = a.slice_start[slice];
    double sum[RB];
#pragma unroll
    for (int p = 0; p < RB; ++p) sum[p] = 0.0;
    for (uint32_t k = 0; k < len; ++k) {
        const uint32_t col = a.cols[(size_t)(slot0 + k) * NPW + j];
        const double *blk = a.vals + ((size_t)(slot0 + k) * WAVE + (size_t)j * RB) * CB;
#pragma unroll
        for (int p = 0; p < RB; ++p)
#pragma unroll
            for (int q = 0; q < CB; ++q) sum[p] = sum[p] + fabs(blk[p * CB + q] * x[((size_t)col * CB + q) * M + g.m]);
    }
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const double bound = (double)(len * CB) * 2.220446049250313e-16 * sum[p];
        out[((size_t)row * RB + p) * M + g.m] = bound * bound;
    }
}

// The Chebyshev start for M columns (crates/solidfem-solve/src/multigrid/cycle.rs:591-610):
// z = D^-1 b, d = z / theta, x = d. One thread per block row and column.
template <int RB, typename S, typename V>
__global__ __launch_bounds__(256) void cheb_start_batch_kernel(uint32_t rows, uint32_t M, const S *__restrict__ dinv,
                                                               const V *__restrict__ b, V theta, V *__restrict__ d,
                                                               V *__restrict__ x) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)rows * M) return;
    const size_t row = t / M, m = t - row * M;
    V bv[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) bv[q] = b[(row * RB + q) * M + m];
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const S *dr = dinv + row * RB * RB + p * RB;
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(dr[q]) * bv[q];
        const V dv = z / theta;
        d[(row * RB + p) * M + m] = dv;
        x[(row * RB + p) * M + m] = dv;
    }
}

// The finest level's right-hand sides rounded in from f64 and the start on them (convert_start_kernel
// per column). One thread per block row and column.
template <int RB, typename S, typename V>
__global__ __launch_bounds__(256) void convert_start_batch_kernel(uint32_t rows, uint32_t M, const double *__restrict__ r,
                                                                  V *__restrict__ b, const S *__restrict__ dinv, V theta,
                                                                  V *__restrict__ d, V *__restrict__ x) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)rows * M) return;
    const uint32_t row = (uint32_t)(t / M), m = (uint32_t)(t - (size_t)row * M);
    V bv[RB][1];
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        const size_t at = ((size_t)row * RB + q) * M + m;
        bv[q][0] = (V)r[at];
        b[at] = bv[q][0];
    }
    start_columns<RB, 1, S, V>(Start<S, V>{dinv, theta, d, x}, row, m, M, bv);
}

// ---- few columns of a small system ----

// rows_sum for M columns (a compile-time count, as row_product_few's): a wavefront (one workgroup) takes
// RPW block rows, 64 / RPW lanes each; every lane loads a block and the M columns of the x entries it
// meets and forms their terms into LDS, then lane c adds chain c's terms in stored order: row entry and column c % (RB M) of row c / (RB M),
// RPW RB M <= 64. One round trip per 64 / RPW blocks, where a lane walking its row pays one per few. A
// block of six rows is shared by two lanes, three rows each: four columns' steps of the 603k-DOF
// plate's level 2 (334 rows) take 5.3 us (17.9 with lanes walking rows), and batches of four solve in
// 28.6 ms for 40.3 (55k-DOF plate), 14.9 for 18.6 (300k-DOF block), 10.6 for 14.2 (115k-DOF tube).
template <int RB, int RPW>
constexpr int ROWS_BATCH_BLOCKS = WAVE / RPW / (RB / 3);  // blocks of a row at a time
template <int RB, int CB, typename V, int RPW>
constexpr int ROWS_BATCH_STRIDE = ROWS_BATCH_BLOCKS<RB, RPW> * CB + 16 / sizeof(V);  // entries of a chain's room
template <int RB, int M, int RPW, typename V>
constexpr size_t ROWS_BATCH_LDS = (size_t)RPW * RB * M * ROWS_BATCH_STRIDE<RB, RB, V, RPW> * sizeof(V);  // all that a launch takes
template <int RB, int CB, int M, int RPW, typename S, typename V>
__device__ __forceinline__ V rows_sum_batch(const Bsr<S> &a, V *terms, int g, int sl, uint32_t start, uint32_t len,
                                            const V *__restrict__ x) {
    constexpr int PARTS = RB / 3, LW = ROWS_BATCH_BLOCKS<RB, RPW>, STRIDE = ROWS_BATCH_STRIDE<RB, CB, V, RPW>;
    const int at = sl / PARTS, p0 = sl % PARTS * 3;
    const uint32_t longest = longest_of_wave<RPW>(len), chain = threadIdx.x;
    const bool adds = chain < (uint32_t)(RPW * RB * M);
    const uint32_t chain_len = (uint32_t)__shfl((int)len, adds ? (int)(chain / (RB * M)) * (WAVE / RPW) : 0, WAVE);
    V sum = (V)0;
    for (uint32_t k0 = 0; k0 < longest; k0 += LW) {
        const uint32_t k = k0 + at;
        if (k < len) {
            const uint32_t col = a.cols[start + k];
            S v[3 * CB];
            V xv[CB][M];
            const S *blk = a.vals + ((size_t)(start + k) * RB + p0) * CB;
#pragma unroll
            for (int e = 0; e < 3 * CB; ++e) v[e] = blk[e];
#pragma unroll
            for (int q = 0; q < CB; ++q) load_few<M, V>(x + ((size_t)col * CB + q) * M, xv[q]);
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int q = 0; q < CB; ++q)
                        terms[((g * RB + p0 + p) * M + m) * STRIDE + at * CB + q] = widen<V>(v[p * CB + q]) * xv[q][m];
        }
        __syncthreads();
        if (adds && k0 < chain_len)
            sum = add_terms<4>(sum, (const V *)terms + (size_t)chain * STRIDE, (chain_len - k0 < (uint32_t)LW ? chain_len - k0 : (uint32_t)LW) * CB);
        __syncthreads();
    }
    return sum;
}

template <int RB, int CB, int M, int RPW, typename S, typename V>
__global__ __launch_bounds__(64) void rows_batch_kernel(Bsr<S> a, int epi, const V *__restrict__ x, V *__restrict__ y,
                                                        const V *__restrict__ b, Start<S, V> then) {
    constexpr int LW = WAVE / RPW;
    // the chains' terms, and after the sums (rows_sum_batch ends at a barrier) the block rows' values
    extern __shared__ __align__(16) unsigned char rows_terms[];
    V *terms = reinterpret_cast<V *>(rows_terms), *values = terms;
    const uint32_t lane = threadIdx.x, first = (a.reverse ? xcd_reversed_block() : blockIdx.x) * RPW;
    const uint32_t row = first + lane / LW;
    const uint32_t start = row < a.rows ? a.starts[row] : 0u, len = row < a.rows ? a.starts[row + 1] - start : 0u;
    // this lane's chain: row entry p of `own`, column m
    constexpr uint32_t per = RB * M;
    const uint32_t within = lane % per, p = within / M, m = within - p * M, own = first + lane / per;
    const bool owner = lane < RPW * per && own < a.rows;
    const size_t out = owner ? ((size_t)own * RB + p) * M + m : 0;
    const V before = !owner || epi == EPI_STORE ? (V)0 : b[out];
    const V sum = rows_sum_batch<RB, CB, M, RPW, S, V>(a, terms, (int)(lane / LW), (int)(lane % LW), start, len, x);
    V value = (V)0;
    if (owner) {
        value = epi == EPI_STORE ? sum : before - sum;
        y[out] = value;
    }
    if (!then.dinv) return;  // uniform
    values[lane] = value;
    __syncthreads();
    if (owner) {
        const S *drow = then.dinv + (size_t)own * RB * RB + (size_t)p * RB;
        const V *row_values = values + lane - within + m;
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * row_values[q * M];
        const V dv = z / then.theta;
        then.d[out] = dv;
        then.x[out] = dv;
    }
}

// A restriction's few, long rows for M columns: a workgroup per block row of six. Three wavefronts load
// the next CHUNK blocks and the M columns of the x entries they meet (a block shared by 192 / CHUNK
// threads) and form their terms into LDS; the fourth adds the chunk before, a lane per chain (row entry
// and column), in stored order. Bound by that chain of additions: 73 rows of 350 blocks, five columns,
// f32: 9.0 us a launch, against 19.0 for the staged product. Batches of two to four solve in 0.85 to
// 0.97 times the time (300k-DOF block, four columns: 14.9 -> 12.9 ms).
constexpr uint32_t WIDE_BATCH_THREADS = 256, WIDE_BATCH_LDS = 65536 - 512;
template <int CB, int M, typename V>
struct WideRowsBatch {
    static constexpr int stride(int chunk) { return chunk * CB + 16 / (int)sizeof(V); }  // entries of a chain's room
    static constexpr uint32_t bytes(int chunk) { return 2u * 6 * M * stride(chunk) * sizeof(V); }
    // the longest chunk whose two buffers fit the LDS; FITS: whether any does
    static constexpr int CHUNK = bytes(64) <= WIDE_BATCH_LDS ? 64 : 32;
    static constexpr bool FITS = bytes(CHUNK) <= WIDE_BATCH_LDS;
    static constexpr int STRIDE = stride(CHUNK), PARTS = 192 / CHUNK, RP = 6 / PARTS;
};
template <int CB, int M, typename S, typename V>
__global__ __launch_bounds__(256) void wide_rows_batch_kernel(Bsr<S> a, const V *__restrict__ x, V *__restrict__ y, Start<S, V> then) {
    using W = WideRowsBatch<CB, M, V>;
    constexpr int RB = 6, RP = W::RP, STRIDE = W::STRIDE;
    constexpr uint32_t CHUNK = W::CHUNK, CHAINS = RB * M;
    __shared__ __align__(16) V terms[2][CHAINS * STRIDE];
    __shared__ V values[WAVE];
    const uint32_t row = a.reverse ? xcd_reversed_block() : blockIdx.x;  // one workgroup per row: row < a.rows
    const uint32_t start = a.starts[row], len = a.starts[row + 1] - start;
    const uint32_t t = threadIdx.x, k = t / W::PARTS, p0 = t % W::PARTS * RP;
    const bool loads = t < 192;  // k < CHUNK
    const uint32_t chain = t - 192, p = chain / M, m = chain - p * M;
    const bool adds = !loads && chain < CHAINS;
    const size_t out = (size_t)row * CHAINS + chain;
    S drow[RB];
    if (then.dinv && adds) {
#pragma unroll
        for (int q = 0; q < RB; ++q) drow[q] = then.dinv[(size_t)row * RB * RB + (size_t)p * RB + q];
    }
    S v[RP * CB];
    V xv[CB][M];
    auto fetch = [&](uint32_t at, uint32_t col) {
        if (loads && at < len) {
            const S *blk = a.vals + ((size_t)(start + at) * RB + p0) * CB;
#pragma unroll
            for (int e = 0; e < RP * CB; ++e) v[e] = blk[e];
#pragma unroll
            for (int q = 0; q < CB; ++q) load_few<M, V>(x + ((size_t)col * CB + q) * M, xv[q]);
        }
    };
    uint32_t col = loads && k < len ? a.cols[start + k] : 0u;
    fetch(k, col);
    col = loads && k + CHUNK < len ? a.cols[start + k + CHUNK] : 0u;
    V sum = (V)0;
    int buf = 0;
    for (uint32_t k0 = 0; k0 < len; k0 += CHUNK, buf ^= 1) {
        if (loads && k0 + k < len) {
#pragma unroll
            for (int r = 0; r < RP; ++r)
#pragma unroll
                for (int m1 = 0; m1 < M; ++m1)
#pragma unroll
                    for (int q = 0; q < CB; ++q)
                        terms[buf][((p0 + r) * M + m1) * STRIDE + k * CB + q] = widen<V>(v[r * CB + q]) * xv[q][m1];
        }
        const uint32_t k1 = k0 + CHUNK, k2 = k1 + CHUNK;
        if (k1 < len) {
            fetch(k1 + k, col);
            if (loads && k2 + k < len) col = a.cols[start + k2 + k];
        }
        // one barrier per chunk, as in wide_rows_kernel
        __syncthreads();
        if (adds) sum = add_terms<4>(sum, (const V *)terms[buf] + chain * STRIDE, (len - k0 < CHUNK ? len - k0 : CHUNK) * CB);
    }
    if (adds) {
        y[out] = sum;
        values[chain] = sum;
    }
    if (!then.dinv) return;  // uniform
    __syncthreads();
    if (adds) {
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * values[q * M + m];
        const V dv = z / then.theta;
        then.d[out] = dv;
        then.x[out] = dv;
    }
}

template <int RB, int M, int RPW, typename S, typename V>
__global__ __launch_bounds__(64) void cheb_rows_batch_kernel(Bsr<S> a, const S *__restrict__ dinv, const V *__restrict__ d_in,
                                                             const V *__restrict__ r_in, V keep, V step, V *__restrict__ d_out,
                                                             V *__restrict__ r_out, V *__restrict__ x, V *__restrict__ sum_into,
                                                             double *__restrict__ widen_into) {
    constexpr int LW = WAVE / RPW;
    // the chains' terms, and after the sums the block rows' residuals
    extern __shared__ __align__(16) unsigned char rows_terms[];
    V *terms = reinterpret_cast<V *>(rows_terms), *r_new = terms;
    const uint32_t lane = threadIdx.x, first = (a.reverse ? xcd_reversed_block() : blockIdx.x) * RPW;
    const uint32_t row = first + lane / LW;
    const uint32_t start = row < a.rows ? a.starts[row] : 0u, len = row < a.rows ? a.starts[row + 1] - start : 0u;
    constexpr uint32_t per = RB * M;
    const uint32_t within = lane % per, p = within / M, m = within - p * M, own = first + lane / per;
    const bool owner = lane < RPW * per && own < a.rows;
    const size_t i = owner ? ((size_t)own * RB + p) * M + m : 0;
    V r_old = (V)0, d_old = (V)0, x_old = (V)0, into = (V)0;
    S drow[RB];
    if (owner) {
        r_old = r_in[i];
        d_old = d_in[i];
        x_old = x[i];
        if (sum_into) into = sum_into[i];
#pragma unroll
        for (int q = 0; q < RB; ++q) drow[q] = dinv[(size_t)own * RB * RB + (size_t)p * RB + q];
    }
    const V sum = rows_sum_batch<RB, RB, M, RPW, S, V>(a, terms, (int)(lane / LW), (int)(lane % LW), start, len, d_in);
    r_new[lane] = r_old - sum;
    __syncthreads();
    if (!owner) return;
    const V *row_r = r_new + lane - within + m;
    V z = (V)0;
#pragma unroll
    for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * row_r[q * M];
    const V dn = keep * d_old + step * z;
    const V xn = x_old + dn;
    d_out[i] = dn;
    r_out[i] = r_new[lane];
    x[i] = xn;
    if (sum_into) {
        const V total = into + xn;
        sum_into[i] = total;
        if (widen_into) widen_into[i] = (double)total;
    }
}

// One later Chebyshev step for M columns, fused as cheb_step_kernel: ad = A d_in;
// r_out = r_in - ad; z = D^-1 r_out (the lane holds its block row's residuals); d_out = keep d_in
// + step z; x += d_out; with `sum_into`, sum_into += x (cycle.rs:611-650, :534-536, :655-674).
template <int RB, int BATCH, typename S, typename V, int CPL>
__global__ __launch_bounds__(256) void cheb_step_batch_kernel(Sliced<S> a, int log2g, uint32_t M, const S *__restrict__ dinv,
                                                              const V *__restrict__ d_in, const V *__restrict__ r_in, V keep,
                                                              V step, V *__restrict__ d_out, V *__restrict__ r_out,
                                                              V *__restrict__ x, V *__restrict__ sum_into,
                                                              double *__restrict__ widen_into) {
    constexpr int NPW = Shape<RB>::NPW;
    const GroupLane g = group_lane(log2g, a.order);
    const uint32_t m0 = (uint32_t)g.m * CPL;
    if (g.pos >= a.slices * (uint32_t)NPW || m0 >= M) return;
    const uint32_t row = a.perm[g.pos];
    if (row == NONE) return;
    const uint32_t slice = g.pos / NPW;
    const int j = (int)(g.pos - slice * NPW);
    V ad[RB][CPL];
    rows_product_columns<RB, RB, BATCH, S, V, CPL>(a, a.slice_start[slice], a.row_len[g.pos], j, (int)m0, M, d_in, ad);
    // the CPL columns of each row entry move as one vector
    V r_new[RB][CPL];
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        V r[CPL];
        load_columns<CPL, V>(r_in + ((size_t)row * RB + p) * M + m0, r);
#pragma unroll
        for (int c = 0; c < CPL; ++c) r_new[p][c] = r[c] - ad[p][c];
    }
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const S *drow = dinv + (size_t)row * RB * RB + (size_t)p * RB;
        const size_t i = ((size_t)row * RB + p) * M + m0;
        V dold[CPL], xold[CPL], dn[CPL], xn[CPL];
        load_columns<CPL, V>(d_in + i, dold);
        load_columns<CPL, V>(x + i, xold);
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            V z = (V)0;
#pragma unroll
            for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * r_new[q][c];
            dn[c] = keep * dold[c] + step * z;
            xn[c] = xold[c] + dn[c];
        }
        store_columns<CPL, V>(d_out + i, dn);
        store_columns<CPL, V>(r_out + i, r_new[p]);
        store_columns<CPL, V>(x + i, xn);
        if (sum_into) {
            V acc[CPL];
            load_columns<CPL, V>(sum_into + i, acc);
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[c] = acc[c] + xn[c];
            store_columns<CPL, V>(sum_into + i, acc);
            if (widen_into) {
                double w[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) w[c] = (double)acc[c];
                store_columns<CPL, double>(widen_into + i, w);
            }
        }
    }
}

// The coarsest solve as a product with the f64 inverse for M columns (coarse_inverse_kernel per
// column): out[i][m] = sum over k ascending of inv(i, k) b[k][m], from zero. A block takes R rows
// (coarse_rows: R * M' = 256 with M' the power of two at or above M, so one sum per thread) and all
// the columns: thread t is row t % R, column t / R. Tiles of 32 k of the inverse's R rows and of
// b pass through two LDS buffers, the next tile's loads in flight while the current one is summed.
constexpr int COARSE_TILE_K = 32;
constexpr int COARSE_STAGE = COARSE_TILE_K * 64 / 256;  // tile entries per thread, R and M at most 64
__host__ __device__ inline uint32_t coarse_rows(uint32_t M) {
    uint32_t p = 1;
    while (p < M) p *= 2;
    return p >= 4 ? 256 / p : 64;
}
template <typename V>
__global__ __launch_bounds__(256) void coarse_inverse_batch_kernel(uint32_t n, uint32_t M, uint32_t R, const double *__restrict__ inv,
                                                                   const V *__restrict__ rhs, V *__restrict__ out) {
    __shared__ double as[2][COARSE_TILE_K * 64];
    __shared__ double bs[2][COARSE_TILE_K * 64];
    const uint32_t t = threadIdx.x, r = t % R, m = t / R;
    const uint32_t i0 = blockIdx.x * R, i = i0 + r;
    double pa[COARSE_STAGE], pb[COARSE_STAGE];
    // tile k0's entries e = t + 256 j: inverse entry (k0 + e / R, i0 + e % R), b entry k0 * M + e
    auto fetch = [&](uint32_t k0) {
        const uint32_t kn = n - k0 < (uint32_t)COARSE_TILE_K ? n - k0 : (uint32_t)COARSE_TILE_K;
#pragma unroll
        for (int j = 0; j < COARSE_STAGE; ++j) {
            const uint32_t e = t + 256 * j, kk = e / R, rr = e % R;
            pa[j] = kk < kn && i0 + rr < n ? inv[(size_t)(k0 + kk) * n + i0 + rr] : 0.0;
            pb[j] = e < kn * M ? (double)rhs[(size_t)k0 * M + e] : 0.0;
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int j = 0; j < COARSE_STAGE; ++j) {
            as[buf][t + 256 * j] = pa[j];
            bs[buf][t + 256 * j] = pb[j];
        }
    };
    fetch(0);
    put(0);
    __syncthreads();
    double sum = 0.0;
    int buf = 0;
    for (uint32_t k0 = 0; k0 < n; k0 += COARSE_TILE_K) {
        const uint32_t kn = n - k0 < (uint32_t)COARSE_TILE_K ? n - k0 : (uint32_t)COARSE_TILE_K;
        const bool more = k0 + COARSE_TILE_K < n;
        if (more) fetch(k0 + COARSE_TILE_K);
        if (m < M && i < n)
            for (uint32_t kk = 0; kk < kn; ++kk) sum = sum + as[buf][kk * R + r] * bs[buf][kk * M + m];
        if (more) put(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    if (m < M && i < n) out[(size_t)i * M + m] = (V)sum;
}

// The same product where it has few sums (row, column), too few to fill the chip with a thread each:
// a workgroup takes eight of them, all threads form a chunk of their terms into LDS at once, and a row
// of 16 lanes adds each sum's terms in ascending k (add_row_terms). n = 377 rows and 5 columns took
// 20 us with the tiles above, 12 workgroups in a chain of round trips.
constexpr uint32_t COARSE_SUMS = 8, COARSE_SUMS_CHUNK = 512;
// Sums up to which this form is taken, two waves of the chip's workgroups. n = 774, an iteration of a
// 220k-DOF plate: 16 columns 882 us (908 with the tiles), 32 1344 (1329), 64 2418 (2363).
constexpr size_t COARSE_SUMS_MOST = 16384;
template <typename V>
__global__ __launch_bounds__(256) void coarse_inverse_sums_kernel(uint32_t n, uint32_t M, const double *__restrict__ inv,
                                                                  const V *__restrict__ rhs, V *__restrict__ out) {
    __shared__ __align__(16) double terms[COARSE_SUMS][COARSE_SUMS_CHUNK + 2];
    const uint32_t t = threadIdx.x, first = blockIdx.x * COARSE_SUMS, count = n * M;
    double sum = 0.0;
    for (uint32_t k0 = 0; k0 < n; k0 += COARSE_SUMS_CHUNK) {
        constexpr uint32_t PER = COARSE_SUMS_CHUNK / 256;
        double a[COARSE_SUMS][PER], bk[COARSE_SUMS][PER];
#pragma unroll
        for (uint32_t r = 0; r < COARSE_SUMS; ++r) {
            const uint32_t e = first + r < count ? first + r : count - 1, i = e / M, m = e - i * M;
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                const uint32_t k = k0 + t + 256 * j;
                a[r][j] = k < n ? inv[(size_t)i * n + k] : 0.0;
                bk[r][j] = k < n ? (double)rhs[(size_t)k * M + m] : 0.0;
            }
        }
        if (k0) __syncthreads();  // the chunk before has been added
#pragma unroll
        for (uint32_t r = 0; r < COARSE_SUMS; ++r)
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) terms[r][t + 256 * j] = a[r][j] * bk[r][j];
        __syncthreads();
        if (t < COARSE_SUMS * 16)
            sum = add_row_terms(sum, (const double *)terms[t / 16], n - k0 < COARSE_SUMS_CHUNK ? n - k0 : COARSE_SUMS_CHUNK);
    }
    if (t < COARSE_SUMS * 16 && t % 16 == 0 && first + t / 16 < count) out[first + t / 16] = (V)sum;
}

// ---- conjugate gradient, M columns -----------------------------------------------------------

// Batched dot products whose every column is bit for bit the single-column TREE dot
// (dot_partials_kernel then dot_final_kernel): block `blk` forms, for each thread slot t of the
// single kernel and each column, the same grid-stride sum from zero; the sums are staged in LDS
// and reduced by the same pairs as the single kernel's shuffle butterfly (lane l with l + off for
// off = 32 .. 1, lane 0's value), then its four wave sums in order from zero. Columns read
// coalesced: thread u takes column u % M of slots t = u / M, u / M + 256 / M, ..., eight slots at a
// time, so that each grid-stride step has their sixteen loads in flight together.
constexpr int DOT_CHUNK = 8;
// The sums of a block's DOT_THREADS slots per column, from LDS, into the block's partials.
__device__ __forceinline__ void reduce_slots(double *ls, uint32_t M, double *__restrict__ partials) {
    const uint32_t u = threadIdx.x;
    __syncthreads();
    // the butterfly of wave_sum, as pairs: s[l] = s[l] + s[l + off] for l < off
    for (uint32_t off = WAVE / 2; off > 0; off >>= 1) {
        const uint32_t work = (DOT_THREADS / WAVE) * off * M;
        for (uint32_t e = u; e < work; e += DOT_THREADS) {
            const uint32_t m = e % M, rest = e / M, l = rest % off, w = rest / off;
            const uint32_t t = w * WAVE + l;
            ls[t * M + m] = ls[t * M + m] + ls[(t + off) * M + m];
        }
        __syncthreads();
    }
    for (uint32_t m = u; m < M; m += DOT_THREADS) {
        double s = 0.0;
        for (int w = 0; w < DOT_THREADS / WAVE; ++w) s = s + ls[(size_t)w * WAVE * M + m];
        partials[(size_t)blockIdx.x * M + m] = s;
    }
}

template <int MODE>
__global__ __launch_bounds__(DOT_THREADS) void dot_partials_batch_kernel(size_t n, uint32_t M, const double *__restrict__ a,
                                                                          const double *__restrict__ b,
                                                                          double *__restrict__ partials) {
    extern __shared__ double ls[];  // DOT_THREADS x M
    const uint32_t u = threadIdx.x;
    const uint32_t groups = DOT_THREADS / M;
    const size_t stride = (size_t)gridDim.x * DOT_THREADS;
    if (u < groups * M) {
        const uint32_t m = u % M;
        for (uint32_t t0 = u / M; t0 < (uint32_t)DOT_THREADS; t0 += DOT_CHUNK * groups) {
            double v[DOT_CHUNK];
#pragma unroll
            for (int j = 0; j < DOT_CHUNK; ++j) v[j] = 0.0;
            for (size_t base = (size_t)blockIdx.x * DOT_THREADS; base < n; base += stride) {
                double x[DOT_CHUNK], y[DOT_CHUNK];
#pragma unroll
                for (int j = 0; j < DOT_CHUNK; ++j) {
                    const size_t i = base + t0 + (size_t)j * groups;
                    const bool live = t0 + j * groups < (uint32_t)DOT_THREADS && i < n;
                    x[j] = live ? a[i * M + m] : 0.0;
                    y[j] = MODE == 0 && live ? b[i * M + m] : 0.0;
                }
#pragma unroll
                for (int j = 0; j < DOT_CHUNK; ++j)  // each slot's terms in ascending i, as alone
                    if (t0 + j * groups < (uint32_t)DOT_THREADS && base + t0 + (size_t)j * groups < n)
                        v[j] = v[j] + (MODE == 0 ? x[j] * y[j] : x[j]);
            }
#pragma unroll
            for (int j = 0; j < DOT_CHUNK; ++j)
                if (t0 + j * groups < (uint32_t)DOT_THREADS) ls[(t0 + j * groups) * M + m] = v[j];
        }
    }
    reduce_slots(ls, M, partials);
}

// What a batched final sum feeds, per column: STORE writes the column's `out` field (`field` is a
// byte offset into PcgScalars); RZ forms rz_next, beta and rz as dot_finish does. Columns whose
// `mask` entry is zero are left as they are.
static __global__ __launch_bounds__(DOT_THREADS) void dot_final_batch_kernel(int parts, uint32_t M, const double *__restrict__ partials,
                                                                             int kind, uint32_t field, PcgScalars *s,
                                                                             const uint32_t *__restrict__ mask, PcgScalars *mirror,
                                                                             uint32_t tag) {
    const uint32_t m = blockIdx.x;
    double v = 0.0;
    for (int i = threadIdx.x; i < parts; i += blockDim.x) v = v + partials[(size_t)i * M + m];
    const double total = block_sum(v);
    if (threadIdx.x == 0) {
        PcgScalars *c = s + m;
        if (!mask || mask[m]) {
            if (kind == FINAL_STORE) *(double *)((char *)c + field) = total;
            else dot_finish(FINAL_RZ, total, nullptr, c);
        }
        // a column's scalars for the host, as dot_final_kernel's
        if (mirror) mirror_scalars(c, mirror + m, tag);
    }
}

// The scalars of all M columns for the host (the serial order's readback).
static __global__ void mirror_columns_kernel(uint32_t M, const PcgScalars *s, PcgScalars *mirror, uint32_t tag) {
    const uint32_t m = threadIdx.x;
    if (m < M) mirror_scalars(s + m, mirror + m, tag);
}

// For few columns, the final sums formed by every block of the kernel that uses them, as tree_total
// does for one: a launch less each. FUSED_COLUMNS: each block reads every column's 512 partials, which
// at eight columns costs what it saves on a 300k-DOF block (733 us an iteration against 736 with sums of
// their own; one column 345 against 353) and less on smaller systems (plate of 55k DOFs 289 against 300).
constexpr uint32_t FUSED_COLUMNS = 8;
// M is a compile-time count, so that every column's partials are in flight at once.
template <uint32_t M>
__device__ __forceinline__ void tree_totals(const double *__restrict__ partials, double (&totals)[FUSED_COLUMNS]) {
    __shared__ double wsum[FUSED_COLUMNS][DOT_THREADS / WAVE];
    static_assert(DOT_BLOCKS == 2 * DOT_THREADS, "two partials a thread");
    double first[M], second[M];
#pragma unroll
    for (uint32_t m = 0; m < M; ++m) {
        first[m] = partials[(size_t)threadIdx.x * M + m];
        second[m] = partials[(size_t)(threadIdx.x + DOT_THREADS) * M + m];
    }
#pragma unroll
    for (uint32_t m = 0; m < M; ++m) {
        const double v = wave_sum((0.0 + first[m]) + second[m]);  // dot_final_batch_kernel's sums
        if (threadIdx.x % WAVE == 0) wsum[m][threadIdx.x / WAVE] = v;
    }
    __syncthreads();
    if (threadIdx.x < M) {
        double t = 0.0;
        for (int w = 0; w < DOT_THREADS / WAVE; ++w) t = t + wsum[threadIdx.x][w];
        totals[threadIdx.x] = t;
    }
    __syncthreads();
}

// pcg_update_fused_kernel for M <= FUSED_COLUMNS columns: p . A p from its partials, the update of
// pcg_update_batch_kernel, and the partials of the new r . r over dot_partials_batch_kernel's slots.
template <uint32_t M>
__global__ __launch_bounds__(DOT_THREADS) void pcg_update_fused_batch_kernel(size_t n, PcgScalars *__restrict__ s, uint32_t slot,
                                                                                    const uint32_t *__restrict__ active,
                                                                                    const double *__restrict__ pap_partials,
                                                                                    const double *__restrict__ p,
                                                                                    const double *__restrict__ ap, double *__restrict__ x,
                                                                                    double *__restrict__ r, double *__restrict__ rr_partials) {
    extern __shared__ double ls[];  // DOT_THREADS x M
    __shared__ double totals[FUSED_COLUMNS];
    tree_totals<M>(pap_partials, totals);
    const uint32_t u = threadIdx.x, groups = DOT_THREADS / M, m = u % M;
    const double curvature = totals[m], rz = rz_in(s + m, slot);
    const bool live_column = active[m] != 0;
    const bool valid = !(isnan(curvature) || curvature <= 0.0 || !isfinite(rz));
    const double alpha = rz / curvature;
    if (blockIdx.x == 0 && u < M) {
        s[m].curvature = curvature;
        if (live_column) {
            s[m].valid = valid ? 1 : 0;
            s[m].alpha = alpha;
        }
    }
    const bool moves = live_column && valid;
    const size_t stride = (size_t)gridDim.x * DOT_THREADS;
    if (u < groups * M) {
        for (uint32_t t0 = u / M; t0 < (uint32_t)DOT_THREADS; t0 += DOT_CHUNK * groups) {
            double v[DOT_CHUNK];
#pragma unroll
            for (int j = 0; j < DOT_CHUNK; ++j) v[j] = 0.0;
            for (size_t base = (size_t)blockIdx.x * DOT_THREADS; base < n; base += stride) {
                double rv[DOT_CHUNK], xv[DOT_CHUNK], pv[DOT_CHUNK], av[DOT_CHUNK];
#pragma unroll
                for (int j = 0; j < DOT_CHUNK; ++j) {
                    const size_t i = base + t0 + (size_t)j * groups;
                    if (t0 + j * groups < (uint32_t)DOT_THREADS && i < n) {
                        rv[j] = r[i * M + m];
                        if (moves) {
                            xv[j] = x[i * M + m];
                            pv[j] = p[i * M + m];
                            av[j] = ap[i * M + m];
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < DOT_CHUNK; ++j) {
                    const size_t i = base + t0 + (size_t)j * groups;
                    if (t0 + j * groups < (uint32_t)DOT_THREADS && i < n) {
                        if (moves) {
                            x[i * M + m] = xv[j] + alpha * pv[j];
                            rv[j] = rv[j] + (-alpha) * av[j];
                            r[i * M + m] = rv[j];
                        }
                        v[j] = v[j] + rv[j] * rv[j];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < DOT_CHUNK; ++j)
                if (t0 + j * groups < (uint32_t)DOT_THREADS) ls[(t0 + j * groups) * M + m] = v[j];
        }
    }
    reduce_slots(ls, M, rr_partials);
}

// pcg_direction_fused_kernel for M <= FUSED_COLUMNS columns: r . z from its partials, beta, then
// p = z + beta p in the active columns. Block 0 stores the next r . z in the other slot.
template <uint32_t M>
__global__ __launch_bounds__(DOT_THREADS) void pcg_direction_fused_batch_kernel(size_t n, PcgScalars *__restrict__ s,
                                                                                       uint32_t slot, const uint32_t *__restrict__ active,
                                                                                       const double *__restrict__ rz_partials,
                                                                                       const double *__restrict__ z, double *__restrict__ p) {
    __shared__ double totals[FUSED_COLUMNS];
    __shared__ double betas[FUSED_COLUMNS];
    tree_totals<M>(rz_partials, totals);
    if (threadIdx.x < M) {
        const uint32_t m = threadIdx.x;
        const double beta = totals[m] / rz_in(s + m, slot);
        betas[m] = beta;
        if (blockIdx.x == 0 && active[m]) {
            rz_in(s + m, slot ^ 1u) = totals[m];
            s[m].beta = beta;
        }
    }
    __syncthreads();
    const size_t stride = (size_t)gridDim.x * DOT_THREADS;
    for (size_t e = (size_t)blockIdx.x * DOT_THREADS + threadIdx.x; e < n * M; e += stride) {
        const uint32_t m = (uint32_t)(e % M);
        if (active[m]) p[e] = z[e] + betas[m] * p[e];
    }
}

// REFERENCE order for M columns: one thread per column sums in index order from zero
// (crates/solidfem-solve/src/pcg.rs:285-291).
template <int MODE>
__global__ void dot_serial_batch_kernel(size_t n, uint32_t M, const double *__restrict__ a, const double *__restrict__ b,
                                        int kind, uint32_t field, PcgScalars *s, const uint32_t *__restrict__ mask) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    double sum = 0.0;
    for (size_t i = 0; i < n; ++i) sum = sum + (MODE == 0 ? a[i * M + m] * b[i * M + m] : a[i * M + m]);
    if (mask && !mask[m]) return;
    PcgScalars *c = s + m;
    if (kind == FINAL_STORE) *(double *)((char *)c + field) = sum;
    else dot_finish(FINAL_RZ, sum, nullptr, c);
}

// pcg_update_kernel per column; columns whose `active` entry is zero are not touched.
static __global__ void pcg_update_batch_kernel(size_t n, uint32_t M, PcgScalars *__restrict__ s, const uint32_t *__restrict__ active,
                                               const double *__restrict__ p, const double *__restrict__ ap,
                                               double *__restrict__ x, double *__restrict__ r) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * M) return;
    const uint32_t m = (uint32_t)(e % M);
    if (!active[m]) return;
    const double curvature = s[m].curvature, rz = s[m].rz;
    const bool valid = !(isnan(curvature) || curvature <= 0.0 || !isfinite(rz));
    const double alpha = rz / curvature;
    if (e < M) {
        s[m].valid = valid ? 1 : 0;
        s[m].alpha = alpha;
    }
    if (!valid) return;
    x[e] = x[e] + alpha * p[e];
    r[e] = r[e] + (-alpha) * ap[e];
}

// p = z + beta p per active column.
static __global__ void pcg_direction_batch_kernel(size_t n, uint32_t M, const PcgScalars *__restrict__ s,
                                                  const uint32_t *__restrict__ active, const double *__restrict__ z,
                                                  double *__restrict__ p) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * M) return;
    const uint32_t m = (uint32_t)(e % M);
    if (active[m]) p[e] = z[e] + s[m].beta * p[e];
}

// dst = src in the columns whose mask entry is set.
template <typename T>
__global__ void copy_columns_kernel(size_t n, uint32_t M, const uint32_t *__restrict__ mask, const T *__restrict__ src,
                                    T *__restrict__ dst) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n * M && mask[e % M]) dst[e] = src[e];
}

// Column m of a row-interleaved array from a plain vector.
template <typename T>
__global__ void set_column_kernel(size_t n, uint32_t M, uint32_t m, const T *__restrict__ src, T *__restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i * M + m] = src[i];
}
template <typename T>
__global__ void get_column_kernel(size_t n, uint32_t M, uint32_t m, const T *__restrict__ src, T *__restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i * M + m];
}

// Zeroes the masked columns of a row-interleaved array.
template <typename T>
__global__ void zero_columns_kernel(size_t n, uint32_t M, const uint32_t *__restrict__ mask, T *__restrict__ dst) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n * M && mask[e % M]) dst[e] = (T)0;
}

// Zeroes the scalars of the masked columns.
static __global__ void zero_scalars_kernel(uint32_t M, const uint32_t *__restrict__ mask, PcgScalars *s) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < M && mask[m]) s[m] = PcgScalars{};
}

// Column-major (column m at m * n) to row-interleaved, and back.
template <typename T>
__global__ void interleave_kernel(size_t n, uint32_t M, const T *__restrict__ cm, T *__restrict__ il) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * M) return;
    const size_t i = e / M, m = e - i * M;
    il[e] = cm[m * n + i];
}
template <typename T>
__global__ void deinterleave_kernel(size_t n, uint32_t M, const T *__restrict__ il, T *__restrict__ cm) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * M) return;
    const size_t m = e / n, i = e - m * n;
    cm[e] = il[i * M + m];
}

// z = r * inverse diagonal for M columns (preconditioner.rs:237-247).
static __global__ void jacobi_batch_kernel(size_t n, uint32_t M, const double *__restrict__ inv, const double *__restrict__ r,
                                           double *__restrict__ z) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n * M) z[e] = r[e] * inv[e / M];
}

}  // namespace dev
}  // namespace sf
