// Device kernels of the solve path for gfx950 (CDNA4, wave64).
//
// Sliced block layout ("node slices"). A block sparse matrix of RB x CB blocks is cut into
// slices of NPW = 64 / RB block rows (21 nodes of 3 rows, 10 of 6, 64 scalar rows), one
// wavefront per slice and one lane per scalar row. Within a slice, the k-th block of every row
// is stored side by side: block columns at cols[(start + k) * NPW + j] and values at
// vals[((start + k) * 64 + j * RB + p) * CB + q] for row j, block row p, block column q. A lane's
// CB values of a block are contiguous, one vector load, and a wavefront's loads of one slot cover
// 64 * CB consecutive values; the RB lanes of a row read the same column index (one fetch), and
// every lane sums its own row's blocks in stored order, column by column, from zero: the
// summation order of the reference's block product
// (crates/solidfem-solve/src/multigrid/block.rs:136-154), so the result is the same bits.
// BATCH blocks are loaded before their terms are added, in order, so BATCH loads are in flight
// per lane whatever the latency; the batch depth changes no bit and is chosen per matrix by timing.
// Rows are permuted inside windows so that a slice's rows have similar block counts; perm[]
// maps a slice position back to the block row.
//
// Every kernel is compiled with -ffp-contract=off: no multiply-add is fused, as the reference
// refuses mul_add (clippy.toml:8-9), so the device repeats the reference's roundings.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace sf {
namespace dev {

constexpr int WAVE = 64;
constexpr uint32_t NONE = 0xffffffffu;

template <int RB>
struct Shape {
    static constexpr int NPW = WAVE / RB;  // block rows per slice
    static constexpr int LANES = NPW * RB; // lanes holding a scalar row
};

template <typename T>
struct Sliced {
    const uint32_t *slice_start;  // slices + 1, in block slots per row
    const uint32_t *row_len;      // per slice position: blocks in the row (0 for padding)
    const uint32_t *perm;         // per slice position: block row, NONE for padding
    const uint32_t *cols;         // per block slot and slice row
    const T *vals;                // per block slot, block column and lane
    uint32_t slices;
    uint32_t order;               // workgroup -> slice order: ORDER_* bits (slice_of)
};

// Workgroup-to-slice orders; none changes a bit of any result, only which workgroups run
// together and where. XCD_RUNS gives each XCD one contiguous run of slices; XCD_WINDOWS gives
// each XCD whole sort windows (8 workgroups of 4 slices), so the rows a window permutes share one
// L2; REVERSE walks the slices from the end (alternate passes over a matrix then start where the
// last one ended, in the cache).
enum : uint32_t { ORDER_XCD_RUNS = 1, ORDER_XCD_WINDOWS = 2, ORDER_REVERSE = 4, ORDER_GROUP_RUNS = 8, ORDER_GROUP_CHUNKS = 16 };
// With ORDER_GROUP_CHUNKS, bits 24-31 of an order hold log2 of the chunk (workgroups per XCD).
constexpr uint32_t ORDER_CHUNK_SHIFT = 24;

template <typename V, typename S>
__device__ __forceinline__ V widen(S s) {
    return (V)(double)s;
}

// Workgroups are dispatched to the 8 XCDs in turn (workgroup b to XCD b mod 8). The renumberings
// below are bijections on [0, gridDim.x).
__device__ __forceinline__ uint32_t xcd_runs_block() {
    constexpr uint32_t XCDS = 8;
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    const uint32_t x = b % XCDS, local = b / XCDS, base = nb / XCDS, rem = nb % XCDS;
    return x * base + (x < rem ? x : rem) + local;
}
__device__ __forceinline__ uint32_t xcd_windows_block() {
    // within each group of 64 workgroups, XCD x takes logical workgroups 8x .. 8x + 7
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    if (b >= nb - nb % 64) return b;
    const uint32_t r = b % 64;
    return b - r + (r % 8) * 8 + r / 8;
}
// Within each group of 8 W workgroups, XCD x takes the W consecutive logical workgroups
// x W .. x W + W - 1 (W = 2^lw); the tail past the last whole group keeps its order.
__device__ __forceinline__ uint32_t xcd_chunks_block(uint32_t lw) {
    const uint32_t nb = gridDim.x, b = blockIdx.x, group = 8u << lw;
    if (b >= nb - nb % group) return b;
    const uint32_t r = b & (group - 1u);
    return b - r + (r & 7u) * (1u << lw) + (r >> 3);
}
// The slice a wavefront works on under `order` (4 wavefronts of 64 lanes per workgroup).
__device__ __forceinline__ uint32_t slice_of(uint32_t order) {
    const uint32_t block = (order & ORDER_XCD_RUNS) ? xcd_runs_block() : (order & ORDER_XCD_WINDOWS) ? xcd_windows_block() : blockIdx.x;
    const uint32_t waves = blockDim.x / WAVE;
    uint32_t slice = block * waves + threadIdx.x / WAVE;
    if (order & ORDER_REVERSE) slice = gridDim.x * waves - 1 - slice;
    return slice;
}

// Sum of one lane's row of A x, from zero in stored order: the row product of the reference.
// The column indices of the next batch are loaded with the current batch's values, so each
// batch costs one dependent memory round trip.
template <int RB, int CB, int BATCH, typename S, typename V>
__device__ __forceinline__ V row_product(const Sliced<S> &a, uint32_t slot0, uint32_t len, int j, int lane,
                                         const V *__restrict__ x) {
    constexpr int NPW = Shape<RB>::NPW;
    V sum = (V)0;
    const uint32_t *cp = a.cols + (size_t)slot0 * NPW + j;
    const S *vp = a.vals + ((size_t)slot0 * WAVE + lane) * CB;
    const uint32_t full = len - len % BATCH;
    uint32_t c[BATCH];
    if (full) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) c[b] = cp[(size_t)b * NPW];
    }
    for (uint32_t k = 0; k < full; k += BATCH) {
        S v[BATCH][CB];
        V xv[BATCH][CB];
        uint32_t cn[BATCH];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) v[b][q] = vp[(size_t)(k + b) * WAVE * CB + q];
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) xv[b][q] = x[(size_t)c[b] * CB + q];
        if (k + BATCH < full) {
#pragma unroll
            for (int b = 0; b < BATCH; ++b) cn[b] = cp[(size_t)(k + BATCH + b) * NPW];
        }
#pragma unroll
        for (int b = 0; b < BATCH; ++b)
#pragma unroll
            for (int q = 0; q < CB; ++q) sum = sum + widen<V>(v[b][q]) * xv[b][q];
#pragma unroll
        for (int b = 0; b < BATCH; ++b) c[b] = cn[b];
    }
    for (uint32_t k = full; k < len; ++k) {
        const uint32_t col = cp[(size_t)k * NPW];
#pragma unroll
        for (int q = 0; q < CB; ++q) sum = sum + widen<V>(vp[(size_t)k * WAVE * CB + q]) * x[(size_t)col * CB + q];
    }
    return sum;
}

enum Epilogue { EPI_STORE = 0, EPI_RESIDUAL = 1, EPI_ADD = 2 };

// The Chebyshev start (cycle.rs:591-610) on a vector a kernel has just produced, so that the
// smoothing that follows needs no launch of its own: z = D^-1 y summed over the block row in
// order from zero, d = z / theta, x = d. A null `dinv` means no start.
template <typename S, typename V>
struct Start {
    const S *dinv;
    V theta;
    V *d;
    V *x;
};

// y = A x (STORE), y = b - A x (RESIDUAL) or y = y + A x (ADD): the block products, the
// residual (crates/solidfem-solve/src/multigrid/cycle.rs:548-564), the gather restriction over
// the stored transpose (crates/solidfem-solve/src/gpu/layout.rs:249-291) and the prolongation
// with correction (cycle.rs:512-521); optionally followed by the Chebyshev start on y, the RB
// values of a block row shuffled in from its lanes.
template <int RB, int CB, int BATCH, typename S, typename V, int EPI>
__global__ __launch_bounds__(256) void spmv_kernel(Sliced<S> a, const V *__restrict__ x, V *__restrict__ y,
                                                   const V *__restrict__ b, Start<S, V> start) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t slice = slice_of(a.order);
    if (slice >= a.slices) return;  // whole wave leaves together
    const int lane = threadIdx.x % WAVE;
    const int j = lane / RB, p = lane - j * RB;
    const bool in_wave = j < NPW;
    const uint32_t pos = slice * NPW + (in_wave ? j : 0);
    const uint32_t row = in_wave ? a.perm[pos] : NONE;
    const bool live = row != NONE;
    const size_t out = live ? (size_t)row * RB + p : 0;
    V value = (V)0;
    if (live) {
        const V sum = row_product<RB, CB, BATCH, S, V>(a, a.slice_start[slice], a.row_len[pos], j, lane, x);
        if (EPI == EPI_STORE) value = sum;
        else if (EPI == EPI_RESIDUAL) value = b[out] - sum;
        else value = y[out] + sum;
        y[out] = value;
    }
    if (start.dinv) {  // uniform: every lane takes part in the shuffle
        const S *drow = start.dinv + (live ? (size_t)row * RB * RB + (size_t)p * RB : 0);
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) {
            const V yq = __shfl(value, (in_wave ? j * RB : 0) + q, WAVE);
            if (live) z = z + widen<V>(drow[q]) * yq;
        }
        if (live) {
            const V dv = z / start.theta;
            start.d[out] = dv;
            start.x[out] = dv;
        }
    }
}

// A block matrix in plain block rows: row r's blocks at [starts[r], starts[r + 1]), their
// row-major RB x CB values contiguous. Used for matrices with few, long rows.
template <typename T>
struct Bsr {
    const uint32_t *starts;  // rows + 1
    const uint32_t *cols;
    const T *vals;
    uint32_t rows;
    uint32_t reverse;  // nonzero: each XCD takes its workgroups' rows in reverse order (xcd_reversed_block)
};

// Workgroup b runs on XCD b mod 8. Each XCD takes the same rows as in dispatch order, in reverse:
// block x + 8 l becomes x + 8 (c - 1 - l), c the XCD's count of blocks. A pass that follows a
// forward pass over the same matrix then starts with the rows that XCD's L2 holds last.
__device__ __forceinline__ uint32_t xcd_reversed_block() {
    const uint32_t nb = gridDim.x, b = blockIdx.x, x = b % 8u, l = b / 8u;
    const uint32_t count = (nb - x + 7u) / 8u;
    return x + 8u * (count - 1u - l);
}

// The longest row among a wavefront's RPW rows (each row's length is uniform over its lanes).
template <int RPW>
__device__ __forceinline__ uint32_t longest_of_wave(uint32_t len) {
#pragma unroll
    for (int o = WAVE / RPW; o < WAVE; o <<= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)len, o, WAVE);
        len = other > len ? other : len;
    }
    return len;
}

// `n` terms from `t` (LDS, 16-byte aligned) added in order onto `sum`. READS 16-byte reads are one
// group; two groups alternate, the next one's reads issued before this one's additions (the barrier
// keeps the compiler from moving them back), so the chain of additions never waits on LDS. The last
// group is read whole -- `t` has room up to a multiple of a group -- and what lies past `n` is
// replaced by -0.0, which added to any value leaves it as it is.
template <int READS, typename V>
__device__ __forceinline__ V add_terms(V sum, const V *t, uint32_t n) {
    typedef V Quad __attribute__((ext_vector_type(16 / sizeof(V))));
    constexpr uint32_t W = 16 / sizeof(V), GROUP = W * READS;
    const uint32_t groups = (n + GROUP - 1) / GROUP;
    if (groups == 0) return sum;
    auto read = [&](Quad(&q)[READS], uint32_t g) {
        const Quad *p = reinterpret_cast<const Quad *>(t) + (g < groups ? g : groups - 1) * READS;
#pragma unroll
        for (int u = 0; u < READS; ++u) q[u] = p[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const Quad(&q)[READS], uint32_t g) {
        if ((g + 1) * GROUP <= n) {
#pragma unroll
            for (int u = 0; u < READS; ++u)
#pragma unroll
                for (uint32_t v = 0; v < W; ++v) sum = sum + q[u][v];
        } else if (g < groups) {
#pragma unroll
            for (int u = 0; u < READS; ++u)
#pragma unroll
                for (uint32_t v = 0; v < W; ++v) sum = sum + (g * GROUP + u * W + v < n ? q[u][v] : (V)-0.0);
        }
    };
    Quad a[READS], b[READS];
    read(a, 0);
    for (uint32_t g = 0; g < groups; g += 2) {
        read(b, g + 1);
        add(a, g);
        read(a, g + 2);
        add(b, g + 1);
    }
    return sum;
}

// Adds onto acc, in order, the 16 bytes of terms that lanes FIRST .. FIRST + 3 of the lane's row of 16
// hold, one instruction a term: the term comes from its lane with the addition. For double that is
// fma(t, 1, acc), the same value, the product being exact. One block of instructions: between two
// blocks the compiler would put a wait state each. The sum is written before the block's inputs are all
// read, so its register is its own (an early clobber), also where it starts with an input's value.
template <int FIRST>
__device__ __forceinline__ void add_from_lanes(float &acc, float x, float y, float z, float w) {
#define SF_ADD(N)                                                                          \
    "v_add_f32_dpp %0, %1, %0 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"           \
    "v_add_f32_dpp %0, %2, %0 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"           \
    "v_add_f32_dpp %0, %3, %0 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"           \
    "v_add_f32_dpp %0, %4, %0 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" SF_ADD(5) SF_ADD(6) SF_ADD(7) SF_ADD(8)
        : "+&v"(acc)
        : "v"(x), "v"(y), "v"(z), "v"(w), "n"(FIRST), "n"(FIRST + 1), "n"(FIRST + 2), "n"(FIRST + 3));
#undef SF_ADD
}
template <int FIRST>
__device__ __forceinline__ void add_from_lanes(double &acc, double x, double y) {
#define SF_ADD(N)                                                                             \
    "v_fmac_f64_dpp %0, %1, %3 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"             \
    "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" SF_ADD(4) SF_ADD(5) SF_ADD(6) SF_ADD(7)
        : "+&v"(acc)
        : "v"(x), "v"(y), "v"(1.0), "n"(FIRST), "n"(FIRST + 1), "n"(FIRST + 2), "n"(FIRST + 3));
#undef SF_ADD
}
template <int FIRST, typename Quad>
__device__ __forceinline__ void add_from_lanes(float &acc, const Quad &q) {
    add_from_lanes<FIRST>(acc, q[0], q[1], q[2], q[3]);
}
template <int FIRST, typename Quad>
__device__ __forceinline__ void add_from_lanes(double &acc, const Quad &q) {
    add_from_lanes<FIRST>(acc, q[0], q[1]);
}
// Adds onto three sums, in order, the three terms each that lanes FIRST .. FIRST + 3 of the lane's row
// of 16 hold in their registers, as add_from_lanes. The sums take turns, so none waits for its own last
// addition.
template <int FIRST>
__device__ __forceinline__ void add_three_from_lanes(double (&acc)[3], const double (&t)[3][3]) {
#define SF_ADD(A, B, C, N)                                                                  \
    "v_fmac_f64_dpp %0, %" #A ", %16 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"    \
    "v_fmac_f64_dpp %1, %" #B ", %16 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"    \
    "v_fmac_f64_dpp %2, %" #C ", %16 row_newbcast:%" #N " row_mask:0xf bank_mask:0xf\n"
#define SF_LANE(N) SF_ADD(3, 6, 9, N) SF_ADD(4, 7, 10, N) SF_ADD(5, 8, 11, N)
    asm("s_nop 1\n" SF_LANE(12) SF_LANE(13) SF_LANE(14) SF_LANE(15)
        : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2])
        : "v"(t[0][0]), "v"(t[0][1]), "v"(t[0][2]), "v"(t[1][0]), "v"(t[1][1]), "v"(t[1][2]), "v"(t[2][0]), "v"(t[2][1]), "v"(t[2][2]),
          "n"(FIRST), "n"(FIRST + 1), "n"(FIRST + 2), "n"(FIRST + 3), "v"(1.0));
#undef SF_LANE
#undef SF_ADD
}
// add_terms with a row of 16 lanes per sum (four sums a wavefront, every lane of it active, `n` the
// same for all four): one 16-byte read per lane brings 16 lanes' terms, and each addition takes its
// term from the lane that holds it. Where few lanes add, a 16-byte LDS read is what a lane waits on:
// 33-40 cycles for two doubles or four floats, against 5 to 6 for an addition. A lane of its own per
// sum took 16.6 cycles a double, 10 a float. `t` has room up to a multiple of 16 reads; what lies past
// `n` is replaced by -0.0. The sum is in every lane of the row.
template <typename V>
__device__ __forceinline__ V add_row_terms(V sum, const V *t, uint32_t n) {
    constexpr uint32_t W = 16 / sizeof(V), GROUP = 16 * W;
    typedef V Quad __attribute__((ext_vector_type(16 / sizeof(V))));
    const uint32_t c = threadIdx.x % 16u, groups = (n + GROUP - 1) / GROUP;
    if (groups == 0) return sum;
    const Quad *p = reinterpret_cast<const Quad *>(t) + c;
    Quad next = p[0];
    for (uint32_t g = 0; g < groups; ++g) {
        Quad q = next;
        next = p[(g + 1 < groups ? g + 1 : g) * 16];
        const uint32_t left = n - g * GROUP;
        if (left < GROUP) {
#pragma unroll
            for (uint32_t v = 0; v < W; ++v) q[v] = c * W + v < left ? q[v] : (V)-0.0;
        }
        add_from_lanes<0>(sum, q);
        if (left > 4 * W) add_from_lanes<4>(sum, q);
        if (left > 8 * W) add_from_lanes<8>(sum, q);
        if (left > 12 * W) add_from_lanes<12>(sum, q);
    }
    return sum;
}

// The sums of RPW block rows of one wavefront (one workgroup), 64 / RPW lanes each: every lane loads
// U blocks and the x entries they meet, all in flight at once, and forms their terms A[p][q] x[q] into
// LDS; then lane p of a row's group adds row p's terms in stored block order and column order, from
// zero -- the summation of spmv_kernel and of the reference, so the same bits, with one memory round
// trip per U * 64 / RPW blocks instead of one per few blocks. The sum is lane p's of each group.
template <int RB, int CB, typename V, int RPW, int U>
struct RowTerms {
    static constexpr int LW = WAVE / RPW, CHUNK = LW * U;
    V t[RPW][RB][CHUNK * CB + 16 / sizeof(V)];  // rows on different banks
};
template <int RB, int CB, int RPW, int U, typename S, typename V>
__device__ __forceinline__ V rows_sum(const Bsr<S> &a, RowTerms<RB, CB, V, RPW, U> &terms, int g, int sl, uint32_t start, uint32_t len,
                                      const V *__restrict__ x) {
    using T = RowTerms<RB, CB, V, RPW, U>;
    const uint32_t longest = longest_of_wave<RPW>(len);
    if constexpr (RB == 3 && CB == 3 && RPW == 4 && U == 1 && std::is_same<V, double>::value) {
        // A block row is a row of 16 lanes: every lane of it adds all three sums, each term coming from
        // the register of the lane that formed it, and no LDS takes part: the product of a plate of 20,800
        // rows takes 10.2 us, 11.4 through LDS. (In f32, where an LDS read brings four terms, it lost: a
        // step 9.4 against 9.0 us.)
        V sums[3] = {(V)0, (V)0, (V)0};
        for (uint32_t k0 = 0; k0 < longest; k0 += 16) {
            V t[3][3];
            const uint32_t k = k0 + sl;
            if (k < len) {
                const uint32_t col = a.cols[start + k];
                const S *blk = a.vals + (size_t)(start + k) * 9;
                S v[9];
#pragma unroll
                for (int e = 0; e < 9; ++e) v[e] = blk[e];
                V xv[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) xv[q] = x[(size_t)col * 3 + q];
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int q = 0; q < 3; ++q) t[p][q] = widen<V>(v[p * 3 + q]) * xv[q];
            } else {
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int q = 0; q < 3; ++q) t[p][q] = (V)-0.0;  // changes no sum
            }
            const uint32_t left = longest - k0;  // uniform
            add_three_from_lanes<0>(sums, t);
            if (left > 4) add_three_from_lanes<4>(sums, t);
            if (left > 8) add_three_from_lanes<8>(sums, t);
            if (left > 12) add_three_from_lanes<12>(sums, t);
        }
        return sl == 0 ? sums[0] : sl == 1 ? sums[1] : sums[2];
    }
    V sum = (V)0;
    for (uint32_t k0 = 0; k0 < longest; k0 += T::CHUNK) {
        uint32_t col[U];
        S v[U][RB * CB];
        V xv[U][CB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = k0 + sl + u * T::LW;
            if (k < len) {
                col[u] = a.cols[start + k];
                const S *blk = a.vals + (size_t)(start + k) * RB * CB;
#pragma unroll
                for (int e = 0; e < RB * CB; ++e) v[u][e] = blk[e];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + sl + u * T::LW < len) {
#pragma unroll
                for (int q = 0; q < CB; ++q) xv[u][q] = x[(size_t)col[u] * CB + q];
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + sl + u * T::LW < len) {
#pragma unroll
                for (int p = 0; p < RB; ++p)
#pragma unroll
                    for (int q = 0; q < CB; ++q) terms.t[g][p][(sl + u * T::LW) * CB + q] = widen<V>(v[u][p * CB + q]) * xv[u][q];
            }
        __syncthreads();
        if (sl < RB && k0 < len)
            sum = add_terms<4>(sum, (const V *)terms.t[g][sl], (len - k0 < (uint32_t)T::CHUNK ? len - k0 : (uint32_t)T::CHUNK) * CB);
        __syncthreads();
    }
    return sum;
}

// y = A x or y = b - A x (as spmv_kernel) by rows_sum, for matrices with few or long rows: the
// stored transposes of the prolongators, whose rows gather every fine row of an aggregate's
// neighbourhood, the coarse levels, and systems too small to fill the chip with a lane per row.
template <int RB, int CB, typename S, typename V, int EPI, int RPW, int U>
__global__ __launch_bounds__(64) void long_rows_kernel(Bsr<S> a, const V *__restrict__ x, V *__restrict__ y,
                                                       const V *__restrict__ b, Start<S, V> then) {
    constexpr int LW = WAVE / RPW;
    __shared__ __align__(16) RowTerms<RB, CB, V, RPW, U> terms;
    __shared__ V values[RPW][RB];
    const int lane = threadIdx.x, g = lane / LW, sl = lane % LW;
    const uint32_t row = (a.reverse ? xcd_reversed_block() : blockIdx.x) * RPW + (uint32_t)g;
    const bool live = row < a.rows;
    const uint32_t start = live ? a.starts[row] : 0u, len = live ? a.starts[row + 1] - start : 0u;
    const bool owner = live && sl < RB;
    const size_t out = (size_t)row * RB + (owner ? sl : 0);
    // what the epilogue reads is fetched before the sums
    const V before = !owner || EPI == EPI_STORE ? (V)0 : b[out];
    S drow[RB];
    if (then.dinv && owner) {
#pragma unroll
        for (int q = 0; q < RB; ++q) drow[q] = then.dinv[(size_t)row * RB * RB + (size_t)sl * RB + q];
    }
    const V sum = rows_sum<RB, CB, RPW, U, S, V>(a, terms, g, sl, start, len, x);
    if (owner) {
        const V value = EPI == EPI_STORE ? sum : before - sum;
        y[out] = value;
        values[g][sl] = value;
    }
    if (then.dinv) {  // uniform
        __syncthreads();
        if (owner) {
            V z = (V)0;
#pragma unroll
            for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * values[g][q];
            const V dv = z / then.theta;
            then.d[out] = dv;
            then.x[out] = dv;
        }
    }
}

// long_rows_kernel with one workgroup of four wavefronts per block row, for matrices whose rows
// are so long (hundreds of blocks) and so few that one wavefront per row leaves the chip idle
// through a chain of round trips. All four wavefronts load CHUNK blocks' values and x entries at
// once and put their terms into one of two LDS buffers; then each row of 16 lanes of the first
// wavefronts adds one of the block row's RB rows' terms in stored order (add_row_terms) while the
// next chunk's loads are in flight (its block columns were fetched a chunk before that). Bound by the
// ordered chain of additions: 73 rows of 350 blocks, f32, took 21 us a wavefront per row, 11 us
// here with a lane per sum and 10.2 with a row of 16 lanes per sum.
template <int RB, int CB, typename V>
struct WideRows {
    static constexpr int THREADS = 256;
    // a block is shared by PARTS threads, RB / PARTS rows each, so that both LDS buffers stay under 40 KB
    static constexpr int PARTS = CB * sizeof(V) <= 12 ? 1 : CB * sizeof(V) <= 24 ? 2 : 3;
    static constexpr int CHUNK = PARTS == 1 ? 256 : PARTS == 2 ? 128 : 64;
    static constexpr int STRIDE = CHUNK * CB + 16 / sizeof(V);  // rows on different banks, 16-byte aligned
    static_assert(RB % PARTS == 0 && CHUNK * PARTS <= THREADS, "whole rows per thread");
};
template <int RB, int CB, typename S, typename V>
__global__ __launch_bounds__(256) void wide_rows_kernel(Bsr<S> a, const V *__restrict__ x, V *__restrict__ y, Start<S, V> then) {
    using W = WideRows<RB, CB, V>;
    constexpr int RP = RB / W::PARTS;
    __shared__ __align__(16) V terms[2][RB][W::STRIDE];
    __shared__ V values[RB];
    const uint32_t row = a.reverse ? xcd_reversed_block() : blockIdx.x;  // one workgroup per row: row < a.rows
    const uint32_t start = a.starts[row], len = a.starts[row + 1] - start;
    const uint32_t t = threadIdx.x, k = t / W::PARTS, p0 = (t % W::PARTS) * RP;
    const bool loads = k < (uint32_t)W::CHUNK;
    // the row of 16 lanes t / 16 adds row p of the block row (whole wavefronts: rows past RB repeat the last)
    const bool adds = t / WAVE < (uint32_t)(RB + 3) / 4;
    const uint32_t p = t / 16 < (uint32_t)RB ? t / 16 : RB - 1;
    const bool owner = t / 16 < (uint32_t)RB && t % 16 == 0;
    const size_t out = (size_t)row * RB + p;
    // what the start reads is fetched before the sums
    S drow[RB];
    if (then.dinv && owner) {
#pragma unroll
        for (int q = 0; q < RB; ++q) drow[q] = then.dinv[(size_t)row * RB * RB + (size_t)p * RB + q];
    }
    S v[RP * CB];
    V xv[CB];
    auto fetch = [&](uint32_t at, uint32_t col) {
        if (loads && at < len) {
            const S *blk = a.vals + ((size_t)(start + at) * RB + p0) * CB;
#pragma unroll
            for (int e = 0; e < RP * CB; ++e) v[e] = blk[e];
#pragma unroll
            for (int q = 0; q < CB; ++q) xv[q] = x[(size_t)col * CB + q];
        }
    };
    uint32_t col = loads && k < len ? a.cols[start + k] : 0u;
    fetch(k, col);
    col = loads && k + W::CHUNK < len ? a.cols[start + k + W::CHUNK] : 0u;
    V sum = (V)0;
    int buf = 0;
    for (uint32_t k0 = 0; k0 < len; k0 += W::CHUNK, buf ^= 1) {
        if (loads && k0 + k < len) {
#pragma unroll
            for (int r = 0; r < RP; ++r)
#pragma unroll
                for (int q = 0; q < CB; ++q) terms[buf][p0 + r][k * CB + q] = widen<V>(v[r * CB + q]) * xv[q];
        }
        const uint32_t k1 = k0 + W::CHUNK, k2 = k1 + W::CHUNK;
        if (k1 < len) {
            fetch(k1 + k, col);
            if (loads && k2 + k < len) col = a.cols[start + k2 + k];
        }
        // one barrier per chunk: this buffer is written again two chunks on, after the next barrier,
        // which the adding wavefronts reach only once they have read it
        __syncthreads();
        if (adds) sum = add_row_terms(sum, (const V *)terms[buf][p], (len - k0 < (uint32_t)W::CHUNK ? len - k0 : (uint32_t)W::CHUNK) * CB);
    }
    if (owner) {
        y[out] = sum;
        values[p] = sum;
    }
    if (then.dinv) {  // uniform
        __syncthreads();
        if (owner) {
            V z = (V)0;
#pragma unroll
            for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * values[q];
            const V dv = z / then.theta;
            then.d[out] = dv;
            then.x[out] = dv;
        }
    }
}

// The fused Chebyshev step of cheb_step_kernel by rows_sum: lane p of a row's group holds A d_in, and
// the RB residuals of the block row meet in LDS for the block-Jacobi product (summed over q in order
// from zero). The same bits as cheb_step_kernel.
template <int RB, typename S, typename V, int RPW, int U>
__global__ __launch_bounds__(64) void cheb_rows_kernel(Bsr<S> a, const S *__restrict__ dinv, const V *__restrict__ d_in,
                                                       const V *__restrict__ r_in, V keep, V step, V *__restrict__ d_out,
                                                       V *__restrict__ r_out, V *__restrict__ x, V *__restrict__ sum_into,
                                                       double *__restrict__ widen_into) {
    constexpr int LW = WAVE / RPW;
    __shared__ __align__(16) RowTerms<RB, RB, V, RPW, U> terms;
    __shared__ V r_new[RPW][RB];
    const int lane = threadIdx.x, g = lane / LW, sl = lane % LW;
    const uint32_t row = (a.reverse ? xcd_reversed_block() : blockIdx.x) * RPW + (uint32_t)g;
    const bool live = row < a.rows;
    const uint32_t start = live ? a.starts[row] : 0u, len = live ? a.starts[row + 1] - start : 0u;
    const bool owner = live && sl < RB;
    const size_t i = (size_t)row * RB + (owner ? sl : 0);
    // what the step reads besides the matrix is fetched before the sums
    V r_old = (V)0, d_old = (V)0, x_old = (V)0, into = (V)0;
    S drow[RB];
    if (owner) {
        r_old = r_in[i];
        d_old = d_in[i];
        x_old = x[i];
        if (sum_into) into = sum_into[i];
#pragma unroll
        for (int q = 0; q < RB; ++q) drow[q] = dinv[(size_t)row * RB * RB + (size_t)sl * RB + q];
    }
    const V sum = rows_sum<RB, RB, RPW, U, S, V>(a, terms, g, sl, start, len, d_in);
    if (owner) r_new[g][sl] = r_old - sum;
    __syncthreads();
    if (owner) {
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(drow[q]) * r_new[g][q];
        const V dn = keep * d_old + step * z;
        const V xn = x_old + dn;
        d_out[i] = dn;
        r_out[i] = r_new[g][sl];
        x[i] = xn;
        if (sum_into) {
            const V total = into + xn;
            sum_into[i] = total;
            if (widen_into) widen_into[i] = (double)total;
        }
    }
}

// Per scalar row, the rounding bound term of CsrMatrix::multiply_rounding_bound
// (crates/solidfem-solve/src/csr.rs:142-154): (terms * eps) * sum |a x|, squared.
template <int RB, int CB>
__global__ __launch_bounds__(256) void rounding_bound_kernel(Sliced<double> a, const double *__restrict__ x,
                                                             double *__restrict__ out) {
    constexpr int NPW = Shape<RB>::NPW;
    const uint32_t slice = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (slice >= a.slices) return;
    const int lane = threadIdx.x % WAVE;
    const int j = lane / RB, p = lane - j * RB;
    if (j >= NPW) return;
    const uint32_t pos = slice * NPW + j;
    const uint32_t row = a.perm[pos];
    if (row == NONE) return;
    const uint32_t len = a.row_len[pos], slot0 = a.slice_start[slice];
    double sum = 0.0;
    for (uint32_t k = 0; k < len; ++k) {
        const uint32_t col = a.cols[(size_t)(slot0 + k) * NPW + j];
        for (int q = 0; q < CB; ++q) sum = sum + fabs(a.vals[((size_t)(slot0 + k) * WAVE + lane) * CB + q] * x[(size_t)col * CB + q]);
    }
    const double bound = (double)(len * CB) * 2.220446049250313e-16 * sum;
    out[(size_t)row * RB + p] = bound * bound;
}

// Scalars of a solve, resident on the device.
struct PcgScalars {
    double rz;         // r . z
    double curvature;  // p . A p
    double rr;         // r . r (recursive residual)
    double rz_next;
    double true_rr;    // ||b - A x||^2
    double bound2;     // sum of squared row rounding bounds
    double alpha;
    double beta;
    int32_t valid;     // the curvature test of pcg.rs:219-227 passed
    uint32_t tag;      // host copies only: which readback the copy answers, written last
};

// Copies the scalars to host memory for the host to read without an event: every field first,
// then, after a system-scope fence, the tag the host waits for.
__device__ __forceinline__ void mirror_scalars(const PcgScalars *s, PcgScalars *mirror, uint32_t tag) {
    mirror->rz = s->rz;
    mirror->curvature = s->curvature;
    mirror->rr = s->rr;
    mirror->rz_next = s->rz_next;
    mirror->true_rr = s->true_rr;
    mirror->bound2 = s->bound2;
    mirror->alpha = s->alpha;
    mirror->beta = s->beta;
    mirror->valid = s->valid;
    __threadfence_system();
    __hip_atomic_store(&mirror->tag, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Deterministic dot products. TREE order is a fixed two-stage reduction: DOT_BLOCKS blocks each
// sum a fixed grid-stride pattern through a fixed shuffle tree into one partial, then one block
// sums the partials in the same fixed pattern (a second kernel: no atomics and no fences; a
// one-launch form whose last block finishes the sum measured slower, its per-block release fences
// costing more than the launch they save).
// REFERENCE order is one thread summing in index order from zero, exactly
// crates/solidfem-solve/src/pcg.rs:285-291.
constexpr int DOT_BLOCKS = 512;
constexpr int DOT_THREADS = 256;

__device__ __forceinline__ double wave_sum(double v) {
    // fixed butterfly: the same pairs add in the same order on every run
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) v = v + __shfl_xor(v, off, WAVE);
    return v;
}

__device__ __forceinline__ double block_sum(double v) {
    __shared__ double wsum[DOT_THREADS / WAVE];
    v = wave_sum(v);
    if ((threadIdx.x % WAVE) == 0) wsum[threadIdx.x / WAVE] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < DOT_THREADS / WAVE; ++w) s = s + wsum[w];
    return s;  // valid in thread 0
}

// The final sum of a TREE dot product left to a kernel that has nothing to do with it: its first
// workgroup (of DOT_THREADS threads) forms the sum as dot_final_kernel does, stores it and copies the
// scalars to the host, while the others do the kernel's own work. Null partials: no sum.
struct FinalSum {
    const double *partials;
    double *out;
    PcgScalars *s;
    PcgScalars *mirror;
    uint32_t tag;
};
// Whether this workgroup formed the sum (and has no other work); `block` is its number among the rest.
__device__ __forceinline__ bool final_sum(const FinalSum &f, uint32_t &block) {
    block = blockIdx.x;
    if (!f.partials) return false;
    if (blockIdx.x > 0) {
        --block;
        return false;
    }
    double v = 0.0;
    for (int i = threadIdx.x; i < DOT_BLOCKS; i += DOT_THREADS) v = v + f.partials[i];
    const double total = block_sum(v);
    if (threadIdx.x == 0) {
        *f.out = total;
        if (f.mirror) mirror_scalars(f.s, f.mirror, f.tag);
    }
    return true;
}

// The Chebyshev start (cycle.rs:591-610): z = D^-1 b, d = z / theta, x = d; with a solve's r . r left to it.
template <int RB, typename S, typename V>
__global__ __launch_bounds__(256) void cheb_start_kernel(uint32_t rows, const S *__restrict__ dinv, const V *__restrict__ b,
                                                         V theta, V *__restrict__ d, V *__restrict__ x, FinalSum sum) {
    uint32_t block;
    if (final_sum(sum, block)) return;
    const size_t i = (size_t)block * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * RB) return;
    const size_t row = i / RB, p = i - row * RB;
    const S *dr = dinv + row * RB * RB + p * RB;
    V z = (V)0;
#pragma unroll
    for (int q = 0; q < RB; ++q) z = z + widen<V>(dr[q]) * b[row * RB + q];
    const V dv = z / theta;
    d[i] = dv;
    x[i] = dv;
}

// One later Chebyshev step, fused (cycle.rs:611-650): ad = A d_in; r_out = r_in - ad;
// z = D^-1 r_out (the RB residuals of a block row shuffled in from its lanes, summed from zero,
// cycle.rs:655-674); d_out = keep d_in + step z; x += d_out. With `sum_into` set, the step is the
// last of a post-smoothing and also adds the smoothed correction to the cycle's x
// (cycle.rs:534-536): sum_into += x.
template <int RB, int BATCH, typename S, typename V>
__global__ __launch_bounds__(256) void cheb_step_kernel(Sliced<S> a, const S *__restrict__ dinv, const V *__restrict__ d_in,
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
    V ad = (V)0;
    if (live) ad = row_product<RB, RB, BATCH, S, V>(a, a.slice_start[slice], a.row_len[pos], j, lane, d_in);
    const size_t i = live ? (size_t)row * RB + p : 0;
    const V r_new = live ? r_in[i] - ad : (V)0;
    // every lane takes part in the shuffle; padding lanes carry zeros and store nothing
    const S *drow = dinv + (live ? (size_t)row * RB * RB + (size_t)p * RB : 0);
    V z = (V)0;
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        const V rq = __shfl(r_new, (in_wave ? j * RB : 0) + q, WAVE);
        if (live) z = z + widen<V>(drow[q]) * rq;
    }
    if (!live) return;
    const V dn = keep * d_in[i] + step * z;
    const V xn = x[i] + dn;
    d_out[i] = dn;
    r_out[i] = r_new;
    x[i] = xn;
    if (sum_into) {
        const V total = sum_into[i] + xn;
        sum_into[i] = total;
        if (widen_into) widen_into[i] = (double)total;  // the cycle's correction, widened out
    }
}

// x = x + y (cycle.rs:541-545), for a post-smoothing of degree one.
template <typename V>
__global__ void add_kernel(size_t n, V *__restrict__ x, const V *__restrict__ y) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + y[i];
}

// The finest level's right-hand side rounded in from f64 (the conversion of cycle.rs:226-243)
// and the Chebyshev start on it (cheb_start_kernel), one thread per block row; with a solve's r . r left
// to it.
template <int RB, typename S, typename V>
__global__ __launch_bounds__(256) void convert_start_kernel(uint32_t rows, const double *__restrict__ r, V *__restrict__ b,
                                                            const S *__restrict__ dinv, V theta, V *__restrict__ d,
                                                            V *__restrict__ x, FinalSum sum) {
    uint32_t block;
    if (final_sum(sum, block)) return;
    const size_t row = (size_t)block * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    V bv[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        bv[q] = (V)r[row * RB + q];
        b[row * RB + q] = bv[q];
    }
#pragma unroll
    for (int p = 0; p < RB; ++p) {
        const S *dr = dinv + row * RB * RB + p * RB;
        V z = (V)0;
#pragma unroll
        for (int q = 0; q < RB; ++q) z = z + widen<V>(dr[q]) * bv[q];
        const V dv = z / theta;
        d[row * RB + p] = dv;
        x[row * RB + p] = dv;
    }
}

template <typename To, typename From>
__global__ void convert_kernel(size_t n, const From *__restrict__ in, To *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (To)in[i];
}

// The coarsest level's direct solve with the f64 Cholesky factor (block.rs:357-373), the
// right-hand side widened from V and the solution rounded to V (cycle.rs:475-486). `packed` is the
// factor by columns (column k holds rows k..n-1 at offset k n - k (k - 1) / 2). Forward substitution
// runs right-looking: once x_k is final every later row subtracts its term, so each row still
// subtracts in ascending k, the reference's order. Back substitution also subtracts each row's terms
// in ascending k, which can only start once every later x is known: the lanes form the negated
// products of all but the latest x while that one is still being computed, and every row of 16 lanes
// folds them in order (add_row_terms), so the row's value needs no exchange before its division.
//
// The first wavefront solves, alone and with no barrier inside a panel; the other three bring the
// next panel of `width` columns into the other LDS buffer meanwhile, so no step waits on global
// memory. A factor that fits one buffer is one panel, read once for both substitutions. Forward, a
// block of 64 rows stays in registers, one per lane, for its own columns, then the later rows take
// those columns' terms. Not bound by its chain: n = 90 takes 67 us, of which its n^2 / 2 dependent
// subtractions (2.5 ns) and 2 n divisions (42 ns) are 17; the rest is what each row of the back
// substitution does around them (products to LDS and back, the division, x to LDS, a fence each). With every
// step through LDS and a lane folding the products it took 104. One V-cycle call that is this solve alone
// (25 us of it copies): n = 108 110 us (156 before), 360 0.60 ms (1.02), 756 2.25 (3.89), 1296 6.3 (12.5).
constexpr uint32_t COARSE_MAX = 3072;
constexpr uint32_t COARSE_THREADS = 256;
constexpr uint32_t COARSE_PANEL = 5600;  // entries of one of the two panel buffers
__host__ __device__ constexpr size_t packed_column(uint32_t n, uint32_t k) { return (size_t)k * n - ((size_t)k * (k - 1)) / 2; }
// Columns per panel and LDS bytes: the whole factor where it fits two buffers' room, else two panels.
__host__ __device__ constexpr uint32_t coarse_panel_width(uint32_t n) {
    return packed_column(n, n) <= 2 * COARSE_PANEL ? n : COARSE_PANEL / n;
}
// Entries of one of the two product buffers: whole groups of add_row_terms.
__host__ __device__ constexpr uint32_t coarse_products(uint32_t n) { return (n + 31) / 32 * 32; }
constexpr size_t coarse_solve_lds(uint32_t n) {
    return ((coarse_panel_width(n) == n ? packed_column(n, n) + packed_column(n, n) % 2 : 2 * COARSE_PANEL) + (size_t)n + n % 2 + 2 * coarse_products(n)) * sizeof(double);
}
// Orders this wavefront's LDS accesses before and after this point (LDS serves a wavefront's
// accesses in order, so only the compiler has to be kept from moving them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// v of `lane`, the same lane for the whole wavefront.
__device__ __forceinline__ double lane_value(double v, uint32_t lane) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    const uint32_t low = __builtin_amdgcn_readlane((uint32_t)bits, lane), high = __builtin_amdgcn_readlane((uint32_t)(bits >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)high << 32 | low);
}
// Several right-hand sides (row-interleaved, `stride` columns) take one workgroup each.
template <typename V>
__global__ __launch_bounds__(COARSE_THREADS) void coarse_solve_kernel(uint32_t n, const double *__restrict__ packed,
                                                                      const V *__restrict__ rhs, V *__restrict__ out, uint32_t stride) {
    extern __shared__ __align__(16) double smem[];
    const uint32_t width = coarse_panel_width(n), panels = (n + width - 1) / width;
    const size_t whole = packed_column(n, n);
    double *xs = smem + (panels == 1 ? whole + whole % 2 : 2 * (size_t)COARSE_PANEL), *prod = xs + n + n % 2;
    const uint32_t t = threadIdx.x, room = coarse_products(n);
    rhs += blockIdx.x;
    out += blockIdx.x;
    // panel p into its buffer, by the threads from `first` on
    auto bring = [&](uint32_t p, uint32_t first) {
        const uint32_t k0 = p * width, k1 = k0 + width < n ? k0 + width : n;
        const size_t at = packed_column(n, k0), entries = packed_column(n, k1) - at;
        double *to = smem + (size_t)(p & 1u) * COARSE_PANEL;
        const uint32_t step = COARSE_THREADS - first;
        for (size_t e = t - first; e < entries; e += 8 * (size_t)step) {
            double v[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) v[u] = e + u * step < entries ? packed[at + e + u * step] : 0.0;
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                if (e + u * step < entries) to[e + u * step] = v[u];
        }
    };
    bring(0, 0);
    for (uint32_t i = t; i < n; i += COARSE_THREADS) xs[i] = (double)rhs[(size_t)i * stride];
    // adding -0.0 changes nothing, and a buffer's products grow by two a step: what lies past them is
    // never anything else
    for (uint32_t i = t; i < 2 * room; i += COARSE_THREADS) prod[i] = -0.0;
    __syncthreads();
    for (uint32_t p = 0; p < panels; ++p) {
        const uint32_t k0 = p * width, k1 = k0 + width < n ? k0 + width : n;
        if (t >= WAVE) {
            if (p + 1 < panels) bring(p + 1, WAVE);
        } else {
            const double *panel = smem + (size_t)(p & 1u) * COARSE_PANEL;
            const double *col = panel;  // col[i - k] = L[i][k]
            for (uint32_t kb = k0; kb < k1; kb += WAVE) {
                const uint32_t ke = k1 - kb < (uint32_t)WAVE ? k1 : kb + WAVE, i = kb + t;
                const double *const block = col;
                double y = i < n ? xs[i] : 0.0;
                double diagonal = col[0], below = i < n ? col[t] : 0.0;
                for (uint32_t k = kb; k < ke; ++k) {
                    // the next column's entries are read before this one's division
                    const double d = diagonal, l = below;
                    col += n - k;
                    if (k + 1 < ke) {
                        diagonal = col[0];
                        below = i > k && i < n ? col[i - k - 1] : 0.0;
                    }
                    const double xv = lane_value(y, k - kb) / d;
                    if (i == k) y = xv;
                    else if (i > k) y = y - l * xv;
                }
                if (i < n) xs[i] = y;
                wave_lds_fence();
                for (uint32_t later = kb + WAVE + t; later < n; later += WAVE) {
                    double v = xs[later];
                    const double *c = block;
#pragma unroll 8
                    for (uint32_t k = kb; k < ke; ++k) {
                        v = v - c[later - k] * xs[k];
                        c += n - k;
                    }
                    xs[later] = v;
                }
                wave_lds_fence();
            }
        }
        __syncthreads();
    }
    double latest = 0.0;  // x of the row below the current one
    for (uint32_t p = panels; p-- > 0;) {
        const uint32_t k0 = p * width, k1 = k0 + width < n ? k0 + width : n;
        if (t >= WAVE) {
            if (p > 0) bring(p - 1, WAVE);
        } else {
            const double *col = smem + (size_t)(p & 1u) * COARSE_PANEL + (packed_column(n, k1) - packed_column(n, k0));
            // row ii's products with every x but the latest: k from ii + 2; c is its column
            auto products = [&](uint32_t ii, const double *c) {
                double *to = prod + (ii & 1u) * room;
                for (uint32_t k = ii + 2 + t; k < n; k += 2 * WAVE) {
                    const bool more = k + WAVE < n;
                    const double l0 = c[k - ii], x0 = xs[k], l1 = more ? c[k + WAVE - ii] : 0.0, x1 = more ? xs[k + WAVE] : 0.0;
                    to[k - ii - 2] = -(l0 * x0);
                    if (more) to[k + WAVE - ii - 2] = -(l1 * x1);
                }
            };
            products(k1 - 1, col - (n - (k1 - 1)));
            double d_next = col[-(int)(n - (k1 - 1))], first_next = k1 < n ? col[1 - (int)(n - (k1 - 1))] : 0.0, y_next = xs[k1 - 1];
            for (uint32_t ii = k1; ii-- > k0;) {
                col -= n - ii;
                const double d = d_next, first = first_next, y = y_next;
                if (ii > k0) {
                    const double *c = col - (n - (ii - 1));
                    products(ii - 1, c);  // with the x of row ii + 1 by now
                    d_next = c[0];
                    first_next = c[1];
                    y_next = xs[ii - 1];
                }
                wave_lds_fence();
                double v = ii + 1 < n ? y + -(first * latest) : y;
                v = add_row_terms(v, (const double *)(prod + (ii & 1u) * room), ii + 2 < n ? n - ii - 2 : 0u);
                latest = v / d;
                wave_lds_fence();
                if (t == 0) xs[ii] = latest;
                wave_lds_fence();
            }
        }
        __syncthreads();
    }
    for (uint32_t i = t; i < n; i += COARSE_THREADS) out[(size_t)i * stride] = (V)xs[i];
}

// The explicit inverse of a coarse factor, L^-T L^-1. First linv = L^-1 by forward substitution
// for all columns at once: row k is finished (divided by L[k][k]), then every later row i takes the
// term L[i][k] linv[k][j] off its entries j <= k. Entry (i, j) thus computes ((i == j) - sum over k
// from j to i - 1 of L[i][k] linv[k][j], subtracted in ascending k) / L[i][i]; `lt` holds L by columns
// (lt[k n + i] = L[i][k]), linv starts as the identity. DENSE_PANEL rows are taken at a time: the
// panel's own rows, one thread a column, then every later row takes the panel's terms in ascending k.
// Then entry (i, j) of the inverse = sum over k from max(i, j) of linv[k][i] linv[k][j], added in
// ascending k from zero, stored at inv[j n + i], by tiles staged through LDS; entries (i, j) and
// (j, i) add the same products, so tiles on one side give both. A step per row took 2 n launches.
constexpr uint32_t DENSE_PANEL = 32;  // columns or rows of a dense coarse level taken at a time
static __global__ __launch_bounds__(64) void factor_inverse_panel_kernel(uint32_t n, uint32_t k0, uint32_t w, const double *__restrict__ lt,
                                                                        double *__restrict__ linv) {
    // d[k][r] = L[k0 + r][k0 + k]; past a last panel's w rows the identity, which leaves its zeros as they
    // are, so that every step's loop is whole
    __shared__ double d[DENSE_PANEL][DENSE_PANEL], v[DENSE_PANEL][64];
    const uint32_t t = threadIdx.x;
    for (uint32_t e = t; e < DENSE_PANEL * DENSE_PANEL; e += 64) {
        const uint32_t k = e / DENSE_PANEL, r = e % DENSE_PANEL;
        d[k][r] = r < k ? 0.0 : r < w ? lt[(size_t)(k0 + k) * n + k0 + r] : r == k ? 1.0 : 0.0;
    }
    __syncthreads();
    const uint32_t j = blockIdx.x * 64 + t;
    if (j >= k0 + w) return;
    // column j of the panel, in LDS: a loop short enough to stay in the instruction cache, where the
    // unrolled one over registers (30 KB of instructions run once) took 70 us a panel. Where the column
    // starts within the panel, the rows above its diagonal are zeros and stay so.
    for (uint32_t r = 0; r < DENSE_PANEL; ++r) v[r][t] = r < w ? linv[(size_t)(k0 + r) * n + j] : 0.0;
#pragma unroll 1
    for (uint32_t k = 0; k < DENSE_PANEL; ++k) {
        const double vk = v[k][t] / d[k][k];
        v[k][t] = vk;
#pragma unroll 4
        for (uint32_t r = k + 1; r < DENSE_PANEL; ++r) v[r][t] = v[r][t] - d[k][r] * vk;
    }
    for (uint32_t r = 0; r < w; ++r) linv[(size_t)(k0 + r) * n + j] = v[r][t];
}
static __global__ __launch_bounds__(256) void factor_inverse_trailing_kernel(uint32_t n, uint32_t k0, uint32_t w, const double *__restrict__ lt,
                                                                            double *__restrict__ linv) {
    __shared__ double l[DENSE_PANEL][DENSE_PANEL], x[DENSE_PANEL][DENSE_PANEL];  // by k
    const uint32_t t = threadIdx.x, i0 = k0 + w + blockIdx.y * DENSE_PANEL, j0 = blockIdx.x * DENSE_PANEL;
    for (uint32_t e = t; e < w * DENSE_PANEL; e += 256) {
        const uint32_t k = e / DENSE_PANEL, c = e % DENSE_PANEL;
        l[k][c] = i0 + c < n ? lt[(size_t)(k0 + k) * n + i0 + c] : 0.0;
        x[k][c] = j0 + c < k0 + w ? linv[(size_t)(k0 + k) * n + j0 + c] : 0.0;
    }
    __syncthreads();
    for (uint32_t e = t; e < DENSE_PANEL * DENSE_PANEL; e += 256) {
        const uint32_t r = e / DENSE_PANEL, c = e % DENSE_PANEL, i = i0 + r, j = j0 + c;
        if (i >= n || j >= k0 + w) continue;
        double v = linv[(size_t)i * n + j];
        for (uint32_t k = j > k0 ? j - k0 : 0; k < w; ++k) v = v - l[k][r] * x[k][c];  // j <= k0 + k
        linv[(size_t)i * n + j] = v;
    }
}
static __global__ __launch_bounds__(256) void factor_inverse_entries_kernel(uint32_t n, const double *__restrict__ linv,
                                                                           double *__restrict__ inv) {
    if (blockIdx.x > blockIdx.y) return;  // j0 <= i0: the other side is its mirror
    __shared__ double a[DENSE_PANEL][DENSE_PANEL], b[DENSE_PANEL][DENSE_PANEL];  // by k
    const uint32_t t = threadIdx.x, i0 = blockIdx.y * DENSE_PANEL, j0 = blockIdx.x * DENSE_PANEL;
    constexpr uint32_t PER = DENSE_PANEL * DENSE_PANEL / 256;
    const uint32_t c = t % DENSE_PANEL, j = j0 + c;
    double v[PER] = {};
    for (uint32_t k0 = i0; k0 < n; k0 += DENSE_PANEL) {
        for (uint32_t e = t; e < DENSE_PANEL * DENSE_PANEL; e += 256) {
            const uint32_t k = e / DENSE_PANEL, r = e % DENSE_PANEL;
            a[k][r] = k0 + k < n && i0 + r < n ? linv[(size_t)(k0 + k) * n + i0 + r] : 0.0;
            b[k][r] = k0 + k < n && j0 + r < n ? linv[(size_t)(k0 + k) * n + j0 + r] : 0.0;
        }
        __syncthreads();
        const uint32_t w = n - k0 < DENSE_PANEL ? n - k0 : DENSE_PANEL;
#pragma unroll
        for (uint32_t u = 0; u < PER; ++u) {
            const uint32_t r = t / DENSE_PANEL + u * (256 / DENSE_PANEL), first = i0 + r > j ? i0 + r : j;
            for (uint32_t k = first > k0 ? first - k0 : 0; k < w; ++k) v[u] = v[u] + a[k][r] * b[k][c];
        }
        __syncthreads();
    }
#pragma unroll
    for (uint32_t u = 0; u < PER; ++u) {
        const uint32_t i = i0 + t / DENSE_PANEL + u * (256 / DENSE_PANEL);
        if (i < n && j < n) {
            inv[(size_t)j * n + i] = v[u];
            inv[(size_t)i * n + j] = v[u];
        }
    }
}

// The coarsest level's solve as a product with the f64 inverse, the right-hand side widened from V:
// out = inv b, COARSE_ROWS rows per workgroup. inv is symmetric bit for bit (entry (i, j) and entry (j, i) add
// the same products in the same order), so a row's entries are read as its column's, contiguous. All
// threads form a chunk of the rows' terms into LDS with every load in flight at once; then row r of 16
// lanes of the first wavefront adds row r's terms in ascending k from zero. Bound by that chain of n
// additions; n = 438 took 17.5 us with one lane per row walking its column.
constexpr uint32_t COARSE_ROWS = 4, COARSE_CHUNK = 1024;
template <typename V>
__global__ __launch_bounds__(256) void coarse_inverse_kernel(uint32_t n, const double *__restrict__ inv, const V *__restrict__ rhs,
                                                             V *__restrict__ out) {
    __shared__ __align__(16) double terms[COARSE_ROWS][COARSE_CHUNK + 2];
    const uint32_t t = threadIdx.x, i0 = blockIdx.x * COARSE_ROWS;
    const uint32_t rows = n - i0 < COARSE_ROWS ? n - i0 : COARSE_ROWS;
    double sum = 0.0;
    for (uint32_t k0 = 0; k0 < n; k0 += COARSE_CHUNK) {
        constexpr uint32_t PER = COARSE_CHUNK / 256;
        double a[COARSE_ROWS][PER], bk[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            const uint32_t k = k0 + t + 256 * j;
            bk[j] = k < n ? (double)rhs[k] : 0.0;
#pragma unroll
            for (uint32_t r = 0; r < COARSE_ROWS; ++r) a[r][j] = k < n && r < rows ? inv[(size_t)(i0 + r) * n + k] : 0.0;
        }
        if (k0) __syncthreads();  // the chunk before has been added
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j)
#pragma unroll
            for (uint32_t r = 0; r < COARSE_ROWS; ++r) terms[r][t + 256 * j] = a[r][j] * bk[j];
        __syncthreads();
        if (t < WAVE) sum = add_row_terms(sum, (const double *)terms[t / 16], n - k0 < COARSE_CHUNK ? n - k0 : COARSE_CHUNK);
    }
    if (t < WAVE && t % 16 == 0 && t / 16 < rows) out[i0 + t / 16] = (V)sum;
}

// ---- conjugate gradient vectors -------------------------------------------------------------

// MODE 0: a . b; MODE 1: sum of a.
template <int MODE>
__global__ __launch_bounds__(DOT_THREADS) void dot_partials_kernel(size_t n, const double *__restrict__ a,
                                                                    const double *__restrict__ b, double *__restrict__ partials) {
    double v = 0.0;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) v = v + (MODE == 0 ? a[i] * b[i] : a[i]);
    const double s = block_sum(v);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// What the final sum feeds: STORE writes it to `out`; RZ makes it the next r.z and forms
// beta = rz_next / rz, rz = rz_next (pcg.rs:258-260).
enum DotFinal { FINAL_STORE = 0, FINAL_RZ = 1 };

__device__ __forceinline__ void dot_finish(int kind, double total, double *out, PcgScalars *s) {
    if (kind == FINAL_STORE) {
        *out = total;
    } else {
        s->rz_next = total;
        s->beta = total / s->rz;
        s->rz = total;
    }
}

// `mirror`, when given, is host memory that receives a copy of the scalars once the sum is stored,
// tagged `tag`: the host waits for the tag instead of an event or a separate copy.
static __global__ __launch_bounds__(DOT_THREADS) void dot_final_kernel(int parts, const double *__restrict__ partials, int kind,
                                                                 double *out, PcgScalars *s, PcgScalars *mirror, uint32_t tag) {
    double v = 0.0;
    for (int i = threadIdx.x; i < parts; i += blockDim.x) v = v + partials[i];
    const double total = block_sum(v);
    if (threadIdx.x == 0) {
        dot_finish(kind, total, out, s);
        if (mirror) mirror_scalars(s, mirror, tag);
    }
}

template <int MODE>
__global__ void dot_serial_kernel(size_t n, const double *__restrict__ a, const double *__restrict__ b, int kind,
                                  double *out, PcgScalars *s, PcgScalars *mirror, uint32_t tag) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double sum = 0.0;
    for (size_t i = 0; i < n; ++i) sum = sum + (MODE == 0 ? a[i] * b[i] : a[i]);
    dot_finish(kind, sum, out, s);
    if (mirror) mirror_scalars(s, mirror, tag);
}

// The update of pcg.rs:219-230: the curvature test, then x += alpha p and r += (-alpha) A p.
static __global__ void pcg_update_kernel(size_t n, PcgScalars *__restrict__ s, const double *__restrict__ p,
                                  const double *__restrict__ ap, double *__restrict__ x, double *__restrict__ r) {
    const double curvature = s->curvature, rz = s->rz;
    const bool valid = !(isnan(curvature) || curvature <= 0.0 || !isfinite(rz));
    const double alpha = rz / curvature;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        s->valid = valid ? 1 : 0;
        s->alpha = alpha;
    }
    if (!valid || i >= n) return;
    x[i] = x[i] + alpha * p[i];
    r[i] = r[i] + (-alpha) * ap[i];
}

// The total of a TREE dot product formed by every block of a consumer kernel of DOT_THREADS
// threads, exactly as dot_final_kernel forms it (the same partials summed in the same order):
// the consumer needs no separate final launch and the bits do not change.
__device__ __forceinline__ double tree_total(const double *__restrict__ partials) {
    double v = 0.0;
    for (int i = threadIdx.x; i < DOT_BLOCKS; i += blockDim.x) v = v + partials[i];
    const double total = block_sum(v);
    __shared__ double shared_total;
    if (threadIdx.x == 0) shared_total = total;
    __syncthreads();
    return shared_total;
}

// The slot of PcgScalars that holds the current r.z in the fused TREE iteration: the direction
// kernel reads it in every block while block 0 stores the next one, so the two alternate.
__device__ __forceinline__ double &rz_in(PcgScalars *s, uint32_t slot) { return slot ? s->rz_next : s->rz; }

// pcg.rs:216-230 with both reductions around it fused, for TREE order, on DOT_BLOCKS blocks of
// DOT_THREADS: p . A p summed from its partials as dot_final_kernel does, the curvature test,
// x += alpha p and r += (-alpha) A p, and the partials of the new r . r over the same grid-stride
// rows as dot_partials_kernel -- the same bits as the separate launches.
static __global__ __launch_bounds__(DOT_THREADS) void pcg_update_fused_kernel(size_t n, PcgScalars *__restrict__ s, uint32_t slot,
                                                                              const double *__restrict__ pap_partials,
                                                                              const double *__restrict__ p,
                                                                              const double *__restrict__ ap, double *__restrict__ x,
                                                                              double *__restrict__ r, double *__restrict__ rr_partials) {
    const double curvature = tree_total(pap_partials);
    const double rz = rz_in(s, slot);
    const bool valid = !(isnan(curvature) || curvature <= 0.0 || !isfinite(rz));
    const double alpha = rz / curvature;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->curvature = curvature;
        s->valid = valid ? 1 : 0;
        s->alpha = alpha;
    }
    double v = 0.0;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        double ri = r[i];
        if (valid) {
            x[i] = x[i] + alpha * p[i];
            ri = ri + (-alpha) * ap[i];
            r[i] = ri;
        }
        v = v + ri * ri;
    }
    __syncthreads();  // block_sum's shared words were read by tree_total
    const double part = block_sum(v);
    if (threadIdx.x == 0) rr_partials[blockIdx.x] = part;
}

// pcg.rs:256-263 fused for TREE order, on DOT_BLOCKS blocks of DOT_THREADS: r . z summed from its
// partials as dot_final_kernel does, beta = rz_next / rz, then p = z + beta p. Block 0 stores the
// next r . z in the other slot.
static __global__ __launch_bounds__(DOT_THREADS) void pcg_direction_fused_kernel(size_t n, PcgScalars *__restrict__ s,
                                                                                 uint32_t slot,
                                                                                 const double *__restrict__ rz_partials,
                                                                                 const double *__restrict__ z,
                                                                                 double *__restrict__ p) {
    const double total = tree_total(rz_partials);
    const double beta = total / rz_in(s, slot);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        rz_in(s, slot ^ 1u) = total;
        s->beta = beta;
    }
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = z[i] + beta * p[i];
}

// p = z + beta p (pcg.rs:261-263), beta formed by the r.z reduction.
static __global__ void pcg_direction_kernel(size_t n, const PcgScalars *__restrict__ s, const double *__restrict__ z,
                                            double *__restrict__ p) {
    const double beta = s->beta;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = z[i] + beta * p[i];
}

// Jacobi: z = r * inverse diagonal (preconditioner.rs:237-247).
static __global__ void jacobi_kernel(size_t n, const double *__restrict__ inv, const double *__restrict__ r, double *__restrict__ z) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z[i] = r[i] * inv[i];
}

// A sliced matrix's block columns row after row (Bsr's order), from the slots they lie in: one thread a row.
template <int NPW>
__global__ void plain_columns_kernel(size_t positions, const uint32_t *__restrict__ slice_start, const uint32_t *__restrict__ row_len,
                                     const uint32_t *__restrict__ perm, const uint32_t *__restrict__ cols, const uint32_t *__restrict__ starts,
                                     uint32_t *__restrict__ out) {
    const size_t pos = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= positions) return;
    const uint32_t row = perm[pos];
    if (row == NONE) return;
    const uint32_t slice = (uint32_t)(pos / NPW), j = (uint32_t)(pos % NPW), to = starts[row], len = row_len[pos];
    for (uint32_t k = 0; k < len; ++k) out[to + k] = cols[((size_t)slice_start[slice] + k) * NPW + j];
}

// Sliced values from a row-major block array: slot i of the sliced layout takes value
// src[map[i]] rounded to T (the precision conversion of block.rs:26-35).
template <typename T>
__global__ void gather_convert_kernel(size_t n, const uint32_t *__restrict__ block_of_slot, int rb, int cb,
                                      const double *__restrict__ src, T *__restrict__ dst) {
    // dst index = ((slot * 64 + lane) * cb + q), lane = j * rb + p ; map gives the source block
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t q = i % cb;
    const size_t lane = (i / cb) % WAVE;
    const size_t slot_row = i / ((size_t)WAVE * cb);  // the slot
    const int npw = WAVE / rb;
    const int j = (int)(lane / rb), p = (int)(lane % rb);
    if (j >= npw) {
        dst[i] = (T)0;
        return;
    }
    const uint32_t blk = block_of_slot[slot_row * npw + j];
    dst[i] = blk == NONE ? (T)0 : (T)src[(size_t)blk * rb * cb + (size_t)p * cb + q];
}

// A plain copy, 16 bytes per lane per step, grid-stride.
static __global__ void stream_copy_kernel(size_t n16, const uint4 *__restrict__ src, uint4 *__restrict__ dst) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

// A plain read, 16 bytes per lane per step, grid-stride; one word per lane is written so the
// loads stay.
static __global__ void stream_read_kernel(size_t n16, const uint4 *__restrict__ src, uint32_t *__restrict__ sink) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0;
    for (size_t i = t; i < n16; i += stride) {
        const uint4 v = src[i];
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    sink[t] = acc;
}

}  // namespace dev
}  // namespace sf
