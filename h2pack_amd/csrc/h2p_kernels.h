// Global kernels of the MI355X H2 engine (matvec path).
//
// Vector spaces on the device:
//   xin   = [ px (N, permuted input) | y0 (S, skeleton coefficients) ]
//   y1    = S skeleton accumulators (downward sweep)
//   arena = partial outputs of the grouped B/D block launch
// Skeleton offsets are assigned so that the children of every node occupy a
// contiguous range in child order; the stacked operand of a non-leaf U is
// therefore one contiguous slice of y0 / y1.
#pragma once
#include <type_traits>

#include "h2p_device.h"

namespace h2p {

// One B or D block of the grouped launch.
struct BlkTask {
    long long data_off;   // AOT: element offset of the row-major block
    long long out0, out1; // arena offsets of the two partial outputs (out1 < 0: none)
    int nrow, ncol;       // block dimensions in vector entries (points * kd)
    int c0, c1;           // JIT: first point of each set in the unified coordinates
    int n0, n1;           // JIT: point counts
    int in0, in1;         // xin offsets of the operands (in0: ncol long, in1: nrow long)
    int flags;            // bit 0: has out1; bits 1, 2: H2P_BLK_FAR, H2P_BLK_FAST
    int shift;            // index into the shift table, added to set 1's coordinates
                          // (periodic images; entry 0 is the zero shift)
};

// The two point sets' bounding boxes are apart: no coincident pair, and for
// RPY no pair within the sum of two radii.
#define H2P_BLK_FAR 2
// Gaussian, Matern: no kernel value of the block is below 2^-1000.
#define H2P_BLK_FAST 4

// Upward-sweep task: y0[out] = U^T in, U row-major nrow x r.
// Workgroups that a launch has to reach with a chunk width, else it takes the
// next narrower one (see group_sum): {256, 64} outputs, then 16.
#define H2P_FWD_MIN_WG 256    // upward sweep (256, 128 and 64 columns, then 16)
#define H2P_RED_MIN_WG {1024, 256}
#define H2P_BWD_MIN_WG {512, 256}
#define H2P_LEAF_MIN_WG {1024, 256}
#define H2P_LEAF_OWN_MIN_WG {256, 256}   // every chunk sums the leaf's partials again
struct FwdTask {
    long long u_off;
    int nrow, r, in_off, out_off;
    int col0;         // first of the output columns this task computes
    int ncol;         // at most this many columns from col0: 16, 64, 128 or 256
};

// Segmented reduction into y1: y1[dst + e] = sum_k arena[contrib[k] + e] for
// the w elements from e0 (e < len).
struct RedTask {
    int dst, len, cbeg, cend;
    int e0, w;        // w: 256, 64 or 16
};

// ---------------------------------------------------------------------------
__global__ void k_gather(const double *__restrict__ x, const int *__restrict__ idx,
                         double *__restrict__ out, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = x[idx[i]];
}

// v + arena[contrib[k] + e] for k = kb, kb + step, ... < ke, added in list
// order.  The offsets and values of H2P_GATHER_AHEAD entries are loaded
// before their adds, so that many loads are in flight instead of one
// offset-then-value chain per entry; the last batch repeats the last entry
// and adds zeros for it.
#define H2P_GATHER_AHEAD 8
__device__ __forceinline__ double ordered_gather_sum(double v, const long long *__restrict__ contrib,
                                                     const double *__restrict__ arena, int kb, int ke, int step,
                                                     int e) {
    int k = kb;
    for (; k + (H2P_GATHER_AHEAD - 1) * step < ke; k += H2P_GATHER_AHEAD * step) {
        double a[H2P_GATHER_AHEAD];
#pragma unroll
        for (int u = 0; u < H2P_GATHER_AHEAD; u++) a[u] = arena[contrib[k + u * step] + e];
#pragma unroll
        for (int u = 0; u < H2P_GATHER_AHEAD; u++) v += a[u];
    }
    if (k < ke) {
        double a[H2P_GATHER_AHEAD];
#pragma unroll
        for (int u = 0; u < H2P_GATHER_AHEAD; u++) {
            const int ku = k + u * step;
            const double x = arena[contrib[ku < ke ? ku : k] + e];
            a[u] = ku < ke ? x : 0.0;
        }
#pragma unroll
        for (int u = 0; u < H2P_GATHER_AHEAD; u++) v += a[u];
    }
    return v;
}

// The sweeps and sums below give every workgroup of 256 threads a chunk of W
// consecutive outputs and deal the terms of each output's sum to 256 / W
// groups of threads, whose sums are added in group order.  W = 256 (one
// thread per output) is the least overhead where a launch has enough
// workgroups; a level of a few nodes with long sums takes W = 64 or 16 so
// that all CUs have loads in flight and the chain of dependent batches is
// short (the host picks W per launch; 16 doubles are one 128-byte line).
// The sweeps are bound by HBM where a level has hundreds of nodes and by
// the chain of one workgroup's loads where it has a few.  us per matvec, 256
// rows a workgroup everywhere -> widths by launch: periodic RPY N = 10k 807
// -> 591, RPY N = 20k 472 -> 431, 10 CG iterations on three Matern matrices
// of 24k points and fewer 5927 -> 5640.  Widths 256 / 64 / 16 of the downward
// sweep of RPY N = 20k (64 nodes x 938 rows): 462 / 442 / 460; of the leaf
// outputs of the periodic matrix (64 leaves x 469 rows) 64 / 16: 597 / 605.
//
// The group sums of one output, added in group order; valid in threads < W.
template <int W>
__device__ __forceinline__ double group_sum(double v, double *part) {
    if constexpr (W == 256) return v;
    __syncthreads();   // part may still be read by an earlier call
    part[threadIdx.x] = v;
    __syncthreads();
    double s = part[threadIdx.x & (W - 1)];
#pragma unroll
    for (int g = 1; g < 256 / W; g++) s += part[g * W + (threadIdx.x & (W - 1))];
    return s;
}

// group of a thread; wave-uniform (and said so) from W = 64 on
template <int W>
__device__ __forceinline__ int group_of() {
    return W >= H2P_WAVE ? __builtin_amdgcn_readfirstlane(threadIdx.x / W) : threadIdx.x / W;
}

// sum_i M[i * ld] v[i] over i < n for this thread's column (M points at it):
// each group takes a contiguous range of i, 16 values loaded before their
// FMAs; the last batch repeats the last entry with factors of zero.  ok:
// the thread has a column (a wave without one skips the loads).
template <int W>
__device__ __forceinline__ double group_dot(const double *__restrict__ M, int ld, int n, const double *v, bool ok,
                                            double *part) {
    constexpr int G = 256 / W;
    const int q = (n + G - 1) / G, i0 = group_of<W>() * q, i1 = min(n, i0 + q);
    double a0 = 0.0, a1 = 0.0;
    if (ok) {
        int i = i0;
        for (; i + 15 < i1; i += 16) {
            double u[16];
#pragma unroll
            for (int j = 0; j < 16; j++) u[j] = M[(long long)(i + j) * ld];
#pragma unroll
            for (int j = 0; j < 16; j += 2) {
                a0 += u[j] * v[i + j];
                a1 += u[j + 1] * v[i + j + 1];
            }
        }
        for (; i < i1; i += 8) {
            double u[8];
#pragma unroll
            for (int j = 0; j < 8; j++) u[j] = M[(long long)min(i + j, i1 - 1) * ld];
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const bool k0 = i + j < i1, k1 = i + j + 1 < i1;
                a0 += (k0 ? u[j] : 0.0) * (k0 ? v[i + j] : 0.0);
                a1 += (k1 ? u[j + 1] : 0.0) * (k1 ? v[i + j + 1] : 0.0);
            }
        }
    }
    return group_sum<W>(a0 + a1, part);
}

// The contributions [kb, ke) of element e, dealt to the groups in turn.
template <int W>
__device__ __forceinline__ double group_gather(const long long *__restrict__ contrib, const double *__restrict__ arena,
                                               int kb, int ke, int e, bool ok, double *part) {
    double v = 0.0;
    if (ok) v = ordered_gather_sum(0.0, contrib, arena, kb + group_of<W>(), ke, 256 / W, e);
    return group_sum<W>(v, part);
}

#define H2P_BY_WIDTH(w, F, ...)        \
    do {                               \
        if ((w) == 256) F<256>(__VA_ARGS__); \
        else if ((w) == 64) F<64>(__VA_ARGS__); \
        else F<16>(__VA_ARGS__);       \
    } while (0)

// Fixed-order segmented reduction of the block partials into y1.
template <int W>
__device__ __forceinline__ void reduce_y1_w(const RedTask &t, const long long *__restrict__ contrib,
                                            const double *__restrict__ arena, double *__restrict__ y1, double *part) {
    const int e = t.e0 + (threadIdx.x & (W - 1));
    const double v = group_gather<W>(contrib, arena, t.cbeg, t.cend, e, e < t.len, part);
    if (threadIdx.x < W && e < t.len) y1[t.dst + e] = v;
}

__device__ __forceinline__ void reduce_y1_body(const RedTask &t, const long long *__restrict__ contrib,
                                               const double *__restrict__ arena, double *__restrict__ y1) {
    __shared__ double part[256];
    H2P_BY_WIDTH(t.w, reduce_y1_w, t, contrib, arena, y1, part);
}

__global__ void __launch_bounds__(256) k_reduce_y1(const RedTask *__restrict__ tasks,
                                                   const long long *__restrict__ contrib,
                                                   const double *__restrict__ arena,
                                                   double *__restrict__ y1) {
    reduce_y1_body(tasks[blockIdx.x], contrib, arena, y1);
}

// ---------------------------------------------------------------------------
// Sweep kernels.
//
// Upward sweep (src/H2Pack_matvec.c:95-177): one workgroup per node and
// column chunk of its U (256 columns, or 128 / 64 / 16 on a level with fewer
// workgroups than CUs, so a node with a large basis spreads over several
// workgroups).  Chunks of 64 columns and more: lanes own the columns (NS
// strips of 64, only the strips that hold columns), the four waves take
// contiguous quarters of the rows and load UR = 32 / NS rows x NS strips
// before their FMAs (32 loads in flight per wave whatever the chunk width, 24
// at NS = 3; then 8-row batches, then single rows; rows in order), and the
// four wave partials are added in LDS in a fixed order: a column's sum has
// the same bits at each of these widths.  Chunks of 16 columns deal the rows to
// 16 groups of threads instead (group_dot), another order of the same sum;
// the width is fixed at upload, so a handle's results do not change.
// R rows x NS strips loaded, then their FMAs in row order.
template <int R, int NS>
__device__ __forceinline__ void fwd2_rows(const double *__restrict__ Ut, int ld, const double *__restrict__ in, int i,
                                          const int *cc, double *acc) {
    double u[R][NS];
#pragma unroll
    for (int a = 0; a < R; a++)
#pragma unroll
        for (int k = 0; k < NS; k++) u[a][k] = Ut[(long long)(i + a) * ld + cc[k]];
#pragma unroll
    for (int a = 0; a < R; a++) {
        const double v = in[i + a];
#pragma unroll
        for (int k = 0; k < NS; k++) acc[k] += u[a][k] * v;
    }
}

template <int NS>
__device__ __forceinline__ void fwd2_strips(const FwdTask &t, const double *__restrict__ U,
                                            double *__restrict__ xin, double (*red)[4][H2P_WAVE]) {
    constexpr int UR = NS == 3 ? 8 : 32 / NS;
    // the wave index is the same on every lane: said so, the row addresses
    // stay scalar and each load needs only its column offset per lane
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double *Ut = U + t.u_off;
    const double *in = xin + t.in_off;
    const int q = (t.nrow + 3) >> 2;
    const int i0 = w * q, i1 = min(t.nrow, i0 + q);
    const int cs = t.col0;
    double acc[NS];
    int cc[NS];
    bool ok[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        acc[k] = 0.0;
        cc[k] = cs + k * H2P_WAVE + lane;
        ok[k] = cc[k] < t.r;
        cc[k] = ok[k] ? cc[k] : 0;
    }
    int i = i0;
    for (; i + UR - 1 < i1; i += UR) fwd2_rows<UR, NS>(Ut, t.r, in, i, cc, acc);
    if (UR > 8)
        for (; i + 7 < i1; i += 8) fwd2_rows<8, NS>(Ut, t.r, in, i, cc, acc);
    for (; i < i1; i++) {
        const double v = in[i];
#pragma unroll
        for (int k = 0; k < NS; k++) acc[k] += Ut[(long long)i * t.r + cc[k]] * v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NS; k++) red[k][w][lane] = acc[k];
    __syncthreads();
    if (w == 0) {
#pragma unroll
        for (int k = 0; k < NS; k++)
            if (ok[k])
                xin[t.out_off + cc[k]] = (red[k][0][lane] + red[k][1][lane]) + (red[k][2][lane] + red[k][3][lane]);
    }
}

__device__ __forceinline__ void fwd2_body(const FwdTask &t, const double *__restrict__ U,
                                          double *__restrict__ xin) {
    __shared__ double red[4][4][H2P_WAVE];
    if (t.ncol == 16) {   // 16 columns x 16 groups of rows
        const int c = t.col0 + (threadIdx.x & 15);
        const double v = group_dot<16>(U + t.u_off + c, t.r, t.nrow, xin + t.in_off, c < t.r, &red[0][0][0]);
        if (threadIdx.x < 16 && c < t.r) xin[t.out_off + c] = v;
        return;
    }
    const int ns = (min(t.r - t.col0, t.ncol) + H2P_WAVE - 1) / H2P_WAVE;
    if (ns <= 1) fwd2_strips<1>(t, U, xin, red);
    else if (ns == 2) fwd2_strips<2>(t, U, xin, red);
    else if (ns == 3) fwd2_strips<3>(t, U, xin, red);
    else fwd2_strips<4>(t, U, xin, red);
}

__global__ void __launch_bounds__(256) k_fwd2(const FwdTask *__restrict__ tasks,
                                              const double *__restrict__ U,
                                              double *__restrict__ xin) {
    fwd2_body(tasks[blockIdx.x], U, xin);
}

// Downward sweep (src/H2Pack_matvec.c:767-861), one workgroup per w-row chunk of a node:
// yp[child rows] = U (y1 + yp)[node], U^T stored row-major, so that the lanes'
// rows are contiguous for each column.  The push-down buffer yp is written
// exactly once per row (each child has one parent).
struct BwdTask2 {
    long long ut_off;
    int nrow, r, y1_off, push, out_off, row0;
    int w, pad;       // w: 256, 64 or 16
};
#define H2P_MAXR 2048

template <int W>
__device__ __forceinline__ void bwd2_w(const BwdTask2 &t, const double *__restrict__ UT, const double *yv,
                                       double *__restrict__ yp, double *part) {
    const int row = t.row0 + (threadIdx.x & (W - 1));
    const double v = group_dot<W>(UT + t.ut_off + row, t.nrow, t.r, yv, row < t.nrow, part);
    if (threadIdx.x < W && row < t.nrow) yp[t.out_off + row] = v;
}

__device__ __forceinline__ void bwd2_body(const BwdTask2 &t, const double *__restrict__ UT,
                                          const double *__restrict__ y1, double *__restrict__ yp) {
    __shared__ double yv[H2P_MAXR], part[256];
    for (int c = threadIdx.x; c < t.r; c += blockDim.x)
        yv[c] = y1[t.y1_off + c] + (t.push ? yp[t.y1_off + c] : 0.0);
    __syncthreads();
    H2P_BY_WIDTH(t.w, bwd2_w, t, UT, yv, yp, part);
}

__global__ void __launch_bounds__(256, 8) k_bwd2(const BwdTask2 *__restrict__ tasks,
                                              const double *__restrict__ UT,
                                              const double *__restrict__ y1,
                                              double *__restrict__ yp) {
    bwd2_body(tasks[blockIdx.x], UT, y1, yp);
}

// Leaf outputs (src/H2Pack_matvec.c:767-861 for the leaves, and the backward
// permutation y[fwd[i]] = py[i] of src/H2Pack_matvec.c:1156-1159), one
// workgroup per w-row chunk of a leaf: the leaf's skeleton value is its
// block partials plus its parent's push-down; then U y1 plus the point
// partials go straight to the caller's order.  The skeleton partials were
// summed into y1 with the inner nodes' (own = 0), or, in a tree whose leaves
// are all there is to sum, are summed here (own = 1), which saves a launch.
struct LeafTask2 {
    long long ut_off;
    int nrow, r, s_off, push, vec_s;
    int cb1, ce1;   // contributions in skeleton space (length r; own = 1)
    int cb0, ce0;   // contributions in point space (length nrow)
    int own, row0;
    int w;          // 256, 64 or 16
};
// A leaf's output row i is
//   (U y1)_i + (its point-space contributions) + shift x_i;
// shift != 0 adds shift * x (a diagonal nugget applied outside the H2
// product, as the PCG wrapper of examples/SPDHSS-H2/pcg_tests.c:15-21 does);
// px holds x in the permuted order.
// own = 1 with a small rank (r <= blockDim / 2): the contributions are dealt
// to G = blockDim / r groups of r threads (group g sums contributions g,
// g + G, ...), and the G group sums are added in group order; part holds
// blockDim doubles.  The caller synchronises before reading yv.
__device__ __forceinline__ void leaf_stage_y1(const LeafTask2 &t, const long long *__restrict__ contrib,
                                              const double *__restrict__ arena, const double *__restrict__ y1,
                                              const double *__restrict__ yp, double *yv, double *part) {
    if (!t.own) {
        for (int c = threadIdx.x; c < t.r; c += blockDim.x)
            yv[c] = y1[t.s_off + c] + (t.push ? yp[t.s_off + c] : 0.0);
        return;
    }
    const int G = t.r > 0 ? min(8, (int)blockDim.x / t.r) : 1;
    if (G <= 1) {
        for (int c = threadIdx.x; c < t.r; c += blockDim.x)
            yv[c] = ordered_gather_sum(t.push ? yp[t.s_off + c] : 0.0, contrib, arena, t.cb1, t.ce1, 1, c);
        return;
    }
    const int g = threadIdx.x / t.r, c = threadIdx.x - g * t.r;
    if (g < G) part[g * t.r + c] = ordered_gather_sum(0.0, contrib, arena, t.cb1 + g, t.ce1, G, c);
    __syncthreads();
    for (int c2 = threadIdx.x; c2 < t.r; c2 += blockDim.x) {
        double v = t.push ? yp[t.s_off + c2] : 0.0;
        for (int g2 = 0; g2 < G; g2++) v += part[g2 * t.r + c2];
        yv[c2] = v;
    }
}

template <int W>
__device__ __forceinline__ double leaf_u_row(const LeafTask2 &t, const double *__restrict__ UT, const double *yv,
                                             double *part) {
    const int row = t.row0 + (threadIdx.x & (W - 1));
    return group_dot<W>(UT + t.ut_off + row, t.nrow, t.r, yv, row < t.nrow, part);
}

// the output row of thread < W from its U part u
template <int W>
__device__ __forceinline__ void leaf_out_row(const LeafTask2 &t, const long long *__restrict__ contrib,
                                             const double *__restrict__ arena, const double *__restrict__ px,
                                             double shift, const int *__restrict__ fwd, double *__restrict__ y,
                                             double u, double *part) {
    const int row = t.row0 + (threadIdx.x & (W - 1));
    const double d = group_gather<W>(contrib, arena, t.cb0, t.ce0, row, row < t.nrow, part);
    if (threadIdx.x < W && row < t.nrow) {
        double v = u + d;
        if (shift != 0.0) v += shift * px[t.vec_s + row];
        y[fwd[t.vec_s + row]] = v;
    }
}

template <int W>
__device__ __forceinline__ void leaf_final2_w(const LeafTask2 &t, const long long *__restrict__ contrib,
                                              const double *__restrict__ arena, const double *__restrict__ UT,
                                              const double *yv, const int *__restrict__ fwd, double *__restrict__ y,
                                              const double *__restrict__ px, double shift, double *part) {
    const double u = leaf_u_row<W>(t, UT, yv, part);
    leaf_out_row<W>(t, contrib, arena, px, shift, fwd, y, u, part);
}

__device__ __forceinline__ void leaf_final2_body(const LeafTask2 &t, const long long *__restrict__ contrib,
                                                 const double *__restrict__ arena,
                                                 const double *__restrict__ UT,
                                                 const double *__restrict__ y1,
                                                 const double *__restrict__ yp,
                                                 const int *__restrict__ fwd, double *__restrict__ y,
                                                 const double *__restrict__ px, double shift) {
    __shared__ double yv[H2P_MAXR], part[256];
    leaf_stage_y1(t, contrib, arena, y1, yp, yv, part);
    __syncthreads();
    H2P_BY_WIDTH(t.w, leaf_final2_w, t, contrib, arena, UT, yv, fwd, y, px, shift, part);
}

__global__ void __launch_bounds__(256, 8) k_leaf_final2(const LeafTask2 *__restrict__ tasks,
                                                     const long long *__restrict__ contrib,
                                                     const double *__restrict__ arena,
                                                     const double *__restrict__ UT,
                                                     const double *__restrict__ y1,
                                                     const double *__restrict__ yp,
                                                     const int *__restrict__ fwd,
                                                     double *__restrict__ y,
                                                     const double *__restrict__ px, double shift) {
    leaf_final2_body(tasks[blockIdx.x], contrib, arena, UT, y1, yp, fwd, y, px, shift);
}

// The leaf outputs in two launches, for handles whose D blocks are still
// running during the downward sweep: k_leaf_u writes (U y1)_i to yt (in
// the permuted order, no D contribution needed), k_leaf_d adds the
// point-space contributions once the D blocks are done.  Same operations in
// the same order as k_leaf_final2, so the same bits.
template <int W>
__device__ __forceinline__ void leaf_u_w(const LeafTask2 &t, const double *__restrict__ UT, const double *yv,
                                         double *__restrict__ yt, double *part) {
    const double u = leaf_u_row<W>(t, UT, yv, part);
    const int row = t.row0 + (threadIdx.x & (W - 1));
    if (threadIdx.x < W && row < t.nrow) yt[t.vec_s + row] = u;
}

__global__ void __launch_bounds__(256, 8) k_leaf_u(const LeafTask2 *__restrict__ tasks,
                                                const long long *__restrict__ contrib,
                                                const double *__restrict__ arena,
                                                const double *__restrict__ UT,
                                                const double *__restrict__ y1,
                                                const double *__restrict__ yp, double *__restrict__ yt) {
    __shared__ double yv[H2P_MAXR], part[256];
    const LeafTask2 t = tasks[blockIdx.x];
    leaf_stage_y1(t, contrib, arena, y1, yp, yv, part);
    __syncthreads();
    H2P_BY_WIDTH(t.w, leaf_u_w, t, UT, yv, yt, part);
}

template <int W>
__device__ __forceinline__ void leaf_d_w(const LeafTask2 &t, const long long *__restrict__ contrib,
                                         const double *__restrict__ arena, const double *__restrict__ px,
                                         double shift, const int *__restrict__ fwd, double *__restrict__ y,
                                         const double *__restrict__ yt, double *part) {
    const int row = min(t.row0 + (int)(threadIdx.x & (W - 1)), t.nrow - 1);
    leaf_out_row<W>(t, contrib, arena, px, shift, fwd, y, yt[t.vec_s + row], part);
}

__global__ void __launch_bounds__(256) k_leaf_d(const LeafTask2 *__restrict__ tasks,
                                                const long long *__restrict__ contrib,
                                                const double *__restrict__ arena,
                                                const double *__restrict__ yt,
                                                const int *__restrict__ fwd, double *__restrict__ y,
                                                const double *__restrict__ px, double shift) {
    __shared__ double part[256];
    const LeafTask2 t = tasks[blockIdx.x];
    H2P_BY_WIDTH(t.w, leaf_d_w, t, contrib, arena, px, shift, fwd, y, yt, part);
}

// ---------------------------------------------------------------------------
// Grouped bi-GEMV over stored blocks (AOT), the products of
// CBLAS_BI_GEMV (src/H2Pack_matvec.c:26-65) as used by the intermediate
// (:303-381) and dense (:864-934) phases.  One workgroup per block: lanes
// own columns (NS strips of 64), the four waves take every fourth row; the
// row sums are wave reductions, the column sums are reduced across waves in
// LDS in a fixed order.
template <typename TS, int NS>
__device__ __forceinline__ void blk_aot_pass(const BlkTask &t, int cbase, int ncols,
                                             const TS *__restrict__ A,
                                             const double *__restrict__ xin,
                                             double *__restrict__ arena,
                                             double (*red)[4][H2P_WAVE], bool first) {
    // TS = double: FP64 products.  TS = float (FP32-mixed): blocks stored and
    // multiplied in FP32; row sums leave the pass as FP32 into FP64 partials,
    // column sums are FP32 over 16 rows and folded into FP64 registers.
    // Each wave takes four consecutive rows per iteration (4 x NS loads in
    // flight per lane) and reduces the four row sums with one butterfly.
    // The wave index is the same on every lane: said so, the row addresses
    // stay scalar and each load needs only its column offset per lane.
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    TS x0[NS], acc1[NS];
    double acc1d[NS];
    int cc[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int c = k * H2P_WAVE + lane;
        const bool ok = c < ncols;
        cc[k] = ok ? c : 0;
        x0[k] = ok ? (TS)xin[t.in0 + cbase + c] : (TS)0;
        acc1[k] = (TS)0;
        acc1d[k] = 0.0;
    }
    const double *in1 = xin + t.in1;
    const bool has1 = t.flags & 1;
    int tile = 0;
    for (int r0 = 4 * w; r0 < t.nrow; r0 += 16) {
        TS p[4], v1[4], a[4][NS];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = min(r0 + q, t.nrow - 1);     // rows past the end repeat the last row
            const bool ok = r0 + q < t.nrow;
            const TS *row = A + (long long)i * t.ncol + cbase;
#pragma unroll
            for (int k = 0; k < NS; k++) a[q][k] = row[cc[k]];
            v1[q] = (has1 && ok) ? (TS)in1[i] : (TS)0;
            p[q] = (TS)0;
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int k = 0; k < NS; k++) {
                p[q] += a[q][k] * x0[k];
                acc1[k] += a[q][k] * v1[q];
            }
        const TS s = wave_sum4<TS>(p[0], p[1], p[2], p[3]);
        const int myrow = r0 + ((lane >> 4) & 3);
        if ((lane & 15) == 0 && myrow < t.nrow) {
            double *o = arena + t.out0 + myrow;
            if (first) *o = (double)s;
            else *o += (double)s;
        }
        if constexpr (sizeof(TS) == 4) {
            if (++tile == 4) {
                tile = 0;
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    acc1d[k] += (double)acc1[k];
                    acc1[k] = (TS)0;
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NS; k++) acc1d[k] += (double)acc1[k];
    if (has1) {
#pragma unroll
        for (int k = 0; k < NS; k++) red[k][w][lane] = acc1d[k];
        __syncthreads();
        for (int c = threadIdx.x; c < ncols; c += blockDim.x) {
            const int k = c >> 6, l = c & 63;
            arena[t.out1 + cbase + c] = (red[k][0][l] + red[k][1][l]) + (red[k][2][l] + red[k][3][l]);
        }
        __syncthreads();
    }
}

#define H2P_AOT_MAXNS 4
template <typename TS>
__device__ __forceinline__ void blocks_aot_body(const BlkTask &t, const TS *__restrict__ blob,
                                                const double *__restrict__ xin,
                                                double *__restrict__ arena) {
    __shared__ double red[H2P_AOT_MAXNS][4][H2P_WAVE];
    const TS *A = blob + t.data_off;
    for (int cb = 0; cb < t.ncol; cb += H2P_AOT_MAXNS * H2P_WAVE) {
        const int nc = min(t.ncol - cb, H2P_AOT_MAXNS * H2P_WAVE);
        const int ns = (nc + 63) >> 6;
        const bool first = (cb == 0);
        if (ns <= 1) blk_aot_pass<TS, 1>(t, cb, nc, A, xin, arena, red, first);
        else if (ns <= 2) blk_aot_pass<TS, 2>(t, cb, nc, A, xin, arena, red, first);
        else if (ns <= 3) blk_aot_pass<TS, 3>(t, cb, nc, A, xin, arena, red, first);
        else blk_aot_pass<TS, 4>(t, cb, nc, A, xin, arena, red, first);
        // the next column pass adds into out0 rows written by the same lanes
        __syncthreads();
    }
}

template <typename TS>
__global__ void __launch_bounds__(256) k_blocks_aot(const BlkTask *__restrict__ tasks,
                                                    const TS *__restrict__ blob,
                                                    const double *__restrict__ xin,
                                                    double *__restrict__ arena) {
    blocks_aot_body<TS>(tasks[blockIdx.x], blob, xin, arena);
}

__global__ void k_f64_to_f32(const double *__restrict__ in, float *__restrict__ out, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) out[i] = (float)in[i];
}

// Orders the LDS accesses of one wave (LDS operations of a wave complete in
// issue order; the fences keep the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NW>
__device__ __forceinline__ void jitm_sync() {
    if constexpr (NW == 4) __syncthreads();
    else wave_lds_sync();
}

// ---------------------------------------------------------------------------
// Grouped kernel-evaluating bi-matvec for RPY (JIT), the krnl_bimv products
// of src/H2Pack_matvec.c:586-764 (B) and :1002-1145 (D) with the 3x3 tensor
// K = t1 I + t2 u u^T per point pair.
//  * Source points live in lanes, NS strips of 64 per pass, with their
//    coordinates (plus the task's periodic shift), radius and its
//    reciprocal in registers.
//  * Target points are staged in LDS per chunk (coordinates, radius, its
//    reciprocal, the transposed product's input); each wave takes four
//    targets per iteration and reduces their twelve row sums with three
//    butterflies (one per component).
//  * Lanes without a source point use a valid point with zero coefficients.
#define H2P_JIT_ROWS 256                 // target rows staged per chunk (all JIT launches)
#define H2P_RPY_MAXNS 2
// FP32-mixed: coordinates relative to the task's first target point (the
// differences taken in FP64, once per point, then rounded), the tensor and
// the products in FP32; row sums leave the pass as FP32 into the FP64
// partials, column sums are FP32 over 16 rows per lane and folded into FP64
// registers.  (FP64: the tiled launch below.)
struct RpyRow { float x, y, z, a, ia, v0, v1, v2; };

template <int NS>
__device__ __forceinline__ void rpy_pass(const BlkTask &t, int pbase, int npts,
                                         const double *__restrict__ cx, long long cstride, const KParam &kp,
                                         const double *__restrict__ shifts, const double *__restrict__ xin,
                                         double *__restrict__ arena, RpyRow *rows,
                                         double (*red)[3][4][H2P_WAVE], bool first) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // rows of cx: x, y, z, radius, reciprocal radius
    const double *cy = cx + cstride, *cz = cx + 2 * cstride, *ca = cx + 3 * cstride, *cia = cx + 4 * cstride;
    // set 1 may be a periodic image: its coordinates plus the task's shift
    double hx = shifts[3 * t.shift], hy = shifts[3 * t.shift + 1], hz = shifts[3 * t.shift + 2];
    const double ox = cx[t.c0], oy = cy[t.c0], oz = cz[t.c0];
    float sx[NS], sy[NS], sz[NS], sa[NS], isa[NS], x0[NS][3], acc1[NS][3];
    double acc1d[NS][3];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int p = k * H2P_WAVE + lane;
        const bool ok = p < npts;
        const int g = t.c1 + pbase + (ok ? p : 0);
        sx[k] = (float)(cx[g] + hx - ox);
        sy[k] = (float)(cy[g] + hy - oy);
        sz[k] = (float)(cz[g] + hz - oz);
        sa[k] = (float)ca[g];
        isa[k] = (float)cia[g];
#pragma unroll
        for (int b = 0; b < 3; b++) {
            x0[k][b] = ok ? (float)xin[t.in0 + (pbase + p) * 3 + b] : 0.0f;
            acc1[k][b] = 0.0f;
            acc1d[k][b] = 0.0;
        }
    }
    const bool has1 = t.flags & 1;
    const float C = (float)kp.p1;
    int tile = 0;
    for (int rc = 0; rc < t.n0; rc += H2P_JIT_ROWS) {
        const int nr = min(t.n0 - rc, H2P_JIT_ROWS);
        const int nr_pad = (nr + 15) & ~15;
        __syncthreads();
        for (int q = threadIdx.x; q < nr_pad; q += blockDim.x) {
            const bool ok = q < nr;
            const int g = t.c0 + rc + (ok ? q : 0);
            RpyRow r;
            r.x = (float)(cx[g] - ox);
            r.y = (float)(cy[g] - oy);
            r.z = (float)(cz[g] - oz);
            r.a = (float)ca[g];
            r.ia = (float)cia[g];
            const bool v = ok && has1;
            r.v0 = v ? (float)xin[t.in1 + (rc + q) * 3] : 0.0f;
            r.v1 = v ? (float)xin[t.in1 + (rc + q) * 3 + 1] : 0.0f;
            r.v2 = v ? (float)xin[t.in1 + (rc + q) * 3 + 2] : 0.0f;
            rows[q] = r;
        }
        __syncthreads();
        for (int r0 = 4 * w; r0 < nr_pad; r0 += 16) {
            float p[4][3];
            // one target at a time (the barriers bound the registers the
            // scheduler may spend on interleaving targets)
#pragma unroll
            for (int a = 0; a < 4; a++) {
                __builtin_amdgcn_sched_barrier(0);
                const RpyRow R = rows[r0 + a];
                p[a][0] = p[a][1] = p[a][2] = 0.0f;
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    const bool ok = (k * H2P_WAVE + lane) < npts;
                    float t1, t2, ux, uy, uz;
                    rpy_coef_rcp(R.x - sx[k], R.y - sy[k], R.z - sz[k], R.a, sa[k], R.ia, isa[k], C,
                                 t1, t2, ux, uy, uz);
                    t1 = ok ? t1 : 0.0f;
                    t2 = ok ? t2 : 0.0f;
                    // K = t1 I + t2 u u^T (symmetric)
                    const float ud0 = ux * x0[k][0] + uy * x0[k][1] + uz * x0[k][2];
                    const float ud1 = ux * R.v0 + uy * R.v1 + uz * R.v2;
                    p[a][0] += t1 * x0[k][0] + t2 * ux * ud0;
                    p[a][1] += t1 * x0[k][1] + t2 * uy * ud0;
                    p[a][2] += t1 * x0[k][2] + t2 * uz * ud0;
                    acc1[k][0] += t1 * R.v0 + t2 * ux * ud1;
                    acc1[k][1] += t1 * R.v1 + t2 * uy * ud1;
                    acc1[k][2] += t1 * R.v2 + t2 * uz * ud1;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int myrow = r0 + ((lane >> 4) & 3);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float s = wave_sum4<float>(p[0][c], p[1][c], p[2][c], p[3][c]);
                if ((lane & 15) == 0 && myrow < nr) {
                    double *o = arena + t.out0 + (rc + myrow) * 3 + c;
                    if (first) *o = (double)s;
                    else *o += (double)s;
                }
            }
            if (++tile == 4) {
                tile = 0;
#pragma unroll
                for (int k = 0; k < NS; k++)
#pragma unroll
                    for (int b = 0; b < 3; b++) {
                        acc1d[k][b] += (double)acc1[k][b];
                        acc1[k][b] = 0.0f;
                    }
            }
        }
    }
    if (has1) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                red[k][b][w][lane] = acc1d[k][b] + (double)acc1[k][b];
            }
        __syncthreads();
        for (int q = threadIdx.x; q < npts * 3; q += blockDim.x) {
            const int pnt = q / 3, b = q - pnt * 3;
            const int k = pnt >> 6, l = pnt & 63;
            arena[t.out1 + (pbase + pnt) * 3 + b] =
                (red[k][b][0][l] + red[k][b][1][l]) + (red[k][b][2][l] + red[k][b][3][l]);
        }
    }
}

// FP64 RPY in tiles: a step covers 8 target x 16 source points, lane l the
// pairs (4 k + l / 16, l % 16), k = 0, 1.
//  * A pass covers up to 16 H2P_RPYT_NT source points, as evenly split over
//    a block's passes as tiles allow (ranks of ~76 points are 5 tiles; lanes
//    over 64 sources would leave 40% of them idle).  The points of both sets
//    are staged in LDS, one array per component, so that a step reads its
//    sources conflict-free and its targets by broadcast.
//  * Row sums stay in the lane over the pass's tiles and are reduced over the
//    16 lanes by DPP moves, column sums stay in registers over all rows.
//  * The kernel is evaluated on the difference vector d itself, K = t1 I +
//    g d d^T: no unit vector.  Blocks whose bounding boxes are further apart
//    than two radii (flag H2P_BLK_FAR, set at upload) have only the far form,
//      t1 = 1/r + (s / 3) / r^3,  g = (1 - s / r^2) / r^3,  s = a^2 + b^2,
//    with 3 C / 4 folded into the staged inputs: 41 slots of the FP64 pipe
//    per pair with both products, against 61 in the general form with its
//    three regimes.
//  * ONE (periodic handles): blocks act one way only.
// Two launch units as in the norm-form kernels below: four waves share a
// large block's rows, or take one small block each.
// Bound by the FP64 pipe.  N = 20k at 20% volume fraction, us per launch: lanes
// over 64 sources with the general form on every pair 796, this form 258;
// periodic N = 10k: 1077 and 450.
#define H2P_RPYT_NT 6
#define H2P_RPYT_ROWS 64                      // targets staged per chunk (four workgroups' LDS fit a CU)
#define H2P_RPYT_WAVE 96                      // a wave unit's most targets and sources
#define H2P_RPYT_COMP 8                       // x y z a 1/a v0 v1 v2 (far: a^2 in place of a)
#define H2P_RPYT_LDS (H2P_RPYT_COMP * (H2P_RPYT_ROWS + 16 * H2P_RPYT_NT))   // doubles per unit

// Whether an RPY task runs as a wave unit.
__host__ __device__ inline bool rpy_wave_task(int n0, int n1) {
    return n0 <= H2P_RPYT_WAVE && n1 <= 16 * H2P_RPYT_NT;
}

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// Sums over the 16 lanes of each lane group of two per-lane values; lanes
// with bit 3 clear return the sum of v0, the others that of v1.  Row
// rotation by 8, half-row mirror and quad permutations: VALU only.
__device__ __forceinline__ double group16_sum2(double v0, double v1) {
    const bool b3 = threadIdx.x & 8;
    double a = (b3 ? v1 : v0) + dpp_move<0x128>(b3 ? v0 : v1);
    a += dpp_move<0x141>(a);
    a += dpp_move<0x4e>(a);
    a += dpp_move<0xb1>(a);
    return a;
}

// Stages points [0, n) of a set (padded with repeats and zero inputs to np).
template <bool FAR>
__device__ __forceinline__ void rpyt_stage(double *dst, int ld, int n, int np, int tid, int nthr, int c,
                                           const double *__restrict__ cx, long long cstride, double hx, double hy,
                                           double hz, const double *__restrict__ v, double vs) {
    for (int q = tid; q < np; q += nthr) {
        const bool ok = q < n;
        const long long g = c + (ok ? q : 0);
        const double a = cx[3 * cstride + g];
        dst[q] = cx[g] + hx;
        dst[ld + q] = cx[cstride + g] + hy;
        dst[2 * ld + q] = cx[2 * cstride + g] + hz;
        dst[3 * ld + q] = FAR ? a * a : a;
        if (!FAR) dst[4 * ld + q] = cx[4 * cstride + g];
#pragma unroll
        for (int b = 0; b < 3; b++) dst[(5 + b) * ld + q] = (ok && v) ? v[3 * q + b] * vs : 0.0;
    }
}

template <int NT, int NW, bool FAR, bool ONE>
__device__ __forceinline__ void rpyt_pass(const BlkTask &t, int pbase, int npts, const double *__restrict__ cx,
                                          long long cstride, double C, const double *__restrict__ shifts,
                                          const double *__restrict__ xin, double *__restrict__ arena, double *lds,
                                          double *red, bool first) {
    constexpr int LR = H2P_RPYT_ROWS, LC = 16 * H2P_RPYT_NT;
    const int lane = threadIdx.x & 63, w = NW == 4 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int tid = NW == 4 ? threadIdx.x : lane;
    const int li = lane & 15, lg = lane >> 4;
    double *rows = lds, *cols = lds + H2P_RPYT_COMP * LR;
    const double vs = FAR ? 0.75 * C : 1.0;
    const double *sh = shifts + 3 * t.shift;
    const bool has1 = !ONE && (t.flags & 1);
    rpyt_stage<FAR>(cols, LC, npts, 16 * NT, tid, NW * H2P_WAVE, t.c1 + pbase, cx, cstride, sh[0], sh[1], sh[2],
                    xin + t.in0 + 3 * pbase, vs);
    double acc[NT][3];
#pragma unroll
    for (int c = 0; c < NT; c++)
#pragma unroll
        for (int b = 0; b < 3; b++) acc[c][b] = 0.0;
    for (int rc = 0; rc < t.n0; rc += LR) {
        const int nr = min(t.n0 - rc, LR);
        const int nstep = (nr + 7) >> 3;
        jitm_sync<NW>();
        rpyt_stage<FAR>(rows, LR, nr, 8 * nstep, tid, NW * H2P_WAVE, t.c0 + rc, cx, cstride, 0.0, 0.0, 0.0,
                        has1 ? xin + t.in1 + 3 * rc : nullptr, vs);
        jitm_sync<NW>();
        for (int st = w; st < nstep; st += NW) {
            double r[2][8], p[2][3];
            // an offset the compiler cannot see through: otherwise it keeps
            // every tile's sources in registers across the steps and spills
            int o0 = li;
            asm volatile("" : "+v"(o0));
#pragma unroll
            for (int k = 0; k < 2; k++) {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (!(FAR && e == 4) && !(ONE && e >= 5)) r[k][e] = rows[e * LR + 8 * st + 4 * k + lg];
                p[k][0] = p[k][1] = p[k][2] = 0.0;
            }
#pragma unroll
            for (int c = 0; c < NT; c++) {
                double s[8];
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (!(FAR && e == 4)) s[e] = cols[e * LC + 16 * c + o0];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    double dx = r[k][0] - s[0], dy = r[k][1] - s[1], dz = r[k][2] - s[2], t1, g;
                    if constexpr (FAR) {
                        const double y = rsqrt_refined(__builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx)));
                        const double y2 = y * y, sr = (r[k][3] + s[3]) * y2, y3 = y * y2;
                        t1 = __builtin_fma(y * sr, 1.0 / 3.0, y);
                        g = __builtin_fma(-sr, y3, y3);
                    } else {
                        double ux, uy, uz;
                        rpy_coef_rcp(dx, dy, dz, r[k][3], s[3], r[k][4], s[4], C, t1, g, ux, uy, uz);
                        dx = ux;
                        dy = uy;
                        dz = uz;
                    }
                    const double w0 = g * __builtin_fma(dz, s[7], __builtin_fma(dy, s[6], dx * s[5]));
                    p[k][0] = __builtin_fma(w0, dx, __builtin_fma(t1, s[5], p[k][0]));
                    p[k][1] = __builtin_fma(w0, dy, __builtin_fma(t1, s[6], p[k][1]));
                    p[k][2] = __builtin_fma(w0, dz, __builtin_fma(t1, s[7], p[k][2]));
                    if constexpr (!ONE) {
                        const double w1 = g * __builtin_fma(dz, r[k][7], __builtin_fma(dy, r[k][6], dx * r[k][5]));
                        acc[c][0] = __builtin_fma(w1, dx, __builtin_fma(t1, r[k][5], acc[c][0]));
                        acc[c][1] = __builtin_fma(w1, dy, __builtin_fma(t1, r[k][6], acc[c][1]));
                        acc[c][2] = __builtin_fma(w1, dz, __builtin_fma(t1, r[k][7], acc[c][2]));
                        // pinned here: the compiler would sink the sums past the
                        // row stores and keep every pair's t1, g and d alive
                        asm volatile("" : "+v"(acc[c][0]), "+v"(acc[c][1]), "+v"(acc[c][2]));
                    }
                    asm volatile("" : "+v"(p[k][0]), "+v"(p[k][1]), "+v"(p[k][2]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int row = 8 * st + 4 * ((lane >> 3) & 1) + lg;
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const double v = group16_sum2(p[0][b], p[1][b]);
                if ((lane & 7) == 0 && row < nr) {
                    double *o = arena + t.out0 + 3 * (rc + row) + b;
                    *o = first ? v : *o + v;
                }
            }
        }
    }
    if (!has1) return;
    // column sums: (g0 + g1) + (g2 + g3) over the lane groups, then the waves in order
#pragma unroll
    for (int c = 0; c < NT; c++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
            double v = acc[c][b] + __shfl_xor(acc[c][b], 16, H2P_WAVE);
            v += __shfl_xor(v, 32, H2P_WAVE);
            const int j = 16 * c + li;
            if constexpr (NW == 4) {
                if (lg == 0) red[(w * 3 + b) * LC + j] = v;
            } else {
                if (lg == 0 && j < npts) arena[t.out1 + 3 * (pbase + j) + b] = v;
            }
        }
    if constexpr (NW == 4) {
        __syncthreads();
        for (int q = threadIdx.x; q < 3 * npts; q += blockDim.x) {
            const int j = q / 3, b = q - 3 * j;
            arena[t.out1 + 3 * pbase + q] = (red[b * LC + j] + red[(3 + b) * LC + j]) +
                                            (red[(6 + b) * LC + j] + red[(9 + b) * LC + j]);
        }
    }
}

template <int NW, bool FAR, bool ONE>
__device__ __forceinline__ void rpyt_task(const BlkTask &t, const double *__restrict__ cx, long long cstride,
                                          double C, const double *__restrict__ shifts,
                                          const double *__restrict__ xin, double *__restrict__ arena, double *lds,
                                          double *red) {
    const int ntile = (t.n1 + 15) >> 4, npass = (ntile + H2P_RPYT_NT - 1) / H2P_RPYT_NT;
    const int per = (ntile + npass - 1) / npass;   // tiles per pass, evenly
    for (int c0 = 0; c0 < ntile; c0 += per) {
        const int pb = 16 * c0, np = min(t.n1 - pb, 16 * per);
        const bool first = c0 == 0;
        switch ((np + 15) >> 4) {
#define H2P_RPYT_CASE(n) \
            case n: rpyt_pass<n, NW, FAR, ONE>(t, pb, np, cx, cstride, C, shifts, xin, arena, lds, red, first); break;
            H2P_RPYT_CASE(1) H2P_RPYT_CASE(2) H2P_RPYT_CASE(3)
            H2P_RPYT_CASE(4) H2P_RPYT_CASE(5) H2P_RPYT_CASE(6)
#undef H2P_RPYT_CASE
            default: break;
        }
        jitm_sync<NW>();
    }
}

// Launch unit u: u < nbig runs task u on the whole workgroup, later units
// tasks nbig + 4 (u - nbig) + w, one per wave.
template <bool ONE>
__device__ __forceinline__ void blocks_rpy_unit(const BlkTask *__restrict__ tasks, int u, int nbig, int ntask,
                                                const double *__restrict__ cx, long long cstride, double C,
                                                const double *__restrict__ shifts, const double *__restrict__ xin,
                                                double *__restrict__ arena) {
    __shared__ double lds[4 * H2P_RPYT_LDS];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (u < nbig) {
        const BlkTask t = tasks[u];
        double *red = lds + H2P_RPYT_LDS;   // 4 x 3 x 16 NT doubles
        if (t.flags & H2P_BLK_FAR) rpyt_task<4, true, ONE>(t, cx, cstride, C, shifts, xin, arena, lds, red);
        else rpyt_task<4, false, ONE>(t, cx, cstride, C, shifts, xin, arena, lds, red);
    } else {
        const int i = nbig + 4 * (u - nbig) + w;
        if (i >= ntask) return;
        const BlkTask t = tasks[i];
        double *l = lds + w * H2P_RPYT_LDS;
        if (t.flags & H2P_BLK_FAR) rpyt_task<1, true, ONE>(t, cx, cstride, C, shifts, xin, arena, l, nullptr);
        else rpyt_task<1, false, ONE>(t, cx, cstride, C, shifts, xin, arena, l, nullptr);
    }
}

template <bool ONE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_blocks_rpy(const BlkTask *__restrict__ tasks, int nbig, int ntask, const double *__restrict__ cx,
             long long cstride, double C, const double *__restrict__ shifts, const double *__restrict__ xin,
             double *__restrict__ arena) {
    blocks_rpy_unit<ONE>(tasks, blockIdx.x, nbig, ntask, cx, cstride, C, shifts, xin, arena);
}

// FP32-mixed RPY.
__device__ __forceinline__ void blocks_rpy32(const BlkTask &t, const double *__restrict__ cx, long long cstride,
                                             const KParam &kp, const double *__restrict__ shifts,
                                             const double *__restrict__ xin, double *__restrict__ arena) {
    __shared__ RpyRow rows[H2P_JIT_ROWS];
    __shared__ double red[H2P_RPY_MAXNS][3][4][H2P_WAVE];
    for (int pb = 0; pb < t.n1; pb += H2P_RPY_MAXNS * H2P_WAVE) {
        const int np = min(t.n1 - pb, H2P_RPY_MAXNS * H2P_WAVE);
        const bool first = (pb == 0);
        if (np <= H2P_WAVE) rpy_pass<1>(t, pb, np, cx, cstride, kp, shifts, xin, arena, rows, red, first);
        else rpy_pass<2>(t, pb, np, cx, cstride, kp, shifts, xin, arena, rows, red, first);
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) k_blocks_rpy32(const BlkTask *__restrict__ tasks,
                                                      const double *__restrict__ cx, long long cstride, KParam kp,
                                                      const double *__restrict__ shifts,
                                                      const double *__restrict__ xin, double *__restrict__ arena) {
    blocks_rpy32(tasks[blockIdx.x], cx, cstride, kp, shifts, xin, arena);
}

// The root's periodic block (H2P_matvec_periodic, src/H2Pack_matvec_periodic.c:
// 455-470): y1[root] = per_blk y0[root], one wave per row, lanes over the
// columns, fixed-order wave reduction.
__global__ void __launch_bounds__(256) k_root_block(const double *__restrict__ per, int r,
                                                    const double *__restrict__ y0,
                                                    double *__restrict__ y1) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= r) return;
    const double *a = per + (long long)row * r;
    double s = 0.0;
    for (int c = lane; c < r; c += H2P_WAVE) s += a[c] * y0[c];
    s = wave_sum(s);
    if (lane == 0) y1[row] = s;
}

// ---------------------------------------------------------------------------
// FP64 norm-form kernels (Gaussian, Matern) with the distances on the matrix
// cores.  The squared distances of a tile of 16 target rows x 16 source
// columns are one v_mfma_f64_16x16x4f64,
//     q[i][j] = |r_i|^2 + sum_k A[i][k] B[k][j],
//     A[i] = (1, r_i),  B[.][j] = (|s_j|^2, -2 s_j),
// with |r_i|^2 as the accumulator input (the same terms, in the same order,
// as the VALU form |r|^2 + |s|^2 - 2 r.s), so the VALU only evaluates the
// kernel and the two products of each pair.  MFMA layout, lane l: it
// supplies A[l % 16][l / 16] and B[l / 16][l % 16] and receives
// q[4 r + l / 16][l % 16] in register r.
//  * A pass covers up to H2P_JITM_NT tiles of 16 source columns, staged in
//    LDS (B operand and input value); each lane keeps one column partial
//    sum per tile in registers.
//  * Target rows are staged in LDS in chunks; the NW cooperating waves take
//    the 16-row tiles w, w + NW, ...; per tile a lane accumulates four row
//    sums (rows 4 r + l / 16) over its columns, reduced over the 16 lanes
//    of each group once per tile.
//  * Column partial sums are reduced at the end of the pass over the four
//    lane groups (and, with NW = 4, the four waves) in a fixed order.
//  * Padded rows repeat a valid row with input 0 and padded columns a valid
//    source with input 0, so every kernel value is finite and the padding
//    adds exact zeros.
// Two launch units share one kernel: a workgroup unit (NW = 4) runs one
// large block; a wave unit runs four small blocks (n0 <= H2P_JITW_ROWS,
// n1 <= 16 H2P_JITM_NT), one per wave, with wave-private LDS and no
// workgroup barriers, so the short blocks do not wait on each other.
// Bound by the FP64 pipe and by the wait for the table: the four values of a
// lane's tile are evaluated together, their four table reads in flight
// before the polynomials, and blocks whose values stay normal (H2P_BLK_FAST, 94%
// of the pairs at N = 1M) add the exponent by an integer operation.  53 instead
// of 57 VALU operations per tile (Matern: 85 instead of 97), 65 with staging and
// reductions (65.5); matvec N = 1M Gaussian 13.63 -> 13.49 ms, CG on three Matern
// matrices of 12-24k points 6.36 -> 5.93 ms per 10 iterations.  A 1024-entry table
// with a polynomial of one degree less (49 operations) measured slower, 14.5 ms:
// 8 KB of table to copy per workgroup and more bank conflicts; several units per
// workgroup, to copy it once, 14.8 ms.
#define H2P_JITM_NT 8

// Runs a tile body for the rows that hold points: lane group g's register r
// holds tile row 4 r + g, so with vr valid rows the registers r >= ceil(vr /
// 4) hold only padding (a repeated point with input 0, whose products add
// exact zeros) and are skipped.  Same results, fewer kernel evaluations in a
// block's last row tile.
template <typename F>
__device__ __forceinline__ void tile_rows(int vr, F &&body) {
    if (vr <= 4) body(std::integral_constant<int, 1>{});
    else if (vr <= 8) body(std::integral_constant<int, 2>{});
    else body(std::integral_constant<int, 4>{});
}
#define H2P_JITW_ROWS 80
struct JitmRow { double a[4]; };   // (1, x, y, z) of a target; (|s|^2, -2 s) of a source
struct JitmNV { double n, v; };    // |r|^2 and the transposed product's input

// LDS of the norm-form kernels, in doubles: the workgroup unit uses rows
// (4 + 2) x H2P_JIT_ROWS, sources 5 x 16 NT and the wave partials 4 x 16 NT; a
// wave unit gives each wave (4 + 2) x H2P_JITW_ROWS + 5 x 16 NT.
#define H2P_JITM_LDS_WG (6 * H2P_JIT_ROWS + 5 * 16 * H2P_JITM_NT + 4 * 16 * H2P_JITM_NT)
#define H2P_JITM_LDS_WAVE (6 * H2P_JITW_ROWS + 5 * 16 * H2P_JITM_NT)
#define H2P_JITM_LDS (H2P_JITM_LDS_WG > 4 * H2P_JITM_LDS_WAVE ? H2P_JITM_LDS_WG : 4 * H2P_JITM_LDS_WAVE)

template <int KID, int NT, int NW, bool FAST>
__device__ __forceinline__ void jitm_pass(const BlkTask &t, int pbase, int npts,
                                          const double *__restrict__ cx, long long cstride,
                                          double scale, double ox, double oy, double oz,
                                          const double *__restrict__ xin, double *__restrict__ arena,
                                          JitmRow *rowa, JitmNV *rownv, JitmRow *srcb, double *srcx,
                                          double *red, const double *e2x, bool first) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS;
    const int lane = threadIdx.x & 63, w = NW == 4 ? (threadIdx.x >> 6) : 0;
    const int tid = NW == 4 ? threadIdx.x : lane;
    const int li = lane & 15, lg = lane >> 4;
    const double *cy = cx + cstride, *cz = cx + 2 * cstride;
    // the pass's sources: B operand (|s|^2, -2 s) and input value
    for (int q = tid; q < NT * 16; q += NW * H2P_WAVE) {
        const bool ok = q < npts;
        const int g = t.c1 + pbase + (ok ? q : 0);
        const double ux = (cx[g] - ox) * scale, uy = (cy[g] - oy) * scale, uz = (cz[g] - oz) * scale;
        JitmRow b;
        b.a[0] = ux * ux + uy * uy + uz * uz;
        b.a[1] = -2.0 * ux;
        b.a[2] = -2.0 * uy;
        b.a[3] = -2.0 * uz;
        srcb[q] = b;
        srcx[q] = ok ? xin[t.in0 + pbase + q] : 0.0;
    }
    double c2 = H2P_E2X_C2;
    asm volatile("" : "+v"(c2));   // stays in a vector register
    double acc[NT];
#pragma unroll
    for (int c = 0; c < NT; c++) acc[c] = 0.0;
    const bool has1 = t.flags & 1;
    for (int rc = 0; rc < t.n0; rc += ROWS) {
        const int nr = min(t.n0 - rc, ROWS);
        const int ntile = (nr + 15) >> 4;
        jitm_sync<NW>();
        for (int q = tid; q < ntile * 16; q += NW * H2P_WAVE) {
            const bool ok = q < nr;
            const int g = t.c0 + rc + (ok ? q : 0);
            const double ux = (cx[g] - ox) * scale, uy = (cy[g] - oy) * scale, uz = (cz[g] - oz) * scale;
            JitmRow ra;
            ra.a[0] = 1.0;
            ra.a[1] = ux;
            ra.a[2] = uy;
            ra.a[3] = uz;
            rowa[q] = ra;
            JitmNV e;
            e.n = ux * ux + uy * uy + uz * uz;
            e.v = (ok && has1) ? xin[t.in1 + rc + q] : 0.0;
            rownv[q] = e;
        }
        jitm_sync<NW>();
        for (int tt = w; tt < ntile; tt += NW) {
            const double a = rowa[tt * 16 + li].a[lg];
            // one base for all tiles, opaque so that it stays one
            unsigned o = li;
            asm volatile("" : "+v"(o));
            const double *sx = srcx + o, *sb = (const double *)srcb + 4 * o + lg;
            d4 cn;
            double v[4], p[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const JitmNV e = rownv[tt * 16 + 4 * r + lg];
                cn[r] = e.n;
                v[r] = e.v;
                p[r] = 0.0;
            }
            // the scheduling barriers keep the compiler from hoisting all NT
            // products ahead of the VALU work (each live result costs 8
            // registers); other waves cover the product's latency
            auto tile = [&](auto nrq) {
                constexpr int NR = decltype(nrq)::value;
#pragma unroll
                for (int c = 0; c < NT; c++) {
                    const double xc = sx[c * 16];
                    const d4 q = __builtin_amdgcn_mfma_f64_16x16x4f64(a, sb[c * 64], cn, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    double kv[NR];
                    kjit<KID, FAST, NR>(q, e2x, c2, kv);
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        p[r] += kv[r] * xc;
                        acc[c] += kv[r] * v[r];
                    }
                    // Matern: pinned here, or the compiler sinks the column sums past
                    // the row stores, keeps every kernel value alive and spills
                    // (the Gaussian fits and is 1.5% faster left alone)
                    if constexpr (KID == KM) asm volatile("" : "+v"(acc[c]));
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            tile_rows(nr - tt * 16, tile);
            const double s = group16_sum4(p[0], p[1], p[2], p[3]);
            const int myrow = tt * 16 + 4 * ((lane >> 2) & 3) + lg;
            if ((lane & 3) == 0 && myrow < nr) {
                double *o = arena + t.out0 + rc + myrow;
                if (first) *o = s;
                else *o += s;
            }
        }
    }
    if (!has1) return;
    // (g0 + g1) + (g2 + g3) over the four lane groups, then the waves in order
#pragma unroll
    for (int c = 0; c < NT; c++) {
        double s = acc[c] + __shfl_xor(acc[c], 16, H2P_WAVE);
        s += __shfl_xor(s, 32, H2P_WAVE);
        const int j = c * 16 + li;
        if constexpr (NW == 4) {
            if (lg == 0) red[w * 16 * H2P_JITM_NT + j] = s;
        } else {
            if (lg == 0 && j < npts) arena[t.out1 + pbase + j] = s;
        }
    }
    if constexpr (NW == 4) {
        constexpr int LC = 16 * H2P_JITM_NT;
        __syncthreads();
        for (int j = threadIdx.x; j < npts; j += blockDim.x)
            arena[t.out1 + pbase + j] = (red[j] + red[LC + j]) + (red[2 * LC + j] + red[3 * LC + j]);
    }
}

template <int KID, int NW, bool FAST>
__device__ __forceinline__ void jitm_task(const BlkTask &t, const double *__restrict__ cx,
                                          long long cstride, double scale,
                                          const double *__restrict__ xin, double *__restrict__ arena,
                                          double *lds, const double *e2x) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS;
    JitmRow *rowa = (JitmRow *)lds;
    JitmNV *rownv = (JitmNV *)(lds + 4 * ROWS);
    JitmRow *srcb = (JitmRow *)(lds + 6 * ROWS);
    double *srcx = lds + 6 * ROWS + 4 * 16 * H2P_JITM_NT;
    double *red = srcx + 16 * H2P_JITM_NT;   // workgroup unit only
    const double ox = cx[t.c0], oy = cx[cstride + t.c0], oz = cx[2 * cstride + t.c0];
    const int ntile = (t.n1 + 15) >> 4, npass = (ntile + H2P_JITM_NT - 1) / H2P_JITM_NT;
    const int per = npass > 0 ? (ntile + npass - 1) / npass : 1;   // tiles per pass, evenly
    for (int c0 = 0; c0 < ntile; c0 += per) {
        const int pb = 16 * c0, np = min(t.n1 - pb, 16 * per);
        const bool first = c0 == 0;
        switch ((np + 15) >> 4) {
#define H2P_JITM_CASE(n) \
            case n: jitm_pass<KID, n, NW, FAST>(t, pb, np, cx, cstride, scale, ox, oy, oz, xin, arena, rowa, rownv, srcb, srcx, red, e2x, first); break;
            H2P_JITM_CASE(1) H2P_JITM_CASE(2) H2P_JITM_CASE(3) H2P_JITM_CASE(4)
            H2P_JITM_CASE(5) H2P_JITM_CASE(6) H2P_JITM_CASE(7) H2P_JITM_CASE(8)
#undef H2P_JITM_CASE
            default: break;
        }
        jitm_sync<NW>();
    }
}

// Launch unit u of a tiled launch: u < nbig runs task u on the whole
// workgroup, later units run tasks nbig + 4 (u - nbig) + w, one per wave.
// The exp2_neg128x table is copied into LDS first (one copy per workgroup).
template <int KID>
__device__ __forceinline__ void blocks_jitm_unit(const BlkTask *__restrict__ tasks, int u, int nbig, int ntask,
                                                 const double *__restrict__ cx, long long cstride,
                                                 double scale, const double *__restrict__ xin,
                                                 double *__restrict__ arena) {
    __shared__ double lds[H2P_JITM_LDS];
    __shared__ double e2x[H2P_E2_N];
    if (threadIdx.x < H2P_E2_N) e2x[threadIdx.x] = e2x_entry(c_e2tab[threadIdx.x], threadIdx.x);
    __syncthreads();
    if (u < nbig) {
        const BlkTask t = tasks[u];
        if (t.flags & H2P_BLK_FAST) jitm_task<KID, 4, true>(t, cx, cstride, scale, xin, arena, lds, e2x);
        else jitm_task<KID, 4, false>(t, cx, cstride, scale, xin, arena, lds, e2x);
    } else {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int i = nbig + 4 * (u - nbig) + w;
        if (i >= ntask) return;
        const BlkTask t = tasks[i];
        double *l = lds + w * H2P_JITM_LDS_WAVE;
        if (t.flags & H2P_BLK_FAST) jitm_task<KID, 1, true>(t, cx, cstride, scale, xin, arena, l, e2x);
        else jitm_task<KID, 1, false>(t, cx, cstride, scale, xin, arena, l, e2x);
    }
}

// ---------------------------------------------------------------------------
// FP64 Coulomb in the same tiling and launch units, with the distances from
// coordinate differences on the VALU: 1/r has the kernel's diagonal value at
// r = 0, so r = 0 must be exact.
//  * A pass's sources are staged in LDS, one array per component; a lane
//    reads its column's point once per tile for its four rows, whose
//    coordinates stay in registers.
//  * Blocks whose bounding boxes are apart (H2P_BLK_FAR) have no coincident
//    pair and skip the test for one (3 of 19 slots per pair).
// Bound by the FP64 pipe.  N = 200k, density 10 (1.4e9 pairs): B launches 2127
// us with sources in 64-lane strips (ranks of ~80 points leave a third of them
// idle), 1223 us in tiles; D launches 272 and 135.
#define H2P_JITC_LDS_WG (4 * H2P_JIT_ROWS + 4 * 16 * H2P_JITM_NT + 4 * 16 * H2P_JITM_NT)
#define H2P_JITC_LDS_WAVE (4 * H2P_JITW_ROWS + 4 * 16 * H2P_JITM_NT)
#define H2P_JITC_LDS (H2P_JITC_LDS_WG > 4 * H2P_JITC_LDS_WAVE ? H2P_JITC_LDS_WG : 4 * H2P_JITC_LDS_WAVE)

template <int NT, int NW, bool FAR>
__device__ __forceinline__ void jitc_pass(const BlkTask &t, int pbase, int npts, const double *__restrict__ cx,
                                          long long cstride, double diag, const double *__restrict__ xin,
                                          double *__restrict__ arena, double *rows, double *cols, double *red,
                                          bool first) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS, LC = 16 * H2P_JITM_NT;
    const int lane = threadIdx.x & 63, w = NW == 4 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int tid = NW == 4 ? threadIdx.x : lane;
    const int li = lane & 15, lg = lane >> 4;
    const bool has1 = t.flags & 1;
    // one set in LDS: x, y, z, input value (padding repeats a point, input 0)
    auto stage = [&](double *dst, int ld, int n, int np, int c, const double *v) {
        for (int q = tid; q < np; q += NW * H2P_WAVE) {
            const bool ok = q < n;
            const long long g = c + (ok ? q : 0);
            dst[q] = cx[g];
            dst[ld + q] = cx[cstride + g];
            dst[2 * ld + q] = cx[2 * cstride + g];
            dst[3 * ld + q] = (ok && v) ? v[q] : 0.0;
        }
    };
    stage(cols, LC, npts, 16 * NT, t.c1 + pbase, xin + t.in0 + pbase);
    double acc[NT];
#pragma unroll
    for (int c = 0; c < NT; c++) acc[c] = 0.0;
    for (int rc = 0; rc < t.n0; rc += ROWS) {
        const int nr = min(t.n0 - rc, ROWS);
        const int ntile = (nr + 15) >> 4;
        jitm_sync<NW>();
        stage(rows, ROWS, nr, 16 * ntile, t.c0 + rc, has1 ? xin + t.in1 + rc : nullptr);
        jitm_sync<NW>();
        for (int tt = w; tt < ntile; tt += NW) {
            double rx[4], ry[4], rz[4], rv[4], p[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int q = tt * 16 + 4 * r + lg;
                rx[r] = rows[q];
                ry[r] = rows[ROWS + q];
                rz[r] = rows[2 * ROWS + q];
                rv[r] = rows[3 * ROWS + q];
                p[r] = 0.0;
            }
            // an offset the compiler cannot see through, or it keeps every
            // tile's sources in registers across the row tiles
            int o = li;
            asm volatile("" : "+v"(o));
            auto tile = [&](auto nrq) {
                constexpr int NR = decltype(nrq)::value;
#pragma unroll
                for (int c = 0; c < NT; c++) {
                    const double sx = cols[16 * c + o], sy = cols[LC + 16 * c + o], sz = cols[2 * LC + 16 * c + o],
                                 sv = cols[3 * LC + 16 * c + o];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const double dx = rx[r] - sx, dy = ry[r] - sy, dz = rz[r] - sz;
                        const double q = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
                        double kv = rsqrt_refined(q);   // NaN at q = 0, replaced
                        if constexpr (!FAR) kv = q == 0.0 ? diag : kv;
                        p[r] = __builtin_fma(kv, sv, p[r]);
                        acc[c] = __builtin_fma(kv, rv[r], acc[c]);
                        asm volatile("" : "+v"(acc[c]));   // not sunk past the row stores
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            tile_rows(nr - tt * 16, tile);
            const double s = group16_sum4(p[0], p[1], p[2], p[3]);
            const int myrow = tt * 16 + 4 * ((lane >> 2) & 3) + lg;
            if ((lane & 3) == 0 && myrow < nr) {
                double *o2 = arena + t.out0 + rc + myrow;
                if (first) *o2 = s;
                else *o2 += s;
            }
        }
    }
    if (!has1) return;
    // (g0 + g1) + (g2 + g3) over the lane groups, then the waves in order
#pragma unroll
    for (int c = 0; c < NT; c++) {
        double s = acc[c] + __shfl_xor(acc[c], 16, H2P_WAVE);
        s += __shfl_xor(s, 32, H2P_WAVE);
        const int j = 16 * c + li;
        if constexpr (NW == 4) {
            if (lg == 0) red[w * LC + j] = s;
        } else {
            if (lg == 0 && j < npts) arena[t.out1 + pbase + j] = s;
        }
    }
    if constexpr (NW == 4) {
        __syncthreads();
        for (int j = threadIdx.x; j < npts; j += blockDim.x)
            arena[t.out1 + pbase + j] = (red[j] + red[LC + j]) + (red[2 * LC + j] + red[3 * LC + j]);
    }
}

template <int NW, bool FAR>
__device__ __forceinline__ void jitc_task(const BlkTask &t, const double *__restrict__ cx, long long cstride,
                                          double diag, const double *__restrict__ xin, double *__restrict__ arena,
                                          double *lds) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS;
    double *cols = lds + 4 * ROWS, *red = cols + 4 * 16 * H2P_JITM_NT;   // red: workgroup unit only
    const int ntile = (t.n1 + 15) >> 4, npass = (ntile + H2P_JITM_NT - 1) / H2P_JITM_NT;
    const int per = npass > 0 ? (ntile + npass - 1) / npass : 1;   // tiles per pass, evenly
    for (int c0 = 0; c0 < ntile; c0 += per) {
        const int pb = 16 * c0, np = min(t.n1 - pb, 16 * per);
        const bool first = c0 == 0;
        switch ((np + 15) >> 4) {
#define H2P_JITC_CASE(n) \
            case n: jitc_pass<n, NW, FAR>(t, pb, np, cx, cstride, diag, xin, arena, lds, cols, red, first); break;
            H2P_JITC_CASE(1) H2P_JITC_CASE(2) H2P_JITC_CASE(3) H2P_JITC_CASE(4)
            H2P_JITC_CASE(5) H2P_JITC_CASE(6) H2P_JITC_CASE(7) H2P_JITC_CASE(8)
#undef H2P_JITC_CASE
            default: break;
        }
        jitm_sync<NW>();
    }
}

__device__ __forceinline__ void blocks_jitc_unit(const BlkTask *__restrict__ tasks, int u, int nbig, int ntask,
                                                 const double *__restrict__ cx, long long cstride, double diag,
                                                 const double *__restrict__ xin, double *__restrict__ arena) {
    __shared__ double lds[H2P_JITC_LDS];
    if (u < nbig) {
        const BlkTask t = tasks[u];
        if (t.flags & H2P_BLK_FAR) jitc_task<4, true>(t, cx, cstride, diag, xin, arena, lds);
        else jitc_task<4, false>(t, cx, cstride, diag, xin, arena, lds);
    } else {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int i = nbig + 4 * (u - nbig) + w;
        if (i >= ntask) return;
        const BlkTask t = tasks[i];
        double *l = lds + w * H2P_JITC_LDS_WAVE;
        if (t.flags & H2P_BLK_FAR) jitc_task<1, true>(t, cx, cstride, diag, xin, arena, l);
        else jitc_task<1, false>(t, cx, cstride, diag, xin, arena, l);
    }
}

// ---------------------------------------------------------------------------
// FP32-mixed scalar kernels (Coulomb, Gaussian, Matern) in the same tiling
// and launch units, with the distances on the VALU from coordinate
// differences (FP32 keeps differences for accuracy, and Coulomb's r = 0 stays
// exact).  Lane l takes column l % 16 of a tile and rows 4 r + l / 16.
// Kernel values and products in FP32; a pass's row sums (up to
// 16 H2P_JITM_NT columns) leave it as FP32 into the FP64 partial outputs;
// each lane's column sums are FP32 over one staged row chunk and are then
// folded into FP64 registers.
struct JitfPt { float x, y, z, v; };   // prepared coordinates and input value

// A workgroup unit's pass covers up to H2P_JITF_NT tiles of 16 columns
// (one source per thread), a wave unit's up to H2P_JITM_NT: the wider pass
// halves the per-column-tile cost of the row reductions and row staging.
// LDS in doubles: workgroup unit rows 2 H2P_JIT_ROWS, sources 2 x 16 NT,
// wave partials 4 x NT x 16; a wave unit 2 H2P_JITW_ROWS + 2 x 16 NT per wave.
#define H2P_JITF_NT 16
#define H2P_JITF_LDS_WG (2 * H2P_JIT_ROWS + 2 * 16 * H2P_JITF_NT + 4 * H2P_JITF_NT * 16)
#define H2P_JITF_LDS_WAVE (2 * H2P_JITW_ROWS + 2 * 16 * H2P_JITM_NT)
#define H2P_JITF_LDS (H2P_JITF_LDS_WG > 4 * H2P_JITF_LDS_WAVE ? H2P_JITF_LDS_WG : 4 * H2P_JITF_LDS_WAVE)

template <int KID, int NT, int NW>
__device__ __forceinline__ void jitf_pass(const BlkTask &t, int pbase, int npts,
                                          const double *__restrict__ cx, long long cstride,
                                          double scale, double diag, double ox, double oy, double oz,
                                          const double *__restrict__ xin, double *__restrict__ arena,
                                          JitfPt *rows, JitfPt *srcs, double *red, bool first) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS;
    const int lane = threadIdx.x & 63, w = NW == 4 ? (threadIdx.x >> 6) : 0;
    const int tid = NW == 4 ? threadIdx.x : lane;
    const int li = lane & 15, lg = lane >> 4;
    const double *cy = cx + cstride, *cz = cx + 2 * cstride;
    const float dg = (float)diag;
    for (int q = tid; q < NT * 16; q += NW * H2P_WAVE) {
        const bool ok = q < npts;
        const int g = t.c1 + pbase + (ok ? q : 0);
        JitfPt e;
        e.x = (float)((cx[g] - ox) * scale);
        e.y = (float)((cy[g] - oy) * scale);
        e.z = (float)((cz[g] - oz) * scale);
        e.v = ok ? (float)xin[t.in0 + pbase + q] : 0.0f;
        srcs[q] = e;
    }
    float acc[NT];
#pragma unroll
    for (int c = 0; c < NT; c++) acc[c] = 0.0f;
    const bool has1 = t.flags & 1;
    for (int rc = 0; rc < t.n0; rc += ROWS) {
        const int nr = min(t.n0 - rc, ROWS);
        const int ntile = (nr + 15) >> 4;
        jitm_sync<NW>();
        for (int q = tid; q < ntile * 16; q += NW * H2P_WAVE) {
            const bool ok = q < nr;
            const int g = t.c0 + rc + (ok ? q : 0);
            JitfPt e;
            e.x = (float)((cx[g] - ox) * scale);
            e.y = (float)((cy[g] - oy) * scale);
            e.z = (float)((cz[g] - oz) * scale);
            e.v = (ok && has1) ? (float)xin[t.in1 + rc + q] : 0.0f;
            rows[q] = e;
        }
        jitm_sync<NW>();
        for (int tt = w; tt < ntile; tt += NW) {
            float rx[4], ry[4], rz[4], rv[4], p[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const JitfPt e = rows[tt * 16 + 4 * r + lg];
                rx[r] = e.x;
                ry[r] = e.y;
                rz[r] = e.z;
                rv[r] = e.v;
                p[r] = 0.0f;
            }
            // one column tile at a time (the barriers bound the registers
            // the scheduler may spend on interleaving tiles)
            auto tile = [&](auto nrq) {
                constexpr int NR = decltype(nrq)::value;
#pragma unroll
                for (int c = 0; c < NT; c++) {
                    const JitfPt e = srcs[c * 16 + li];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const float dx = rx[r] - e.x, dy = ry[r] - e.y, dz = rz[r] - e.z;
                        const float kv = kprep<KID>(dx * dx + dy * dy + dz * dz, dg);
                        p[r] += kv * e.v;
                        acc[c] += kv * rv[r];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            tile_rows(nr - tt * 16, tile);
            const float s = group16_sum4(p[0], p[1], p[2], p[3]);
            const int myrow = tt * 16 + 4 * ((lane >> 2) & 3) + lg;
            if ((lane & 3) == 0 && myrow < nr) {
                double *o = arena + t.out0 + rc + myrow;
                if (first) *o = (double)s;
                else *o += (double)s;
            }
        }
        if (has1) {
            // the chunk's FP32 column sums in FP64, (g0 + g1) + (g2 + g3)
            // over the four lane groups, added in chunk order to the wave's
            // sums (in LDS for a workgroup unit, in the output for a wave unit)
#pragma unroll
            for (int c = 0; c < NT; c++) {
                double v = (double)acc[c];
                v += __shfl_xor(v, 16, H2P_WAVE);
                v += __shfl_xor(v, 32, H2P_WAVE);
                acc[c] = 0.0f;
                const int j = c * 16 + li;
                double *o = NW == 4 ? red + (w * NT + c) * 16 + li : arena + t.out1 + pbase + j;
                if (lg == 0 && (NW == 4 || j < npts)) *o = rc == 0 ? v : *o + v;
            }
        }
    }
    if (!has1) return;
    if constexpr (NW == 4) {   // the four waves in order
        __syncthreads();
        for (int j = threadIdx.x; j < npts; j += blockDim.x) {
            const int c = j >> 4, m = j & 15;
            double s = red[c * 16 + m];
#pragma unroll
            for (int w2 = 1; w2 < 4; w2++) s += red[(w2 * NT + c) * 16 + m];
            arena[t.out1 + pbase + j] = s;
        }
    }
}

template <int KID, int NW>
__device__ __forceinline__ void jitf_task(const BlkTask &t, const double *__restrict__ cx,
                                          long long cstride, double scale, double diag,
                                          const double *__restrict__ xin, double *__restrict__ arena,
                                          double *lds) {
    constexpr int ROWS = NW == 4 ? H2P_JIT_ROWS : H2P_JITW_ROWS;
    constexpr int NTX = NW == 4 ? H2P_JITF_NT : H2P_JITM_NT;
    JitfPt *rows = (JitfPt *)lds;
    JitfPt *srcs = (JitfPt *)(lds + 2 * ROWS);
    double *red = lds + 2 * ROWS + 2 * 16 * NTX;   // workgroup unit only
    const double ox = cx[t.c0], oy = cx[cstride + t.c0], oz = cx[2 * cstride + t.c0];
    for (int pb = 0; pb < t.n1; pb += NTX * 16) {
        const int np = min(t.n1 - pb, NTX * 16);
        const bool first = (pb == 0);
        const int nt = (np + 15) >> 4;
#define H2P_JITF_CASE(n) \
            case n: jitf_pass<KID, n, NW>(t, pb, np, cx, cstride, scale, diag, ox, oy, oz, xin, arena, rows, srcs, red, first); break;
        if constexpr (NW == 4) {
            switch (nt) {
                H2P_JITF_CASE(1) H2P_JITF_CASE(2) H2P_JITF_CASE(3) H2P_JITF_CASE(4)
                H2P_JITF_CASE(5) H2P_JITF_CASE(6) H2P_JITF_CASE(7) H2P_JITF_CASE(8)
                H2P_JITF_CASE(9) H2P_JITF_CASE(10) H2P_JITF_CASE(11) H2P_JITF_CASE(12)
                H2P_JITF_CASE(13) H2P_JITF_CASE(14) H2P_JITF_CASE(15) H2P_JITF_CASE(16)
                default: break;
            }
        } else {
            switch (nt) {
                H2P_JITF_CASE(1) H2P_JITF_CASE(2) H2P_JITF_CASE(3) H2P_JITF_CASE(4)
                H2P_JITF_CASE(5) H2P_JITF_CASE(6) H2P_JITF_CASE(7) H2P_JITF_CASE(8)
                default: break;
            }
        }
#undef H2P_JITF_CASE
        jitm_sync<NW>();
    }
}

template <int KID>
__device__ __forceinline__ void blocks_jitf_unit(const BlkTask *__restrict__ tasks, int u, int nbig, int ntask,
                                                 const double *__restrict__ cx, long long cstride,
                                                 double scale, double diag, const double *__restrict__ xin,
                                                 double *__restrict__ arena) {
    __shared__ double lds[H2P_JITF_LDS];
    if (u < nbig) {
        jitf_task<KID, 4>(tasks[u], cx, cstride, scale, diag, xin, arena, lds);
    } else {
        const int w = threadIdx.x >> 6;
        const int i = nbig + 4 * (u - nbig) + w;
        if (i < ntask)
            jitf_task<KID, 1>(tasks[i], cx, cstride, scale, diag, xin, arena, lds + w * H2P_JITF_LDS_WAVE);
    }
}

// Whether a task of the tiled launches runs as a wave unit.
__host__ __device__ inline bool jitm_wave_task(int n0, int n1) {
    return n0 <= H2P_JITW_ROWS && n1 <= 16 * H2P_JITM_NT;
}

// Launch unit u of the grouped kernel-evaluating launch.
template <int KID, typename T>
__device__ __forceinline__ void blocks_jit2_unit(const BlkTask *__restrict__ tasks, int u, int nbig, int ntask,
                                                 const double *__restrict__ cx, long long cstride,
                                                 double scale, double diag, const double *__restrict__ xin,
                                                 double *__restrict__ arena) {
    if constexpr (sizeof(T) == 4) {
        blocks_jitf_unit<KID>(tasks, u, nbig, ntask, cx, cstride, scale, diag, xin, arena);
    } else if constexpr (KID == KG || KID == KM) {
        blocks_jitm_unit<KID>(tasks, u, nbig, ntask, cx, cstride, scale, xin, arena);
    } else {
        static_assert(KID == KC, "scalar kernels only");
        blocks_jitc_unit(tasks, u, nbig, ntask, cx, cstride, diag, xin, arena);
    }
}

// Occupancy build of the grouped launch: the same body compiled for at
// least WPE waves per SIMD, so with fewer registers per lane.  Same
// arithmetic, same results.  PART (0: B blocks, 1: D blocks) only names the
// launch, so that the two launches of a matvec are told apart in profiles.
template <int KID, typename T, int WPE, int PART>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_blocks_jit2_occ(const BlkTask *__restrict__ tasks, int nbig, int ntask, const double *__restrict__ cx,
                  long long cstride, double scale, double diag, const double *__restrict__ xin,
                  double *__restrict__ arena) {
    blocks_jit2_unit<KID, T>(tasks, blockIdx.x, nbig, ntask, cx, cstride, scale, diag, xin, arena);
}

template <typename TS, int WPE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_blocks_aot_occ(const BlkTask *__restrict__ tasks, const TS *__restrict__ blob,
                 const double *__restrict__ xin, double *__restrict__ arena) {
    blocks_aot_body<TS>(tasks[blockIdx.x], blob, xin, arena);
}

template <int KID, typename T, int PART>
__global__ void __launch_bounds__(256) k_blocks_jit2(const BlkTask *__restrict__ tasks, int nbig, int ntask,
                                                     const double *__restrict__ cx,
                                                     long long cstride, double scale, double diag,
                                                     const double *__restrict__ xin,
                                                     double *__restrict__ arena) {
    blocks_jit2_unit<KID, T>(tasks, blockIdx.x, nbig, ntask, cx, cstride, scale, diag, xin, arena);
}

// ---------------------------------------------------------------------------
// Device-side evaluation of AOT blocks (H2P_build_B_AOT / H2P_build_D_AOT,
// src/H2Pack_build.c:789-889, 1034-1140): one workgroup per block, threads
// over the row-major entries.
template <int KID, int KD, typename TS>
__global__ void __launch_bounds__(256) k_build_blocks(const BlkTask *__restrict__ tasks,
                                                      const double *__restrict__ cx,
                                                      long long cstride, KParam kp,
                                                      TS *__restrict__ blob) {
    // values are evaluated in FP64 and stored as TS
    const BlkTask t = tasks[blockIdx.x];
    const double *cy = cx + cstride, *cz = cx + 2 * cstride, *ca = cx + 3 * cstride;
    TS *A = blob + t.data_off;
    const long long total = (long long)t.n0 * t.n1;
    for (long long e = threadIdx.x; e < total; e += blockDim.x) {
        int i = (int)(e / t.n1), j = (int)(e - (long long)i * t.n1);
        int gi = t.c0 + i, gj = t.c1 + j;
        double dx = cx[gi] - cx[gj], dy = cy[gi] - cy[gj], dz = cz[gi] - cz[gj];
        if constexpr (KD == 1) {
            A[e] = (TS)kval<KID>(dx * dx + dy * dy + dz * dz, kp);
        } else {
            double t1, t2, ux, uy, uz;
            rpy_coef(dx, dy, dz, ca[gi], ca[gj], kp.p1, t1, t2, ux, uy, uz);
            double u[3] = {ux, uy, uz};
            const long long ld = (long long)t.n1 * 3;
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
                for (int b = 0; b < 3; b++)
                    A[(long long)(3 * i + a) * ld + 3 * j + b] = (TS)(t2 * u[a] * u[b] + (a == b ? t1 : 0.0));
        }
    }
}

// ---------------------------------------------------------------------------
// Direct FP64 n-body rows (examples/direct_nbody.h): grid = (target blocks of
// 256, source chunks); partial sums per chunk, reduced in a fixed order.
template <int KID, int KD>
__global__ void __launch_bounds__(256) k_nbody_partial(const double *__restrict__ src, long long sld, int n_src,
                                                       const double *__restrict__ x,
                                                       const double *__restrict__ dst, long long dld, int n_dst,
                                                       KParam kp, int chunk, double *__restrict__ part) {
    __shared__ double s[4][256];
    __shared__ double sxv[3][256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int js = blockIdx.y * chunk, je = min(n_src, js + chunk);
    double tx = 0, ty = 0, tz = 0, ta = 0;
    if (i < n_dst) {
        tx = dst[i]; ty = dst[dld + i]; tz = dst[2 * dld + i];
        if constexpr (KD == 3) ta = dst[3 * dld + i];
    }
    double acc[KD];
#pragma unroll
    for (int a = 0; a < KD; a++) acc[a] = 0.0;
    for (int j0 = js; j0 < je; j0 += 256) {
        int j = j0 + threadIdx.x;
        __syncthreads();
        if (j < je) {
            s[0][threadIdx.x] = src[j]; s[1][threadIdx.x] = src[sld + j]; s[2][threadIdx.x] = src[2 * sld + j];
            if constexpr (KD == 3) s[3][threadIdx.x] = src[3 * sld + j];
#pragma unroll
            for (int b = 0; b < KD; b++) sxv[b][threadIdx.x] = x[(long long)j * KD + b];
        }
        __syncthreads();
        int n = min(256, je - j0);
        for (int q = 0; q < n; q++) {
            double dx = tx - s[0][q], dy = ty - s[1][q], dz = tz - s[2][q];
            if constexpr (KD == 1) {
                acc[0] += kval<KID>(dx * dx + dy * dy + dz * dz, kp) * sxv[0][q];
            } else {
                double t1, t2, ux, uy, uz;
                rpy_coef(dx, dy, dz, ta, s[3][q], kp.p1, t1, t2, ux, uy, uz);
                double ud = ux * sxv[0][q] + uy * sxv[1][q] + uz * sxv[2][q];
                acc[0] += t1 * sxv[0][q] + t2 * ux * ud;
                acc[1] += t1 * sxv[1][q] + t2 * uy * ud;
                acc[2] += t1 * sxv[2][q] + t2 * uz * ud;
            }
        }
    }
    if (i < n_dst)
#pragma unroll
        for (int a = 0; a < KD; a++) part[((long long)blockIdx.y * n_dst + i) * KD + a] = acc[a];
}

__global__ void k_nbody_reduce(const double *__restrict__ part, int nchunk, int len,
                               double *__restrict__ y) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= len) return;
    double s = 0.0;
    for (int c = 0; c < nchunk; c++) s += part[(long long)c * len + e];
    y[e] = s;
}

}  // namespace h2p
