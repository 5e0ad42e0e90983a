// Multi-RHS H2 product (H2P_matmul, src/H2Pack_matmul.c:455-583) on MFMA.
//
// Every phase of the matmul is a list of tasks of one form,
//     dst (M x nv)  (+)=  sum_s  op(A_s) (M x K_s) * X_s (K_s x nv),
// evaluated in the pull formulation of H2P_matmul_intmd_mult /
// H2P_matmul_dense_mult (one task per destination, each source block applied
// to the destination side only), so every output row has one writer and no
// partial buffers are needed:
//   upward   : Y0[node]      = U^T[node] * (PX[leaf rows] | Y0[children])
//   coupling : Y1[node]      = sum op(B) * (Y0[other] | PX[other leaf rows])
//   downward : Y1[children] += U[node] * Y1[node]           (level by level)
//   leaves   : PY[leaf rows] = U[leaf] * Y1[leaf] + sum op(D) * PX + sum op(B) * Y0
// A_s is a dense block (U, U^T, or a stored B/D block, transposed for the
// negative entries of the pair-to-block CSR) or, in JIT mode, kernel values:
// the kernels are symmetric, so op(B) = K(dst set, src set).  Panels are
// row-major with a row length of nvp (vectors padded to a multiple of 16).
//
// Work split.  A destination is cut into tasks of MM_PIECE (32) rows, or 16
// points = 48 rows for the evaluated 3x3 kernel; the four waves of a
// workgroup share a task's rows and deal its inner entries round-robin in
// chunks of 16 (4 points for the 3x3 kernel), and their four accumulator
// sets are added in wave order at the end.  So a wave needs nothing from the
// others before that: no barrier and no LDS staging in the inner loop, and
// a task's longest chain is a quarter of its sources.
//
// Operands stay in registers.  v_mfma_f64_16x16x4f64: lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and receives D[4 r + l / 16][l % 16]
// in register r.  Four such products consume 16 inner entries, and any
// assignment of the 16 entries to (step, lane group) does, as long as A and X
// use the same one:
//   dense A    : step r, lane group g take entry 4 g + r, so a lane reads 32
//                consecutive bytes of its row (transposed blocks: each step
//                reads 16 consecutive rows' entries, 128 bytes per group);
//   evaluated A: step r, lane group g take entry 4 r + g.  A lane evaluates
//                source 4 r + g against destination l % 16 for r = 0 .. 3,
//                the A operands of the four steps: kernel values go from the
//                evaluation into the product without leaving the lane.
#pragma once
#include "h2p_device.h"

namespace h2p {

enum { MM_PX = 0, MM_Y0 = 1, MM_Y1 = 2, MM_PY = 3 };
enum { MM_A_U = 0, MM_A_UT = 1, MM_A_BD = 2, MM_A_JIT = 3 };

#define H2P_MM_MAXNVP 64
#define H2P_MM_NVARIANT 4      // accepted; only bit 0 (the task order) has an effect
#define H2P_MM_PIECE 32       // rows of a task
#define H2P_MM_PIECE3 48      // rows of a task with evaluated 3x3 blocks

// One source block of a destination (shared by the destination's tasks).
struct MMSrc {
    long long a_off;   // dense: element offset of op(A)'s first row in its blob
    int kind;          // MM_A_*
    int trans;         // dense: op(A) = A^T
    int lda;           // dense: row length of the stored A
    int K;             // inner dimension (vector entries)
    int c1;            // JIT: first source point (unified coordinates)
    int x_space, x_off;
    int shift;         // JIT: shift-table entry added to the source points (periodic images)
};

// M destination rows from row m0 of a destination; its sources in
// [sbeg, smid) are dense, those in [smid, send) evaluated.
struct MMTask {
    int dst_space, dst_off, M, accumulate;
    int sbeg, smid, send;
    int m0;            // first row within the destination (dense sources' row offset)
    int c0;            // JIT: first destination point of this task (unified coordinates)
    int pad;
};

struct MMPanels {
    double *p[4];      // PX, Y0, Y1, PY
    int nvp;           // padded row length
};

// the operands of a launch beside its tasks
struct MMArgs {
    const MMSrc *srcs;
    const double *U, *UT;
    const void *BD;            // stored blocks (double, or float for the FP32 products)
    const double *cx;          // unified coordinates, one row per dimension
    long long cstride;
    const double *shifts;
    double scale;              // the FP64 kernels' factor (kmm_scale)
    KParam kp;
    MMPanels P;
};

// x x + y y + z z with its roundings fixed, so that every kernel that forms a
// kernel value gets the same bits
__device__ __forceinline__ double mm_sq3(double x, double y, double z) {
    return __builtin_fma(z, z, __builtin_fma(x, x, y * y));
}

typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// Walks the chunks of a source list that belong to one wave: chunk indices
// run through the sources one after the other and wave w takes w, w + 4, ...
// All members are the same on every lane.
template <int CH>
struct MMCursor {
    int si, c, nch, send;
    MMSrc s;
    __device__ __forceinline__ void settle(const MMSrc *__restrict__ srcs) {
        while (c >= nch) {
            c -= nch;
            if (++si >= send) return;
            s = srcs[si];
            nch = (s.K + CH - 1) / CH;
        }
    }
    __device__ __forceinline__ void start(const MMSrc *__restrict__ srcs, int beg, int end, int w) {
        si = beg;
        send = end;
        c = w;
        nch = 0;
        if (si < send) {
            s = srcs[si];
            nch = (s.K + CH - 1) / CH;
            settle(srcs);
        }
    }
    __device__ __forceinline__ bool live() const { return si < send; }
    __device__ __forceinline__ void next(const MMSrc *__restrict__ srcs) {
        c += 4;
        settle(srcs);
    }
};

// Destination row of entry `lane row` i of tile t: consecutive rows, or for
// the 3x3 kernel one tensor component of 16 points per tile.
template <bool ROW3>
__device__ __forceinline__ int mm_row(int t, int i) {
    return ROW3 ? 3 * i + t : 16 * t + i;
}

// A operand of one 16-entry chunk of a dense source: a[t][r] = op(A)[row][kc + 4 lg + r],
// rows past the task's last repeat it, entries past K repeat the last.
template <int MT, bool ROW3>
__device__ __forceinline__ void mm_load_a(const double *__restrict__ blob, const MMSrc &s, int m0, int M, int kc,
                                          int li, int lg, double (*a)[4]) {
    const bool full = kc + 16 <= s.K;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int row = m0 + min(mm_row<ROW3>(t, li), M - 1);
        if (!s.trans) {
            const double *p = blob + s.a_off + (long long)row * s.lda + kc + 4 * lg;
            if (full) {
                const d2u u = *(const d2u *)p, v = *(const d2u *)(p + 2);
                a[t][0] = u.x;
                a[t][1] = u.y;
                a[t][2] = v.x;
                a[t][3] = v.y;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) a[t][r] = p[min(4 * lg + r, s.K - 1 - kc) - 4 * lg];
            }
        } else {
            const double *p = blob + s.a_off + row;
#pragma unroll
            for (int r = 0; r < 4; r++) a[t][r] = p[(long long)min(kc + 4 * lg + r, s.K - 1) * s.lda];
        }
    }
}

// X operand rows: x[r][n] = X[row(r)][16 n + li] with row(r) = kc + k0 + kr r,
// zero past K.  NT column tiles of the panel are live (GUARD: fewer than
// NVT may be).
template <int NVT, bool GUARD>
__device__ __forceinline__ void mm_load_x(const double *__restrict__ X, int nvp, int nt, int K, int kc, int k0, int kr,
                                          int li, double (*x)[NVT]) {
    const bool full = kc + 16 <= K;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int k = kc + k0 + kr * r;
        const double *p = X + (long long)(full ? k : min(k, K - 1)) * nvp + li;
#pragma unroll
        for (int n = 0; n < NVT; n++) {
            if (GUARD && n >= nt) continue;
            const double v = p[16 * n];
            x[r][n] = (full || k < K) ? v : 0.0;
        }
    }
}

// The dense sources [sbeg, send) of a task: a software pipeline over the
// wave's chunks, the next chunk's operands in flight during the products.
template <int MT, bool ROW3, int NVT, bool GUARD>
__device__ __forceinline__ void mm_dense(const MMTask &t, int sbeg, int send, const MMArgs &A, int nt, int w, int li,
                                         int lg, d4 (*acc)[NVT]) {
    MMCursor<16> cu;
    cu.start(A.srcs, sbeg, send, w);
    if (!cu.live()) return;
    double a[MT][4], x[4][NVT];
    auto fetch = [&](const MMSrc &s, int c) {
        const double *blob = s.kind == MM_A_U ? A.U : s.kind == MM_A_UT ? A.UT : (const double *)A.BD;
        mm_load_a<MT, ROW3>(blob, s, t.m0, t.M, 16 * c, li, lg, a);
        const double *X = A.P.p[s.x_space] + (long long)s.x_off * A.P.nvp;
        mm_load_x<NVT, GUARD>(X, A.P.nvp, nt, s.K, 16 * c, 4 * lg, 1, li, x);
    };
    fetch(cu.s, cu.c);
    while (cu.live()) {
        double a0[MT][4], x0[4][NVT];
#pragma unroll
        for (int q = 0; q < MT; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) a0[q][r] = a[q][r];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int n = 0; n < NVT; n++) x0[r][n] = x[r][n];
        cu.next(A.srcs);
        if (cu.live()) fetch(cu.s, cu.c);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int n = 0; n < NVT; n++) {
                if (GUARD && n >= nt) continue;
#pragma unroll
                for (int q = 0; q < MT; q++)
                    acc[q][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[q][r], x0[r][n], acc[q][n], 0, 0, 0);
            }
    }
}

// The evaluated sources of a task, scalar kernels: 16 sources x 32
// destinations per chunk, kernel values straight into the products.  The
// distances are coordinate differences on the VALU (6 operations a pair): a
// leaf or a skeleton can hold points far apart, and |r|^2 + |s|^2 - 2 r.s,
// one matrix product for the tile, is off by the square of its extent
// (times 2^-53): two groups of a leaf 8e4 lengthscales apart gave products off
// by 1e-7, now 1e-15, and 7.6e-15 -> 5.0e-16 for Matern points in a cube of
// side 10 (l = 2).  us per product, squares -> differences: Gaussian
// N = 40k x16 1153 -> 1296, N = 17k x64 959 -> 1035; Matern 1383 -> 1556 and
// 960 -> 1029.
template <int KID, int NVT, bool GUARD>
__device__ __forceinline__ void mm_jit1(const MMTask &t, const MMArgs &A, int nt, int w, int li, int lg,
                                        const double *e2t, d4 (*acc)[NVT]) {
    const double *cx = A.cx, *cy = A.cx + A.cstride, *cz = A.cx + 2 * A.cstride;
    const double scale = A.scale, diag = A.kp.p0;
    MMCursor<16> cu;
    cu.start(A.srcs, t.smid, t.send, w);
    if (!cu.live()) return;
    // destinations of the two tiles: point 16 q + li
    double dx[2], dy[2], dz[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int g = t.c0 + min(16 * q + li, t.M - 1);
        dx[q] = cx[g];
        dy[q] = cy[g];
        dz[q] = cz[g];
    }
    // sources of a chunk: points 4 r + lg
    double sx[4], sy[4], sz[4];
    auto fetch = [&](const MMSrc &s, int c) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int g = s.c1 + min(16 * c + 4 * r + lg, s.K - 1);
            sx[r] = cx[g];
            sy[r] = cy[g];
            sz[r] = cz[g];
        }
    };
    fetch(cu.s, cu.c);
    const bool two = t.M > 16;
    while (cu.live()) {
        double x[4][NVT];
        mm_load_x<NVT, GUARD>(A.P.p[cu.s.x_space] + (long long)cu.s.x_off * A.P.nvp, A.P.nvp, nt, cu.s.K, 16 * cu.c,
                              lg, 4, li, x);
        double px[4], py[4], pz[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            px[r] = sx[r];
            py[r] = sy[r];
            pz[r] = sz[r];
        }
        cu.next(A.srcs);
        if (cu.live()) fetch(cu.s, cu.c);
        auto tile = [&](int q) {
            double kv[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const double ex = dx[q] - px[r], ey = dy[q] - py[r], ez = dz[q] - pz[r];
                kv[r] = kmm<KID>(mm_sq3(ex, ey, ez), scale, diag, e2t);
            }
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int n = 0; n < NVT; n++) {
                    if (GUARD && n >= nt) continue;
                    acc[q][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv[r], x[r][n], acc[q][n], 0, 0, 0);
                }
        };
        tile(0);
        if (two) tile(1);
    }
}

// The evaluated sources of a task, 3x3 kernel: 4 source points x 16
// destination points per chunk.  Lane l evaluates the pair (destination
// l % 16, source l / 16) once; its six distinct tensor entries are the A
// operands of nine products, one per component pair.
template <int NVT, bool GUARD>
__device__ __forceinline__ void mm_jit3(const MMTask &t, const MMArgs &A, int nt, int w, int li, int lg,
                                        d4 (*acc)[NVT]) {
    const double *cx = A.cx;
    const long long cs = A.cstride;
    MMCursor<12> cu;
    cu.start(A.srcs, t.smid, t.send, w);
    if (!cu.live()) return;
    double d[5], sp[5];
    {
        const int g = t.c0 + min(li, t.M / 3 - 1);
#pragma unroll
        for (int k = 0; k < 5; k++) d[k] = cx[k * cs + g];
    }
    auto fetch = [&](const MMSrc &s, int c) {
        const int g = s.c1 + min(4 * c + lg, s.K / 3 - 1);
#pragma unroll
        for (int k = 0; k < 5; k++) sp[k] = cx[k * cs + g];
#pragma unroll
        for (int k = 0; k < 3; k++) sp[k] += A.shifts[3 * s.shift + k];
    };
    fetch(cu.s, cu.c);
    while (cu.live()) {
        double x[3][NVT];
        {
            const int np = cu.s.K / 3, p = 4 * cu.c + lg;
            const double *X = A.P.p[cu.s.x_space] + (long long)(cu.s.x_off + 3 * min(p, np - 1)) * A.P.nvp + li;
#pragma unroll
            for (int b = 0; b < 3; b++)
#pragma unroll
                for (int n = 0; n < NVT; n++) {
                    if (GUARD && n >= nt) continue;
                    const double v = X[(long long)b * A.P.nvp + 16 * n];
                    x[b][n] = p < np ? v : 0.0;
                }
        }
        const double ex = d[0] - sp[0], ey = d[1] - sp[1], ez = d[2] - sp[2], ra = sp[3], rb = sp[4];
        cu.next(A.srcs);
        if (cu.live()) fetch(cu.s, cu.c);
        double t1, t2, ux, uy, uz;
        rpy_coef_rcp(ex, ey, ez, d[3], ra, d[4], rb, A.kp.p1, t1, t2, ux, uy, uz);
        const double gx = t2 * ux, gy = t2 * uy, gz = t2 * uz;
        const double kxx = gx * ux + t1, kxy = gx * uy, kxz = gx * uz, kyy = gy * uy + t1, kyz = gy * uz,
                     kzz = gz * uz + t1;
        const double k3[3][3] = {{kxx, kxy, kxz}, {kxy, kyy, kyz}, {kxz, kyz, kzz}};
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int n = 0; n < NVT; n++) {
                if (GUARD && n >= nt) continue;
#pragma unroll
                for (int a = 0; a < 3; a++)
                    acc[a][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(k3[a][b], x[b][n], acc[a][n], 0, 0, 0);
            }
    }
}

// Adds the four waves' accumulators in wave order, a column tile at a time
// through LDS (3 MT x 256 doubles), and writes the task's rows.
template <int MT, bool ROW3, int NVT, bool GUARD>
__device__ __forceinline__ void mm_finish(const MMTask &t, const MMPanels &P, int nt, int w, int lane, d4 (*acc)[NVT],
                                          d4 *lds) {
    double *dst = P.p[t.dst_space] + (long long)t.dst_off * P.nvp;
    const int li = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int n = 0; n < NVT; n++) {
        if (GUARD && n >= nt) continue;
        if (n > 0) __syncthreads();
        if (w > 0)
#pragma unroll
            for (int q = 0; q < MT; q++) lds[((w - 1) * MT + q) * H2P_WAVE + lane] = acc[q][n];
        __syncthreads();
        if (w > 0) continue;
#pragma unroll
        for (int q = 0; q < MT; q++) {
            d4 v = acc[q][n];
#pragma unroll
            for (int k = 0; k < 3; k++) v += lds[(k * MT + q) * H2P_WAVE + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mm_row<ROW3>(q, 4 * r + lg);
                if (m < t.M) {
                    double *o = dst + (long long)m * P.nvp + 16 * n + li;
                    *o = t.accumulate ? *o + v[r] : v[r];
                }
            }
        }
    }
}

// Dense tasks (U phases, stored blocks).
template <int NVT, bool GUARD>
__device__ __forceinline__ void mmd_body(const MMTask &t, const MMArgs &A) {
    __shared__ d4 lds[3 * 2 * H2P_WAVE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nt = GUARD ? A.P.nvp >> 4 : NVT;
    d4 acc[2][NVT];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int n = 0; n < NVT; n++) acc[q][n] = (d4){0.0, 0.0, 0.0, 0.0};
    mm_dense<2, false, NVT, GUARD>(t, t.sbeg, t.smid, A, nt, w, lane & 15, lane >> 4, acc);
    mm_finish<2, false, NVT, GUARD>(t, A.P, nt, w, lane, acc, lds);
}

// Tasks with evaluated sources (after any dense ones).
template <int KID, int NVT, bool GUARD>
__device__ __forceinline__ void mmj_body(const MMTask &t, const MMArgs &A) {
    constexpr bool R3 = KID == KR;
    constexpr int MT = R3 ? 3 : 2;
    __shared__ d4 lds[3 * MT * H2P_WAVE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nt = GUARD ? A.P.nvp >> 4 : NVT;
    d4 acc[MT][NVT];
#pragma unroll
    for (int q = 0; q < MT; q++)
#pragma unroll
        for (int n = 0; n < NVT; n++) acc[q][n] = (d4){0.0, 0.0, 0.0, 0.0};
    if (t.smid > t.sbeg) mm_dense<MT, R3, NVT, GUARD>(t, t.sbeg, t.smid, A, nt, w, lane & 15, lane >> 4, acc);
    if constexpr (R3) {
        mm_jit3<NVT, GUARD>(t, A, nt, w, lane & 15, lane >> 4, acc);
    } else if constexpr (KID == KC) {
        mm_jit1<KID, NVT, GUARD>(t, A, nt, w, lane & 15, lane >> 4, nullptr, acc);
    } else {
        __shared__ double e2t[H2P_E2_N];
        if (threadIdx.x < H2P_E2_N) e2t[threadIdx.x] = c_e2tab[threadIdx.x];
        __syncthreads();
        mm_jit1<KID, NVT, GUARD>(t, A, nt, w, lane & 15, lane >> 4, e2t, acc);
    }
    mm_finish<MT, R3, NVT, GUARD>(t, A.P, nt, w, lane, acc, lds);
}

// ---------------------------------------------------------------------------
// FP32-mixed products (handles of precision FP32MIX): the B and D sources
// -- kernel values evaluated in FP32 (JIT: the FP64 coordinate difference and
// squared distance rounded once to FP32, then the hardware exp2 / rsqrt as
// in the FP32-mixed matvec) or blocks stored in FP32 (AOT) -- and their
// operand rows rounded to FP32 run on v_mfma_f32_16x16x4f32; the FP32 tile
// sums of every 16 inner entries (four products, counted from the start of
// each source) are folded into FP64 accumulators, and the output panels
// stay FP64.  The U phases keep the FP64 kernel.  Only B/D sources reach
// this kernel (the host splits the leaf tasks into a U part and a B/D part).
//
// Lane layouts: v_mfma_f32_16x16x4f32 takes A[l % 16][l / 16] and
// B[l / 16][l % 16] like the FP64 product, but returns D[4 (l / 16) + r]
// [l % 16] in register r, where the FP64 product returns row 4 r + l / 16.
// Feeding the A rows in the order sigma(4 a + b) = 4 b + a makes the FP32
// tile land in the FP64 accumulator layout, so the fold is lane-local.
// Inner entry of step r, lane group g: 4 r + g for both kinds of source.
__device__ __forceinline__ int mm32_sigma(int i) { return 4 * (i & 3) + (i >> 2); }

template <int KID, int NVT, bool GUARD>
__device__ __forceinline__ void mm32_body(const MMTask &t, const MMArgs &A) {
    __shared__ d4 lds[3 * 2 * H2P_WAVE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4, ls = mm32_sigma(li);
    const int nt = GUARD ? A.P.nvp >> 4 : NVT;
    d4 acc[2][NVT];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int n = 0; n < NVT; n++) acc[q][n] = (d4){0.0, 0.0, 0.0, 0.0};
    const double *cx = A.cx, *cy = A.cx + A.cstride, *cz = A.cx + 2 * A.cstride;
    const float p0 = (float)A.kp.p0;
    const bool two = t.M > 16;
    MMCursor<16> cu;
    cu.start(A.srcs, t.sbeg, t.send, w);
    // the next chunk's coordinates (JIT, KID >= 0) or block entries (KID < 0)
    double dx[2], dy[2], dz[2], sx[4], sy[4], sz[4];
    float a[2][4];
    auto fetch = [&](const MMSrc &s, int c) {
        if constexpr (KID >= 0) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int g = s.c1 + min(16 * c + 4 * r + lg, s.K - 1);
                sx[r] = cx[g];
                sy[r] = cy[g];
                sz[r] = cz[g];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int row = t.m0 + min(16 * q + ls, t.M - 1);
                const float *p = (const float *)A.BD + s.a_off;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int k = min(16 * c + 4 * r + lg, s.K - 1);
                    a[q][r] = s.trans ? p[(long long)k * s.lda + row] : p[(long long)row * s.lda + k];
                }
            }
        }
    };
    if constexpr (KID >= 0) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int g = t.c0 + min(16 * q + ls, t.M - 1);
            dx[q] = cx[g];
            dy[q] = cy[g];
            dz[q] = cz[g];
        }
    }
    if (cu.live()) fetch(cu.s, cu.c);
    while (cu.live()) {
        double xd[4][NVT];
        mm_load_x<NVT, GUARD>(A.P.p[cu.s.x_space] + (long long)cu.s.x_off * A.P.nvp, A.P.nvp, nt, cu.s.K, 16 * cu.c,
                              lg, 4, li, xd);
        double px[4], py[4], pz[4];
        float a0[2][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if constexpr (KID >= 0) {
                px[r] = sx[r];
                py[r] = sy[r];
                pz[r] = sz[r];
            } else {
                a0[0][r] = a[0][r];
                a0[1][r] = a[1][r];
            }
        }
        cu.next(A.srcs);
        if (cu.live()) fetch(cu.s, cu.c);
        float x[4][NVT];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int n = 0; n < NVT; n++) {
                if (GUARD && n >= nt) continue;
                x[r][n] = (float)xd[r][n];
            }
        auto tile = [&](int q) {
            float kv[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if constexpr (KID >= 0) {
                    const double ex = dx[q] - px[r], ey = dy[q] - py[r], ez = dz[q] - pz[r];
                    const double r2 = mm_sq3(ex, ey, ez);
                    kv[r] = kvalf<KID>((float)r2, p0);
                } else {
                    kv[r] = a0[q][r];
                }
            }
#pragma unroll
            for (int n = 0; n < NVT; n++) {
                if (GUARD && n >= nt) continue;
                f4 a32 = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int r = 0; r < 4; r++) a32 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[r], x[r][n], a32, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[q][n][r] += (double)a32[r];
            }
        };
        tile(0);
        if (two) tile(1);
    }
    mm_finish<2, false, NVT, GUARD>(t, A.P, nt, w, lane, acc, lds);
}

template <int NVT>
__global__ void __launch_bounds__(256) k_mmd(const MMTask *__restrict__ tasks, MMArgs A) {
    mmd_body<NVT, false>(tasks[blockIdx.x], A);
}

template <int KID, int NVT>
__global__ void __launch_bounds__(256) k_mmj(const MMTask *__restrict__ tasks, MMArgs A) {
    mmj_body<KID, NVT, false>(tasks[blockIdx.x], A);
}

// One column tile: 104 VGPRs by the compiler's own choice (4 waves per SIMD);
// five waves hide the operand loads better (Matern N = 105k x8: 3.90 -> 3.80
// ms).  Asking for a wave more of the wider or the FP64 builds spills and
// measured slower (Coulomb N = 80k x20 2.52 -> 4.89 ms).
template <int KID, int NVT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NVT == 1 ? 5 : 1, 8)))
k_mm32(const MMTask *__restrict__ tasks, MMArgs A) {
    mm32_body<KID, NVT, false>(tasks[blockIdx.x], A);
}

// Caller panel (original order, row- or column-major, ld) -> PX (permuted,
// row-major nvp, zero padding), for columns [v0, v0 + nv).
__global__ void k_mm_gather(const double *__restrict__ X, long long ldx, int row_major, int v0, int nv,
                            const int *__restrict__ fwd, int N, double *__restrict__ PX, int nvp) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long long)N * nvp) return;
    const int i = (int)(e / nvp), c = (int)(e - (long long)i * nvp);
    double v = 0.0;
    if (c < nv) {
        const long long src = fwd[i];
        v = row_major ? X[src * ldx + v0 + c] : X[(long long)(v0 + c) * ldx + src];
    }
    PX[e] = v;
}

// PY -> caller panel: Y[fwd[i], v0 + c] = PY[i, c] (the backward permutation).
__global__ void k_mm_scatter(const double *__restrict__ PY, int nvp, const int *__restrict__ fwd, int N,
                             double *__restrict__ Y, long long ldy, int row_major, int v0, int nv) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long long)N * nv) return;
    const int i = (int)(e / nv), c = (int)(e - (long long)i * nv);
    const long long dstr = fwd[i];
    const double v = PY[(long long)i * nvp + c];
    if (row_major) Y[dstr * ldy + v0 + c] = v;
    else Y[(long long)(v0 + c) * ldy + dstr] = v;
}

}  // namespace h2p
