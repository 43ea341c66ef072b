// FP64 complex Cholesky factorisation and solve on gfx950 for the shifted
// S-matrix (S + eps I) x = g of a stochastic-reconfiguration step.  The
// reference has no counterpart (its get_S_matrix, S_matrix.cu:10-58, only
// builds S).  Matrices are row-major, n x n complex<double>; the factor
// overwrites the lower triangle (A = L L^H).
//
// Blocked right-looking factorisation, block columns of CB = 128 in panels of
// NB = 32, with FP64 MFMA for the updates:
//   k_chol_trail   rank-128 update of the trailing matrix by the last block column
//   k_chol_panel   a panel's solve X L_kk^H = A_ik and its update of the rest of
//                  the block column
// each of which also factors the next 32 x 32 diagonal block (potrf32);
// then blocked forward and backward substitution (k_trsv_forward, _backward).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "linalg_kernels.hpp"

namespace rbmhip {

constexpr int NB = 32;

// Lane j's value of a complex double, broadcast to the whole wavefront (j is
// wave-uniform).
RBM_DI double lane_bcast(double v, int j) {
    const int2 r = *reinterpret_cast<int2*>(&v);
    int2 q;
    q.x = __builtin_amdgcn_readlane(r.x, j);
    q.y = __builtin_amdgcn_readlane(r.y, j);
    return *reinterpret_cast<double*>(&q);
}
RBM_DI cx<double> lane_bcast(cx<double> v, int j) { return mk(lane_bcast(v.re, j), lane_bcast(v.im, j)); }

// sqrt(d) and 1 / sqrt(d) of a positive d: the hardware's reciprocal square root
// and one third-order and one second-order correction step, where that can
// neither overflow nor lose bits, else the library's.
RBM_DI void sqrt_pair(double d, double& sd, double& rs) {
    if (d > 1e-200 && d < 1e200) {
        double y = __builtin_amdgcn_rsq(d);
        double e = __builtin_fma(-d * y, y, 1.0);
        y = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
        e = __builtin_fma(-d * y, y, 1.0);
        rs = __builtin_fma(y * e, 0.5, y);
        sd = d * rs;
        sd = __builtin_fma(__builtin_fma(-sd, sd, d), 0.5 * rs, sd);
    } else {
        sd = sqrt(d);
        rs = 1.0 / sd;
    }
}

typedef double doublex4 __attribute__((ext_vector_type(4)));
// a complex value as one 16-byte word: as a struct, arrays of them that loads
// fill ahead of their use end up in scratch memory
typedef double doublex2 __attribute__((ext_vector_type(2)));
RBM_DI doublex2 load2(const cx<double>* p) { return *reinterpret_cast<const doublex2*>(p); }
RBM_DI void store2(cx<double>* p, doublex2 v) { *reinterpret_cast<doublex2*>(p) = v; }
constexpr int CB = 128;        // block column
constexpr int CLD = NB + 1;    // LDS stride of 32-column panels

// acc += X Y^H for one 16 x 16 tile and 4 columns, x and y this lane's X[l % 16]
// [l / 16] and Y[l % 16][l / 16]
RBM_DI void mfma_herk(doublex4& re, doublex4& im, cx<double> x, cx<double> y) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.re, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.re, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.im, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.re, y.im, im, 0, 0, 0);
}

// 256 threads factor the 32 x 32 block L (lower triangle; rows past the matrix
// are the identity) in place and write its lower triangle to A[k0:, k0:].
// Thread (i, g) = (t % 32, t / 32) holds row i, columns 8 q + g; step j = 8 q + g
// passes the finished column through L, one barrier each.  A pivot that is not
// positive sets *info = index + 1, if none had, and is replaced by 1 so that the
// factorisation runs to the end.  Compact loops: unrolled over j the code of one
// use, 40 KiB, took longer to fetch than to execute (n = 32: 40 us against 12).
// Columns past the matrix are left out, as in the substitutions (n = 1, a whole
// call: 70 us with all of them, 54 so).
RBM_DI void potrf_store(int n, int k0, cx<double> (*L)[CLD], cx<double>* __restrict__ A, int* __restrict__ info) {
    const int i = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    cx<double> a[4];
#pragma unroll
    for (int q = 0; q < 4; q++) a[q] = L[i][8 * q + g];
    int bad = 0;
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll 1
        for (int gj = 0; gj < (n - k0 - 8 * q < 8 ? n - k0 - 8 * q : 8); gj++) {   // the identity's columns are done
            const int j = 8 * q + gj;
            if (wave == gj >> 1) {
                double d = lane_bcast(a[q].re, j + 32 * (gj & 1)), sd, rs;
                if (!(d > 0.0)) {
                    if (!bad) bad = k0 + j + 1;
                    d = 1.0;
                }
                sqrt_pair(d, sd, rs);
                if (g == gj && i >= j) L[i][j] = i == j ? mk(sd, 0.0) : mk(a[q].re * rs, a[q].im * rs);
            }
            __syncthreads();
            const cx<double> x = L[i][j];
#pragma unroll
            for (int u = q; u < 4; u++) {
                const cx<double> y = L[8 * u + g][j];
                a[u].re = __builtin_fma(-x.re, y.re, __builtin_fma(-x.im, y.im, a[u].re));
                a[u].im = __builtin_fma(-x.im, y.re, __builtin_fma(x.re, y.im, a[u].im));
            }
        }
    // the wavefronts' first bad pivots; the smallest is the block's
    __shared__ int bads[4];
    if ((threadIdx.x & 63) == 0) bads[wave] = bad;
    __syncthreads();
    if (threadIdx.x == 0 && *info == 0) {
        int b = 0;
        for (int w = 0; w < 4; w++)
            if (bads[w] && (!b || bads[w] < b)) b = bads[w];
        if (b) *info = b;
    }
    for (int t = threadIdx.x; t < NB * NB; t += 256) {
        const int r = t / NB, l = t % NB;
        if (k0 + r < n && l <= r) A[(int64_t)(k0 + r) * n + k0 + l] = L[r][l];
    }
}

// ROWS x 32 rows of X solve X L^H = X in place (LDS), thread (i, g) as above in
// rows i, i + 32, ...; rd = 1 / diagonal.  Each x_j gets its terms in the order
// of a sequential substitution.
template <int ROWS>
RBM_DI void trsm32(const cx<double> (*L)[CLD], const double* rd, cx<double> (*X)[CLD]) {
    const int i = threadIdx.x & 31, g = threadIdx.x >> 5;
    cx<double> a[ROWS][4];
#pragma unroll
    for (int p = 0; p < ROWS; p++)
#pragma unroll
        for (int q = 0; q < 4; q++) a[p][q] = X[32 * p + i][8 * q + g];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll 1
        for (int gj = 0; gj < 8; gj++) {
            const int j = 8 * q + gj;
            if (g == gj) {
                const double r = rd[j];
#pragma unroll
                for (int p = 0; p < ROWS; p++) X[32 * p + i][j] = mk(a[p][q].re * r, a[p][q].im * r);
            }
            __syncthreads();
            cx<double> y[4];
#pragma unroll
            for (int u = q; u < 4; u++) y[u] = L[8 * u + g][j];
#pragma unroll
            for (int p = 0; p < ROWS; p++) {
                const cx<double> x = X[32 * p + i][j];
#pragma unroll
                for (int u = q; u < 4; u++) {
                    a[p][u].re = __builtin_fma(-x.re, y[u].re, __builtin_fma(-x.im, y[u].im, a[p][u].re));
                    a[p][u].im = __builtin_fma(-x.im, y[u].re, __builtin_fma(x.re, y[u].im, a[p][u].im));
                }
            }
        }
    __syncthreads();
}

// Column panel c .. c + 31 (its diagonal block factored): rows below solve
// X L_cc^H = A, and the rest of the block column, columns c + 32 .. bend,
// subtracts X X^H.  A workgroup has 32 rows and solves for itself the up to 96
// rows of the block column's diagonal block that its update needs, all in one
// sweep of 32 steps; the update is FP64 MFMA, a wavefront 16 rows by
// half the columns.  Those shared
// rows live in D (CB x CB, the diagonal block at K0), where every workgroup may
// read the unsolved columns c .. c + 31 while their owner writes solved ones to
// A.  Workgroup 0, when the next diagonal block is in this block column, updates
// and factors that block alone.
//
// 5328 x 5328: 19 us a panel, a chain of barriers and LDS round trips (34 with a
// launch each for factor, solve by 32 lanes a row, and update).
__global__ __launch_bounds__(256) void k_chol_panel(int n, int c, int K0, int bend, cx<double>* __restrict__ A,
                                                    cx<double>* __restrict__ D, int* __restrict__ info) {
    __shared__ cx<double> X[NB + CB - NB][CLD];   // own rows, then the shared ones
    __shared__ cx<double> Lc[NB][CLD];
    __shared__ double rdiag[NB];
    cx<double>(*Xo)[CLD] = X, (*Xt)[CLD] = X + NB;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c1 = c + NB, nt = bend - c1;
    const bool has_next = nt > 0;
    const bool next = has_next && blockIdx.x == 0;
    const int r0 = next ? c1 : c1 + NB * ((int)blockIdx.x - (has_next ? 1 : 0));
    const int l = tid & 31;
    const int passes = has_next ? CB / 8 : NB / 8;
#pragma unroll 16
    for (int u = 0; u < passes; u++) {   // 8 rows at a time
        const int s = 8 * u + (tid >> 5), r = u < NB / 8 ? r0 + s : c1 + s - NB;
        const bool live = u < NB / 8 ? r < n : r < bend;
        const doublex2 v = load2(live && r >= bend ? A + (int64_t)r * n + c + l : D + (live ? r - K0 : 0) * CB + (c - K0) + l);
        store2(&X[s][l], live ? v : doublex2{0.0, 0.0});
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int i = 8 * u + (tid >> 5);
        const doublex2 v = load2(A + (int64_t)(c + i) * n + c + (l <= i ? l : i));
        store2(&Lc[i][l], l <= i ? v : doublex2{0.0, 0.0});
        if (i == l) rdiag[i] = 1.0 / Lc[i][i].re;
    }
    __syncthreads();
    if (next || !has_next) trsm32<1>(Lc, rdiag, X);
    else trsm32<CB / NB>(Lc, rdiag, X);
    const int row = lane & 15, kq = lane >> 4;
    if (next) {
        const int ti = 16 * (wave >> 1), tj = 16 * (wave & 1);
        doublex4 re{0., 0., 0., 0.}, im{0., 0., 0., 0.};
        doublex2 d[4];
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] = load2(D + (c1 + ti + kq + 4 * v - K0) * CB + (c1 + tj + row - K0));
#pragma unroll
        for (int k = 0; k < NB; k += 4) mfma_herk(re, im, Xo[ti + row][k + kq], Xo[tj + row][k + kq]);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = ti + kq + 4 * v, l = tj + row;
            cx<double> e = mk(i == l ? 1.0 : 0.0, 0.0);
            if (c1 + i < bend && l <= i) e = mk(d[v][0] - re[v], d[v][1] - im[v]);
            Xt[i][l] = e;
        }
        __syncthreads();
        potrf_store(n, c1, Xt, A, info);
        return;
    }
    for (int t = tid; t < NB * NB; t += 256) {
        const int i = t / NB, l = t % NB;
        if (r0 + i < n) store2(A + (int64_t)(r0 + i) * n + c + l, load2(&Xo[i][l]));
    }
    if (!has_next) return;
    constexpr int BT = (CB - NB) / 32;
    const int ti = 16 * (wave & 1), tj = 16 * BT * (wave >> 1);
    const int i0 = r0 + ti + kq, l0 = c1 + tj + row;
    doublex2 e[BT][4];   // on their way during the products
#pragma unroll
    for (int b = 0; b < BT; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = i0 + 4 * v, l = l0 + 16 * b;
            const bool own = i < n && l <= i && l < bend;
            e[b][v] = load2(own && i >= bend ? A + (int64_t)i * n + l : D + (own ? (i - K0) * CB + (l - K0) : 0));
        }
    doublex4 re[BT], im[BT];
#pragma unroll
    for (int b = 0; b < BT; b++) re[b] = im[b] = doublex4{0., 0., 0., 0.};
#pragma unroll 2
    for (int k = 0; k < NB; k += 4) {
        const cx<double> xi = Xo[ti + row][k + kq];
#pragma unroll
        for (int b = 0; b < BT; b++)
            if (tj + 16 * b < nt) mfma_herk(re[b], im[b], xi, Xt[tj + 16 * b + row][k + kq]);
    }
#pragma unroll
    for (int b = 0; b < BT; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = i0 + 4 * v, l = l0 + 16 * b;
            if (i >= n || l > i || l >= bend || i < c1 + NB) continue;   // the next diagonal block is workgroup 0's
            store2(i < bend ? D + (i - K0) * CB + (l - K0) : A + (int64_t)i * n + l,
                   e[b][v] - doublex2{re[b][v], im[b][v]});
        }
}

// Trailing update A_il -= X_i X_l^H by the CB columns from kc (kc < 0: none), rows
// i >= columns l >= base, one 64 x 64 tile of the lower triangle per workgroup:
// FP64 MFMA, 32 x 32 a wavefront, 16 columns at a time through LDS with the next
// 16 on their way.  The next block column's diagonal block, rows below bend, goes
// to D, except its first 32 x 32, which workgroup 0 updates alone and factors
// while the others work.
// Above 32 rows of tiles (then the block column, 4 MiB, outgrows a die's L2)
// squares of 4 x 4 tiles go to one die, the dies in turn along a row of squares.
// n = 5328: 4.4 ms a factorisation, 51 TFLOP/s for the largest update (of 78.6)
// falling with its size; as 64 x 64 tiles on the vector units 8.6.
constexpr int TR_K = 16, TR_LD = TR_K + 1;
__global__ __launch_bounds__(256, 3) void k_chol_trail(int n, int kc, int base, int bend, int tiles, int group,
                                                       cx<double>* __restrict__ A,
                                                    cx<double>* __restrict__ D, int* __restrict__ info) {
    __shared__ cx<double> P[2][64][TR_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, kq = lane >> 4;
    if (blockIdx.x == 0) {
        const int ti = 16 * (wave >> 1), tj = 16 * (wave & 1);
        doublex4 re{0., 0., 0., 0.}, im{0., 0., 0., 0.};
        doublex2 d[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = ti + kq + 4 * v, l = tj + row;
            d[v] = load2(A + (base + i < n && l <= i ? (int64_t)(base + i) * n + base + l : 0));
        }
        if (kc >= 0) {
            const cx<double>* xi = A + (int64_t)(base + ti + row < n ? base + ti + row : n - 1) * n + kc + kq;
            const cx<double>* xj = A + (int64_t)(base + tj + row < n ? base + tj + row : n - 1) * n + kc + kq;
#pragma unroll 8
            for (int k = 0; k < CB; k += 4) mfma_herk(re, im, xi[k], xj[k]);
        }
        cx<double>(*L)[CLD] = reinterpret_cast<cx<double>(*)[CLD]>(&P[0][0][0]);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = ti + kq + 4 * v, l = tj + row;
            cx<double> e = mk(i == l ? 1.0 : 0.0, 0.0);
            if (base + i < n && l <= i) e = mk(d[v][0] - re[v], d[v][1] - im[v]);
            L[i][l] = e;
        }
        __syncthreads();
        potrf_store(n, base, L, A, info);
        return;
    }
    int t = (int)blockIdx.x - 1, sub = 0;
    if (group > 1) {
        const int per = group * group, seq = t / 8;
        sub = seq % per;
        t = seq / per * 8 + t % 8;
    }
    int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((bi + 1) * (bi + 2) / 2 <= t) bi++;
    while (bi * (bi + 1) / 2 > t) bi--;
    const int bj = group * (t - bi * (bi + 1) / 2) + sub % group;
    bi = group * bi + sub / group;
    if (bj > bi || bi >= tiles) return;
    const int r0 = base + 64 * bi, c0 = base + 64 * bj;
    doublex4 re[2][2], im[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) re[a][b] = im[a][b] = doublex4{0., 0., 0., 0.};
    if (kc >= 0) {
        const int k = tid & 15, ri = tid >> 4;
        const cx<double>*src[2][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = r0 + ri + 16 * u, l = c0 + ri + 16 * u;
            src[0][u] = A + (int64_t)(i < n ? i : n - 1) * n + kc + k;
            src[1][u] = A + (int64_t)(l < n ? l : n - 1) * n + kc + k;
        }
        doublex2 f[2][4];
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int u = 0; u < 4; u++) f[o][u] = load2(src[o][u]);
        const int wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
        for (int k0 = 0; k0 < CB; k0 += TR_K) {
            __syncthreads();
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int u = 0; u < 4; u++) store2(&P[o][ri + 16 * u][k], f[o][u]);
            __syncthreads();
            const int kn = k0 + TR_K < CB ? k0 + TR_K : 0;   // without a branch, which would make each load wait
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int u = 0; u < 4; u++) f[o][u] = load2(src[o][u] + kn);
#pragma unroll
            for (int kk = 0; kk < TR_K; kk += 4) {
                cx<double> x[2], y[2];
#pragma unroll
                for (int a = 0; a < 2; a++) x[a] = P[0][wr + 16 * a + row][kk + kq];
#pragma unroll
                for (int b = 0; b < 2; b++) y[b] = P[1][wc + 16 * b + row][kk + kq];
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 2; b++) mfma_herk(re[a][b], im[a][b], x[a], y[b]);
            }
        }
    }
    // eight loads in flight: one at a time the sixteen round trips of a tile cost
    // as much as its products
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int i0 = r0 + 32 * (wave >> 1) + 16 * a + kq, l0 = c0 + 32 * (wave & 1) + row;
        doublex2 e[2][4];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + 4 * v, l = l0 + 16 * b;
                // in the lower triangle, and not in workgroup 0's block
                const bool own = i < n && l <= i && i >= base + NB;
                e[b][v] = load2(A + (own ? (int64_t)i * n + l : 0));
            }
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + 4 * v, l = l0 + 16 * b;
                if (i >= n || l > i || i < base + NB) continue;
                store2(i < bend ? D + (i - base) * CB + (l - base) : A + (int64_t)i * n + l,
                       e[b][v] - doublex2{re[a][b][v], im[a][b][v]});
            }
    }
}

// ---------------------------------------------------------------------------
// Products C = X^T Y of row-major K x ld operands on FP32 MFMA: the per-layer
// gradient products of PsiDeep (all tiles, split over K).
// A 256-thread workgroup computes a 128 x 128 tile as 2 x 2 waves of 64 x 64,
// each 2 x 2 v_mfma_f32_32x32x2f32 tiles (lane l supplies A[l % 32][l / 32]
// and B[l / 32][l % 32]; accumulator v of lane l is row
// 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32).  K advances 16 rows per LDS
// stage; the next stage's rows are loaded into registers while the current
// one is multiplied.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int GR_T = 128, GR_K = 16, GR_LD = GR_T + 4;

// C[m0.., n0..] = X[k_begin..k_end)^T Y[k_begin..k_end) for one 128 x 128 tile
RBM_DI void tile_tn(const float* __restrict__ X, int ldx, int m0, const float* __restrict__ Y, int ldy, int n0,
                    int k_begin, int k_end, float* __restrict__ C, int ldc) {
    __shared__ float As[GR_K][GR_LD];
    __shared__ float Bs[GR_K][GR_LD];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // staging: 16 rows x 128 columns per operand = 512 float4; thread tid loads
    // float4 q = tid and tid + 256 of each (row q / 32, column 4 (q % 32))
    const int q0 = tid, q1 = tid + 256;
    const int r0 = q0 >> 5, c0 = (q0 & 31) * 4, r1 = q1 >> 5, c1 = (q1 & 31) * 4;
    float4 ra0, ra1, rb0, rb1;
#define GR_FETCH(k0)                                                                        \
    ra0 = *reinterpret_cast<const float4*>(X + (int64_t)((k0) + r0) * ldx + m0 + c0);        \
    ra1 = *reinterpret_cast<const float4*>(X + (int64_t)((k0) + r1) * ldx + m0 + c1);        \
    rb0 = *reinterpret_cast<const float4*>(Y + (int64_t)((k0) + r0) * ldy + n0 + c0);        \
    rb1 = *reinterpret_cast<const float4*>(Y + (int64_t)((k0) + r1) * ldy + n0 + c1);
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x16{};
    GR_FETCH(k_begin)
    for (int k0 = k_begin; k0 < k_end; k0 += GR_K) {
        __syncthreads();
        *reinterpret_cast<float4*>(&As[r0][c0]) = ra0;
        *reinterpret_cast<float4*>(&As[r1][c1]) = ra1;
        *reinterpret_cast<float4*>(&Bs[r0][c0]) = rb0;
        *reinterpret_cast<float4*>(&Bs[r1][c1]) = rb1;
        __syncthreads();
        if (k0 + GR_K < k_end) { GR_FETCH(k0 + GR_K) }
#pragma unroll
        for (int kk = 0; kk < GR_K; kk += 2) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) a[i] = As[kk + (lane >> 5)][wm + 32 * i + (lane & 31)];
#pragma unroll
            for (int j = 0; j < 2; j++) b[j] = Bs[kk + (lane >> 5)][wn + 32 * j + (lane & 31)];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
#undef GR_FETCH
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = m0 + wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const int col = n0 + wn + 32 * j + (lane & 31);
                C[(int64_t)row * ldc + col] = acc[i][j][v];
            }
}

// Split-K product: workgroup (x, z) covers tile x of the (ldx / 128) x (ldy / 128)
// grid over rows [z Kper, (z + 1) Kper); out[z] is ldx x ldy.
__global__ __launch_bounds__(256) void k_gemm_tn(int ldx, int ldy, int Kper, const float* __restrict__ X,
                                                 const float* __restrict__ Y, float* __restrict__ out) {
    const int tn = ldy / GR_T;
    const int bm = blockIdx.x / tn, bn = blockIdx.x % tn;
    const int k0 = (int)blockIdx.z * Kper;
    tile_tn(X, ldx, bm * GR_T, Y, ldy, bn * GR_T, k0, k0 + Kper, out + (int64_t)blockIdx.z * ldx * ldy, ldy);
}

// acc[i] += sum_z part[z n + i], the split partials added in FP64 in a fixed order
__global__ __launch_bounds__(256) void k_accum_splits_f64(int64_t n, int splits, const float* __restrict__ part,
                                                          double* __restrict__ acc) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int z = 0; z < splits; z++) s += (double)part[(int64_t)z * n + i];
        acc[i] += s;
    }
}

hipError_t launch_accum_splits_f64(int64_t n, int splits, const float* part, double* acc, hipStream_t stream) {
    int64_t g = (n + 255) / 256;
    if (g > 4096) g = 4096;
    if (g < 1) g = 1;
    hipLaunchKernelGGL(k_accum_splits_f64, dim3((unsigned)g), dim3(256), 0, stream, n, splits, part, acc);
    return hipGetLastError();
}

hipError_t launch_gemm_tn_splitk(int ldx, int ldy, int64_t K, int splits, const float* X, const float* Y, float* out,
                                 hipStream_t stream) {
    if (ldx <= 0 || ldy <= 0 || ldx % GR_T || ldy % GR_T || splits < 1 || K <= 0 || K % ((int64_t)GR_K * splits) ||
        K > ((int64_t)1 << 30))
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)((ldx / GR_T) * (ldy / GR_T)), 1, (unsigned)splits);
    hipLaunchKernelGGL(k_gemm_tn, grid, dim3(256), 0, stream, ldx, ldy, (int)(K / splits), X, Y, out);
    return hipGetLastError();
}

hipError_t launch_cholesky(int n, cx<double>* A, cx<double>* D, int* info, hipStream_t stream) {
    for (int K0 = 0; K0 < n; K0 += CB) {
        const int bend = n - K0 < CB ? n : K0 + CB;
        // the first block column only takes its diagonal block over
        const int tiles = ((K0 ? n : bend) - K0 + 63) / 64;
        const int group = tiles > 32 ? 4 : 1, rows = (tiles + group - 1) / group, squares = rows * (rows + 1) / 2;
        const int blocks = group > 1 ? (squares + 7) / 8 * 8 * group * group : squares;
        hipLaunchKernelGGL(k_chol_trail, dim3((unsigned)(1 + blocks)), dim3(256), 0, stream, n, K0 ? K0 - CB : -1, K0,
                           bend, tiles, group, A, D, info);
        for (int c = K0; c < bend && c + NB < n; c += NB)
            hipLaunchKernelGGL(k_chol_panel, dim3((unsigned)((n - c - 1) / NB + (c + NB < bend ? 1 : 0))), dim3(256),
                               0, stream, n, c, K0, bend, A, D, info);
    }
    return hipGetLastError();
}

// Blocked substitution, one launch per block of CB: the rows outside the solved
// blocks subtract the products of the block solved last (p0 ..; p0 < 0: none),
// and workgroup 0, which has the next block (k0 ..), then solves that.  Its
// triangle is in LDS by the time its right-hand side is complete, and wavefront
// s solves 32 rows with its part of the triangle in registers: a launch of its
// own for each 32 rows' solve and another for their update took 5.1 ms for
// n = 5328, this 2.1, most of it the chain through workgroup 0.
// The triangle is packed by rows; rows past the matrix are the identity.
RBM_DI int tri(int i, int l) { return i * (i + 1) / 2 + l; }
constexpr int TRI = CB * (CB + 1) / 2;
constexpr int TRSV_LDS = (TRI + 4 * CB) * (int)sizeof(cx<double>);

RBM_DI void trsv_load(int n, int k0, const cx<double>* __restrict__ A, cx<double>* Ls) {
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
#pragma unroll 16
    for (int i = wave; i < CB; i += 4) {
        const int r = k0 + i < n ? k0 + i : n - 1;   // columns stay within row r: l <= i
        const cx<double>* a = A + (int64_t)r * n + k0;
        const int l0 = lane < r - k0 ? lane : r - k0, l1 = lane + 64 < r - k0 ? lane + 64 : r - k0;
        const doublex2 v0 = load2(a + l0), v1 = load2(a + l1);
        const bool in = k0 + i < n;
        if (lane <= i) store2(Ls + tri(i, lane), in ? v0 : doublex2{i == lane ? 1.0 : 0.0, 0.0});
        if (lane + 64 <= i) store2(Ls + tri(i, lane + 64), in ? v1 : doublex2{i == lane + 64 ? 1.0 : 0.0, 0.0});
    }
}

// L y = x: x_i -= L_ip y_p below, then block k0
__global__ __launch_bounds__(512) void k_trsv_forward(int n, int p0, int k0, const cx<double>* __restrict__ A,
                                                      cx<double>* __restrict__ x) {
    extern __shared__ cx<double> trsv_lds[];
    cx<double>*Ls = trsv_lds, *xs = trsv_lds + TRI, *ys = xs + CB;   // block k0's triangle, its x, the solved block's y
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool solve = blockIdx.x == 0;
    const bool first_half = tid < 256;   // subtracts the products, the others load the triangle
    if (solve) {
        if (!first_half) trsv_load(n, k0, A, Ls);
        if (tid < CB) xs[tid] = k0 + tid < n ? x[k0 + tid] : mk(0.0, 0.0);
    }
    if (p0 >= 0) {
        if (tid < CB) ys[tid] = x[p0 + tid];
        __syncthreads();
        // 16 lanes a row, 8 columns each
        const int q = tid & 15, first = solve ? k0 : k0 + CB + 64 * ((int)blockIdx.x - 1);
        for (int g = 0; first_half && g < (solve ? CB / 64 : 1); g++) {
            doublex2 f[4][8];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = first + 64 * g + 16 * u + (tid >> 4);
                const cx<double>* a = A + (int64_t)(i < n ? i : n - 1) * n + p0 + q;
#pragma unroll
                for (int m = 0; m < 8; m++) f[u][m] = load2(a + 16 * m);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = first + 64 * g + 16 * u + (tid >> 4);
                cx<double> s = mk(0.0, 0.0);
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const cx<double> y = ys[q + 16 * m];
                    s.re = __builtin_fma(f[u][m][0], y.re, __builtin_fma(-f[u][m][1], y.im, s.re));
                    s.im = __builtin_fma(f[u][m][0], y.im, __builtin_fma(f[u][m][1], y.re, s.im));
                }
                s = row_sum16(s);
                if (q == 0 && i < n) {
                    if (solve) xs[i - k0] = mk(xs[i - k0].re - s.re, xs[i - k0].im - s.im);
                    else x[i] = mk(x[i].re - s.re, x[i].im - s.im);
                }
            }
        }
    }
    if (!solve) return;
    __syncthreads();
    // rows scaled by their diagonal, so that a step is a broadcast and two FMAs
    const int j = lane & 31;
    const double rd = 1.0 / Ls[tri(32 * (wave & 3) + j, 32 * (wave & 3) + j)].re;
    doublex2 L[NB];
#pragma unroll
    for (int m = 0; m < NB; m++) {
        const doublex2 a = load2(Ls + tri(32 * (wave & 3) + j, 32 * (wave & 3) + (m < j ? m : 0)));
        L[m] = m < j ? a * rd : doublex2{0.0, 0.0};
    }
    for (int s = 0; s < CB / NB && k0 + NB * s < n; s++) {   // identity rows past the matrix are left
        if (wave == s) {
            cx<double> v = mk(xs[32 * s + j].re * rd, xs[32 * s + j].im * rd);
#pragma unroll
            for (int m = 0; m < NB; m++) {
                const cx<double> y = lane_bcast(v, m);
                v.re = __builtin_fma(-L[m][0], y.re, __builtin_fma(L[m][1], y.im, v.re));
                v.im = __builtin_fma(-L[m][0], y.im, __builtin_fma(-L[m][1], y.re, v.im));
            }
            if (lane < NB) xs[32 * s + j] = v;
        }
        __syncthreads();
        // rows below in the block: 8 lanes a row, 4 columns each
        for (int i = 32 * (s + 1) + (tid >> 3); i < CB && k0 + i < n; i += 64) {
            cx<double> u = mk(0.0, 0.0);
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const int l = 32 * s + (tid & 7) + 8 * m;
                const cx<double> a = Ls[tri(i, l)], y = xs[l];
                u.re = __builtin_fma(a.re, y.re, __builtin_fma(-a.im, y.im, u.re));
                u.im = __builtin_fma(a.re, y.im, __builtin_fma(a.im, y.re, u.im));
            }
#pragma unroll
            for (int off = 4; off > 0; off >>= 1) {
                u.re += __shfl_xor(u.re, off);
                u.im += __shfl_xor(u.im, off);
            }
            if ((tid & 7) == 0) xs[i] = mk(xs[i].re - u.re, xs[i].im - u.im);
        }
        __syncthreads();
    }
    if (tid < CB && k0 + tid < n) x[k0 + tid] = xs[tid];
}

// L^H y = x: x_i -= sum_m conj(L_mi) y_m above, m over the solved block, then
// block k0
__global__ __launch_bounds__(512) void k_trsv_backward(int n, int p0, int k0, const cx<double>* __restrict__ A,
                                                       cx<double>* __restrict__ x) {
    extern __shared__ cx<double> trsv_lds[];
    cx<double>*Ls = trsv_lds, *xs = trsv_lds + TRI, *ys = xs + CB, *ps = ys + CB;   // ps: 4 x 64 partial sums
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool solve = blockIdx.x == 0;
    const bool first_half = tid < 256;   // subtracts the products, the others load the triangle
    if (solve) {
        if (!first_half) trsv_load(n, k0, A, Ls);
        if (tid < CB) xs[tid] = k0 + tid < n ? x[k0 + tid] : mk(0.0, 0.0);
    }
    if (p0 >= 0) {
        if (tid < CB) ys[tid] = p0 + tid < n ? x[p0 + tid] : mk(0.0, 0.0);
        __syncthreads();
        // a column a lane, 32 rows a wavefront
        const int first = solve ? k0 : 64 * ((int)blockIdx.x - 1);
        for (int g = 0; g < (solve ? CB / 64 : 1); g++) {
            const int i = first + 64 * g + lane;
            if (first_half) {
                doublex2 f[NB];
#pragma unroll
                for (int m = 0; m < NB; m++) {
                    const int r = p0 + 32 * wave + m;   // past the matrix: times ys = 0
                    f[m] = load2(A + (int64_t)(r < n ? r : n - 1) * n + i);
                }
                cx<double> s = mk(0.0, 0.0);
#pragma unroll
                for (int m = 0; m < NB; m++) {
                    const cx<double> y = ys[32 * wave + m];
                    s.re = __builtin_fma(f[m][0], y.re, __builtin_fma(f[m][1], y.im, s.re));
                    s.im = __builtin_fma(f[m][0], y.im, __builtin_fma(-f[m][1], y.re, s.im));
                }
                ps[64 * wave + lane] = s;
            }
            __syncthreads();
            if (wave == 0) {
                cx<double> t = ps[lane];
#pragma unroll
                for (int z = 1; z < 4; z++) t = mk(t.re + ps[64 * z + lane].re, t.im + ps[64 * z + lane].im);
                if (solve) xs[i - k0] = mk(xs[i - k0].re - t.re, xs[i - k0].im - t.im);
                else x[i] = mk(x[i].re - t.re, x[i].im - t.im);
            }
            __syncthreads();
        }
    }
    if (!solve) return;
    __syncthreads();
    // rows scaled by their diagonal, so that a step is a broadcast and two FMAs
    const int j = lane & 31;
    const double rd = 1.0 / Ls[tri(32 * (wave & 3) + j, 32 * (wave & 3) + j)].re;
    doublex2 L[NB];
#pragma unroll
    for (int m = 0; m < NB; m++) {
        const doublex2 a = load2(Ls + tri(32 * (wave & 3) + m, 32 * (wave & 3) + (m > j ? j : 0)));
        L[m] = m > j ? a * rd : doublex2{0.0, 0.0};
    }
    for (int s = (n - k0 < CB ? n - k0 - 1 : CB - 1) / NB; s >= 0; s--) {
        if (wave == s) {
            cx<double> v = mk(xs[32 * s + j].re * rd, xs[32 * s + j].im * rd);
#pragma unroll
            for (int m = NB - 1; m >= 0; m--) {
                const cx<double> y = lane_bcast(v, m);
                v.re = __builtin_fma(-L[m][0], y.re, __builtin_fma(-L[m][1], y.im, v.re));
                v.im = __builtin_fma(-L[m][0], y.im, __builtin_fma(L[m][1], y.re, v.im));
            }
            if (lane < NB) xs[32 * s + j] = v;
        }
        __syncthreads();
        // columns above in the block: four threads a column, 8 rows each
        if (tid < 4 * 32 * s) {
            const int i = tid >> 2;
            cx<double> u = mk(0.0, 0.0);
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const int r = 32 * s + 4 * m + (tid & 3);
                const cx<double> a = Ls[tri(r, i)], y = xs[r];
                u.re = __builtin_fma(a.re, y.re, __builtin_fma(a.im, y.im, u.re));
                u.im = __builtin_fma(a.re, y.im, __builtin_fma(-a.im, y.re, u.im));
            }
#pragma unroll
            for (int off = 2; off > 0; off >>= 1) {
                u.re += __shfl_xor(u.re, off);
                u.im += __shfl_xor(u.im, off);
            }
            if ((tid & 3) == 0) xs[i] = mk(xs[i].re - u.re, xs[i].im - u.im);
        }
        __syncthreads();
    }
    if (tid < CB && k0 + tid < n) x[k0 + tid] = xs[tid];
}

hipError_t launch_cholesky_solve(int n, const cx<double>* L, cx<double>* x, hipStream_t stream) {
    for (const void* f : {(const void*)&k_trsv_forward, (const void*)&k_trsv_backward}) {
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, TRSV_LDS);
        if (e != hipSuccess) return e;
    }
    const int nblk = (n + CB - 1) / CB;
    for (int b = 0; b < nblk; b++) {
        const int k0 = b * CB, rest = b ? n - k0 - CB : 0;
        hipLaunchKernelGGL(k_trsv_forward, dim3((unsigned)(1 + (rest > 0 ? (rest + 63) / 64 : 0))), dim3(512), TRSV_LDS,
                           stream, n, b ? k0 - CB : -1, k0, L, x);
    }
    for (int b = nblk - 1; b >= 0; b--) {
        const int k0 = b * CB;
        hipLaunchKernelGGL(k_trsv_backward, dim3((unsigned)(1 + (b < nblk - 1 ? k0 / 64 : 0))), dim3(512), TRSV_LDS, stream,
                           n, b < nblk - 1 ? k0 + CB : -1, k0, L, x);
    }
    return hipGetLastError();
}

}  // namespace rbmhip
