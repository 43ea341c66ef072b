// The centred S of a stochastic-reconfiguration step on the bfloat16 matrix
// cores (the reference only builds S, S_matrix.cu:10-58): second moments by
// pairs of spins and pairs of units (k_pair_moments), and the Gram product of
// the O_k rows (k_gram_lower_bf3) for small models and where moments cancel.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "linalg_kernels.hpp"

namespace rbmhip {

// ---------------------------------------------------------------------------
// Gram product G = A^T A of the S-matrix rows (lower 128 x 128 tiles) on the
// bfloat16 matrix cores with FP32 accuracy.  Every FP32 value of A arrives
// split exactly into three bfloat16 parts, x = hi + mid + lo (hi = bf16(x),
// mid = bf16(x - hi), lo = x - hi - mid), stored per block of 32 samples as
// [block][part][column][32 samples].  A product x y is the sum of the six part
// products hi hi, hi mid, mid hi, hi lo, lo hi, mid mid, which leaves out
// terms below 2^-24 |x y|, and v_mfma_f32_16x16x32_bf16 sums them in FP32
// like an FP32 GEMM; six bfloat16 products cost 6 / 16 of one FP32 product on
// the matrix cores.  The batch's FP32 tile is added into the FP64 accumulator
// C, so the FP32 error does not grow with the number of batches.
//
// A 128-thread workgroup owns the lower tile (bm, bn) that order[blockIdx.x]
// names (gram_tile_order below), as two waves of 128 x 64 (8 x 4 MFMA tiles; lane l supplies A[l % 16][8 (l /
// 16) + q] and B[8 (l / 16) + q][l % 16], accumulator v of lane l is row 4 (l /
// 16) + v, column l % 16).  The stored layout is the MFMA operand layout: the
// fragment of lane l for a column tile is the 16 bytes of column c0 + l % 16 at
// samples 8 (l / 16) .. + 7, so every fragment is one coalesced 16-byte load
// and no LDS or barrier is needed.  The B fragments of the next block load
// into a second register set at the start of a block and are moved into place
// at its end; the A fragments of row tile i are reloaded for the next block as
// soon as row tile i's 24 MFMAs of this block are issued.  With 128 FP32
// accumulators the wave runs alone on its SIMD.
// Measured against other forms on the 6x6 Heisenberg SR step (21 batches of
// 12 480 samples and one of 64, ld 10 752), in the row-major tile order:
// 150 ms of Gram product per step; staging both column stripes through LDS
// for 2 x 2 waves of 64 x 64, 165-171 ms; 64 x 64 per wave loaded straight
// from memory (two waves per SIMD), 244 ms.  The grouped order below: 147 ms.
// ---------------------------------------------------------------------------
constexpr int GM_T = 128, GB_K = 32;
typedef float gbf32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 gbbf16x8 __attribute__((ext_vector_type(8)));

constexpr int RT = 8;   // row tiles per wave

__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_gram_lower_bf3(int ld, int K, const uint4* __restrict__ A, double* __restrict__ C,
                      const int2* __restrict__ order) {
    const int2 tile = order[blockIdx.x];
    if (tile.x < 0) return;
    const int bm = tile.x, bn = tile.y;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m0 = bm * GM_T, n0 = bn * GM_T + 64 * wave;
    const int nblk = K / GB_K;
    // uint4 index of (block, part, column, chunk): ((blk * 3 + q) * ld + col) * 4 + chunk
    const uint4* pa = A + (int64_t)(m0 + (lane & 15)) * 4 + (lane >> 4);
    const uint4* pb = A + (int64_t)(n0 + (lane & 15)) * 4 + (lane >> 4);
    const int64_t part_stride = (int64_t)ld * 4, blk_stride = 3 * part_stride;
    uint4 fa[RT][3], fb[4][3], fn[4][3];
    gbf32x4 acc[RT][4];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = gbf32x4{0.f, 0.f, 0.f, 0.f};
    // first loads in the order the loop issues them (B, then A by row tile),
    // so that the waits at the loop head hold for the first block too
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int j = 0; j < 4; j++) fb[j][q] = pb[q * part_stride + 64 * j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RT; i++) {
#pragma unroll
        for (int q = 0; q < 3; q++) fa[i][q] = pa[q * part_stride + 64 * i];
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int blk = 0; blk < nblk; blk++) {
        // the last block reloads itself, so that no load is conditional
        const int64_t o = (int64_t)(blk + 1 < nblk ? blk + 1 : blk) * blk_stride;
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) fn[j][q] = pb[o + q * part_stride + 64 * j];
        // the loads stay where they are issued (the scheduler would move them
        // next to their first use)
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PA[6] = {1, 0, 2, 0, 1, 0}, PB[6] = {1, 2, 0, 1, 0, 0};
#pragma unroll
        for (int i = 0; i < RT; i++) {
#pragma unroll
            for (int p = 0; p < 6; p++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(gbbf16x8, fa[i][PA[p]]),
                        __builtin_bit_cast(gbbf16x8, fb[j][PB[p]]), acc[i][j], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 3; q++) fa[i][q] = pa[o + q * part_stride + 64 * i];
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int q = 0; q < 3; q++) fb[j][q] = fn[j][q];
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = m0 + 16 * i + 4 * (lane >> 4) + v;
                const int col = n0 + 16 * j + (lane & 15);
                C[(int64_t)row * ld + col] += (double)acc[i][j][v];
            }
}

// Workgroup order of the lower 128 x 128 tiles.  Workgroup b runs on XCD b mod
// 8, after the earlier workgroups of that XCD, and an XCD holds 64 of these
// workgroups at once (two per CU).  The tiles are listed by 8 x 8 groups (the
// lower triangle of groups row by row, the tiles of a group row by row) and
// XCD x takes the x-th eighth of the list in order, so the 64 workgroups it
// runs at once mostly form one group and read 16 column stripes between them,
// which its L2 holds, instead of up to 128.  Entries past the list are (-1, -1).
int gram_tile_order(int ld, std::vector<int2>& order) {
    const int T = ld / GM_T, G = 8;
    std::vector<int2> list;
    list.reserve((size_t)T * (T + 1) / 2);
    for (int gm = 0; gm * G < T; gm++)
        for (int gn = 0; gn <= gm; gn++)
            for (int bm = gm * G; bm < std::min(T, gm * G + G); bm++)
                for (int bn = gn * G; bn < std::min(bm + 1, gn * G + G); bn++) list.push_back(make_int2(bm, bn));
    const int n = (int)list.size(), per = (n + 7) / 8;
    order.assign((size_t)8 * per, make_int2(-1, -1));
    for (int b = 0; b < 8 * per; b++) {
        const int k = (b % 8) * per + b / 8;
        if (k < n) order[(size_t)b] = list[(size_t)k];
    }
    return n;
}

hipError_t launch_gram_lower(int ld, int K, const uint32_t* A, double* C, const int2* order, int n_order,
                             hipStream_t stream) {
    if (ld <= 0 || ld % GM_T || K <= 0 || K % (2 * GB_K) || n_order <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gram_lower_bf3, dim3((unsigned)n_order), dim3(128), 0, stream, ld, K,
                       reinterpret_cast<const uint4*>(A), C, order);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Second moments of an RBM's log-derivatives from pairs.  With the constant
// spin s_0 = 1, the spins s_1 .. s_N, and the constant unit t_M = 1, every
// O_k is a product s_p T_j, so
//   <conj(O_(p,j)) O_(p',j')> = sum_s w s_p s_p' conj(T_j) T_j'
// depends on the pair (p, p') through s_p s_p' alone, one of 1 + N (N + 1) / 2
// sign rows, and on the pair (j, j') through one of (M + 1)^2 real columns.
// The product of all sign rows with all unit pairs is a GEMM of
// N^2 / 2 x M^2 x samples with one exact +-1 operand, where the Gram product
// of the realified O_k rows takes (2 N M)^2 / 2 x samples products of two
// split operands: 8 times fewer matrix products at N = 36, M = 144 (three
// part products per pair product instead of six, and each pair once).
//
// Operands.  A: the sign rows' bits per 32-sample block (k_pair_planes); a
// lane takes the byte of its K quarter and a 256-entry LDS table turns it
// into the four packed bfloat16 +-1 pairs.  B: columns 2 c + part, part (Re,
// Im) of t_j conj(t_j') for unit pair c = j (j + 1) / 2 + j' (j >= j'), formed
// in FP32 from the centred, sqrt(w)-scaled unit values (k_pair_units, stored
// per 32-sample block as [unit][Re, Im][32 samples], so that a lane loads its
// 8 samples as two 16-byte words) and split exactly into three bfloat16
// parts; v_mfma_f32_16x16x32_bf16 sums the exact products in FP32.
//
// A wavefront owns RT <= 12 row tiles and CT = 3 column tiles of one sample
// split: B is formed once for RT row tiles (about 65 vector instructions per
// column tile and K step against RT x 3 MFMAs of 16 cycles), and the 4 RT CT
// accumulators leave two wavefronts per SIMD; from nine row tiles up some of
// the other registers go to scratch (18, 38, 60, 80 a lane at 9, 10, 11, 12).
// 6x6 Heisenberg, M = 144 (11 row tiles), 65 536 samples: 6.4 ms, 0.92 PFLOP/s of
// bfloat16 products, the matrix pipes busy 39 % of the cycles, and 0.8 ms for
// the operands and the assembly, where the Gram product took 37.6 + 2.7 ms;
// what it waits for now is the loads and vector work of B, formed again by
// each of the 4 row groups.  Every PAIR_FLUSH blocks the FP32
// tile is added into the split's FP64 accumulator, so the FP32 error does not
// grow with the sample count.
// ---------------------------------------------------------------------------
constexpr int PAIR_CT = 3, PAIR_RT_MAX = 12, PAIR_FLUSH = 128;

// bits of the sign rows: row 0 is 1, row 1 + q (q - 1) / 2 + p is s_p s_q for
// 0 <= p < q <= N with s_0 = 1; rows past the last read as 1
__global__ __launch_bounds__(256) void k_pair_planes(int64_t nblk, int N, int rows_p, const uint32_t* __restrict__ planes,
                                                     uint32_t* __restrict__ out) {
    const int rows = 1 + N * (N + 1) / 2;
    for (int64_t b = blockIdx.x; b < nblk; b += gridDim.x)
        for (int r = threadIdx.x; r < rows_p; r += blockDim.x) {
            uint32_t w = 0xFFFFFFFFu;
            if (r >= 1 && r < rows) {
                const int t = r - 1;
                int q = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)t)) * 0.5f);
                while (q * (q - 1) / 2 > t) q--;
                while ((q + 1) * q / 2 <= t) q++;
                const int p = t - q * (q - 1) / 2;
                w = planes[b * N + q - 1];
                if (p > 0) w = ~(w ^ planes[b * N + p - 1]);
            }
            out[b * rows_p + r] = w;
        }
}

// sqrt(w) (T_j - mean_j) for unit j < M, sqrt(w) for the constant unit M, of
// samples [s0, s0 + 32 nblk) (zero past n), in the layout above.  One workgroup
// per block: the records are read along their rows and turned in LDS.
template <typename T>
__global__ __launch_bounds__(256) void k_pair_units(int64_t s0, int64_t n, int M, const cx<T>* __restrict__ Trec,
                                                    const cx<double>* __restrict__ w, const cx<double>* __restrict__ mean,
                                                    float* __restrict__ out) {
    constexpr int UC = 64;   // units per LDS stage
    __shared__ float v[2][UC][33];
    __shared__ float sw[32];
    const int64_t base = s0 + (int64_t)blockIdx.x * 32;
    if (threadIdx.x < 32) sw[threadIdx.x] = base + threadIdx.x < n ? (float)sqrt(w[base + threadIdx.x].re) : 0.0f;
    for (int j0 = 0; j0 <= M; j0 += UC) {
        __syncthreads();
        for (int t = threadIdx.x; t < 32 * UC; t += blockDim.x) {
            const int jj = t & (UC - 1), k = t / UC, j = j0 + jj;
            float re = 0.0f, im = 0.0f;
            if (j < M && base + k < n) {
                const cx<T> x = Trec[(base + k) * M + j];
                re = sw[k] * (float)(x.re - (T)mean[j].re);
                im = sw[k] * (float)(x.im - (T)mean[j].im);
            } else if (j == M) {
                re = sw[k];
            }
            v[0][jj][k] = re;
            v[1][jj][k] = im;
        }
        __syncthreads();
        for (int t = threadIdx.x; t < 64 * UC; t += blockDim.x) {
            const int k = t & 31, part = (t >> 5) & 1, jj = t >> 6, j = j0 + jj;
            if (j <= M) out[((int64_t)blockIdx.x * (M + 1) + j) * 64 + part * 32 + k] = v[part][jj][k];
        }
    }
}

RBM_DI uint32_t gb_pair(float lo, float hi) {
    const __bf16 a = (__bf16)lo, b = (__bf16)hi;
    return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}

template <int RT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void k_pair_moments(int64_t nblk, int splits, int groups, int col_groups, int M, int rows_p, int cols_p,
                    const uint32_t* __restrict__ planes, const float* __restrict__ units, double* __restrict__ C) {
    constexpr int CT = PAIR_CT;
    __shared__ uint4 lut[256];
    const int lane = threadIdx.x;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t byte = (uint32_t)(lane + 64 * e);
        uint32_t q4[4];
#pragma unroll
        for (int q = 0; q < 4; q++)
            q4[q] = 0xBF80BF80u ^ (((byte >> (2 * q)) & 1u) << 15) ^ (((byte >> (2 * q + 1)) & 1u) << 31);
        lut[byte] = make_uint4(q4[0], q4[1], q4[2], q4[3]);
    }
    __syncthreads();
    const int kk = lane >> 4, ii = lane & 15;
    // the row groups of one column group and split run next to each other and
    // read the same unit values
    const int grp = blockIdx.x % groups, rest = blockIdx.x / groups;
    const int cg = rest % col_groups, z = rest / col_groups;
    const int row0 = grp * RT * 16, col0 = cg * CT * 16;
    const int part = ii & 1;
    const float sgn = part ? -1.0f : 1.0f;
    const int pairs = (M + 1) * (M + 2) / 2;
    int oj[CT], ojp[CT];   // float offsets of units j and j' of this lane's columns within a block
#pragma unroll
    for (int b = 0; b < CT; b++) {
        int c = (col0 + 16 * b + ii) >> 1;
        if (c >= pairs) c = 0;   // padding columns repeat the first pair; they are never read
        int j = (int)((sqrtf(8.0f * (float)c + 1.0f) - 1.0f) * 0.5f);
        while (j * (j + 1) / 2 > c) j--;
        while ((j + 1) * (j + 2) / 2 <= c) j++;
        oj[b] = j * 64;
        ojp[b] = (c - j * (j + 1) / 2) * 64;
    }
    const int64_t per = (nblk + splits - 1) / splits;
    const int64_t b0 = z * per, b1 = b0 + per < nblk ? b0 + per : nblk;
    double* Cz = C + (int64_t)z * rows_p * cols_p;
    const int64_t ustride = (int64_t)(M + 1) * 64;
    for (int64_t f0 = b0; f0 < b1; f0 += PAIR_FLUSH) {
        const int64_t f1 = f0 + PAIR_FLUSH < b1 ? f0 + PAIR_FLUSH : b1;
        gbf32x4 acc[RT][CT];
#pragma unroll
        for (int a = 0; a < RT; a++)
#pragma unroll
            for (int b = 0; b < CT; b++) acc[a][b] = gbf32x4{0.f, 0.f, 0.f, 0.f};
        for (int64_t blk = f0; blk < f1; blk++) {
            const float* U = units + blk * ustride + 8 * kk;
            const uint32_t* pl = planes + blk * rows_p + row0 + ii;
            uint32_t byte[RT];
#pragma unroll
            for (int a = 0; a < RT; a++) byte[a] = pl[16 * a];
            uint4 bh[CT], bm[CT], bl[CT];
#pragma unroll
            for (int b = 0; b < CT; b++) {
                float x[8], y[8], re[8], im[8];
                const float4* px = reinterpret_cast<const float4*>(U + oj[b] + 32 * part);
                const float4* py = reinterpret_cast<const float4*>(U + oj[b] + 32 * (1 - part));
                const float4* pr = reinterpret_cast<const float4*>(U + ojp[b]);
                const float4* pi = reinterpret_cast<const float4*>(U + ojp[b] + 32);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    *reinterpret_cast<float4*>(x + 4 * h) = px[h];
                    *reinterpret_cast<float4*>(y + 4 * h) = py[h];
                    *reinterpret_cast<float4*>(re + 4 * h) = pr[h];
                    *reinterpret_cast<float4*>(im + 4 * h) = pi[h];
                }
                // Re = re_j re_j' + im_j im_j',  Im = im_j re_j' - re_j im_j'
                uint32_t hi[4], mid[4], lo[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    float v[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const int k = 2 * q + h;
                        v[h] = __builtin_fmaf(x[k], re[k], sgn * (y[k] * im[k]));
                    }
                    hi[q] = gb_pair(v[0], v[1]);
                    const float r0 = v[0] - __uint_as_float(hi[q] << 16), r1 = v[1] - __uint_as_float(hi[q] & 0xFFFF0000u);
                    mid[q] = gb_pair(r0, r1);
                    lo[q] = gb_pair(r0 - __uint_as_float(mid[q] << 16), r1 - __uint_as_float(mid[q] & 0xFFFF0000u));
                }
                bh[b] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                bm[b] = make_uint4(mid[0], mid[1], mid[2], mid[3]);
                bl[b] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
                // one column tile's loads at a time: registers for RT = 12
                __builtin_amdgcn_sched_barrier(0);
            }
            uint4 next = lut[(byte[0] >> (8 * kk)) & 0xFFu];
#pragma unroll
            for (int a = 0; a < RT; a++) {
                const gbbf16x8 A = __builtin_bit_cast(gbbf16x8, next);
                if (a + 1 < RT) next = lut[(byte[a + 1] >> (8 * kk)) & 0xFFu];
#pragma unroll
                for (int b = 0; b < CT; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(gbbf16x8, bl[b]), acc[a][b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < CT; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(gbbf16x8, bm[b]), acc[a][b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < CT; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(gbbf16x8, bh[b]), acc[a][b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int a = 0; a < RT; a++) {
            double* Ca = Cz + (int64_t)(row0 + 16 * a + 4 * kk) * cols_p + col0 + ii;
#pragma unroll
            for (int b = 0; b < CT; b++)
#pragma unroll
                for (int v = 0; v < 4; v++) Ca[(int64_t)v * cols_p + 16 * b] += (double)acc[a][b][v];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

PairShape pair_shape(int N, int M) {
    PairShape s;
    const int tiles = (1 + N * (N + 1) / 2 + 15) / 16;
    s.groups = (tiles + PAIR_RT_MAX - 1) / PAIR_RT_MAX;
    s.rt = (tiles + s.groups - 1) / s.groups;
    s.rows_p = s.groups * s.rt * 16;
    s.col_groups = ((M + 1) * (M + 2) + 16 * PAIR_CT - 1) / (16 * PAIR_CT);
    s.cols_p = s.col_groups * 16 * PAIR_CT;
    return s;
}

hipError_t launch_pair_planes(int64_t nblk, int N, int rows_p, const uint32_t* planes, uint32_t* out, hipStream_t stream) {
    const unsigned g = (unsigned)(nblk < 65535 ? nblk : 65535);
    hipLaunchKernelGGL(k_pair_planes, dim3(g), dim3(256), 0, stream, nblk, N, rows_p, planes, out);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pair_units(int64_t s0, int64_t n, int64_t nblk, int M, const void* Trec, const cx<double>* w,
                             const cx<double>* mean, float* out, hipStream_t stream) {
    if (nblk <= 0 || nblk > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_pair_units<T>), dim3((unsigned)nblk), dim3(256), 0, stream, s0, n, M,
                       reinterpret_cast<const cx<T>*>(Trec), w, mean, out);
    return hipGetLastError();
}
template hipError_t launch_pair_units<float>(int64_t, int64_t, int64_t, int, const void*, const cx<double>*, const cx<double>*,
                                             float*, hipStream_t);
template hipError_t launch_pair_units<double>(int64_t, int64_t, int64_t, int, const void*, const cx<double>*, const cx<double>*,
                                              float*, hipStream_t);

hipError_t launch_pair_moments(const PairShape& s, int64_t nblk, int splits, int M, const uint32_t* planes,
                               const float* units, double* C, hipStream_t stream) {
    if (nblk <= 0 || splits < 1 || s.rt < 1 || s.rt > PAIR_RT_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(s.groups * s.col_groups * splits));
#define RBM_PAIR_CASE(R_)                                                                                              \
    case R_:                                                                                                           \
        hipLaunchKernelGGL((k_pair_moments<R_>), grid, dim3(64), 0, stream, nblk, splits, s.groups, s.col_groups, M,   \
                           s.rows_p, s.cols_p, planes, units, C);                                                      \
        break;
    switch (s.rt) {
        RBM_PAIR_CASE(1) RBM_PAIR_CASE(2) RBM_PAIR_CASE(3) RBM_PAIR_CASE(4) RBM_PAIR_CASE(5) RBM_PAIR_CASE(6)
        RBM_PAIR_CASE(7) RBM_PAIR_CASE(8) RBM_PAIR_CASE(9) RBM_PAIR_CASE(10) RBM_PAIR_CASE(11) RBM_PAIR_CASE(12)
        default: return hipErrorInvalidValue;
    }
#undef RBM_PAIR_CASE
    return hipGetLastError();
}

// Sum of the sample splits into split 0, in order.
__global__ __launch_bounds__(256) void k_pair_sum(int64_t len, int splits, double* __restrict__ C) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < len; i += (int64_t)gridDim.x * blockDim.x) {
        double s = C[i];
        for (int z = 1; z < splits; z++) s += C[(int64_t)z * len + i];
        C[i] = s;
    }
}

RBM_DI int pair_row(int p, int q) {   // sign row of s_p s_q
    if (p == q) return 0;
    const int lo = p < q ? p : q, hi = p < q ? q : p;
    return 1 + hi * (hi - 1) / 2 + lo;
}
// <conj(t_j) t_j'> of sign row r
RBM_DI cx<double> pair_moment(const double* __restrict__ C, int cols_p, int r, int j, int jp) {
    const int hi = j > jp ? j : jp, lo = j > jp ? jp : j;
    const double* c = C + (int64_t)r * cols_p + 2 * (hi * (hi + 1) / 2 + lo);
    const double im = hi == lo ? 0.0 : c[1];
    // the column holds t_hi conj(t_lo)
    return mk(c[0], j > jp ? -im : im);
}

// mean of O_(p,j) = <s_p t_j> + mean_j <s_p>; first[p * (M + 1) + j], times n
__global__ __launch_bounds__(256) void k_pair_first(int N, int M, int cols_p, const cx<double>* __restrict__ mean,
                                                    const double* __restrict__ C, cx<double>* __restrict__ first) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (N + 1) * (M + 1)) return;
    const int p = e / (M + 1), j = e % (M + 1);
    const int r = pair_row(0, p);
    const cx<double> t = conj(pair_moment(C, cols_p, r, j, M));   // <t_j conj(t_M)>
    first[e] = j < M ? t + pair_moment(C, cols_p, r, M, M).re * mean[j] : t;
}

// The columns of the constant unit, sum s_r sqrt(w) conj(t_j) and, for j = M,
// sum s_r w, in FP64 for ensembles whose weights are not all 1.  The assembly
// multiplies them by unit means and takes their products away again, so a
// relative error e of them leaves e |mean|^2 in S, however small the entry.  As
// FP32 sums of FP32-rounded weights they left 9e-5 of sqrt(S_kk S_ll) for a
// plain state with biases around 0.5, 8e-4 at <s> = 0.999 and 0.2 at 0.9999 (12
// spins, 170 units, exact sum), now 3e-7; the Gram product leaves 1e-6 to 6e-6.
// Here every product is exact (two FP32 factors and a sign) and the sums are
// FP64, of the same rounded sqrt(w) and t as the other columns, so that S is the
// covariance of those values.  Weights of 1 don't need it: their sums are whole
// numbers, which the FP32 sums of 4096 samples hold exactly.
// v_mfma_f64_16x16x4f64 as below; MFMA e of a 32-sample block takes samples
// 8 (l / 16) + e, so that a lane's 8 samples are two 16-byte words.  A wavefront
// owns 4 row tiles and 2 column tiles of one sample split; part holds
// splits x rows_p x cols, cols = 2 (M + 1) rounded up to 32.  36 spins, 144
// units, 51 155 samples: 0.8 ms with the sum of the splits beside 5.5 ms of
// k_pair_moments, 30 TFLOP/s with about one wavefront a SIMD (the Gram product
// took 30.6 ms).
typedef double gbf64x4 __attribute__((ext_vector_type(4)));
constexpr int PAIRC_RT = 4, PAIRC_CT = 2;
static int pair_const_cols(int M) { return (2 * (M + 1) + 16 * PAIRC_CT - 1) / (16 * PAIRC_CT) * (16 * PAIRC_CT); }

__global__ __launch_bounds__(64) void k_pair_const(int64_t nblk, int splits, int groups, int M, int rows_p, int cols,
                                                   const uint32_t* __restrict__ planes, const float* __restrict__ units,
                                                   double* __restrict__ part) {
    constexpr int RT = PAIRC_RT, CT = PAIRC_CT;
    const int lane = threadIdx.x, kk = lane >> 4, ii = lane & 15;
    const int col_groups = cols / (16 * CT);
    const int grp = blockIdx.x % groups, rest = blockIdx.x / groups;
    const int col0 = (rest % col_groups) * 16 * CT, z = rest / col_groups;
    const int im = ii & 1;
    int row[RT], off[CT];
#pragma unroll
    for (int a = 0; a < RT; a++) {
        const int r = 16 * (grp * RT + a) + ii;
        row[a] = r < rows_p ? r : ii;   // tiles past the last repeat the first; they are not stored
    }
#pragma unroll
    for (int b = 0; b < CT; b++) {
        const int j = (col0 + 16 * b + ii) >> 1;
        off[b] = (j < M ? j : M) * 64 + 32 * im;
    }
    gbf64x4 acc[RT][CT];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < CT; b++) acc[a][b] = gbf64x4{0.0, 0.0, 0.0, 0.0};
    const int64_t per = (nblk + splits - 1) / splits;
    const int64_t b0 = z * per, b1 = b0 + per < nblk ? b0 + per : nblk;
    const int64_t ustride = (int64_t)(M + 1) * 64;
    for (int64_t blk = b0; blk < b1; blk++) {
        const float* U = units + blk * ustride + 8 * kk;
        float sw[8], t[CT][8];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            *reinterpret_cast<float4*>(sw + 4 * h) = *reinterpret_cast<const float4*>(U + M * 64 + 4 * h);
#pragma unroll
            for (int b = 0; b < CT; b++)
                *reinterpret_cast<float4*>(t[b] + 4 * h) = *reinterpret_cast<const float4*>(U + off[b] + 4 * h);
        }
        uint32_t byte[RT];
#pragma unroll
        for (int a = 0; a < RT; a++) byte[a] = planes[blk * rows_p + row[a]] >> (8 * kk);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            double bv[CT];
#pragma unroll
            for (int b = 0; b < CT; b++) bv[b] = (double)sw[e] * (double)(im ? -t[b][e] : t[b][e]);
#pragma unroll
            for (int a = 0; a < RT; a++) {
                const double av = (byte[a] >> e) & 1u ? 1.0 : -1.0;
#pragma unroll
                for (int b = 0; b < CT; b++) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[b], acc[a][b], 0, 0, 0);
            }
        }
    }
    double* out = part + (int64_t)z * rows_p * cols;
#pragma unroll
    for (int a = 0; a < RT; a++) {
        const int tile = grp * RT + a;
        if (16 * tile >= rows_p) break;
#pragma unroll
        for (int b = 0; b < CT; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) out[(int64_t)(16 * tile + kk + 4 * v) * cols + col0 + 16 * b + ii] += acc[a][b][v];
    }
}

// The splits added in order into the constant unit's columns of C
__global__ __launch_bounds__(256) void k_pair_const_sum(int splits, int M, int rows_p, int cols, int cols_p,
                                                        const double* __restrict__ part, double* __restrict__ C) {
    const int live = 2 * (M + 1);
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= (int64_t)rows_p * live) return;
    const int64_t r = e / live;
    const int col = (int)(e % live);
    double s = 0.0;
    for (int z = 0; z < splits; z++) s += part[((int64_t)z * rows_p + r) * cols + col];
    C[r * cols_p + M * (M + 1) + col] = s;
}

int64_t pair_const_len(const PairShape& s, int M) { return (int64_t)s.rows_p * pair_const_cols(M); }

int pair_const_splits(const PairShape& s, int M, int64_t nblk, int num_cus) {
    // about a wavefront per SIMD, at least 8 blocks each and at most 256 MiB of partials
    const int64_t wp = (int64_t)((s.rows_p / 16 + PAIRC_RT - 1) / PAIRC_RT) * (pair_const_cols(M) / (16 * PAIRC_CT));
    int64_t z = (4ll * num_cus + wp - 1) / wp;
    if (z > nblk / 8) z = nblk / 8;
    if (z > (256ll << 20) / (pair_const_len(s, M) * 8)) z = (256ll << 20) / (pair_const_len(s, M) * 8);
    return z < 1 ? 1 : (int)z;
}

hipError_t launch_pair_const(const PairShape& s, int64_t nblk, int splits, int M, const uint32_t* planes, const float* units,
                             double* part, hipStream_t stream) {
    if (nblk <= 0 || splits < 1 || s.rows_p <= 0 || s.rows_p % 16) return hipErrorInvalidValue;
    const int cols = pair_const_cols(M), groups = (s.rows_p / 16 + PAIRC_RT - 1) / PAIRC_RT;
    hipLaunchKernelGGL(k_pair_const, dim3((unsigned)(groups * (cols / (16 * PAIRC_CT)) * splits)), dim3(64), 0, stream, nblk,
                       splits, groups, M, s.rows_p, cols, planes, units, part);
    return hipGetLastError();
}

hipError_t launch_pair_const_sum(const PairShape& s, int splits, int M, const double* part, double* C, hipStream_t stream) {
    if (splits < 1) return hipErrorInvalidValue;
    const int64_t len = (int64_t)s.rows_p * 2 * (M + 1);
    hipLaunchKernelGGL(k_pair_const_sum, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, stream, splits, M, s.rows_p,
                       pair_const_cols(M), s.cols_p, part, C);
    return hipGetLastError();
}

// S_kl = <conj(O_k - <O_k>) (O_l - <O_l>)> = <conj(O_k) O_l> - (2 - <1>)
// conj(<O_k>) <O_l> with O_(p,j) = s_p (t_j + mean_j), averages over n and <1> =
// sum w / n (1 where psi is normalised); the upper triangle is the conjugate of
// the lower one
__global__ __launch_bounds__(256) void k_pair_assemble(int N, int M, int P, int cols_p, double inv, double eps,
                                                       const cx<double>* __restrict__ mean,
                                                       const cx<double>* __restrict__ first,
                                                       const double* __restrict__ C, cx<double>* __restrict__ S) {
    const int row = blockIdx.y, WN = M + N * M;
    const double twice = 2.0 - inv * pair_moment(C, cols_p, 0, M, M).re;
    auto spin = [&](int k) { return k < M ? 0 : k < WN ? 1 + (k - M) / M : 1 + k - WN; };
    auto unit = [&](int k) { return k < M ? k : k < WN ? (k - M) % M : M; };
    const int rp = spin(row), rj = unit(row);
    for (int col = blockIdx.x * blockDim.x + threadIdx.x; col < P; col += gridDim.x * blockDim.x) {
        const int cp = spin(col), cj = unit(col);
        const bool lower = row >= col;
        const int p = lower ? rp : cp, j = lower ? rj : cj, pl = lower ? cp : rp, jl = lower ? cj : rj;
        const int r = pair_row(p, pl);
        cx<double> m = pair_moment(C, cols_p, r, j, jl);
        const cx<double> mj = j < M ? conj(mean[j]) : mk(0.0, 0.0), ml = jl < M ? mean[jl] : mk(0.0, 0.0);
        // conj(t_j) mean_l + conj(mean_j) t_l + conj(mean_j) mean_l with t_M = 1
        if (jl < M) m = m + pair_moment(C, cols_p, r, j, M) * ml;
        if (j < M) m = m + mj * pair_moment(C, cols_p, r, M, jl);
        if (j < M && jl < M) m = m + pair_moment(C, cols_p, r, M, M).re * (mj * ml);
        cx<double> v = inv * m - (twice * inv * conj(first[p * (M + 1) + j])) * (inv * first[pl * (M + 1) + jl]);
        if (row == col) v = mk(v.re + eps, 0.0);
        S[(int64_t)row * P + col] = lower ? v : conj(v);
    }
}

hipError_t launch_pair_sum(const PairShape& s, int splits, double* C, hipStream_t stream) {
    const int64_t len = (int64_t)s.rows_p * s.cols_p;
    if (splits < 2) return hipSuccess;
    const unsigned g = (unsigned)((len + 255) / 256 < 8192 ? (len + 255) / 256 : 8192);
    hipLaunchKernelGGL(k_pair_sum, dim3(g), dim3(256), 0, stream, len, splits, C);
    return hipGetLastError();
}

// partials[b][j] = sum over chunk b of w |T_j|^2, a thread per unit with eight
// rows' loads in flight
template <typename T>
__global__ __launch_bounds__(256) void k_unit_squares(int64_t n, int M, int64_t chunk, const cx<T>* __restrict__ Trec,
                                                      const cx<double>* __restrict__ w, cx<double>* __restrict__ partials) {
    const int j = threadIdx.x;
    if (j >= M) return;
    const int64_t s0 = blockIdx.x * chunk, s1 = s0 + chunk < n ? s0 + chunk : n;
    double q = 0.0;
#pragma unroll 8
    for (int64_t s = s0; s < s1; s++) {
        const cx<double> t = to_d(Trec[s * M + j]);
        q = fm(w[s].re, fm(t.re, t.re, t.im * t.im), q);
    }
    partials[(int64_t)blockIdx.x * M + j] = mk(q, 0.0);
}

template <typename T>
hipError_t launch_unit_squares(int64_t n, int M, int64_t chunk, const void* Trec, const cx<double>* w, cx<double>* partials,
                               hipStream_t stream) {
    if (n <= 0 || chunk <= 0 || M <= 0 || M > 256) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_unit_squares<T>), dim3((unsigned)((n + chunk - 1) / chunk)), dim3(256), 0, stream, n, M, chunk,
                       reinterpret_cast<const cx<T>*>(Trec), w, partials);
    return hipGetLastError();
}
template hipError_t launch_unit_squares<float>(int64_t, int, int64_t, const void*, const cx<double>*, cx<double>*, hipStream_t);
template hipError_t launch_unit_squares<double>(int64_t, int, int64_t, const void*, const cx<double>*, cx<double>*, hipStream_t);

hipError_t launch_pair_assemble(const PairShape& s, int N, int M, int P, double inv, double eps, const cx<double>* mean,
                                const double* C, cx<double>* first, cx<double>* S, hipStream_t stream) {
    if (P <= 0 || P > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_pair_first, dim3((unsigned)(((N + 1) * (M + 1) + 255) / 256)), dim3(256), 0, stream, N, M, s.cols_p,
                       mean, C, first);
    hipLaunchKernelGGL(k_pair_assemble, dim3((unsigned)((P + 255) / 256), (unsigned)P), dim3(256), 0, stream, N, M, P,
                       s.cols_p, inv, eps, mean, first, C, S);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// get_S_matrix (source/network_functions/S_matrix.cu:10-58, CPU semantics),
// S_kl = inv sum_s O_k(s) conj(O_l(s)), unweighted and uncentred, in FP64: the
// same sign rows and unit pairs as k_pair_moments (T_j as they are, no
// weights), the product on v_mfma_f64_16x16x4f64 (lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16], accumulator v is row l / 16 + 4 v).
// A wavefront owns RT <= 4 row tiles and 2 column tiles of one sample split.
// N = 10, M = 20 (1024 states, 240 x 240): moments, sum and assembly 30 us, where
// one thread per entry running down all states took 608.
// ---------------------------------------------------------------------------
constexpr int PAIR64_RT_MAX = 4, PAIR64_CT = 2;

template <typename T, int RT>
__global__ __launch_bounds__(64) void k_pair_moments_f64(int64_t n, int64_t per, int N, int M, int groups, int col_groups,
                                                         int rows_p, int cols_p, const cx<T>* __restrict__ Trec,
                                                         const uint64_t* __restrict__ spins, double* __restrict__ C) {
    constexpr int CT = PAIR64_CT;
    const int lane = threadIdx.x, kk = lane >> 4, ii = lane & 15;
    const int grp = blockIdx.x % groups, rest = blockIdx.x / groups;
    const int cg = rest % col_groups, z = rest / col_groups;
    const int row0 = grp * RT * 16, col0 = cg * CT * 16;
    const int rows = 1 + N * (N + 1) / 2, pairs = (M + 1) * (M + 2) / 2;
    uint64_t m0[RT], m1[RT];   // the spins of each sign row (rows past the last read as 1)
#pragma unroll
    for (int a = 0; a < RT; a++) {
        const int r = row0 + 16 * a + ii;
        m0[a] = m1[a] = 0;
        if (r >= 1 && r < rows) {
            const int t = r - 1;
            int q = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)t)) * 0.5f);
            while (q * (q - 1) / 2 > t) q--;
            while ((q + 1) * q / 2 <= t) q++;
            const int p = t - q * (q - 1) / 2;
            flip_bit(m0[a], m1[a], q - 1);
            if (p > 0) flip_bit(m0[a], m1[a], p - 1);
        }
    }
    const int part = ii & 1;
    int jh[CT], jl[CT];
#pragma unroll
    for (int b = 0; b < CT; b++) {
        int c = (col0 + 16 * b + ii) >> 1;
        if (c >= pairs) c = 0;   // padding columns repeat the first pair; they are never read
        int j = (int)((sqrtf(8.0f * (float)c + 1.0f) - 1.0f) * 0.5f);
        while (j * (j + 1) / 2 > c) j--;
        while ((j + 1) * (j + 2) / 2 <= c) j++;
        jh[b] = j;
        jl[b] = c - j * (j + 1) / 2;
    }
    gbf64x4 acc[RT][CT];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < CT; b++) acc[a][b] = gbf64x4{0.0, 0.0, 0.0, 0.0};
    const int64_t s_begin = z * per, s_end = s_begin + per < n ? s_begin + per : n;
#pragma unroll 2
    for (int64_t s0 = s_begin; s0 < s_end; s0 += 4) {
        const int64_t s = s0 + kk;
        const bool ok = s < s_end;
        const int64_t sc = ok ? s : s_begin;
        const uint64_t w0 = ~spins[2 * sc], w1 = ~spins[2 * sc + 1];
        const cx<T>* Tr = Trec + sc * M;
        double bv[CT];
#pragma unroll
        for (int b = 0; b < CT; b++) {
            const cx<double> th = jh[b] < M ? to_d(Tr[jh[b] < M ? jh[b] : 0]) : mk(1.0, 0.0);
            const cx<double> tl = jl[b] < M ? to_d(Tr[jl[b] < M ? jl[b] : 0]) : mk(1.0, 0.0);
            // Re, Im of t_j conj(t_j')
            const double v = part ? fm(th.im, tl.re, -(th.re * tl.im)) : fm(th.re, tl.re, th.im * tl.im);
            bv[b] = ok ? v : 0.0;
        }
#pragma unroll
        for (int a = 0; a < RT; a++) {
            const int par = (__popcll(m0[a] & w0) + __popcll(m1[a] & w1)) & 1;
            const double av = par ? -1.0 : 1.0;
#pragma unroll
            for (int b = 0; b < CT; b++) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[b], acc[a][b], 0, 0, 0);
        }
    }
    double* Cz = C + (int64_t)z * rows_p * cols_p;
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < CT; b++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                Cz[(int64_t)(row0 + 16 * a + kk + 4 * v) * cols_p + col0 + 16 * b + ii] = acc[a][b][v];
}

// rows and columns below 2N (alpha, beta) are zero
__global__ __launch_bounds__(256) void k_s_ref_assemble(int N, int M, int P, int cols_p, double inv,
                                                        const double* __restrict__ C, cx<double>* __restrict__ S) {
    const int row = blockIdx.y, WN = M + N * M;
    auto spin = [&](int k) { return k < M ? 0 : k < WN ? 1 + (k - M) / M : 1 + k - WN; };
    auto unit = [&](int k) { return k < M ? k : k < WN ? (k - M) % M : M; };
    const int k = row - 2 * N;
    for (int col = blockIdx.x * blockDim.x + threadIdx.x; col < P; col += gridDim.x * blockDim.x) {
        const int l = col - 2 * N;
        cx<double> v = mk(0.0, 0.0);
        if (k >= 0 && l >= 0) v = inv * conj(pair_moment(C, cols_p, pair_row(spin(k), spin(l)), unit(k), unit(l)));
        S[(int64_t)row * P + col] = v;
    }
}

PairShape pair_shape_f64(int N, int M) {
    PairShape s;
    const int tiles = (1 + N * (N + 1) / 2 + 15) / 16;
    s.groups = (tiles + PAIR64_RT_MAX - 1) / PAIR64_RT_MAX;
    s.rt = (tiles + s.groups - 1) / s.groups;
    s.rows_p = s.groups * s.rt * 16;
    s.col_groups = ((M + 1) * (M + 2) + 16 * PAIR64_CT - 1) / (16 * PAIR64_CT);
    s.cols_p = s.col_groups * 16 * PAIR64_CT;
    return s;
}

template <typename T>
hipError_t launch_s_matrix_ref(const PairShape& s, int64_t n, int splits, int N, int M, int P, const void* Trec,
                               const uint64_t* spins, double inv, double* C, cx<double>* S, hipStream_t stream) {
    if (n <= 0 || splits < 1 || P <= 0 || P > 65535 || s.rt < 1 || s.rt > PAIR64_RT_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(s.groups * s.col_groups * splits));
    const int64_t per = ((n + splits - 1) / splits + 3) / 4 * 4;
    if (per * (splits - 1) >= n) return hipErrorInvalidValue;   // every split has samples
#define RBM_PAIR64_CASE(R_)                                                                                            \
    case R_:                                                                                                           \
        hipLaunchKernelGGL((k_pair_moments_f64<T, R_>), grid, dim3(64), 0, stream, n, per, N, M, s.groups,             \
                           s.col_groups, s.rows_p, s.cols_p, reinterpret_cast<const cx<T>*>(Trec), spins, C);           \
        break;
    switch (s.rt) {
        RBM_PAIR64_CASE(1) RBM_PAIR64_CASE(2) RBM_PAIR64_CASE(3) RBM_PAIR64_CASE(4)
        default: return hipErrorInvalidValue;
    }
#undef RBM_PAIR64_CASE
    const int64_t len = (int64_t)s.rows_p * s.cols_p;
    if (splits > 1)
        hipLaunchKernelGGL(k_pair_sum, dim3((unsigned)((len + 255) / 256 < 8192 ? (len + 255) / 256 : 8192)), dim3(256), 0,
                           stream, len, splits, C);
    hipLaunchKernelGGL(k_s_ref_assemble, dim3((unsigned)((P + 255) / 256), (unsigned)P), dim3(256), 0, stream, N, M, P,
                       s.cols_p, inv, C, S);
    return hipGetLastError();
}
template hipError_t launch_s_matrix_ref<float>(const PairShape&, int64_t, int, int, int, int, const void*, const uint64_t*,
                                               double, double*, cx<double>*, hipStream_t);
template hipError_t launch_s_matrix_ref<double>(const PairShape&, int64_t, int, int, int, int, const void*, const uint64_t*,
                                                double, double*, cx<double>*, hipStream_t);

}  // namespace rbmhip
