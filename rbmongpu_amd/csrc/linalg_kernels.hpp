// FP64 complex Cholesky factorisation and solve (row-major n x n; the factor
// overwrites the lower triangle).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "rbm_device.hpp"

namespace rbmhip {

// A = L L^H in place (lower triangle); *info (zeroed by the caller) receives
// the 1-based index of the first non-positive pivot, 0 if none.
// (D: CHOL_WORK elements of scratch)
constexpr int CHOL_WORK = 128 * 128;
hipError_t launch_cholesky(int n, cx<double>* A, cx<double>* D, int* info, hipStream_t stream);
// x <- (L L^H)^{-1} x with the factor from launch_cholesky
hipError_t launch_cholesky_solve(int n, const cx<double>* L, cx<double>* x, hipStream_t stream);
// C += A^T A on the lower 128 x 128 tiles of the FP64 matrix C (ld x ld) for
// a K x ld FP32 matrix A given split into three bfloat16 parts per 32-row
// block ([block][part][column][32 rows], as launch_o_split3 writes it), the
// product formed on the bfloat16 matrix cores with FP32 accuracy; ld a
// multiple of 128, K of 64.  Tiles above the diagonal are not touched.
// order (n_order entries, from gram_tile_order) assigns the tiles to
// workgroups.
hipError_t launch_gram_lower(int ld, int K, const uint32_t* A, double* C, const int2* order, int n_order,
                             hipStream_t stream);
// Fills order with the workgroup-to-tile map of launch_gram_lower for ld
// (entries (bm, bn) with bn <= bm, or (-1, -1)); returns the number of tiles.
int gram_tile_order(int ld, std::vector<int2>& order);
// Second moments of the O_k by pairs (gram_kernels.hip).  rows_p sign rows
// (row 0 is 1, row 1 + q (q - 1) / 2 + p is s_p s_q for p < q <= N, s_0 = 1) in
// `groups` groups of rt 16-row tiles, cols_p real columns (2 c + part for unit
// pair c = j (j + 1) / 2 + j', j' <= j <= M, unit M constant).
struct PairShape {
    int rt, groups, rows_p, col_groups, cols_p;
};
PairShape pair_shape(int N, int M);
// Sign bits of the rows per 32-sample block (nblk x rows_p words) from the
// spin bit planes (nblk x N words)
hipError_t launch_pair_planes(int64_t nblk, int N, int rows_p, const uint32_t* planes, uint32_t* out, hipStream_t stream);
// sqrt(w) (T_j - mean_j) of samples [s0, s0 + 32 nblk) (zero past n) as
// [block][unit 0..M][Re, Im][32 samples]; Trec holds cx<T>, M per sample
template <typename T>
hipError_t launch_pair_units(int64_t s0, int64_t n, int64_t nblk, int M, const void* Trec, const cx<double>* w,
                             const cx<double>* mean, float* out, hipStream_t stream);
// C[z][row][col] += sum over the blocks of split z (splits equal ranges of the nblk blocks)
hipError_t launch_pair_moments(const PairShape& s, int64_t nblk, int splits, int M, const uint32_t* planes,
                               const float* units, double* C, hipStream_t stream);
// The constant unit's columns in FP64, for weights other than 1: part (splits x
// pair_const_len, zeroed by the caller) += the blocks' sums, and their total into
// C[0] after launch_pair_sum
int64_t pair_const_len(const PairShape& s, int M);
int pair_const_splits(const PairShape& s, int M, int64_t nblk, int num_cus);
hipError_t launch_pair_const(const PairShape& s, int64_t nblk, int splits, int M, const uint32_t* planes, const float* units,
                             double* part, hipStream_t stream);
hipError_t launch_pair_const_sum(const PairShape& s, int splits, int M, const double* part, double* C, hipStream_t stream);
// Adds the splits into C[0]
hipError_t launch_pair_sum(const PairShape& s, int splits, double* C, hipStream_t stream);
// partials[b][j] = sum of w |T_j|^2 over samples b chunk .. (M <= 256 units);
// partials holds ceil(n / chunk) x M
template <typename T>
hipError_t launch_unit_squares(int64_t n, int M, int64_t chunk, const void* Trec, const cx<double>* w, cx<double>* partials,
                               hipStream_t stream);
// S (P x P, eps added on the diagonal) from C[0]; mean holds M values, first
// (N + 1) x (M + 1) scratch
hipError_t launch_pair_assemble(const PairShape& s, int N, int M, int P, double inv, double eps, const cx<double>* mean,
                                const double* C, cx<double>* first, cx<double>* S, hipStream_t stream);
// S_kl = inv sum_s O_k conj(O_l) in FP64 (P x P with the 2N zero rows and
// columns of the axis angles first) over n samples in `splits` equal ranges of
// whole 4-sample steps, none of them empty; C holds splits x rows_p x cols_p
PairShape pair_shape_f64(int N, int M);
template <typename T>
hipError_t launch_s_matrix_ref(const PairShape& s, int64_t n, int splits, int N, int M, int P, const void* Trec,
                               const uint64_t* spins, double inv, double* C, cx<double>* S, hipStream_t stream);
// out[z] = X_z^T Y_z (ldx x ldy) for the row ranges z = 0 .. splits - 1 of
// length K / splits of row-major K x ldx and K x ldy operands (same MFMA
// tiles); ldx and ldy multiples of 128, K a multiple of 16 splits.
hipError_t launch_gemm_tn_splitk(int ldx, int ldy, int64_t K, int splits, const float* X, const float* Y, float* out,
                                 hipStream_t stream);
// acc[i] += sum over z of part[z n + i] (FP64, fixed order)
hipError_t launch_accum_splits_f64(int64_t n, int splits, const float* part, double* acc, hipStream_t stream);

}  // namespace rbmhip
