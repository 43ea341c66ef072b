// Masked autoregressive proposal (MADE, Germain et al. 2015) on gfx950:
// FP32 MFMA training kernels and a bfloat16-weight sampler.  The reference
// has no counterpart; the model is defined in the C ABI header.
//
// Device layout (padded to multiples of 64 so every GEMM tile is full):
//   Np = round_up(N, 64), Hp = round_up(H, 64)
//   W1  Hp x Np  FP32 (zero outside the mask and the padding)
//   b1  Hp,  W2  Np x Hp,  b2  Np
// Inference copies: W1t_bf  N x Hp bfloat16 (row i = column i of W1),
//                   W2_bf   N x Hp bfloat16 (row j of W2).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rbm_device.hpp"

namespace rbmhip {

struct MadeShape {
    int N, H, Np, Hp;
};

inline int made_pad(int x) { return (x + 63) / 64 * 64; }

// degree of hidden unit k: 1 + k mod (N - 1) (0 for N = 1)
__host__ __device__ inline int made_degree(int k, int N) { return N > 1 ? 1 + k % (N - 1) : 0; }

// Number of hidden units of degree <= j: the units output j reads.  Degree d
// (1 <= d <= N - 1) holds q + [d <= r] units, q = H / (N - 1), r = H mod (N - 1).
__host__ __device__ inline int made_prefix(int j, int N, int H) {
    if (N <= 1 || j >= N - 1) return H;
    if (j <= 0) return 0;
    const int q = H / (N - 1), r = H % (N - 1);
    return j * q + (j < r ? j : r);
}

// Hidden unit at position p of the degree-sorted order (ties by unit index);
// positions >= H are the zero padding units and map to themselves.
__host__ __device__ inline int made_sorted_unit(int p, int N, int H) {
    if (N <= 1 || p >= H) return p;
    const int q = H / (N - 1), r = H % (N - 1);
    int d1, t;   // degree - 1 and rank among the units of that degree
    if (p < r * (q + 1)) { d1 = p / (q + 1); t = p % (q + 1); }
    else { const int p2 = p - r * (q + 1); d1 = r + p2 / q; t = p2 % q; }
    return d1 + t * (N - 1);
}

// One training step.  Minibatch row s is sample s of `spins`, or, with draw,
// floor(u n) with u from Philox(seed; ctr = (step, s, 0, 4)); rows B .. Bp (a
// multiple of 64) are padding.  Parameters are one padded block [W1 (Hp x Np),
// b1 (Hp), W2 (Np x Hp), b2 (Np)]; the pass reads the weights from packed copies,
// W1, W2 and W2t (W2 transposed), that the update keeps.
// Left by the pass for the weight gradients, per tile of 16 samples: hT and daT
// [Hp][16], dlT [Np][16], xbits [Np] (bit k of entry i is input i of the tile's
// sample k), bias_part [Hp + Np] and the log q sum.
struct MadeStep {
    int N, B, Bp;
    int64_t n;
    int draw;
    uint32_t step, seed_lo, seed_hi;
    const uint64_t* spins;
    const float *W1, *b1, *W2, *b2, *W2t;
    float inv_batch;
    float *hT, *daT, *dlT;
    uint16_t* xbits;
    float* bias_part;     // (Bp / 16) x (Hp + Np)
    double* loss_part;    // Bp / 16
    float* wgrad_part;    // splits x padded
    int64_t off_b1, off_W2, off_b2, padded;
};
// Adam's arrays and the step's constants (c1, c2: bias corrections), or the
// gradient alone into `grad`
struct MadeUpdate {
    float *params, *m, *v, *grad;
    float c1, c2, lr, beta1, beta2, eps;
};
// packed = [W1, W2, W2t] in the order of the pass (3 Np Hp floats)
hipError_t launch_made_pack(const MadeShape& s, const float* W1, const float* W2, float* packed, hipStream_t stream);
hipError_t launch_made_pass(const MadeShape& s, const MadeStep& p, hipStream_t stream);
// sample splits of the weight gradients for Bp / 16 = tiles
int made_wgrad_splits(const MadeShape& s, int tiles);
hipError_t launch_made_wgrad(const MadeShape& s, const MadeStep& p, int splits, hipStream_t stream);
hipError_t launch_made_update(const MadeShape& s, const MadeUpdate& u, const MadeStep& p, int splits, float* packed,
                              hipStream_t stream);
// p[0 .. n) = 0 (a fill kernel, so the optimiser state can be cleared inside
// captured work)
hipError_t launch_zero(int64_t n, float* p, hipStream_t stream);
// bfloat16 inference copies of W1 (transposed) and W2 in the sampler's layout:
// hidden units in degree-sorted order (made_sorted_unit), row j of either
// matrix as Hp / 2 words, word 32 t + 2 l + b holding pair v = 2 t + b of
// lane l: sorted units 32 v + l (low half) and 32 v + 16 + l (high half);
// b1 permuted to the sorted order.
hipError_t launch_made_inference_weights(const MadeShape& s, const float* W1, const float* b1, const float* W2,
                                         uint16_t* W1t_bf, uint16_t* W2_bf, float* b1_sorted, hipStream_t stream);

struct MadeInf {
    int N, H, Hp;
    const uint16_t* W1t;   // N x Hp, sampler layout
    const uint16_t* W2;    // N x Hp, sampler layout
    const float* b1;       // Hp, degree-sorted (zero padded)
    const float* b2;       // >= N
};
size_t made_sampler_lds(const MadeInf& m);
int made_hidden_per_lane(int Hp);
// Autoregressive sampling of n configurations: proposal g draws its uniforms
// from Philox(seed; ctr = (g_lo, g_hi, call, 0x100 + j / 4)), word j % 4,
// u = (w + 0.5) 2^-32 in FP32, x_j = 1 iff u < sigmoid(l_j).
hipError_t launch_made_sample(const MadeInf& m, int64_t n, uint32_t seed_lo, uint32_t seed_hi, uint32_t call,
                              uint64_t* spins, double* log_q, hipStream_t stream);
// log q of given configurations with the sampler's arithmetic
hipError_t launch_made_log_q(const MadeInf& m, int64_t n, const uint64_t* spins, double* log_q, hipStream_t stream);

// Independent Metropolis-Hastings over precomputed proposals: chain c uses
// proposals t * chains + c for t = 0 .. therm + steps; proposal 0 starts the
// chain and t >= 1 is accepted iff u <= exp(2 (Re lp' - Re lp) + lq - lq'),
// u from Philox(seed; ctr = (c, t, call, 2)) in FP64.  Measured sample k of
// chain c is the configuration held after proposal therm + 1 + k.
// pass 0: runs[c] = number of runs of equal consecutive samples, counts[2c],
//         counts[2c + 1] = acceptances, rejections;
// pass 1: with run_offset[c] (exclusive prefix of runs), run r of chain c is
//         written at run_offset[c] + r: its configuration and its length
//         (run_mult); sample_run[k * chains + c] = the run holding sample k.
hipError_t launch_imh(int chains, int therm, int steps, const uint64_t* prop_spins, const cx<double>* log_psi,
                      const double* log_q, uint32_t seed_lo, uint32_t seed_hi, uint32_t call, int pass, uint32_t* runs,
                      const int64_t* run_offset, uint64_t* run_spins, double* run_mult, int64_t* sample_run,
                      uint32_t* counts, hipStream_t stream);

}  // namespace rbmhip
