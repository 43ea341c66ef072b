// gfx950 kernels of the masked autoregressive proposal (MADE):
//   k_made_pass           forward and backward pass of a training step (FP32 MFMA)
//   k_made_wgrad, k_made_update   weight gradients, bias sums and Adam
//   k_made_inf_weights    bfloat16 inference copies of W1 (transposed) and W2
//   k_made_sample<HPL,S,W1F>  autoregressive sampling / scoring, weights in LDS
//   k_imh                 independent Metropolis-Hastings over precomputed proposals
#include "made_kernels.hpp"

namespace rbmhip {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// Training.  One step of loss = -(1/B) sum_s log q(x_s) is three launches:
//   k_made_pass     forward and backward pass of 16 samples per workgroup
//   k_made_wgrad    weight gradients, split over the batch
//   k_made_update   sums of the splits, masks, Adam
// All products are FP32 MFMA (v_mfma_f32_16x16x4f32: lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16], accumulator v of lane l is
// D[4 (l / 16) + v][l % 16]), with the same FP32 values as a GEMM per product.
//
// In k_made_pass the samples are the columns of D, so a lane's four
// accumulators of one 16-unit tile are four units of one sample: exactly what
// it supplies as B operands (k = l / 16 of four MFMAs, one per v) to the next
// layer when the weights of MFMA v are those of units 16 t + 4 (l / 16) + v,
// which a lane reads as one 16-byte word.  Activations therefore stay in
// registers from the drawn sample to its back-propagated derivative, and the
// inputs come straight from the spin bits.  The pass leaves the activations,
// derivatives and bits that the weight gradients contract, 16 samples of a unit
// in 64 bytes, units of a tile one after the other, so that there a lane's four
// samples are one 16-byte word and 16 units 1 KiB in a row.
//
// N = 100, H = 256, batch 16 384: a step takes 83 us (pass 48, weight
// gradients 27, update 8); the three matrix products of the pass alone are 20
// at the FP32 matrix rate, those of the gradients 14, and the logits' FP32
// functions and bias sums 18 of vector instructions.  It took 257 as 12
// launches (index, gather, five tiled GEMMs through LDS at 34 TFLOP/s, column
// sums, Adam), 86 of them in column sums whose few workgroups ran down the
// batch one row after the other.
// ---------------------------------------------------------------------------
RBM_DI float sigmoidf_acc(float l) { return 1.0f / (1.0f + expf(-l)); }
RBM_DI float softplusf_acc(float l) { return fmaxf(l, 0.0f) + log1pf(expf(-fabsf(l))); }

// Weights in the order in which k_made_pass reads them: 16 x 16 tiles, tile
// (m, t) of a matrix with T tiles a row at 256 (m T + t), in it lane l's four
// weights, row l % 16, columns 4 (l / 16) .., at 4 l.  A load is 1 KiB in a row;
// read from the row-major parameters, 64 bytes of 16 rows a power of two apart,
// the pass took 55 us instead of 48 (N = 100, H = 256, 16 384 samples).
RBM_DI int64_t made_packed(int row, int col, int tiles) {
    return ((int64_t)(row >> 4) * tiles + (col >> 4)) * 256 + ((row & 15) + ((col & 12) << 2)) * 4 + (col & 3);
}

// w[m] = this lane's weights of tile (m0 + m, t)
template <int R> RBM_DI void made_tiles(floatx4* w, const float* __restrict__ W, int tiles, int m0, int t) {
    const float* q = W + (m0 * tiles + t) * 256 + (threadIdx.x & 63) * 4;
#pragma unroll
    for (int m = 0; m < R; m++) w[m] = *reinterpret_cast<const floatx4*>(q + m * tiles * 256);
}

// A workgroup of 4 wavefronts takes 16 samples; wavefront q has the hidden
// tiles q HT / 4 ..: its part of a, the part of l these units give (summed over
// the wavefronts in order through LDS), and its part of da.  The logits' losses
// and derivatives, a long chain of FP32 functions, are shared out the same way,
// so four wavefronts a SIMD overlap them with the others' matrix instructions
// (63 us a pass of 16 384 samples at one wavefront per 16 samples).
// NT, HT: 16-wide tiles of the padded inputs and hidden units.
template <int NT, int HT>
__global__ __launch_bounds__(256, HT <= 16 ? 4 : 2) void k_made_pass(MadeStep p) {
    constexpr int Np = 16 * NT, Hp = 16 * HT, HW = HT / 4, NW = NT / 4;
    __shared__ floatx4 lpart[4][NT][64];
    auto& dls = lpart[0];   // a wavefront replaces the sums it alone has read
    __shared__ double lsum[4];
    const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
    const int q = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int blk = blockIdx.x, s = 16 * blk + r;
    const bool valid = s < p.B;
    uint64_t w0 = 0, w1 = 0;
    if (valid) {
        int64_t src = s;
        if (p.draw) {
            const u32x4 x = philox(p.step, (uint32_t)s, 0u, 4u, p.seed_lo, p.seed_hi);
            src = (int64_t)(((double)x.x + 0.5) * (1.0 / 4294967296.0) * (double)p.n);
            src = src < p.n ? src : p.n - 1;
        }
        w0 = p.spins[2 * src];
        w1 = p.spins[2 * src + 1];
        mask_words(w0, w1, p.N);
    }
    {   // input bits of the 16 samples by spin, a quarter of the spins each
        const uint64_t w = (q * (Np / 4) < 64 ? w0 : w1) >> (q * (Np / 4) & 63);
        uint32_t mine = 0;
        for (int k = 0; k < Np / 4; k++) {
            const uint32_t m = (uint32_t)__ballot((int)((w >> k) & 1u)) & 0xFFFFu;
            mine = lane == k ? m : mine;
        }
        if (lane < Np / 4) p.xbits[(int64_t)blk * Np + q * (Np / 4) + lane] = (uint16_t)mine;
    }
    // a = W1 x + b1.  Of every product the weights of the next 16 inputs are
    // requested before the matrix instructions of the present ones.
    floatx4 a[HW];
#pragma unroll
    for (int m = 0; m < HW; m++) a[m] = *reinterpret_cast<const floatx4*>(p.b1 + 16 * (q * HW + m) + 4 * g);
    {
        floatx4 w[2][HW];
        made_tiles<HW>(w[0], p.W1, NT, q * HW, 0);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t + 1 < NT) made_tiles<HW>(w[(t + 1) & 1], p.W1, NT, q * HW, t + 1);
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t nib = (uint32_t)((t < 4 ? w0 >> (16 * t + 4 * g) : w1 >> (16 * t - 64 + 4 * g)) & 15u);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float x = (nib >> v) & 1u ? 1.0f : 0.0f;
#pragma unroll
                for (int m = 0; m < HW; m++)
                    a[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t & 1][m][v], x, a[m], 0, 0, 0);
            }
        }
    }
    // l = W2 relu(a) + b2
    {
        floatx4 l[NT];
#pragma unroll
        for (int m = 0; m < NT; m++) l[m] = floatx4{0.f, 0.f, 0.f, 0.f};
        float* hT = p.hT + ((int64_t)blk * Hp + 16 * q * HW) * 16 + 64 * g + r;
        floatx4 w[2][4];
        made_tiles<4>(w[0], p.W2, HT, 0, q * HW);
#pragma unroll
        for (int k = 0; k < HW * NW; k++) {   // four output tiles of one hidden tile
            const int t = k / NW, m0 = 4 * (k % NW);
            if (k + 1 < HW * NW) made_tiles<4>(w[(k + 1) & 1], p.W2, HT, 4 * ((k + 1) % NW), q * HW + (k + 1) / NW);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float h = fmaxf(a[t][v], 0.0f);
                if (m0 == 0) hT[256 * t + 16 * v] = h;
#pragma unroll
                for (int m = 0; m < 4; m++)
                    l[m0 + m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[k & 1][m][v], h, l[m0 + m], 0, 0, 0);
            }
        }
#pragma unroll
        for (int m = 0; m < NT; m++) lpart[q][m][lane] = l[m];
    }
    __syncthreads();
    // dl = (sigmoid(l) - x) / B, log q
    double loss = 0.0;
    float* dlT = p.dlT + (int64_t)blk * Np * 16 + 64 * g + r;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const int m = q * NW + k;
        floatx4 l = *reinterpret_cast<const floatx4*>(p.b2 + 16 * m + 4 * g);
#pragma unroll
        for (int z = 0; z < 4; z++) l += lpart[z][m][lane];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int j = 16 * m + 4 * g + v;
            const float x = bit_of(w0, w1, j) ? 1.0f : 0.0f;
            const bool live = valid && j < p.N;
            const float lv = l[v];
            if (live) loss += (double)(x * lv) - (double)softplusf_acc(lv);
            const float d = live ? (sigmoidf_acc(lv) - x) * p.inv_batch : 0.0f;
            l[v] = d;
            dlT[256 * m + 16 * v] = d;
            const float sum = row_sum16(d);
            if (r == 0) p.bias_part[(int64_t)blk * (Hp + Np) + Hp + j] = sum;
        }
        dls[m][lane] = l;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
    if (lane == 0) lsum[q] = loss;
    __syncthreads();
    if (threadIdx.x == 0) p.loss_part[blk] = ((lsum[0] + lsum[1]) + lsum[2]) + lsum[3];
    // da = (W2^T dl) [a > 0]
    floatx4 w[2][HW], d[HW];
#pragma unroll
    for (int m = 0; m < HW; m++) d[m] = floatx4{0.f, 0.f, 0.f, 0.f};
    made_tiles<HW>(w[0], p.W2t, NT, q * HW, 0);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (t + 1 < NT) made_tiles<HW>(w[(t + 1) & 1], p.W2t, NT, q * HW, t + 1);
        __builtin_amdgcn_sched_barrier(0);
        const floatx4 l = dls[t][lane];
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int m = 0; m < HW; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t & 1][m][v], l[v], d[m], 0, 0, 0);
    }
    float* daT = p.daT + ((int64_t)blk * Hp + 16 * q * HW) * 16 + 64 * g + r;
#pragma unroll
    for (int m = 0; m < HW; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float da = a[m][v] > 0.0f ? d[m][v] : 0.0f;
            daT[256 * m + 16 * v] = da;
            const float sum = row_sum16(da);
            if (r == 0) p.bias_part[(int64_t)blk * (Hp + Np) + 16 * (q * HW + m) + 4 * g + v] = sum;
        }
}

// dW1 = da^T x and dW2 = dl^T h.  A workgroup owns a 64 x 64 block of either
// and sample tiles z, z + splits, ..., in turn for its wavefronts, which read 16 samples of 64 + 64 rows per step (64 MFMAs), the
// next step's before them, and add their sums through LDS; part[z] holds both
// gradients at their places in the parameters.  Four wavefronts to a workgroup
// also keep the SIMDs evenly loaded: as single wavefronts they took 28 to 40 us
// (N = 100, H = 256, 16 384 samples) with where the launch before had left room.
template <bool FIRST>
RBM_DI void made_wgrad(const MadeStep& p, int Np, int Hp, int row0, int col0, int t0, int dt, int tiles, float* __restrict__ out,
                       floatx4 (*sums)[16][64]) {
    const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rows = FIRST ? Hp : Np, cols = FIRST ? Np : Hp;
    const float* A = (FIRST ? p.daT : p.dlT) + (row0 + r) * 16 + 4 * g;
    const float* Bm = p.hT + (col0 + r) * 16 + 4 * g;
    const uint16_t* X = p.xbits + col0 + r;
    floatx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 fa[2][4], fb[2][4];
    uint32_t xb[2][4];
    auto fetch = [&](int k, int t) {
#pragma unroll
        for (int i = 0; i < 4; i++) fa[k][i] = *reinterpret_cast<const floatx4*>(A + ((int64_t)t * rows + 16 * i) * 16);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (FIRST) xb[k][j] = X[(int64_t)t * cols + 16 * j];
            else fb[k][j] = *reinterpret_cast<const floatx4*>(Bm + ((int64_t)t * cols + 16 * j) * 16);
        }
    };
    auto step = [&](int k) {
        if (FIRST) {
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) fb[k][j][v] = (xb[k][j] >> (4 * g + v)) & 1u ? 1.0f : 0.0f;
        }
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[k][i][v], fb[k][j][v], acc[i][j], 0, 0, 0);
    };
    int t = t0 + wave * dt;
    dt *= 4;
    if (t < tiles) fetch(0, t);
    for (; t < tiles; t += 2 * dt) {
        if (t + dt < tiles) fetch(1, t + dt);
        __builtin_amdgcn_sched_barrier(0);
        step(0);
        if (t + 2 * dt < tiles) fetch(0, t + 2 * dt);
        __builtin_amdgcn_sched_barrier(0);
        if (t + dt < tiles) step(1);
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) sums[wave][4 * i + j][lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        floatx4 x = sums[0][4 * wave + j][lane];
#pragma unroll
        for (int z = 1; z < 4; z++) x += sums[z][4 * wave + j][lane];
#pragma unroll
        for (int v = 0; v < 4; v++) out[(int64_t)(row0 + 16 * wave + 4 * g + v) * cols + col0 + 16 * j + r] = x[v];
    }
}

// Workgroups go to the 8 dies in turn: all blocks of a split to one die, which
// so reads its samples from memory once, and with a multiple of 8 splits to the
// die whose workgroups of k_made_pass wrote them.
__global__ __launch_bounds__(256) void k_made_wgrad(MadeStep p, int Np, int Hp, int tiles, int splits) {
    __shared__ floatx4 sums[4][16][64];
    const int half = (Np / 64) * (Hp / 64);   // blocks of each gradient
    const int b = ((int)blockIdx.x / 8) % (2 * half), z = (int)blockIdx.x / (16 * half) * 8 + (int)blockIdx.x % 8;
    if (z >= splits) return;
    const bool first = b < half;              // dW1: Hp x Np, dW2: Np x Hp
    const int q = first ? b : b - half, cols = first ? Np / 64 : Hp / 64;
    const int row0 = 64 * (q / cols), col0 = 64 * (q % cols);
    float* out = p.wgrad_part + (int64_t)z * p.padded;
    if (first) made_wgrad<true>(p, Np, Hp, row0, col0, z, splits, tiles, out, sums);
    else made_wgrad<false>(p, Np, Hp, row0, col0, z, splits, tiles, out + p.off_W2, sums);
}

// Gradient of every parameter (the splits and the sample tiles' bias sums
// added in a fixed order, masked entries zero), then Adam (Kingma & Ba 2015),
// or the gradient alone when u.grad is set.  Weights: one thread per
// parameter; biases: workgroups past the weights' take 16 of them with 16
// threads each.
RBM_DI void made_apply(const MadeUpdate& u, int64_t e, float gk) {
    if (u.grad) { u.grad[e] = gk; return; }
    const float mk_ = u.beta1 * u.m[e] + (1.0f - u.beta1) * gk;
    const float vk = u.beta2 * u.v[e] + (1.0f - u.beta2) * gk * gk;
    u.m[e] = mk_;
    u.v[e] = vk;
    u.params[e] -= u.lr * (mk_ * u.c1) / (sqrtf(vk * u.c2) + u.eps);
}

// One weight into the packed copies: W1, W2 and W2 transposed, Np Hp floats each
RBM_DI void made_pack(const MadeShape& sh, bool first, int row, int col, float x, float* __restrict__ packed) {
    const int64_t W = (int64_t)sh.Np * sh.Hp;
    if (first) {
        packed[made_packed(row, col, sh.Np / 16)] = x;
    } else {
        packed[W + made_packed(row, col, sh.Hp / 16)] = x;
        packed[2 * W + made_packed(col, row, sh.Np / 16)] = x;
    }
}

__global__ __launch_bounds__(256) void k_made_update(MadeShape sh, MadeUpdate u, int splits, int tiles, int64_t off_b1,
                                                     int64_t off_W2, int64_t off_b2, int64_t padded, int weight_blocks,
                                                     const float* __restrict__ wpart, const float* __restrict__ bpart,
                                                     float* __restrict__ packed) {
    const int N = sh.N, H = sh.H, Np = sh.Np, Hp = sh.Hp;
    if ((int)blockIdx.x < weight_blocks) {
        const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
        const int64_t W = (int64_t)Np * Hp;
        if (k >= 2 * W) return;
        const bool first = k < W;
        const int64_t e = first ? k : off_W2 + (k - W);
        float x = 0.0f;
#pragma unroll 16
        for (int z = 0; z < splits; z++) x += wpart[(int64_t)z * padded + e];
        const int row = first ? (int)(k / Np) : (int)((k - W) / Hp), col = first ? (int)(k % Np) : (int)((k - W) % Hp);
        const bool ok = first ? row < H && col < N && col < made_degree(row, N) : row < N && col < H && made_degree(col, N) <= row;
        made_apply(u, e, ok ? x : 0.0f);
        if (!u.grad) made_pack(sh, first, row, col, u.params[e], packed);
        return;
    }
    __shared__ float red[16][17];
    const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
    const int k = ((int)blockIdx.x - weight_blocks) * 16 + x;   // b1, then b2
    float s = 0.0f;
#pragma unroll 16
    for (int t = y; t < tiles; t += 16) s += bpart[(int64_t)t * (Hp + Np) + k];
    red[y][x] = s;
    __syncthreads();
    if (y == 0) {
        for (int q = 1; q < 16; q++) s += red[q][x];
        const bool ok = k < Hp ? k < H : k - Hp < N;
        made_apply(u, k < Hp ? off_b1 + k : off_b2 + (k - Hp), ok ? s : 0.0f);
    }
}

__global__ __launch_bounds__(256) void k_made_pack(MadeShape sh, const float* __restrict__ W1, const float* __restrict__ W2,
                                                   float* __restrict__ packed) {
    const int64_t W = (int64_t)sh.Np * sh.Hp;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < 2 * W; k += (int64_t)gridDim.x * blockDim.x) {
        if (k < W) made_pack(sh, true, (int)(k / sh.Np), (int)(k % sh.Np), W1[k], packed);
        else made_pack(sh, false, (int)((k - W) / sh.Hp), (int)((k - W) % sh.Hp), W2[k - W], packed);
    }
}

hipError_t launch_made_pack(const MadeShape& s, const float* W1, const float* W2, float* packed, hipStream_t stream) {
    hipLaunchKernelGGL(k_made_pack, dim3(256), dim3(256), 0, stream, s, W1, W2, packed);
    return hipGetLastError();
}

int made_wgrad_splits(const MadeShape& s, int tiles) {
    // two workgroups a compute unit, at least 4 sample tiles a workgroup
    const int blocks = 2 * (s.Np / 64) * (s.Hp / 64);
    int z = 512 / blocks;
    if (z > tiles / 4) z = tiles / 4;
    if (z > 8) z -= z % 8;
    return z < 1 ? 1 : z;
}

hipError_t launch_made_pass(const MadeShape& sh, const MadeStep& p, hipStream_t stream) {
    if (p.Bp <= 0 || p.Bp % 64 || sh.Np % 64 || sh.Hp % 64) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(p.Bp / 16)), block(256);
#define RBM_PASS_CASE(NT_, HT_)                                                                  \
    if (sh.Np == 16 * NT_ && sh.Hp == 16 * HT_) {                                                \
        hipLaunchKernelGGL((k_made_pass<NT_, HT_>), grid, block, 0, stream, p);                  \
        return hipGetLastError();                                                                \
    }
#define RBM_PASS_ROW(HT_) RBM_PASS_CASE(4, HT_) RBM_PASS_CASE(8, HT_)
    RBM_PASS_ROW(4) RBM_PASS_ROW(8) RBM_PASS_ROW(12) RBM_PASS_ROW(16) RBM_PASS_ROW(20) RBM_PASS_ROW(24) RBM_PASS_ROW(28)
    RBM_PASS_ROW(32)
#undef RBM_PASS_ROW
#undef RBM_PASS_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_made_wgrad(const MadeShape& sh, const MadeStep& p, int splits, hipStream_t stream) {
    const int tiles = p.Bp / 16;
    if (splits < 1 || splits > tiles) return hipErrorInvalidValue;
    const int blocks = 2 * (sh.Np / 64) * (sh.Hp / 64);
    hipLaunchKernelGGL(k_made_wgrad, dim3((unsigned)(blocks * ((splits + 7) / 8 * 8))), dim3(256), 0, stream, p, sh.Np,
                       sh.Hp, tiles, splits);
    return hipGetLastError();
}

hipError_t launch_made_update(const MadeShape& sh, const MadeUpdate& u, const MadeStep& p, int splits, float* packed,
                              hipStream_t stream) {
    const int weight_blocks = (int)((2ll * sh.Np * sh.Hp + 255) / 256), bias_blocks = (sh.Hp + sh.Np) / 16;
    hipLaunchKernelGGL(k_made_update, dim3((unsigned)(weight_blocks + bias_blocks)), dim3(256), 0, stream, sh, u, splits,
                       p.Bp / 16, p.off_b1, p.off_W2, p.off_b2, p.padded, weight_blocks, p.wgrad_part, p.bias_part, packed);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_zero(int64_t n, float* __restrict__ p) {
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) p[k] = 0.0f;
}

hipError_t launch_zero(int64_t n, float* p, hipStream_t stream) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, stream, n, p);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_made_inf_weights(MadeShape s, const float* __restrict__ W1,
                                                          const float* __restrict__ b1, const float* __restrict__ W2,
                                                          uint16_t* __restrict__ W1t, uint16_t* __restrict__ W2b,
                                                          float* __restrict__ b1s) {
    const int64_t total = (int64_t)s.N * s.Hp;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(t / s.Hp), e = (int)(t % s.Hp);
        const int w = e >> 1, half = e & 1;                        // word w = 32 t + 2 l + b
        const int v = 2 * (w >> 5) + (w & 1), l = (w >> 1) & 15;   // pair v = 2 t + b of lane l
        const int p = 32 * v + 16 * half + l;                      // sorted position
        const int k = made_sorted_unit(p, s.N, s.H);
        const __bf16 a = (__bf16)W1[(long)k * s.Np + i];
        const __bf16 b = (__bf16)W2[(long)i * s.Hp + k];
        W1t[t] = __builtin_bit_cast(uint16_t, a);
        W2b[t] = __builtin_bit_cast(uint16_t, b);
    }
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < s.Hp; p += gridDim.x * blockDim.x)
        b1s[p] = b1[made_sorted_unit(p, s.N, s.H)];
}

hipError_t launch_made_inference_weights(const MadeShape& s, const float* W1, const float* b1, const float* W2,
                                         uint16_t* W1t_bf, uint16_t* W2_bf, float* b1_sorted, hipStream_t stream) {
    hipLaunchKernelGGL(k_made_inf_weights, dim3(256), dim3(256), 0, stream, s, W1, b1, W2, W1t_bf, W2_bf, b1_sorted);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Autoregressive sampling (SCORE = false) and scoring (SCORE = true).
// A 16-lane row owns two configurations (one above 256 hidden units),
// interleaved so that their serial per-position chains (dot product, row sum,
// sigmoid, update) overlap and each weight word read from LDS serves both.
// Hidden units are in degree-sorted order: lane l holds sorted units 16 u + l
// (u < HPL) as FP32 pre-activations a[u] and bfloat16 pairs hb[v] of
// relu(a[2v]), relu(a[2v + 1]).  With D_j units of degree <= j, the masks make
// output j read units [0, D_j) only and input j feed units [D_j, Hp) only, so
// per position j (D_j is the same for every lane, and whole 64-unit groups of
// zero weights are skipped):
//   l_j = b2_j + sum_{k < D_j} W2[j][k] relu(a_k)   (v_dot2c_f32_bf16, DPP row sum)
//   x_j drawn (or read), log q += log sigmoid(+-l_j)
//   a_k += x_j W1[k][j] for k >= D_j (an FMA with x_j in {0, 1}: a + W exactly
//   when x_j = 1, a unchanged when x_j = 0), relu(a) repacked in the groups
//   that output j + 1 reads
// Both weight matrices sit in LDS as bfloat16 (N x Hp each, the layout of
// launch_made_inference_weights), W1 expanded to FP32 when it fits (W1F).
// Uniforms: lane l of the row computes Philox blocks l and 16 + l of each of
// its configurations; position j reads word j % 4 of block j / 4 from its lane.
// ---------------------------------------------------------------------------
RBM_DI float dot2_bf16(uint32_t w, uint32_t h, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, h), c, false);
}
// relu as one v_max_f32.  fmaxf(x, 0) compiles to two (a v_max_f32 x, x that
// quiets a possible signalling NaN, then the max with 0); the pre-activations
// here are FMA results, never NaN, and both forms agree on every other value.
RBM_DI float relu(float x) {
    float r;
    asm("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(x));
    return r;
}
// log(1 + e) for e = exp(-|l|) in (0, 1]: the argument lies in (1, 2], so
// v_log_f32 (log2, about 1 ulp there) times ln 2 needs none of the
// denormal-range handling of logf.
RBM_DI float log_1p_e(float e) { return __builtin_amdgcn_logf(1.0f + e) * 0.6931471805599453f; }
RBM_DI uint32_t pack_relu_bf16(float lo, float hi) {
    bf16x2 v;
    v.x = (__bf16)relu(lo);
    v.y = (__bf16)relu(hi);
    return __builtin_bit_cast(uint32_t, v);
}

int made_hidden_per_lane(int Hp) { return Hp / 16; }

// configurations per 16-lane row: two while both fit in the 128 registers a
// 1024-thread workgroup allows (up to 256 hidden units), else one
constexpr int made_cpr(int hpl) { return hpl <= 16 ? 2 : 1; }

RBM_DI float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
RBM_DI float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// W1F: W1 sits in LDS as FP32, expanded from its bfloat16 copy at the start
// (the same values), so the hidden-unit updates need no unpacking; used when
// N x Hp x 6 bytes fit in LDS.  Otherwise W1 stays bfloat16 like W2.
template <int HPL, bool SCORE, bool W1F>
__global__ __launch_bounds__(1024) void k_made_sample(MadeInf m, int64_t n, uint32_t seed_lo, uint32_t seed_hi,
                                                      uint32_t call, const uint64_t* __restrict__ in_spins,
                                                      uint64_t* __restrict__ out_spins, double* __restrict__ log_q) {
    static_assert(HPL % 4 == 0, "hidden units per lane must be a multiple of 4");
    constexpr int C = made_cpr(HPL);
    constexpr int V = HPL / 2;   // bfloat16 pairs per lane
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int N = m.N, Hp = m.Hp;
    uint16_t* sW2 = reinterpret_cast<uint16_t*>(smem_raw + (size_t)N * Hp * (W1F ? 4 : 2));
    {
        const uint4* g1 = reinterpret_cast<const uint4*>(m.W1t);
        const uint4* g2 = reinterpret_cast<const uint4*>(m.W2);
        uint4* l2 = reinterpret_cast<uint4*>(sW2);
        const int nv = N * Hp / 8;
        for (int k = threadIdx.x; k < nv; k += blockDim.x) {
            const uint4 w = g1[k];
            if (W1F) {
                float4* l1 = reinterpret_cast<float4*>(smem_raw) + 2 * k;
                l1[0] = make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
                l1[1] = make_float4(bf16_lo(w.z), bf16_hi(w.z), bf16_lo(w.w), bf16_hi(w.w));
            } else {
                reinterpret_cast<uint4*>(smem_raw)[k] = w;
            }
            l2[k] = g2[k];
        }
    }
    __syncthreads();
    const uint32_t* sW1w = reinterpret_cast<const uint32_t*>(smem_raw);
    const float* sW1f = reinterpret_cast<const float*>(smem_raw);
    const uint32_t* sW2w = reinterpret_cast<const uint32_t*>(sW2);
    const int lane = threadIdx.x & 15, rows = blockDim.x >> 4;
    const int row_base = (threadIdx.x & 63) & ~15;

    for (int64_t g0 = ((int64_t)blockIdx.x * rows + (threadIdx.x >> 4)) * C; g0 < n; g0 += (int64_t)gridDim.x * rows * C) {
        int64_t gc[C];
        uint32_t uw[C][8];
        uint64_t x0[C], x1[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            gc[c] = g0 + c < n ? g0 + c : g0;      // a missing partner repeats the first (not written)
            x0[c] = 0; x1[c] = 0;
            if (SCORE) {
                x0[c] = in_spins[2 * gc[c]];
                x1[c] = in_spins[2 * gc[c] + 1];
            } else {
                const int64_t g = gc[c];
                const u32x4 r0 = philox((uint32_t)g, (uint32_t)(g >> 32), call, 0x100u + lane, seed_lo, seed_hi);
                uw[c][0] = r0.x; uw[c][1] = r0.y; uw[c][2] = r0.z; uw[c][3] = r0.w;
                if (N > 64) {
                    const u32x4 r1 = philox((uint32_t)g, (uint32_t)(g >> 32), call, 0x110u + lane, seed_lo, seed_hi);
                    uw[c][4] = r1.x; uw[c][5] = r1.y; uw[c][6] = r1.z; uw[c][7] = r1.w;
                } else {
                    uw[c][4] = uw[c][5] = uw[c][6] = uw[c][7] = 0u;
                }
                // each word becomes its uniform u = (w + 1/2) 2^-32 once, here,
                // as FP32 bits, instead of at every position that reads it
#pragma unroll
                for (int k = 0; k < 8; k++)
                    uw[c][k] = __float_as_uint(__builtin_fmaf((float)uw[c][k], 2.3283064365386963e-10f,
                                                              1.1641532182693481e-10f));
            }
        }
        float a[C][HPL];
        uint32_t hb[C][V];
        double lq[C];
        // b1 is re-read (cache hits) rather than held in registers for the whole loop
#pragma unroll
        for (int c = 0; c < C; c++) {
            lq[c] = 0.0;
#pragma unroll
            for (int u = 0; u < HPL; u++) a[c][u] = m.b1[16 * u + lane];
#pragma unroll
            for (int v = 0; v < V; v++) hb[c][v] = pack_relu_bf16(a[c][2 * v], a[c][2 * v + 1]);
        }
        // C == 2 sampling: each lane records its own half's configuration
        // (lanes 0-7 configuration 0, lanes 8-15 configuration 1), bits of the
        // current 32-position word in wacc, whole words in own0 / own1
        uint32_t wacc = 0;
        uint64_t own0 = 0, own1 = 0;
        for (int jb = 0; jb < N; jb += 4) {
            uint32_t cur[C][4];
            if (!SCORE) {
                const int b = jb >> 2;
                const int src = row_base | (b & 15);
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        cur[c][q] = (uint32_t)__shfl((int)((b >> 4) ? uw[c][4 + q] : uw[c][q]), src, 64);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int j = jb + q;
                if (j >= N) break;
                const int D = made_prefix(j, N, m.H);
                // pairs 2t, 2t + 1 (64 sorted units) per branch and LDS read
                const uint2* w2 = reinterpret_cast<const uint2*>(sW2w + (size_t)j * (Hp / 2)) + lane;
                const uint2* w1 = reinterpret_cast<const uint2*>(sW1w + (size_t)j * (Hp / 2)) + lane;
                const float4* w1f = reinterpret_cast<const float4*>(sW1f + (size_t)j * Hp) + lane;
                float s0[C], s1[C];
#pragma unroll
                for (int c = 0; c < C; c++) { s0[c] = 0.0f; s1[c] = 0.0f; }
#pragma unroll
                for (int t = 0; t < V / 2; t++) {
                    if (64 * t < D) {
                        const uint2 w = w2[16 * t];
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            s0[c] = dot2_bf16(w.x, hb[c][2 * t], s0[c]);
                            s1[c] = dot2_bf16(w.y, hb[c][2 * t + 1], s1[c]);
                        }
                    }
                }
                const float b2j = m.b2[j];
                float xf[C];
                if constexpr (C == 2) {
                    // The two configurations share one logit / sampling pass: lanes 0-7
                    // of the row carry configuration 0 and lanes 8-15 configuration 1.
                    // Half sums: a = t0[l] + t0[l + 8] (l < 8) or t1[l] + t1[l - 8], then
                    // half-row mirror and two quad permutations add each half's 8 lanes.
                    const bool lo = lane < 8;
                    const float t0 = s0[0] + s1[0], t1 = s0[1] + s1[1];
                    float a = (lo ? t0 : t1) + dpp<0x128>(lo ? t1 : t0);   // row_ror:8
                    a += dpp<0x141>(a);                                     // row_half_mirror
                    a += dpp<0xB1>(a);                                      // quad_perm 1,0,3,2
                    a += dpp<0x4E>(a);                                      // quad_perm 2,3,0,1
                    const float l = a + b2j;
                    const float e = __expf(-fabsf(l));
                    const float L1 = log_1p_e(e);
                    bool x;
                    if (SCORE) {
                        x = lo ? bit_of(x0[0], x1[0], j) != 0 : bit_of(x0[1], x1[1], j) != 0;
                    } else {
                        const float r = __builtin_amdgcn_rcpf(1.0f + e);
                        const float p = l >= 0.0f ? r : e * r;
                        const float u = __uint_as_float(lo ? cur[0][q] : cur[1][q]);
                        x = u < p;
                    }
                    // log sigmoid(l) = -(max(-l, 0) + log(1 + e^-|l|)), log(1 - sigmoid(l)) = -(max(l, 0) + ...)
                    lq[0] -= (double)((x ? fmaxf(-l, 0.0f) : fmaxf(l, 0.0f)) + L1);
                    // each half holds one decision: swap halves to give every lane both
                    const float xm = x ? 1.0f : 0.0f, xo = dpp<0x128>(xm);
                    xf[0] = lo ? xm : xo;
                    xf[1] = lo ? xo : xm;
                    if (!SCORE) wacc |= x ? 1u << (j & 31) : 0u;
                } else {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        const float l = row_sum16(s0[c] + s1[c]) + b2j;
                        const float e = __expf(-fabsf(l));
                        const float L1 = log_1p_e(e);
                        bool x;
                        if (SCORE) {
                            x = bit_of(x0[c], x1[c], j) != 0;
                        } else {
                            const float r = __builtin_amdgcn_rcpf(1.0f + e);
                            const float p = l >= 0.0f ? r : e * r;
                            const float u = __uint_as_float(cur[c][q]);
                            x = u < p;
                            const uint64_t bit = x ? (uint64_t)1 << (j & 63) : 0u;
                            if (j < 64) x0[c] |= bit; else x1[c] |= bit;
                        }
                        lq[c] -= (double)((x ? fmaxf(-l, 0.0f) : fmaxf(l, 0.0f)) + L1);
                        xf[c] = x ? 1.0f : 0.0f;
                    }
                }
                // Only the groups that output j + 1 reads ([0, D_{j+1})) are
                // repacked: a group above that bound is packed by a later
                // update before any output reads it, and a group below D_j
                // receives no more updates.
                const int Dn = made_prefix(j + 1, N, m.H);
#pragma unroll
                for (int t = 0; t < V / 2; t++) {
                    if (64 * t + 64 > D) {
                        // the 4 weights of pairs 2t, 2t + 1 of this lane
                        float wv[4];
                        if (W1F) {
                            const float4 w = w1f[16 * t];
                            wv[0] = w.x; wv[1] = w.y; wv[2] = w.z; wv[3] = w.w;
                        } else {
                            const uint2 w = w1[16 * t];
                            wv[0] = bf16_lo(w.x); wv[1] = bf16_hi(w.x); wv[2] = bf16_lo(w.y); wv[3] = bf16_hi(w.y);
                        }
                        const bool repack = 64 * t < Dn;
#pragma unroll
                        for (int b = 0; b < 2; b++) {
                            const int v = 2 * t + b;
                            const float wlo = wv[2 * b], whi = wv[2 * b + 1];
#pragma unroll
                            for (int c = 0; c < C; c++) {
                                a[c][2 * v] = __builtin_fmaf(xf[c], wlo, a[c][2 * v]);
                                a[c][2 * v + 1] = __builtin_fmaf(xf[c], whi, a[c][2 * v + 1]);
                            }
                        }
                        if (repack) {
#pragma unroll
                            for (int b = 0; b < 2; b++)
#pragma unroll
                                for (int c = 0; c < C; c++)
                                    hb[c][2 * t + b] = pack_relu_bf16(a[c][4 * t + 2 * b], a[c][4 * t + 2 * b + 1]);
                        }
                    }
                }
            }
            // positions jb .. jb + 3 share one 32-bit word (jb is a multiple of 4)
            if (C == 2 && !SCORE && (((jb + 4) & 31) == 0 || jb + 4 >= N)) {
                const int wi = jb >> 5;
                if (wi == 0) own0 |= wacc;
                else if (wi == 1) own0 |= (uint64_t)wacc << 32;
                else if (wi == 2) own1 |= wacc;
                else own1 |= (uint64_t)wacc << 32;
                wacc = 0;
            }
        }
        // configuration c is written by lane 8 c (with two configurations per row,
        // lanes 0-7 accumulated configuration 0's log q in lq[0] and its spins in
        // own0 / own1, lanes 8-15 configuration 1's)
#pragma unroll
        for (int c = 0; c < C; c++) {
            if (lane == 8 * c && g0 + c < n) {
                if (!SCORE) {
                    out_spins[2 * (g0 + c)] = C == 2 ? own0 : x0[c];
                    out_spins[2 * (g0 + c) + 1] = C == 2 ? own1 : x1[c];
                }
                log_q[g0 + c] = C == 2 ? lq[0] : lq[c];
            }
        }
    }
}

#define RBM_HPL_LIST(X) X(4) X(8) X(12) X(16) X(20) X(24) X(28) X(32)

size_t made_sampler_lds(const MadeInf& m) { return (size_t)2 * m.N * m.Hp * sizeof(uint16_t); }

static hipError_t launch_made_common(const MadeInf& m, int64_t n, uint32_t seed_lo, uint32_t seed_hi, uint32_t call,
                                     const uint64_t* in_spins, uint64_t* out_spins, double* log_q, bool score,
                                     hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    if (made_sampler_lds(m) > 160 * 1024) return hipErrorInvalidValue;
    // sampling holds W1 as FP32 when it fits (scoring uses the bfloat16 layout;
    // both read the same weight values)
    const size_t lds_f = (size_t)m.N * m.Hp * 6;
    const bool w1f = !score && lds_f <= 160 * 1024;
    const size_t lds = w1f ? lds_f : made_sampler_lds(m);
    const int hpl = made_hidden_per_lane(m.Hp);
    const int rows = 64;
    int64_t blocks = (n + rows * made_cpr(hpl) - 1) / (rows * made_cpr(hpl));
    int dev = 0, cus = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (blocks > cus) blocks = cus;
    const dim3 grid((unsigned)blocks), block(rows * 16);
#define RBM_MADE_CASE(H)                                                                                           \
    case H:                                                                                                        \
        if (score) {                                                                                               \
            (void)hipFuncSetAttribute((const void*)&k_made_sample<H, true, false>,                                 \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                        \
            hipLaunchKernelGGL((k_made_sample<H, true, false>), grid, block, lds, stream, m, n, seed_lo, seed_hi,    \
                               call, in_spins, out_spins, log_q);                                                   \
        } else if (w1f) {                                                                                          \
            (void)hipFuncSetAttribute((const void*)&k_made_sample<H, false, true>,                                 \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                        \
            hipLaunchKernelGGL((k_made_sample<H, false, true>), grid, block, lds, stream, m, n, seed_lo, seed_hi,   \
                               call, in_spins, out_spins, log_q);                                                   \
        } else {                                                                                                   \
            (void)hipFuncSetAttribute((const void*)&k_made_sample<H, false, false>,                                \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                        \
            hipLaunchKernelGGL((k_made_sample<H, false, false>), grid, block, lds, stream, m, n, seed_lo, seed_hi,  \
                               call, in_spins, out_spins, log_q);                                                   \
        }                                                                                                          \
        break;
    switch (hpl) {
        RBM_HPL_LIST(RBM_MADE_CASE)
        default: return hipErrorInvalidValue;
    }
#undef RBM_MADE_CASE
    return hipGetLastError();
}

hipError_t launch_made_sample(const MadeInf& m, int64_t n, uint32_t seed_lo, uint32_t seed_hi, uint32_t call,
                              uint64_t* spins, double* log_q, hipStream_t stream) {
    return launch_made_common(m, n, seed_lo, seed_hi, call, nullptr, spins, log_q, false, stream);
}

hipError_t launch_made_log_q(const MadeInf& m, int64_t n, const uint64_t* spins, double* log_q, hipStream_t stream) {
    return launch_made_common(m, n, 0, 0, 0, spins, nullptr, log_q, true, stream);
}

// ---------------------------------------------------------------------------
// Independent Metropolis-Hastings, one thread per chain.  A rejected proposal
// repeats the held configuration, so the measured samples of a chain form runs
// of equal configurations.  Pass 0 counts the runs of each chain; pass 1 (with
// run offsets) writes each run's configuration once with its length as the
// multiplicity, and the run of every sample.  Both passes replay the same
// decisions.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_imh(int chains, int therm, int steps, const uint64_t* __restrict__ prop,
                                             const cx<double>* __restrict__ lp, const double* __restrict__ lq,
                                             uint32_t seed_lo, uint32_t seed_hi, uint32_t call, int pass,
                                             uint32_t* __restrict__ runs, const int64_t* __restrict__ run_offset,
                                             uint64_t* __restrict__ run_spins, double* __restrict__ run_mult,
                                             int64_t* __restrict__ sample_run, uint32_t* __restrict__ counts) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= chains) return;
    int64_t cur = c;
    double lpc = lp[cur].re, lqc = lq[cur];
    uint32_t acc = 0, nrun = 0, len = 0;
    const int total = therm + steps;
    const int64_t off = pass ? run_offset[c] : 0;
    for (int t = 1; t <= total; t++) {
        const int64_t g = (int64_t)t * chains + c;
        const double lpg = lp[g].re, lqg = lq[g];
        const double r = 2.0 * (lpg - lpc) + lqc - lqg;
        const u32x4 R = philox((uint32_t)c, (uint32_t)t, call, 2u, seed_lo, seed_hi);
        const double u = ((double)R.x + 0.5) * (1.0 / 4294967296.0);
        const bool accept = u <= exp(r);
        if (accept) {
            cur = g;
            lpc = lpg;
            lqc = lqg;
            acc++;
        }
        if (t > therm) {
            const int k = t - therm - 1;
            if (k == 0 || accept) {
                // a new run starts: close the previous one
                if (pass && nrun > 0) run_mult[off + nrun - 1] = (double)len;
                if (pass) {
                    run_spins[2 * (off + nrun)] = prop[2 * cur];
                    run_spins[2 * (off + nrun) + 1] = prop[2 * cur + 1];
                }
                nrun++;
                len = 0;
            }
            len++;
            if (pass) sample_run[(int64_t)k * chains + c] = off + nrun - 1;
        }
    }
    if (pass) {
        if (nrun > 0) run_mult[off + nrun - 1] = (double)len;
    } else {
        runs[c] = nrun;
        if (counts) {
            counts[2 * c] = acc;
            counts[2 * c + 1] = (uint32_t)total - acc;
        }
    }
}

hipError_t launch_imh(int chains, int therm, int steps, const uint64_t* prop_spins, const cx<double>* log_psi,
                      const double* log_q, uint32_t seed_lo, uint32_t seed_hi, uint32_t call, int pass, uint32_t* runs,
                      const int64_t* run_offset, uint64_t* run_spins, double* run_mult, int64_t* sample_run,
                      uint32_t* counts, hipStream_t stream) {
    hipLaunchKernelGGL(k_imh, dim3((chains + 255) / 256), dim3(256), 0, stream, chains, therm, steps, prop_spins,
                       log_psi, log_q, seed_lo, seed_hi, call, pass, runs, run_offset, run_spins, run_mult, sample_run,
                       counts);
    return hipGetLastError();
}

}  // namespace rbmhip
