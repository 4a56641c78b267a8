// ipf_learned.hip -- the learned return-branch predictor: a 7 -> 64 -> 64 -> 6
// MLP (ReLU, BF16 weights and activations as MFMA operands, FP32
// accumulation) trained on the GPU on pairs the exact return map emits.
//
//   inputs  x = (s1/c, s2/c, s3/c, ln c, phi, psi, alpha): trial principal
//           stresses (descending, from the spectral decomposition of the
//           trial stress), material, accumulated plastic variable;
//   outputs 5 branch logits (elastic, main plane, right edge, left edge,
//           apex) and one regression output for the plastic increment
//           (1e3 * d_alpha of the exact return).
//
// Training: loss = mean cross-entropy of the branch + 0.1 * mean squared
// error of the increment.  One wavefront handles 16 samples at a time with
// __builtin_amdgcn_mfma_f32_16x16x16bf16_1k (16 x 16 x 16 tiles); every
// wavefront accumulates its weight gradients in registers and writes them
// to its own slot, a second kernel sums the slots in a fixed order (the
// gradient is reproducible) and applies Adam to FP32 master weights, then
// refreshes their BF16 copies.
//
// MFMA 16x16x16 operand layout (64 lanes, 4 values per lane):
//   A (16 x 16, row m, column k):  lane = m + 16 * (k / 4), value k % 4
//   B (16 x 16, row k, column n):  lane = n + 16 * (k / 4), value k % 4
//   C (16 x 16, row m, column n):  lane = n + 16 * (m / 4), value m % 4
#include "ipf_kernels.h"
#include "ipf_learned.h"

namespace ipf {

namespace {

constexpr int kWave = 64;
using namespace mlp;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));  // a caller's features: any float address

// round to nearest even (NaN kept quiet)
__device__ __forceinline__ short f2bf(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return (short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}
__device__ __forceinline__ float bf2f(short h) { return __uint_as_float(((uint32_t)(unsigned short)h) << 16); }

// ReLU on the bit pattern -- the int32 maximum with 0 keeps every
// non-negative float and maps negative ones and -0 to +0: one v_max_i32,
// where fmaxf compiles to two v_max_f32 (the first quiets a signalling NaN);
// inference 15 % faster.  A NaN with the sign bit clear passes through (its
// predictions are garbage either way; they only order work).  The derivative
// is 0 at and below 0.
__device__ __forceinline__ float relu(float x) { return __int_as_float(max(__float_as_int(x), 0)); }
__device__ __forceinline__ float relu_grad(float x) { return x > 0.f ? 1.f : 0.f; }

struct WeightsLDS {
    alignas(16) short W1[INP][H];
    alignas(16) short W2[H][H];
    alignas(16) short W3[H][OUTP];
    float b1[H], b2[H], b3[OUTP];
};

// 16 bytes at a time: the matrices start on multiples of 8 values in wbf.
__device__ void load_weights(WeightsLDS& w, const short* __restrict__ wbf, const float* __restrict__ par) {
    static_assert(OFF_W1 % 8 == 0 && OFF_W2 % 8 == 0 && OFF_W3 % 8 == 0, "16-byte rows");
    auto rows = [&](short* dst, const short* src, int n) {
        for (int i = threadIdx.x; i < n / 8; i += blockDim.x)
            reinterpret_cast<int4*>(dst)[i] = reinterpret_cast<const int4*>(src)[i];
    };
    rows(&w.W1[0][0], wbf + OFF_W1, INP * H);
    rows(&w.W2[0][0], wbf + OFF_W2, H * H);
    rows(&w.W3[0][0], wbf + OFF_W3, H * OUTP);
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
        w.b1[i] = par[OFF_B1 + i];
        w.b2[i] = par[OFF_B2 + i];
    }
    for (int i = threadIdx.x; i < OUTP; i += blockDim.x) w.b3[i] = par[OFF_B3 + i];
}

typedef __bf16 bf16x4_hw __attribute__((ext_vector_type(4)));

// Four FP32 values to BF16 with the hardware conversion (v_cvt_pk_bf16_f32:
// round to nearest even, f2bf's result for every finite value).
__device__ __forceinline__ bf16x4 to_bf16x4(f32x4 v) {
    return __builtin_bit_cast(bf16x4, __builtin_convertvector(v, bf16x4_hw));
}

// C += A B over one K step of 16
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 relu4(f32x4 z) {
#pragma unroll
    for (int i = 0; i < 4; i++) z[i] = relu(z[i]);
    return z;
}

// c relu'(z)
__device__ __forceinline__ f32x4 relu_grad4(f32x4 c, f32x4 z) {
#pragma unroll
    for (int i = 0; i < 4; i++) c[i] = c[i] * relu_grad(z[i]);
    return c;
}

__device__ __forceinline__ float sum_bf4(bf16x4 v) { return ((bf2f(v[0]) + bf2f(v[1])) + bf2f(v[2])) + bf2f(v[3]); }

// One wavefront per 16-sample tile (grid-stride); 4 wavefronts per block.
// grad_slots[block][NPAR] receives the block's summed gradient of the mean loss
// over n samples (its wavefronts added in order, in LDS: a quarter of the
// slots to write and to sum), loss_slots[block] its summed loss.
//
// Activations stay in registers.  A C fragment of a transposed product (Z^T:
// lane = sample + 16 (unit / 4), value unit % 4) is an operand of the next
// product over those units, and one of the plain product (Z: lane = unit + 16
// (sample / 4), value sample % 4) is an operand of a weight gradient, a product
// over the samples; the two products take the same operand registers, swapped.
// So each layer is multiplied twice (92 MFMAs a tile) and nothing passes
// through LDS but the 16 x 16 output derivatives, turned once -- against two
// LDS bytes per value and eight 2-byte LDS reads per MFMA before.  Gradient call
// (with the sums): 4,096 samples 38 -> 32 us (bound by two launches and the
// weights' way into registers), 500,000 with the sums as they were before 642
// -> 116, 2 million 1,676 -> 353.
__global__ void __launch_bounds__(4 * kWave)
k_mlp_grad(const short* __restrict__ wbf, const float* __restrict__ par, const float* __restrict__ feat,
           const int* __restrict__ label, const float* __restrict__ target, int64_t n, float* __restrict__ grad_slots,
           double* __restrict__ loss_slots) {
    constexpr int NT = H / 16;
    __shared__ WeightsLDS w;
    __shared__ alignas(16) float G[NPAR];  // read back 16 bytes at a time
    __shared__ alignas(8) short turn[4][16][OUTP];
    __shared__ double wave_loss[4];
    load_weights(w, wbf, par);
    __syncthreads();
    const int wave = threadIdx.x / kWave;
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4, kq = g * 4;
    // weight operands: rows over the inputs (w1, w2, w3), over the outputs (v2, v3)
    bf16x4 w1[NT], w2[NT][NT], w3[NT], v2[NT][NT], v3[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w1[t][i] = w.W1[kq + i][16 * t + r];
            w3[t][i] = w.W3[16 * t + kq + i][r];
            v3[t][i] = w.W3[16 * t + r][kq + i];
#pragma unroll
            for (int u = 0; u < NT; u++) {
                w2[u][t][i] = w.W2[16 * t + kq + i][16 * u + r];
                v2[t][u][i] = w.W2[16 * t + r][16 * u + kq + i];
            }
        }
    }
    const int64_t nw = (int64_t)gridDim.x * 4;
    const int64_t ntile = (n + 15) / 16;
    const float inv_n = 1.f / (float)n;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 g1[NT], g2[NT][NT], g3[NT];
    float gb1[NT], gb2[NT], gb3 = 0.f;  // lane (r, g): column r of tile t, samples 4g..4g+3
#pragma unroll
    for (int a = 0; a < NT; a++) {
        g1[a] = g3[a] = zero;
        gb1[a] = gb2[a] = 0.f;
#pragma unroll
        for (int b = 0; b < NT; b++) g2[a][b] = zero;
    }
    double loss = 0.0;
    for (int64_t tile = (int64_t)blockIdx.x * 4 + wave; tile < ntile; tile += nw) {
        const int64_t s0 = tile * 16, q = s0 + r;
        // inputs: features 4g.. of sample r, and feature r of samples 4g..
        f32x4 xf = zero, xs = zero;
        if (g < 2 && q < n) xf = *reinterpret_cast<const f32x4_any*>(feat + q * FEAT_STRIDE + 4 * g);
        if (g == 1) xf[3] = 0.f;  // IN = 7 features
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (r < IN && s0 + kq + i < n) xs[i] = feat[(s0 + kq + i) * FEAT_STRIDE + r];
        const int y = q < n ? label[q] : 0;
        const float tg = q < n ? target[q] : 0.f;
        const bf16x4 xb = to_bf16x4(xf), xt = to_bf16x4(xs);
        // layer 1: Z1^T and Z1
        bf16x4 h1t[NT], h1n[NT];
        f32x4 z1n[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            f32x4 z = mfma16(w1[t], xb, zero);
#pragma unroll
            for (int i = 0; i < 4; i++) z[i] = z[i] + w.b1[16 * t + kq + i];
            h1t[t] = to_bf16x4(relu4(z));
            z1n[t] = mfma16(xb, w1[t], zero);
            const float b = w.b1[16 * t + r];
#pragma unroll
            for (int i = 0; i < 4; i++) z1n[t][i] = z1n[t][i] + b;
            h1n[t] = to_bf16x4(relu4(z1n[t]));
        }
        // layer 2
        bf16x4 h2t[NT], h2n[NT];
        f32x4 z2t[NT], z2n[NT];
#pragma unroll
        for (int u = 0; u < NT; u++) {
            f32x4 a = zero, b = zero;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                a = mfma16(w2[u][t], h1t[t], a);
                b = mfma16(h1t[t], w2[u][t], b);
            }
            const float bias = w.b2[16 * u + r];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                a[i] = a[i] + w.b2[16 * u + kq + i];
                b[i] = b[i] + bias;
            }
            z2t[u] = a;
            z2n[u] = b;
            h2t[u] = to_bf16x4(relu4(a));
            h2n[u] = to_bf16x4(relu4(b));
        }
        // layer 3: Z3^T, lane (r, g) holds outputs 4g.. of sample r
        f32x4 o = zero;
#pragma unroll
        for (int t = 0; t < NT; t++) o = mfma16(w3[t], h2t[t], o);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = o[i] + w.b3[kq + i];
        // loss and dL/dZ3: every lane of a sample has its six outputs
        float z[OUT];
#pragma unroll
        for (int j = 0; j < 4; j++) z[j] = __shfl(o[j], r, kWave);
        z[4] = __shfl(o[0], r + 16, kWave);
        z[5] = __shfl(o[1], r + 16, kWave);
        float zmax = z[0];
#pragma unroll
        for (int j = 1; j < NBR; j++) zmax = fmaxf(zmax, z[j]);
        float e[NBR], se = 0.f, zy = z[0];
#pragma unroll
        for (int j = 0; j < NBR; j++) {
            e[j] = expf(z[j] - zmax);
            se += e[j];
            if (j == y) zy = z[j];
        }
        const float diff = z[NBR] - tg;
        f32x4 d = zero;
        if (q < n) {
            if (g == 0) {
#pragma unroll
                for (int j = 0; j < 4; j++) d[j] = (e[j] / se - (j == y ? 1.f : 0.f)) * inv_n;
                float l = -(zy - zmax - logf(se));
                l += REG_WEIGHT * diff * diff;
                loss += l;
            } else if (g == 1) {
                d[0] = (e[4] / se - (4 == y ? 1.f : 0.f)) * inv_n;
                d[1] = 2.f * REG_WEIGHT * diff * inv_n;
            }
        }
        const bf16x4 d3t = to_bf16x4(d);
        *reinterpret_cast<bf16x4*>(&turn[wave][r][kq]) = d3t;
        wave_lds_sync();
        bf16x4 d3n;
#pragma unroll
        for (int i = 0; i < 4; i++) d3n[i] = turn[wave][kq + i][r];
        wave_lds_sync();
        gb3 += sum_bf4(d3n);
        // layer 2's derivatives, both ways; dW3 += H2^T D3
        bf16x4 d2t[NT], d2n[NT];
#pragma unroll
        for (int u = 0; u < NT; u++) {
            g3[u] = mfma16(h2n[u], d3n, g3[u]);
            d2t[u] = to_bf16x4(relu_grad4(mfma16(v3[u], d3t, zero), z2t[u]));
            d2n[u] = to_bf16x4(relu_grad4(mfma16(d3t, v3[u], zero), z2n[u]));
            gb2[u] += sum_bf4(d2n[u]);
        }
        // dW2 += H1^T D2; D1 and dW1 += X^T D1
#pragma unroll
        for (int t = 0; t < NT; t++) {
            f32x4 c = zero;
#pragma unroll
            for (int u = 0; u < NT; u++) {
                g2[t][u] = mfma16(h1n[t], d2n[u], g2[t][u]);
                c = mfma16(d2t[u], v2[t][u], c);
            }
            const bf16x4 d1n = to_bf16x4(relu_grad4(c, z1n[t]));
            gb1[t] += sum_bf4(d1n);
            g1[t] = mfma16(xt, d1n, g1[t]);
        }
    }
    // the columns' four sample groups, the samples' losses
    auto over_groups = [&](float v) {
        v += __shfl_xor(v, 16, kWave);
        return v + __shfl_xor(v, 32, kWave);
    };
    gb3 = over_groups(gb3);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        gb1[t] = over_groups(gb1[t]);
        gb2[t] = over_groups(gb2[t]);
    }
#pragma unroll
    for (int k = 8; k > 0; k >>= 1) loss += __shfl_xor(loss, k, kWave);  // lanes 0..15 hold them
    // the block's gradient: C layout element (kq + i, r) of each 16 x 16 tile
    if (lane == 0) wave_loss[wave] = loss;
    for (int t = 0; t < 4; t++) {
        if (wave == t) {
            auto add = [&](int p, float v) { G[p] = t == 0 ? v : G[p] + v; };
#pragma unroll
            for (int nt = 0; nt < H / 16; nt++)
#pragma unroll
                for (int i = 0; i < 4; i++) add(OFF_W1 + (kq + i) * H + nt * 16 + r, g1[nt][i]);
#pragma unroll
            for (int mt = 0; mt < H / 16; mt++)
#pragma unroll
                for (int nt = 0; nt < H / 16; nt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) add(OFF_W2 + (mt * 16 + kq + i) * H + nt * 16 + r, g2[mt][nt][i]);
#pragma unroll
            for (int mt = 0; mt < H / 16; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) add(OFF_W3 + (mt * 16 + kq + i) * OUTP + r, g3[mt][i]);
            if (g == 0) {
#pragma unroll
                for (int u = 0; u < NT; u++) {
                    add(OFF_B1 + 16 * u + r, gb1[u]);
                    add(OFF_B2 + 16 * u + r, gb2[u]);
                }
                add(OFF_B3 + r, gb3);
            }
        }
        __syncthreads();
    }
    float4* out = reinterpret_cast<float4*>(grad_slots + blockIdx.x * (int64_t)NPAR);
    for (int p = threadIdx.x; p < NPAR / 4; p += 4 * kWave) out[p] = reinterpret_cast<const float4*>(G)[p];
    if (threadIdx.x == 0) loss_slots[blockIdx.x] = ((wave_loss[0] + wave_loss[1]) + wave_loss[2]) + wave_loss[3];
}

// Parameters a padded slot never trains: W1 rows >= IN, W3 / b3 columns >= OUT.
__device__ __forceinline__ bool trainable(int p) {
    if (p >= OFF_W1 && p < OFF_B1) return (p - OFF_W1) / H < IN;
    if (p >= OFF_W3 && p < OFF_B3) return (p - OFF_W3) % OUTP < OUT;
    if (p >= OFF_B3) return p - OFF_B3 < OUT;
    return true;
}

// grad[p] = sum of the slots -- 16 threads a parameter, each a run of slots in
// order, then their sums in order -- and optionally one Adam step; block 0
// sums the loss (grad, loss: where wanted, straight into pinned memory).  One thread a parameter took
// 58 us for 256 slots, one load after the other; 64 slots (the block sums of
// the same minibatch) by 16 threads take 4.
constexpr int kRedPar = 16, kRedGroups = 16;
static_assert(NPAR % kRedPar == 0 && NPAR % 4 == 0, "whole blocks");

__global__ void __launch_bounds__(kRedPar * kRedGroups)
k_mlp_reduce(const float* __restrict__ slots, const double* __restrict__ loss_slots, int nslots,
             float* __restrict__ grad, double* __restrict__ loss, float* __restrict__ par, float* __restrict__ m1,
             float* __restrict__ m2, short* __restrict__ wbf, int adam, float lr, float b1, float b2, float eps, float bc1, float bc2) {
    __shared__ float sums[kRedGroups][kRedPar];
    __shared__ double losses[kRedPar * kRedGroups];
    const int t = threadIdx.x, col = t % kRedPar, grp = t / kRedPar;
    const int p = blockIdx.x * kRedPar + col;
    const int per = (nslots + kRedGroups - 1) / kRedGroups;
    const int w0 = min(nslots, grp * per), w1 = min(nslots, w0 + per);
    float s = 0.f;
#pragma unroll 4
    for (int w = w0; w < w1; w++) s += slots[(int64_t)w * NPAR + p];
    sums[grp][col] = s;
    if (blockIdx.x == 0) {
        double l = 0.0;
        for (int w = t; w < nslots; w += kRedPar * kRedGroups) l += loss_slots[w];
        losses[t] = l;
    }
    __syncthreads();
    if (loss && blockIdx.x == 0 && t == 0) {
        double l = 0.0;
        for (int i = 0; i < kRedPar * kRedGroups && i < nslots; i++) l += losses[i];
        *loss = l;
    }
    if (grp != 0) return;
    float g = 0.f;
#pragma unroll
    for (int i = 0; i < kRedGroups; i++) g += sums[i][col];
    if (!trainable(p)) g = 0.f;
    if (grad) grad[p] = g;
    if (!adam) return;
    const float a = b1 * m1[p] + (1.f - b1) * g;
    const float v = b2 * m2[p] + (1.f - b2) * g * g;
    m1[p] = a;
    m2[p] = v;
    float x = par[p];
    if (trainable(p)) x -= lr * (a / bc1) / (sqrtf(v / bc2) + eps);
    par[p] = x;
    wbf[p] = f2bf(x);
}

__global__ void k_mlp_refresh(const float* __restrict__ par, short* __restrict__ wbf) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPAR) wbf[p] = f2bf(par[p]);
}

// C += A B over 32 k with gfx950's 16 x 16 x 32 BF16 MFMA, the operands two
// 16 x 16 x 16 fragments each: A = (a0 | a1), B = (b0 | b1) per lane.  A lane
// group's element e of A and of B address the same k, so the pairs (a0, b0)
// and (a1, b1) -- k steps t and t + 1 of the K = 16 form -- are summed
// together in one instruction instead of two.
__device__ __forceinline__ f32x4 mfma_k32(bf16x4 a0, bf16x4 a1, bf16x4 b0, bf16x4 b1, f32x4 c) {
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef __bf16 bf16x8_hw __attribute__((ext_vector_type(8)));
    const s16x8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
    const s16x8 b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_hw, a), __builtin_bit_cast(bf16x8_hw, b), c,
                                                   0, 0, 0);
}

__device__ __forceinline__ f32x4 load_feat(const float* __restrict__ feat, int64_t q, int64_t n, int g) {
    f32x4 f = {0.f, 0.f, 0.f, 0.f};
    if (g < 2 && q < n) f = *reinterpret_cast<const f32x4_any*>(feat + q * FEAT_STRIDE + 4 * g);
    return f;
}

// Inference over n samples, 16 per wavefront step, every layer computed
// transposed (Z^T = W^T A^T): then the C fragment of one layer's 16 x 16
// output tile -- lane = sample + 16 (hidden / 4), value hidden % 4 -- is
// exactly the B fragment of the next layer's K step over those 16 hidden
// units, so activations stay in registers from input to output, and the
// weights sit in registers as A fragments for the whole grid-stride loop
// (W1^T 4 tiles, W2^T 16, W3^T 4: 48 VGPRs).  Biases start the
// accumulators; the hidden layers' biases are read from LDS per group (32
// VGPRs fewer; 3 waves per SIMD without spills -- a bound of 4 spilled and
// ran slower).  The hidden layers' K = 64 products run as two K = 32 MFMAs
// each (mfma_k32).  Inputs are read as one 16-byte vector per lane
// (features 4g..4g+3 of the lane's sample, g < 2; reading them three groups
// ahead measured 5 % slower), outputs written by the lanes that hold them.
__global__ void __launch_bounds__(4 * kWave)
k_mlp_predict(const short* __restrict__ wbf, const float* __restrict__ par, const float* __restrict__ feat, int64_t n,
              int* __restrict__ branch, float* __restrict__ out) {
    __shared__ f32x4 bias[2 * H / 4];  // b1, b2 in groups of 4 units
    const int lane = threadIdx.x & 63;
    const int s = lane & 15, g = lane >> 4;
    bf16x4 a1[H / 16], a2[H / 16][H / 16], a3[H / 16];
    f32x4 c3;
#pragma unroll
    for (int t = 0; t < H / 16; t++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = 4 * g + i;
            a1[t][i] = wbf[OFF_W1 + k * H + 16 * t + s];
            a3[t][i] = wbf[OFF_W3 + (16 * t + k) * OUTP + s];
#pragma unroll
            for (int t2 = 0; t2 < H / 16; t2++) a2[t2][t][i] = wbf[OFF_W2 + (16 * t + k) * H + 16 * t2 + s];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) c3[i] = par[OFF_B3 + 4 * g + i];
    for (int j = threadIdx.x; j < 2 * H / 4; j += blockDim.x) {
        const int o = j < H / 4 ? OFF_B1 + 4 * j : OFF_B2 + 4 * (j - H / 4);
        bias[j] = f32x4{par[o], par[o + 1], par[o + 2], par[o + 3]};
    }
    __syncthreads();
    const int64_t step = (int64_t)gridDim.x * 4 * 16;
    int64_t s0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
    for (; s0 < n; s0 += step) {
        const int64_t q = s0 + s;
        const bf16x4 xb = to_bf16x4(load_feat(feat, q, n, g));
        bf16x4 h1[H / 16];
#pragma unroll
        for (int t = 0; t < H / 16; t++) {
            f32x4 z = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1[t], xb, bias[4 * t + g], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) z[i] = relu(z[i]);
            h1[t] = to_bf16x4(z);
        }
        bf16x4 h2[H / 16];
#pragma unroll
        for (int t2 = 0; t2 < H / 16; t2++) {
            f32x4 z = bias[H / 4 + 4 * t2 + g];
#pragma unroll
            for (int t = 0; t < H / 16; t += 2) z = mfma_k32(a2[t2][t], a2[t2][t + 1], h1[t], h1[t + 1], z);
#pragma unroll
            for (int i = 0; i < 4; i++) z[i] = relu(z[i]);
            h2[t2] = to_bf16x4(z);
        }
        f32x4 o = c3;
#pragma unroll
        for (int t = 0; t < H / 16; t += 2) o = mfma_k32(a3[t], a3[t + 1], h2[t], h2[t + 1], o);
        // lane (s, g) holds outputs 4g..4g+3 of sample s; logit 4 sits in lane s + 16
        const float o4 = __shfl(o[0], s + 16, kWave);
        if (q < n) {
            if (g == 0) {
                if (branch) {
                    int best = 0;
                    float bv = o[0];
#pragma unroll
                    for (int j = 1; j < 4; j++)
                        if (o[j] > bv) {
                            bv = o[j];
                            best = j;
                        }
                    if (o4 > bv) best = 4;
                    branch[q] = best;
                }
                if (out)
#pragma unroll
                    for (int j = 0; j < 4; j++) out[q * OUT + j] = o[j];
            } else if (g == 1 && out) {
                out[q * OUT + 4] = o[0];
                out[q * OUT + 5] = o[1];
            }
        }
    }
}

// Features and labels of every point from the exact return map at the trial
// state (strain of u, committed plastic strain and alpha); nothing is
// committed.  One wavefront per tile of a group, as k_sigma.
__global__ void __launch_bounds__(kWave)
k_point_features(GroupDev g, int tp, const double* __restrict__ strain, const int64_t* __restrict__ orig,
                 PointState st, float* __restrict__ feat, int* __restrict__ label, float* __restrict__ target) {
    const int64_t tile = blockIdx.x;
    const int lane = threadIdx.x;
    if (lane >= tp) return;
    const int64_t P = g.pt0 + tile * tp + lane;
    const int64_t o = orig[P];
    if (o < 0) return;
    const MatConst& m = tile_material(g, tile);
    const double e3[3] = {strain[3 * o], strain[3 * o + 1], strain[3 * o + 2]};
    const double ep[4] = {st.ep0[P], st.ep1[P], st.ep2[P], st.ep3[P]};
    point_features(e3, ep, st.alpha[P], m, feat + o * FEAT_STRIDE, label[o], target[o]);
}

}  // namespace

void launch_point_features(int shape, const GroupDev& g, const double* strain, const int64_t* orig,
                           const PointState& st, float* feat, int* label, float* target, hipStream_t s) {
    if (g.ntiles == 0) return;
    hipLaunchKernelGGL(k_point_features, dim3((unsigned)g.ntiles), dim3(kWave), 0, s, g, shape_tp(shape), strain,
                       orig, st, feat, label, target);
}

namespace mlp {

void launch_grad(const short* wbf, const float* par, const float* feat, const int* label, const float* target,
                 int64_t n, int nblocks, float* slots, double* loss_slots, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_grad, dim3(nblocks), dim3(4 * kWave), 0, s, wbf, par, feat, label, target, n, slots,
                       loss_slots);
}

void launch_reduce(const float* slots, const double* loss_slots, int nslots, float* grad, double* loss, float* par,
                   float* m1, float* m2, short* wbf, bool adam, float lr, float b1, float b2, float eps, float bc1, float bc2, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_reduce, dim3(NPAR / kRedPar), dim3(kRedPar * kRedGroups), 0, s, slots, loss_slots, nslots,
                       grad, loss, par, m1, m2, wbf, adam ? 1 : 0, lr, b1, b2, eps, bc1, bc2);
}

void launch_refresh(const float* par, short* wbf, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_refresh, dim3((NPAR + 255) / 256), dim3(256), 0, s, par, wbf);
}

void launch_predict(const short* wbf, const float* par, const float* feat, int64_t n, int nblocks, int* branch,
                    float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_predict, dim3(nblocks), dim3(4 * kWave), 0, s, wbf, par, feat, n, branch, out);
}

}  // namespace mlp

}  // namespace ipf

namespace ipf {

namespace {

constexpr int kSortBlock = IPF_SORT_BLOCK;
constexpr int kSortRound = 4 * kSortBlock;  // keys per round of the scatter

__device__ __forceinline__ int clamp_key(int k, int nk) { return (k >= 0 && k < nk) ? k : nk - 1; }

// Counting sort of keys in [0, NK): block b counts the keys of its chunk, then
// every block of the scatter sums the counts before it itself (NK columns of
// at most kSortMaxBlocks rows out of L2) -- no scan between the two launches.
// hist[k * nb + b].
template <int NK>
__global__ void __launch_bounds__(kSortBlock)
k_key_hist(const int* __restrict__ key, int64_t n, int64_t chunk, int* __restrict__ hist) {
    constexpr int NW = kSortBlock / kWave;
    __shared__ int part[NW][NK];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t i0 = (int64_t)blockIdx.x * chunk, i1 = min(n, i0 + chunk);
    int c[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) c[k] = 0;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kSortBlock) {
        const int v = clamp_key(key[i], NK);
#pragma unroll
        for (int k = 0; k < NK; k++) c[k] += v == k;
    }
#pragma unroll
    for (int k = 0; k < NK; k++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) c[k] += __shfl_xor(c[k], o, kWave);
        if (lane == 0) part[wave][k] = c[k];
    }
    __syncthreads();
    if (threadIdx.x < NK) {
        int s = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) s += part[w][threadIdx.x];
        hist[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = s;
    }
}

// Stable scatter of the block's chunk, kSortRound keys at a time, four in a row
// per thread: the counts of the keys before a thread's are one 64-bit scan of
// packed 12-bit fields (at most 256 keys per wavefront).
template <int NK>
__global__ void __launch_bounds__(kSortBlock)
k_key_scatter(const int* __restrict__ key, int64_t n, int64_t chunk, const int* __restrict__ hist,
              int* __restrict__ order) {
    static_assert(NK <= 5, "12-bit fields of one 64-bit word");
    constexpr int NW = kSortBlock / kWave;
    __shared__ unsigned long long wc[2][NW];
    __shared__ int before_part[NW][NK], total_part[NW][NK];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int nb = gridDim.x, me = blockIdx.x;
    const int64_t i0 = (int64_t)me * chunk, i1 = min(n, i0 + chunk);
    int k[4];
    auto request = [&](int64_t i) {  // branch-free: keys past the chunk are read as its last and not used
#pragma unroll
        for (int q = 0; q < 4; q++) k[q] = key[min(i + q, i1 - 1)];
    };
    request(i0 + 4 * (int)threadIdx.x);
    int bs[NK], ts[NK];
#pragma unroll
    for (int j = 0; j < NK; j++) bs[j] = ts[j] = 0;
    for (int b = threadIdx.x; b < nb; b += kSortBlock)
#pragma unroll
        for (int j = 0; j < NK; j++) {
            const int h = hist[(int64_t)j * nb + b];
            ts[j] += h;
            bs[j] += b < me ? h : 0;
        }
#pragma unroll
    for (int j = 0; j < NK; j++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            ts[j] += __shfl_xor(ts[j], o, kWave);
            bs[j] += __shfl_xor(bs[j], o, kWave);
        }
        if (lane == 0) {
            before_part[wave][j] = bs[j];
            total_part[wave][j] = ts[j];
        }
    }
    __syncthreads();
    int before[NK];  // where key j's next element goes
    int base = 0;
#pragma unroll
    for (int j = 0; j < NK; j++) {
        int b = 0, t = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            b += before_part[w][j];
            t += total_part[w][j];
        }
        before[j] = base + b;
        base += t;
    }
    int buf = 0;
    for (int64_t r0 = i0; r0 < i1; r0 += kSortRound, buf ^= 1) {
        const int64_t i = r0 + 4 * (int)threadIdx.x;
        int v[4];
        unsigned long long mine = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            v[q] = i + q < i1 ? clamp_key(k[q], NK) : NK;
            if (v[q] < NK) mine += 1ull << (12 * v[q]);
        }
        if (r0 + kSortRound < i1) request(i + kSortRound);
        unsigned long long incl = mine;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const unsigned long long up = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += up;
        }
        if (lane == kWave - 1) wc[buf][wave] = incl;
        __syncthreads();  // one barrier per round: the next one writes the other buffer
        const unsigned long long excl = incl - mine;
        int pos[NK];
#pragma unroll
        for (int j = 0; j < NK; j++) {
            int round = 0, ahead = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const int c = (int)((wc[buf][w] >> (12 * j)) & 0xfff);
                ahead += w < wave ? c : 0;
                round += c;
            }
            pos[j] = before[j] + ahead + (int)((excl >> (12 * j)) & 0xfff);
            before[j] += round;
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int j = 0; j < NK; j++)
                if (v[q] == j) order[pos[j]++] = (int)(i + q);
    }
}

// The return map of the points in `order` (reference point indexes), one
// point per lane; state and material looked up per point.
__global__ void __launch_bounds__(256)
k_sigma_order(int64_t n, const int* __restrict__ order, const int64_t* __restrict__ new_of,
              const int* __restrict__ pmat, const MatConst* __restrict__ mats, const double* __restrict__ strain,
              double* __restrict__ wsigma, PointState st, int commit) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int64_t o = order[t];
    const int64_t P = new_of[o];
    const MatConst& m = mats[pmat[P]];
    const double e3[3] = {strain[3 * o], strain[3 * o + 1], strain[3 * o + 2]};
    double ep[4] = {st.ep0[P], st.ep1[P], st.ep2[P], st.ep3[P]};
    double alpha = st.alpha[P];
    int mt, br;
    double ws[3];
    point_sigma<false>(e3, ep, alpha, mt, br, m, st.w[P], ws, nullptr);
    wsigma[3 * o + 0] = ws[0];
    wsigma[3 * o + 1] = ws[1];
    wsigma[3 * o + 2] = ws[2];
    if (commit) {
        st.ep0[P] = ep[0];
        st.ep1[P] = ep[1];
        st.ep2[P] = ep[2];
        st.ep3[P] = ep[3];
        st.alpha[P] = alpha;
        st.mtype[P] = (signed char)mt;
        st.branch[P] = (signed char)br;
    }
}

}  // namespace

// Chunks of whole rounds, at most kSortMaxBlocks of them: enough blocks to fill
// the chip, few enough rows that every block can sum them.  1.44 M keys:
// histograms 8.5 + scan by one block 46 + scatter 6.1 us -> 5.9 + 10.3.
constexpr int kSortMaxBlocks = 1024;

static int64_t sort_chunk(int64_t n) {
    const int64_t rounds = (n + kSortRound - 1) / kSortRound;
    return (rounds + kSortMaxBlocks - 1) / kSortMaxBlocks * kSortRound;
}

int key_sort_blocks(int64_t n) { return (int)((n + kSortBlock - 1) / kSortBlock); }

void launch_branch_order(const int* key, int64_t n, int* hist, int* order, hipStream_t s) {
    if (n == 0) return;
    const int64_t chunk = sort_chunk(n);
    const int nb = (int)((n + chunk - 1) / chunk);
    hipLaunchKernelGGL(k_key_hist<IPF_NBRANCH>, dim3(nb), dim3(kSortBlock), 0, s, key, n, chunk, hist);
    hipLaunchKernelGGL(k_key_scatter<IPF_NBRANCH>, dim3(nb), dim3(kSortBlock), 0, s, key, n, chunk, hist, order);
}

void launch_sigma_order(int64_t n, const int* order, const int64_t* new_of, const int* pmat, const MatConst* mats,
                        const double* strain, double* wsigma, const PointState& st, bool commit, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_sigma_order, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, order, new_of, pmat, mats,
                       strain, wsigma, st, commit ? 1 : 0);
}

}  // namespace ipf
