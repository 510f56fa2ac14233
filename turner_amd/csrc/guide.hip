// guide.hip -- training and inference kernels of the learned guiding
// proposal (tn_guide.h) and the tn_guide_* entry points.  No reference
// counterpart: the reference draws indirect directions uniformly
// (lib/sampling.h:20-32).
//
// Every matrix product runs on MFMA with BF16 operands and FP32 accumulation:
//
//   forward   H_l^T  = W_l H_{l-1}^T          A = W_l (BF16 copy), B = LDS rows
//   backward  D_{l-1}^T = W_l^T D_l^T (.) [H_{l-1} > 0]   A = W_l^T (BF16 copy)
//   gradient  dW_l = D_l^T H_{l-1}            K = 64 samples, both from transposed LDS copies
//
// A block sums the gradients of all its sample groups in registers and writes
// one slice; the slices are summed in a fixed order, so a step is
// deterministic.  The per-sample loss gradient with respect to the 40 outputs
// is evaluated in FP32 in log space.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <random>
#include <vector>

#include "tn_guide.h"
#include "tn_scene.h"

namespace tn {
namespace {

constexpr int kGPartial = kGParams + 8;  // a block's gradient slice (+ padding)

__device__ __forceinline__ uint64_t g_splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Writes parameter p's BF16 operand copies (their padding stays zero).
__device__ __forceinline__ void store_operands(uint16_t* __restrict__ wbf, int p, float value) {
    const uint16_t h = to_bf16(value);
    if (p < kGOffB1) {
        wbf[kGW1 + frag_at(p / kGIn, p % kGIn, 2, 4)] = h;
        wbf[kGTW1 + frag16_at(p / kGIn, p % kGIn, 5)] = h;
    } else if (p >= kGOffW2 && p < kGOffB2) {
        const int k = p - kGOffW2;
        wbf[kGW2 + frag_at(k / kGHid, k % kGHid, 2, 4)] = h;
        wbf[kGTW2 + frag16_at(k / kGHid, k % kGHid, 4)] = h;
        wbf[kGWT2 + frag16_at(k % kGHid, k / kGHid, 4)] = h;
    } else if (p >= kGOffW3 && p < kGOffB3) {
        const int k = p - kGOffW3;
        wbf[kGW3 + frag_at(k / kGHid, k % kGHid, 2, 4)] = h;
        wbf[kGTW3 + frag16_at(k / kGHid, k % kGHid, 4)] = h;
        wbf[kGWT3 + frag16_at(k % kGHid, k / kGHid, 4)] = h;
    } else if (p >= kGOffW4 && p < kGOffB4) {
        const int k = p - kGOffW4;
        wbf[kGW4 + frag_at(k / kGHid, k % kGHid, 2, 3)] = h;
        wbf[kGTW4 + frag16_at(k / kGHid, k % kGHid, 4)] = h;
        wbf[kGWT4 + frag16_at(k % kGHid, k / kGHid, 3)] = h;
    }
}

// BF16 operand copies of all FP32 master parameters (wbf zeroed before).
__global__ void k_guide_refresh(const float* __restrict__ theta, uint16_t* __restrict__ wbf) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kGParams) store_operands(wbf, p, theta[p]);
}

__device__ __forceinline__ float3 load3(const float* a, uint32_t i) {
    return make_float3(a[3 * (size_t)i], a[3 * (size_t)i + 1], a[3 * (size_t)i + 2]);
}

// w3 given: q(w) into pdf; else w ~ q from u3 into w3out, q(w) into pdf.  64 points
// per block: one wave for all (NT = 4 tiles of 16) or a wave per tile (NT = 1).
template <int NT>
__global__ __launch_bounds__(256 / NT) void k_guide_eval(GuideView G, const float* __restrict__ p3,
                                                         const float* __restrict__ n3,
                                                         const float* __restrict__ w3,
                                                         const float* __restrict__ u3, uint32_t n,
                                                         float* __restrict__ pdf, float* __restrict__ w3out) {
    __shared__ __align__(16) float rows[64 * kGOut];
    constexpr uint32_t kPoints = 16 * NT;  // of a wave
    const uint32_t first = threadIdx.x / 64u * kPoints, l = threadIdx.x % kPoints;
    const uint32_t i = blockIdx.x * 64u + first + l;
    float* o = rows + first * kGOut;
    const bool act = i < n;
    float3 p = make_float3(0.f, 0.f, 0.f), nn = p;
    if (act) {
        p = load3(p3, i);
        nn = load3(n3, i);
    }
    guide_forward_wave<NT>(G, p, nn, act, o);
    if (!act || threadIdx.x % 64u >= kPoints) return;
    Mixture M;
    mixture_from(o + l * kGOut, M);
    float3 w;
    if (w3) {
        w = load3(w3, i);
    } else {
        w = mixture_sample(M, u3[3 * (size_t)i], u3[3 * (size_t)i + 1], u3[3 * (size_t)i + 2]);
        w3out[3 * (size_t)i] = w.x;
        w3out[3 * (size_t)i + 1] = w.y;
        w3out[3 * (size_t)i + 2] = w.z;
    }
    pdf[i] = mixture_pdf(M, w);
}

int launch_eval(tn_guide* g, const float* p3, const float* n3, const float* w3, const float* u3, uint32_t n, float* pdf,
                float* w3out, hipStream_t stream) {
    const uint32_t blocks = (n + 63) / 64;
    // A wave per tile while a compute unit has at most two blocks: latency is all
    // there is (density of 4,099 points 10.6 us per call against 11.8, of 32,768
    // 11.2 against 12.4); beyond, its idle lanes in the mixture cost more (65,536
    // points 18.4 us against 12.9, 1,048,576 212 against 98).
    if (blocks <= (uint32_t)std::max(g->cus, 1) * 2u) k_guide_eval<1><<<blocks, 256, 0, stream>>>(g->view(), p3, n3, w3, u3, n, pdf, w3out);
    else k_guide_eval<4><<<blocks, 64, 0, stream>>>(g->view(), p3, n3, w3, u3, n, pdf, w3out);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

// four floats at any float's address (callers' arrays need no more)
typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));

// Network outputs for n points with persistent waves: each wave (block) loads
// every weight fragment into registers once and then takes tiles of 16 points
// (points and normals of the next tile in flight), whose outputs it stores from
// the accumulators.  1,048,576 points: 90 us with features, activations and
// outputs in LDS rows, 68 without (54 without the stores, 41 to move the bytes);
// what is left is instruction issue: about 250 vector instructions and 20 sines
// and cosines per tile against 34 matrix ones.  Two to four tiles at a time,
// three waves per SIMD or biases in LDS gave 68 to 71.
__global__ __launch_bounds__(64, 2) void k_guide_forward(GuideView G, const float* __restrict__ p3,
                                                         const float* __restrict__ n3, uint32_t n,
                                                         float* __restrict__ out) {
    const GuideRegs net(G);
    const GuideLane L = guide_lane();
    const uint32_t s = threadIdx.x & 15u;
    const uint32_t tiles = (n + 15) / 16;
    uint32_t tile = blockIdx.x;
    if (tile >= tiles) return;
    uint32_t i = min(tile * 16u + s, n - 1u);
    float3 p = load3(p3, i), nn = load3(n3, i);
    for (;;) {
        const uint32_t next = tile + gridDim.x;
        GuideIn in[1] = {guide_features(G, L, p, nn)};
        if (next < tiles) {
            i = min(next * 16u + s, n - 1u);
            p = load3(p3, i);
            nn = load3(n3, i);
        }
        const uint32_t k = tile * 16u + s;
        guide_network<1>(net, in, [&](int, int o, float4 v) {
            if (k < n) *reinterpret_cast<f4_any*>(out + (size_t)k * kGOut + o) = (f4_any){v.x, v.y, v.z, v.w};
        });
        if (next >= tiles) break;
        tile = next;
    }
}

constexpr int kTrainWaves = 8, kTrainBlock = 64 * kTrainWaves;
constexpr uint32_t kTrainBlocksPerCu = 2;
constexpr int kGStrideIn = kGInPad + 8;  // LDS row strides (u16), padded against bank conflicts
constexpr int kGStrideHid = kGHid + 8;
constexpr int kTStride = 64 + 8;  // row stride (u16) of the transposed [feature][sample] arrays

// d(c * -log q(w)) / d(out) of one of a sample's eight lobes, FP32 in log space:
// lanes that differ in bits 3..5 hold the sample's lobes.  o, d: the lobe's five
// outputs.  Returns -log q.
__device__ __forceinline__ float guide_dout(const float* o, float3 w, float c, float* d) {
    const float kLog2Pi = 1.83787706640934548356f;
    auto sum8 = [](float x) {  // in the lobes' order
        const int first = (int)(threadIdx.x & 7u);
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < kGLobes; ++j) s += __shfl(x, first + 8 * j, 64);
        return s;
    };
    auto max8 = [](float x) {
        x = fmaxf(x, __shfl_xor(x, 8, 64));
        x = fmaxf(x, __shfl_xor(x, 16, 64));
        return fmaxf(x, __shfl_xor(x, 32, 64));
    };
    const float mx = max8(o[0]);
    const float lse = mx + logf(sum8(expf(o[0] - mx)));
    const float inv = 1.0f / fmaxf(sqrtf(o[1] * o[1] + o[2] * o[2] + o[3] * o[3]), 1e-12f);
    const float3 mu = make_float3(o[1] * inv, o[2] * inv, o[3] * inv);
    const float sp = softplusf(o[4]) + kKappaMin;
    const bool live = sp < kKappaMax;
    const float k = fminf(sp, kKappaMax);
    const float cs = mu.x * w.x + mu.y * w.y + mu.z * w.z;
    const float a = o[0] - lse + (logf(k) - kLog2Pi - logf(-expm1f(-2.0f * k)) + k * (cs - 1.0f));
    const float amax = max8(a);
    const float logq = amax + logf(sum8(expf(a - amax)));
    const float gam = expf(a - logq), pi = expf(o[0] - lse);
    d[0] = -(gam - pi) * c;
    const float s = -gam * k * c;
    const float3 dmu = make_float3(s * w.x, s * w.y, s * w.z);
    const float dot = dmu.x * mu.x + dmu.y * mu.y + dmu.z * mu.z;
    d[1] = (dmu.x - dot * mu.x) * inv;
    d[2] = (dmu.y - dot * mu.y) * inv;
    d[3] = (dmu.z - dot * mu.z) * inv;
    // d log vMF / d kappa = 1/k - 2/(e^{2k} - 1) + (cos - 1); series below 0.05
    const float dk = (k < 0.05f ? 1.0f - k * (1.0f / 3.0f) + k * k * k * (1.0f / 45.0f)
                                : 1.0f / k - 2.0f / expm1f(2.0f * k)) +
                     (cs - 1.0f);
    const float sig = 1.0f / (1.0f + expf(-o[4]));
    d[4] = live ? -gam * dk * c * sig : 0.f;
    return -logq;
}

struct TrainSrc {
    // explicit batch (device arrays) ...
    const float* p3;
    const float* n3;
    const float* w3;
    const float* c;
    uint32_t n;
    // ... or n samples drawn from the training set
    const float4* ts;
    const uint32_t* ts_count;
    uint32_t ts_cap;
    uint64_t seed;
    uint32_t subset;       // distinct samples this pass trains on
    uint64_t subset_seed;  // fixes which ones
};

// Two output tiles, mt0 and mt0 + 1, of Y^T = W X^T for 16 samples, K = 16 KT:
// B fragments from their rows (stride in u16), epi(0 or 1, first output,
// accumulator).  In K = 16 steps: a rounding that falls otherwise flips the sign of
// a gradient near zero, and with it a whole Adam step, so the sums keep one order.
template <int KT, class Epi>
__device__ __forceinline__ void train_product(int l, const uint16_t* W, int mt0, const uint16_t* rows, int stride,
                                              Epi epi) {
    const int s = l & 15, grp = l >> 4;
    g_s4 a[2][KT], b[KT];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
            a[mt][kt] = *reinterpret_cast<const g_s4*>(reinterpret_cast<const char*>(W) +
                                                       (8u * (uint32_t)l + 512u * (uint32_t)((mt0 + mt) * KT + kt)));
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) b[kt] = *reinterpret_cast<const g_s4*>(rows + s * stride + 16 * kt + 4 * grp);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        g_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[mt][kt], b[kt], acc, 0, 0, 0);
        epi(mt, 16 * (mt0 + mt) + 4 * grp, acc);
    }
}

// acc += D H^T over the block's 64 samples for one 16 x 16 tile: rows `drow`..
// +15 of D^T against rows `hrow`.. +15 of H^T (both [feature][sample]).
__device__ __forceinline__ void grad_tile(int l, g_f4& acc, const uint16_t* dt, int drow, const uint16_t* ht,
                                          int hrow) {
    const int r = l & 15, grp = l >> 4;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        const g_s4 a = *reinterpret_cast<const g_s4*>(dt + (drow + r) * kTStride + 16 * kt + 4 * grp);
        const g_s4 b = *reinterpret_cast<const g_s4*>(ht + (hrow + r) * kTStride + 16 * kt + 4 * grp);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
}

__device__ __forceinline__ void store_tile(const g_f4& acc, float* __restrict__ out, int o0, int i0, int out_real,
                                           int in_real) {
    const int l = threadIdx.x & 63, grp = l >> 4, i = i0 + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int o = o0 + 4 * grp + r;
        if (o < out_real && i < in_real) out[o * in_real + i] = acc[r];
    }
}

// acc += sums over the block's 64 samples of rows `drow`.. +15 of D^T (every
// column of the tile alike).
__device__ __forceinline__ void bias_tile(int l, g_f4& acc, const uint16_t* dt, int drow) {
    const int r = l & 15, grp = l >> 4;
    const uint32_t one2 = 0x3F803F80u;  // two BF16 ones
    const uint4 o4 = make_uint4(one2, one2, one2, one2);
    g_bf8 ones;
    __builtin_memcpy(&ones, &o4, 16);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
        const g_bf8 a = *reinterpret_cast<const g_bf8*>(dt + (drow + r) * kTStride + 32 * kt + 8 * grp);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, acc, 0, 0, 0);
    }
}
__device__ __forceinline__ void store_bias(const g_f4& acc, float* __restrict__ out, int o0, int out_real) {
    const int l = threadIdx.x & 63, grp = l >> 4;
    if (l & 15) return;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (o0 + 4 * grp + r < out_real) out[o0 + 4 * grp + r] = acc[r];
}

// Gradient slices of a batch.  A block of eight waves takes 64 samples at a time:
// a mini-batch of 16,384 is 256 groups, one per compute unit, so what bounds the
// step is how long one group takes.  Every stage is spread over the block: the
// encoding over eight lanes per sample (half an axis each), the products over
// two waves per 16 samples (half of the outputs each), the loss gradient over
// a lane per lobe, and the weight gradients (K = the block's 64 samples) over
// the waves by output tiles; the activations and deltas are also left
// transposed, so that those read their operands 16 bytes at a time.  The
// gradients stay in registers over all groups of the block: one 64 KB slice per
// block, at most two blocks per compute unit.
// Measured against blocks of four waves that each took 64 samples by themselves,
// with row-major weights: 16,384 samples 37.4 -> 23.8 us (20.7 with K = 32 steps
// and tree sums, which round otherwise; then 33.9 with row-major weights, 31.2
// with four waves); whole step with its update at 64 samples 39.5 -> 20.0, 16,384
// 47.8 -> 29.2, 131,072 104.5 -> 82.9, 1,048,576 897 -> 509 us.
__global__ __launch_bounds__(kTrainBlock, 2 * kTrainBlocksPerCu) void k_guide_train(GuideView G, TrainSrc S,
                                                                                   float* __restrict__ partial,
                                                                                   float* __restrict__ sums) {
    __shared__ __align__(16) uint16_t rowsA[4][16 * kGStrideIn];   // features, H2, D3, D1; outputs
    __shared__ __align__(16) uint16_t rowsB[4][16 * kGStrideHid];  // H1, H3, dO, D2
    __shared__ __align__(16) uint16_t xt[kGInPad * kTStride];
    __shared__ __align__(16) uint16_t ht[3][kGHid * kTStride];
    __shared__ __align__(16) uint16_t dt[2][kGHid * kTStride];
    static_assert(16 * kGOut * sizeof(float) <= sizeof(rowsA[0]), "the outputs fit the feature rows");
    const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int q = wv & 3, half = wv >> 2;  // the wave's 16 samples, its half of the outputs
    uint16_t* ra = rowsA[q];
    uint16_t* rb = rowsB[q];
    g_f4 a4[2] = {}, a3[2] = {}, a2[2] = {}, a1[3] = {}, b4 = {}, b3 = {}, b2 = {}, b1 = {};
    float csum = 0.f, clsum = 0.f;
    const uint32_t groups = (S.n + 63u) / 64u;
    for (uint32_t g = blockIdx.x; g < groups; g += gridDim.x) {
        // Opaque to the compiler, which otherwise keeps every LDS and weight
        // address of the group's straight-line code in a register across groups
        // and spills what the products need.
        int lo = l;
        asm volatile("" : "+v"(lo));
        const int smp = lo & 15, part = lo >> 4, col = 16 * q + smp;  // col: the lane's sample in the group
        const int dsmp = 8 * half + (lo & 7), lobe = lo >> 3, dcol = 16 * q + dsmp;  // in the loss gradient
        const uint32_t i = g * 64u + (uint32_t)col, di = g * 64u + (uint32_t)dcol;
        float3 p = make_float3(0.f, 0.f, 0.f), nn = p, w = p;
        float c = 0.f;
        if (S.ts) {
            const uint32_t cnt = min(*S.ts_count, S.ts_cap);
            if (cnt) {
                // position in this pass's subset of `subset` samples, then the
                // subset's fixed uniform choice from the training set
                const uint32_t j = (uint32_t)(g_splitmix64(S.seed ^ ((uint64_t)i << 20)) % S.subset);
                const uint32_t k = (uint32_t)(g_splitmix64(S.subset_seed ^ ((uint64_t)j << 24)) % cnt);
                const uint32_t dk = (uint32_t)__shfl((int)k, dsmp, 64);
                if (i < S.n) {
                    const float4 a = S.ts[3 * (size_t)k], b = S.ts[3 * (size_t)k + 1];
                    p = make_float3(a.x, a.y, a.z);
                    nn = make_float3(b.x, b.y, b.z);
                }
                if (di < S.n) {
                    const float4 e = S.ts[3 * (size_t)dk + 2];
                    c = S.ts[3 * (size_t)dk].w;
                    w = make_float3(e.x, e.y, e.z);
                }
            }
        } else {
            if (i < S.n) {
                p = load3(S.p3, i);
                nn = load3(S.n3, i);
            }
            if (di < S.n) {
                w = load3(S.w3, di);
                c = S.c[di];
            }
        }
        if (g != blockIdx.x) __syncthreads();  // the last group's weight gradients have read xt
        // features (guide_features): lanes of part 0..2 half an axis each, part 3 the rest
        {
            uint16_t* row = ra + smp * kGStrideIn;
            const float ux = (p.x - G.bmin[0]) * G.inv_ext[0], uy = (p.y - G.bmin[1]) * G.inv_ext[1],
                        uz = (p.z - G.bmin[2]) * G.inv_ext[2];
            if (part < 3) {
                const float u = part == 0 ? ux : (part == 1 ? uy : uz);
                const int k0 = 3 + 2 * kGFreq * part + kGFreq * half;
                uint16_t* t = xt + k0 * kTStride + col;
                float f = half ? 0x1p5f : 0.5f;  // 2^(first frequency - 1)
#pragma unroll
                for (int k = 0; k < kGFreq / 2; ++k) {
                    const float r = __builtin_amdgcn_fractf(f * u);
                    const uint32_t sc = pack_bf16x2(__builtin_amdgcn_sinf(r), __builtin_amdgcn_cosf(r));
                    row[k0 + 2 * k] = (uint16_t)sc;
                    row[k0 + 2 * k + 1] = (uint16_t)(sc >> 16);
                    t[2 * k * kTStride] = (uint16_t)sc;
                    t[(2 * k + 1) * kTStride] = (uint16_t)(sc >> 16);
                    f *= 2.0f;
                }
            } else {
                const int k0 = half ? 75 : 0;
                const float v[3] = {half ? nn.x : ux, half ? nn.y : uy, half ? nn.z : uz};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const uint16_t h = to_bf16(v[k]);
                    row[k0 + k] = h;
                    xt[(k0 + k) * kTStride + col] = h;
                }
                if (half) *reinterpret_cast<uint32_t*>(row + kGIn) = 0u;  // meets zero weights: finite
            }
        }
        __syncthreads();
        // forward, keeping every layer's activations transposed, and packed in
        // registers for the backward pass's masks
        uint2 act[3][2];
        auto hidden = [&](int layer, const float* bvec, uint16_t* rows, int stride) {
            return [=, &act](int mt, int o, g_f4 v) {
                const float4 b = *reinterpret_cast<const float4*>(bvec + o);
                uint2 h;
                h.x = pack_bf16x2(fmaxf(v[0] + b.x, 0.f), fmaxf(v[1] + b.y, 0.f));
                h.y = pack_bf16x2(fmaxf(v[2] + b.z, 0.f), fmaxf(v[3] + b.w, 0.f));
                *reinterpret_cast<uint2*>(rows + smp * stride + o) = h;
                act[layer][mt] = h;
                uint16_t* t = ht[layer] + o * kTStride + col;
                t[0] = (uint16_t)h.x;
                t[kTStride] = (uint16_t)(h.x >> 16);
                t[2 * kTStride] = (uint16_t)h.y;
                t[3 * kTStride] = (uint16_t)(h.y >> 16);
            };
        };
        train_product<5>(lo, G.wbf + kGTW1, 2 * half, ra, kGStrideIn, hidden(0, G.theta + kGOffB1, rb, kGStrideHid));
        __syncthreads();
        train_product<4>(lo, G.wbf + kGTW2, 2 * half, rb, kGStrideHid, hidden(1, G.theta + kGOffB2, ra, kGStrideIn));
        __syncthreads();
        train_product<4>(lo, G.wbf + kGTW3, 2 * half, ra, kGStrideIn, hidden(2, G.theta + kGOffB3, rb, kGStrideHid));
        __syncthreads();
        float* out = reinterpret_cast<float*>(ra);
        // 48 padded outputs: the second half's tiles overlap the first's by one
        train_product<4>(lo, G.wbf + kGTW4, half, rb, kGStrideHid, [&](int mt, int o, g_f4 v) {
            if (o >= kGOut || (half && mt == 0)) return;  // padded rows 40..47
            const float4 b = *reinterpret_cast<const float4*>(G.theta + kGOffB4 + o);
            *reinterpret_cast<float4*>(out + smp * kGOut + o) =
                make_float4(v[0] + b.x, v[1] + b.y, v[2] + b.z, v[3] + b.w);
        });
        __syncthreads();
        // loss gradient: eight samples per wave, a lobe per lane
        {
            float o[5], d[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) o[k] = out[dsmp * kGOut + 5 * lobe + k];
            const float nll = guide_dout(o, w, c, d);
            if (lobe == 0 && c != 0.f) {
                csum += c;
                clsum += c * nll;
            }
            uint16_t* row = rb + dsmp * kGStrideHid;
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const uint16_t h = c != 0.f ? to_bf16(d[k]) : (uint16_t)0;
                row[5 * lobe + k] = h;
                dt[0][(5 * lobe + k) * kTStride + dcol] = h;
            }
            row[kGOut + lobe] = 0;  // columns 40..47 of dO meet zero weights: they must be finite
        }
        __syncthreads();
        // D_{l-1} = (D_l W_l) (.) [H_{l-1} > 0]
        auto back = [&](int layer, uint16_t* rows, int stride, uint16_t* dtr) {
            return [=, &act](int mt, int o, g_f4 v) {
                const uint2 a = act[layer][mt];
                uint2 h;
                h.x = pack_bf16x2((a.x & 0xFFFFu) ? v[0] : 0.f, (a.x >> 16) ? v[1] : 0.f);
                h.y = pack_bf16x2((a.y & 0xFFFFu) ? v[2] : 0.f, (a.y >> 16) ? v[3] : 0.f);
                *reinterpret_cast<uint2*>(rows + smp * stride + o) = h;
                uint16_t* t = dtr + o * kTStride + col;
                t[0] = (uint16_t)h.x;
                t[kTStride] = (uint16_t)(h.x >> 16);
                t[2 * kTStride] = (uint16_t)h.y;
                t[3 * kTStride] = (uint16_t)(h.y >> 16);
            };
        };
        // layer 4 (64 -> 40)
        train_product<3>(lo, G.wbf + kGWT4, 2 * half, rb, kGStrideHid, back(2, ra, kGStrideIn, dt[1]));
        if (half) {
            grad_tile(lo, a4[0], dt[0], 32, ht[2], 16 * q);
            if (q < 3) bias_tile(lo, b4, dt[0], 16 * q);
        } else {
            grad_tile(lo, a4[0], dt[0], 0, ht[2], 16 * q);
            grad_tile(lo, a4[1], dt[0], 16, ht[2], 16 * q);
        }
        __syncthreads();
        // layer 3
        train_product<4>(lo, G.wbf + kGWT3, 2 * half, ra, kGStrideIn, back(1, rb, kGStrideHid, dt[0]));
#pragma unroll
        for (int k = 0; k < 2; ++k) grad_tile(lo, a3[k], dt[1], 16 * q, ht[1], 32 * half + 16 * k);
        if (half) bias_tile(lo, b3, dt[1], 16 * q);
        __syncthreads();
        // layer 2
        train_product<4>(lo, G.wbf + kGWT2, 2 * half, rb, kGStrideHid, back(0, ra, kGStrideIn, dt[1]));
#pragma unroll
        for (int k = 0; k < 2; ++k) grad_tile(lo, a2[k], dt[0], 16 * q, ht[0], 32 * half + 16 * k);
        if (!half) bias_tile(lo, b2, dt[0], 16 * q);
        __syncthreads();
        // layer 1 (78 -> 64)
#pragma unroll
        for (int k = 0; k < 2; ++k) grad_tile(lo, a1[k], dt[1], 16 * q, xt, 48 * half + 16 * k);
        if (half) bias_tile(lo, b1, dt[1], 16 * q);
        else grad_tile(lo, a1[2], dt[1], 16 * q, xt, 32);
    }
    float* P = partial + (size_t)blockIdx.x * kGPartial;
    store_tile(a4[0], P + kGOffW4, 32 * half, 16 * q, kGOut, kGHid);
    if (!half) store_tile(a4[1], P + kGOffW4, 16, 16 * q, kGOut, kGHid);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        store_tile(a3[k], P + kGOffW3, 16 * q, 32 * half + 16 * k, kGHid, kGHid);
        store_tile(a2[k], P + kGOffW2, 16 * q, 32 * half + 16 * k, kGHid, kGHid);
        store_tile(a1[k], P + kGOffW1, 16 * q, 48 * half + 16 * k, kGHid, kGIn);
    }
    if (half) {
        if (q < 3) store_bias(b4, P + kGOffB4, 16 * q, kGOut);
        store_bias(b3, P + kGOffB3, 16 * q, kGHid);
        store_bias(b1, P + kGOffB1, 16 * q, kGHid);
    } else {
        store_tile(a1[2], P + kGOffW1, 16 * q, 32, kGHid, kGIn);
        store_bias(b2, P + kGOffB2, 16 * q, kGHid);
    }
    for (int off = 4; off > 0; off >>= 1) {
        csum += __shfl_xor(csum, off, 64);
        clsum += __shfl_xor(clsum, off, 64);
    }
    __shared__ float red[2][kTrainWaves];
    if (l == 0) {
        red[0][wv] = csum;
        red[1][wv] = clsum;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        float s = 0.f;
        for (int k = 0; k < kTrainWaves; ++k) s += red[threadIdx.x][k];
        sums[2 * blockIdx.x + threadIdx.x] = s;
    }
}

// Sums the blocks' slices in a fixed order (a block of this kernel: 64
// parameters, 16 waves each summing every 16th slice) and, with ADAM, takes the
// step for them (Kingma & Ba 2015, bias corrections bc1 = 1 - b1^t, bc2 = 1 -
// b2^t) and writes their BF16 operand copies; without, stores the gradient in
// theta.  grad = (sum of the slices) / (sum of c); loss = sum(c nll) / sum(c).
// A batch whose weights sum to zero leaves every parameter unchanged (gradient
// 0).  One launch where a reduction to 32 rows, Adam and the refresh of all
// copies took three: 16,384 samples (256 slices, 16.4 MB) 14.6 -> 6.3 us.
constexpr uint32_t kUpdateBlock = 1024, kUpdateGrid = (kGParams + 63) / 64;
template <bool ADAM>
__global__ __launch_bounds__(kUpdateBlock) void k_guide_update(const float* __restrict__ partial,
                                                               const float* __restrict__ sums, uint32_t blocks,
                                                               float* __restrict__ theta, float* __restrict__ m,
                                                               float* __restrict__ v, uint16_t* __restrict__ wbf,
                                                               float lr, float bc1, float bc2,
                                                               float* __restrict__ loss) {
    __shared__ float red[16][64];
    __shared__ float tot[16][2];
    const uint32_t l = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const int p = (int)(blockIdx.x * 64u + l);
    float acc = 0.f;
    if (p < kGParams) {
#pragma unroll 8
        for (uint32_t b = wv; b < blocks; b += 16u) acc += partial[(size_t)b * kGPartial + p];
    }
    red[wv][l] = acc;
    float sc = 0.f, sl = 0.f;
    for (uint32_t b = threadIdx.x; b < blocks; b += kUpdateBlock) {
        sc += sums[2 * b];
        sl += sums[2 * b + 1];
    }
    for (int off = 32; off > 0; off >>= 1) {
        sc += __shfl_xor(sc, off, 64);
        sl += __shfl_xor(sl, off, 64);
    }
    if (l == 0) {
        tot[wv][0] = sc;
        tot[wv][1] = sl;
    }
    __syncthreads();
    if (wv != 0) return;
    sc = sl = acc = 0.f;
    for (int k = 0; k < 16; ++k) {
        sc += tot[k][0];
        sl += tot[k][1];
        acc += red[k][l];
    }
    if (p == 0) {
        loss[0] = sc > 0.f ? sl / sc : 0.f;
        loss[1] = sc;
    }
    if (p >= kGParams) return;
    if (!ADAM) {
        theta[p] = sc > 0.f ? acc / sc : 0.f;
        return;
    }
    if (!(sc > 0.f)) return;
    const float g = acc / sc;
    const float mm = 0.9f * m[p] + 0.1f * g;
    const float vv = 0.999f * v[p] + 0.001f * g * g;
    m[p] = mm;
    v[p] = vv;
    const float t = theta[p] - lr * (mm / bc1) / (sqrtf(vv / bc2) + 1e-8f);
    theta[p] = t;
    store_operands(wbf, p, t);
}

__global__ void k_zero_u32(uint32_t* p) {
    if (threadIdx.x == 0) *p = 0u;
}

uint64_t g_host_mix(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

int check_guide(tn_guide* g) {
    if (!g) return set_error(TN_ERR_INVALID, "NULL guide");
    TN_HIP(hipSetDevice(g->device));
    return TN_OK;
}

// Blocks of a training launch: one 64-sample group each while every compute unit
// has at most two blocks (what LDS holds), then several groups per block.
uint32_t train_blocks(const tn_guide* g, uint32_t n) {
    return std::min((n + 63) / 64, (uint32_t)std::max(g->cus, 1) * kTrainBlocksPerCu);
}

// Per-block gradient slices, then the per-block sums (two words each).
int ensure_partial(tn_guide* g, uint32_t blocks) {
    if (g->partial_blocks >= blocks) return TN_OK;
    if (g->partial) (void)hipFree(g->partial);
    g->partial = nullptr;
    g->partial_blocks = 0;
    TN_HIP(hipMalloc(&g->partial, (size_t)blocks * (kGPartial + 2) * sizeof(float)));
    g->partial_blocks = blocks;
    return TN_OK;
}

float* block_sums(tn_guide* g) { return g->partial + (size_t)g->partial_blocks * kGPartial; }

// Gradient slices and sums of one batch.
int launch_train(tn_guide* g, const TrainSrc& S, uint32_t blocks, hipStream_t stream) {
    k_guide_train<<<blocks, kTrainBlock, 0, stream>>>(g->view(), S, g->partial, block_sums(g));
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int refresh(tn_guide* g, hipStream_t stream) {
    k_guide_refresh<<<(kGParams + 255) / 256, 256, 0, stream>>>(g->theta, g->wbf);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int adam_step(tn_guide* g, uint32_t blocks, hipStream_t stream) {
    const uint32_t t = ++g->steps;
    const float bc1 = (float)(1.0 - std::pow(0.9, (double)t));
    const float bc2 = (float)(1.0 - std::pow(0.999, (double)t));
    k_guide_update<true><<<kUpdateGrid, kUpdateBlock, 0, stream>>>(g->partial, block_sums(g), blocks, g->theta, g->adam_m,
                                                                   g->adam_v, g->wbf, g->lr, bc1, bc2, g->dloss);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int check_batch(const float* p3, const float* n3, const float* w3, const float* c, uint32_t n) {
    if (n && (!p3 || !n3 || !w3 || !c)) return set_error(TN_ERR_INVALID, "NULL batch array");
    if (n > (1u << 26)) return set_error(TN_ERR_LIMIT, "batch of %u samples exceeds 2^26", n);
    return TN_OK;
}

}  // namespace

int guide_reserve_set(tn_guide* g, uint32_t cap, hipStream_t stream) {
    if (cap > g->ts_cap) {
        if (g->ts) (void)hipFree(g->ts);
        g->ts = nullptr;
        g->ts_cap = 0;
        TN_HIP(hipMalloc(&g->ts, (size_t)cap * 3 * sizeof(float4)));
        g->ts_cap = cap;
    }
    k_zero_u32<<<1, 64, 0, stream>>>(g->ts_count);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int guide_train_pending(tn_guide* g, hipStream_t stream) {
    if (!g->pending) return TN_OK;
    const uint32_t n = g->pending;
    g->pending = 0;
    return guide_train_from_set(g, n, stream);
}

int guide_defer_begin(tn_guide* g, hipStream_t stream, bool recording, bool* started) {
    *started = false;
    if (!g->pending) return TN_OK;
    if (!g->tstream) {
        TN_HIP(hipStreamCreateWithFlags(&g->tstream, hipStreamNonBlocking));
        TN_HIP(hipEventCreateWithFlags(&g->ev_fork, hipEventDisableTiming));
        TN_HIP(hipEventCreateWithFlags(&g->ev_join, hipEventDisableTiming));
    }
    TN_HIP(hipMemcpyAsync(g->wbf_snap, g->wbf, kGBf16 * sizeof(uint16_t), hipMemcpyDeviceToDevice, stream));
    TN_HIP(hipMemcpyAsync(g->theta_snap, g->theta, kGParams * sizeof(float), hipMemcpyDeviceToDevice, stream));
    TN_HIP(hipEventRecord(g->ev_fork, stream));
    TN_HIP(hipStreamWaitEvent(g->tstream, g->ev_fork, 0));
    // the kernels take the set's pointers by value, so the swap below
    // leaves this training on the pending set
    const int rc = guide_train_pending(g, g->tstream);
    if (rc) {
        (void)hipStreamSynchronize(g->tstream);
        return rc;
    }
    TN_HIP(hipEventRecord(g->ev_join, g->tstream));
    if (recording) {
        std::swap(g->ts, g->ts_alt);
        std::swap(g->ts_cap, g->ts_alt_cap);
        std::swap(g->ts_count, g->ts_count_alt);
    }
    *started = true;
    return TN_OK;
}

int guide_train_from_set(tn_guide* g, uint32_t train_samples, hipStream_t stream) {
    const uint32_t nb = train_blocks(g, g->batch);
    int rc = ensure_partial(g, nb);
    if (rc) return rc;
    // a uniform subset of train_samples recorded samples, `epochs` passes of
    // mini-batches over it
    const uint64_t draws = (uint64_t)train_samples * std::max(1u, g->epochs);
    const uint32_t steps = (uint32_t)std::max<uint64_t>(1, draws / g->batch);
    const uint64_t subset_seed = g_host_mix(g->seed ^ (0xA5A5A5A5ull + g->passes++));
    for (uint32_t s = 0; s < steps; ++s) {
        TrainSrc S{};
        S.n = g->batch;
        S.ts = g->ts;
        S.ts_count = g->ts_count;
        S.ts_cap = g->ts_cap;
        S.subset = std::max(1u, train_samples);
        S.subset_seed = subset_seed;
        S.seed = g->seed * 0x9E3779B97F4A7C15ull + ((uint64_t)g->steps << 32) + s;
        if ((rc = launch_train(g, S, nb, stream))) return rc;
        if ((rc = adam_step(g, nb, stream))) return rc;
    }
    return TN_OK;
}

}  // namespace tn

using namespace tn;

extern "C" {

int tn_guide_create(const float bmin[3], const float bmax[3], uint64_t seed, tn_guide** out) {
    if (!bmin || !bmax || !out) return set_error(TN_ERR_INVALID, "NULL argument");
    *out = nullptr;
    for (int k = 0; k < 3; ++k)
        if (!(bmax[k] >= bmin[k]) || !std::isfinite(bmin[k]) || !std::isfinite(bmax[k]))
            return set_error(TN_ERR_INVALID, "invalid guide box");
    int dev = 0;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return set_error(TN_ERR_NODEVICE, "no HIP device available");
    TN_HIP(hipGetDevice(&dev));
    tn_guide* g = new tn_guide();
    g->device = dev;
    (void)hipDeviceGetAttribute(&g->cus, hipDeviceAttributeMultiprocessorCount, dev);
    g->seed = seed;
    for (int k = 0; k < 3; ++k) {
        g->bmin[k] = bmin[k];
        g->bmax[k] = bmax[k];
    }
    // Uniform(-1/sqrt(in), 1/sqrt(in)) weights, zero biases.
    std::vector<float> theta(kGParams, 0.f);
    std::mt19937_64 rng(seed);
    const int ins[4] = {kGIn, kGHid, kGHid, kGHid}, outs[4] = {kGHid, kGHid, kGHid, kGOut};
    size_t off = 0;
    for (int L = 0; L < 4; ++L) {
        std::uniform_real_distribution<float> U(-1.0f / std::sqrt((float)ins[L]), 1.0f / std::sqrt((float)ins[L]));
        for (int k = 0; k < ins[L] * outs[L]; ++k) theta[off + k] = U(rng);
        off += (size_t)ins[L] * outs[L] + outs[L];
    }
    auto fail = [&](int rc) {
        tn_guide_destroy(g);
        return rc;
    };
    hipError_t e;
    if ((e = hipMalloc(&g->theta, kGParams * sizeof(float))) != hipSuccess ||
        (e = hipMalloc(&g->adam_m, kGParams * sizeof(float))) != hipSuccess ||
        (e = hipMalloc(&g->adam_v, kGParams * sizeof(float))) != hipSuccess ||
        (e = hipMalloc(&g->wbf, kGBf16 * sizeof(uint16_t))) != hipSuccess ||
        (e = hipMalloc(&g->dloss, 4 * sizeof(float))) != hipSuccess ||
        (e = hipMalloc(&g->ts_count, 4 * sizeof(uint32_t))) != hipSuccess ||
        (e = hipMalloc(&g->wbf_snap, kGBf16 * sizeof(uint16_t))) != hipSuccess ||
        (e = hipMalloc(&g->theta_snap, kGParams * sizeof(float))) != hipSuccess)
        return fail(hip_error(e, "hipMalloc"));
    g->ts_count_alt = g->ts_count + 2;  // words 0 and 2 count the two sets
    if ((e = hipMemset(g->dloss, 0, 4 * sizeof(float))) != hipSuccess ||
        (e = hipMemset(g->ts_count, 0, 4 * sizeof(uint32_t))) != hipSuccess)
        return fail(hip_error(e, "hipMemset"));
    int rc = tn_guide_set_params(g, theta.data());
    if (rc) return fail(rc);
    *out = g;
    return TN_OK;
}

int tn_guide_destroy(tn_guide* g) {
    if (!g) return TN_OK;
    (void)hipSetDevice(g->device);
    (void)hipDeviceSynchronize();
    // ts_count and ts_count_alt are two words of one allocation
    uint32_t* counts = std::min(g->ts_count, g->ts_count_alt ? g->ts_count_alt : g->ts_count);
    for (void* p : {(void*)g->theta, (void*)g->adam_m, (void*)g->adam_v, (void*)g->wbf, (void*)g->partial,
                    (void*)g->dloss, (void*)g->ts, (void*)g->ts_alt, (void*)counts, (void*)g->wbf_snap,
                    (void*)g->theta_snap})
        if (p) (void)hipFree(p);
    if (g->ev_fork) (void)hipEventDestroy(g->ev_fork);
    if (g->ev_join) (void)hipEventDestroy(g->ev_join);
    if (g->tstream) (void)hipStreamDestroy(g->tstream);
    delete g;
    return TN_OK;
}

int tn_guide_flush(tn_guide* g, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    return guide_train_pending(g, (hipStream_t)stream);
}

int tn_guide_get_params(tn_guide* g, float* theta) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (!theta) return set_error(TN_ERR_INVALID, "NULL argument");
    TN_HIP(hipDeviceSynchronize());
    TN_HIP(hipMemcpy(theta, g->theta, kGParams * sizeof(float), hipMemcpyDeviceToHost));
    return TN_OK;
}

int tn_guide_set_params(tn_guide* g, const float* theta) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (!theta) return set_error(TN_ERR_INVALID, "NULL argument");
    for (int k = 0; k < kGParams; ++k)
        if (!std::isfinite(theta[k])) return set_error(TN_ERR_INVALID, "non-finite parameter %d", k);
    TN_HIP(hipDeviceSynchronize());
    TN_HIP(hipMemcpy(g->theta, theta, kGParams * sizeof(float), hipMemcpyHostToDevice));
    TN_HIP(hipMemset(g->adam_m, 0, kGParams * sizeof(float)));
    TN_HIP(hipMemset(g->adam_v, 0, kGParams * sizeof(float)));
    TN_HIP(hipMemset(g->wbf, 0, kGBf16 * sizeof(uint16_t)));
    g->steps = 0;
    rc = refresh(g, nullptr);
    if (rc) return rc;
    TN_HIP(hipDeviceSynchronize());
    return TN_OK;
}

int tn_guide_set_options(tn_guide* g, float lr, uint32_t batch, float mis_guided, uint32_t epochs) {
    if (!g) return set_error(TN_ERR_INVALID, "NULL guide");
    if (!(lr > 0.f) || !std::isfinite(lr)) return set_error(TN_ERR_INVALID, "learning rate must be > 0");
    if (batch == 0 || batch % 64 || batch > (1u << 24))
        return set_error(TN_ERR_INVALID, "batch must be a positive multiple of 64 up to 2^24");
    if (!(mis_guided >= 0.f && mis_guided <= 1.f))
        return set_error(TN_ERR_INVALID, "mis_guided must be in [0, 1]");
    if (epochs == 0 || epochs > 1024) return set_error(TN_ERR_INVALID, "epochs must be in 1..1024");
    g->lr = lr;
    g->batch = batch;
    g->mis_guided = mis_guided;
    g->epochs = epochs;
    return TN_OK;
}

int tn_guide_forward(tn_guide* g, const float* p3, const float* n3, uint32_t n, float* out, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (n && (!p3 || !n3 || !out)) return set_error(TN_ERR_INVALID, "NULL argument");
    if (n > (1u << 30)) return set_error(TN_ERR_LIMIT, "too many points");
    if (!n) return TN_OK;
    const uint32_t grid = std::min<uint32_t>((n + 15) / 16, (uint32_t)std::max(g->cus, 1) * 8);  // resident: 8 one-wave blocks per CU
    k_guide_forward<<<grid, 64, 0, (hipStream_t)stream>>>(g->view(), p3, n3, n, out);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int tn_guide_pdf(tn_guide* g, const float* p3, const float* n3, const float* w3, uint32_t n, float* pdf,
                 void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (n && (!p3 || !n3 || !w3 || !pdf)) return set_error(TN_ERR_INVALID, "NULL argument");
    if (n > (1u << 30)) return set_error(TN_ERR_LIMIT, "too many points");
    if (!n) return TN_OK;
    return launch_eval(g, p3, n3, w3, nullptr, n, pdf, nullptr, (hipStream_t)stream);
}

int tn_guide_sample(tn_guide* g, const float* p3, const float* n3, const float* u3, uint32_t n, float* w3,
                    float* pdf, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (n && (!p3 || !n3 || !u3 || !w3 || !pdf)) return set_error(TN_ERR_INVALID, "NULL argument");
    if (n > (1u << 30)) return set_error(TN_ERR_LIMIT, "too many points");
    if (!n) return TN_OK;
    return launch_eval(g, p3, n3, nullptr, u3, n, pdf, w3, (hipStream_t)stream);
}

int tn_guide_loss_grad(tn_guide* g, const float* p3, const float* n3, const float* w3, const float* c,
                       uint32_t n, float* grad, float* loss, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if ((rc = check_batch(p3, n3, w3, c, n))) return rc;
    if (!grad) return set_error(TN_ERR_INVALID, "NULL gradient");
    if (n == 0) return set_error(TN_ERR_INVALID, "empty batch");
    const uint32_t nb = train_blocks(g, n);
    if ((rc = ensure_partial(g, nb))) return rc;
    hipStream_t s = (hipStream_t)stream;
    TrainSrc S{p3, n3, w3, c, n, nullptr, nullptr, 0, 0, 1, 0};
    if ((rc = launch_train(g, S, nb, s))) return rc;
    k_guide_update<false><<<kUpdateGrid, kUpdateBlock, 0, s>>>(g->partial, block_sums(g), nb, grad, nullptr, nullptr,
                                                               nullptr, 0.f, 1.f, 1.f, g->dloss);
    TN_HIP(hipGetLastError());
    if (loss) {
        TN_HIP(hipMemcpyAsync(loss, g->dloss, sizeof(float), hipMemcpyDeviceToHost, s));
        TN_HIP(hipStreamSynchronize(s));
    }
    return TN_OK;
}

int tn_guide_train_recorded(tn_guide* g, uint32_t train_samples, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if (train_samples == 0) return set_error(TN_ERR_INVALID, "train_samples must be positive");
    if (!g->ts) return set_error(TN_ERR_INVALID, "no recorded training set: render with train_samples > 0 first");
    if ((rc = guide_train_pending(g, (hipStream_t)stream))) return rc;  // a deferred set trains first
    return guide_train_from_set(g, train_samples, (hipStream_t)stream);
}

int tn_guide_train_step(tn_guide* g, const float* p3, const float* n3, const float* w3, const float* c,
                        uint32_t n, float* loss, void* stream) {
    int rc = check_guide(g);
    if (rc) return rc;
    if ((rc = check_batch(p3, n3, w3, c, n))) return rc;
    if (n == 0) return set_error(TN_ERR_INVALID, "empty batch");
    const uint32_t nb = train_blocks(g, n);
    if ((rc = ensure_partial(g, nb))) return rc;
    hipStream_t s = (hipStream_t)stream;
    TrainSrc S{p3, n3, w3, c, n, nullptr, nullptr, 0, 0, 1, 0};
    if ((rc = launch_train(g, S, nb, s))) return rc;
    if ((rc = adam_step(g, nb, s))) return rc;
    if (loss) {
        TN_HIP(hipMemcpyAsync(loss, g->dloss, sizeof(float), hipMemcpyDeviceToHost, s));
        TN_HIP(hipStreamSynchronize(s));
    }
    return TN_OK;
}

int tn_guide_info(tn_guide* g, uint32_t* train_samples, uint32_t* steps, float* last_loss) {
    int rc = check_guide(g);
    if (rc) return rc;
    TN_HIP(hipDeviceSynchronize());
    if (train_samples) {
        uint32_t cnt = 0;
        TN_HIP(hipMemcpy(&cnt, g->ts_count, 4, hipMemcpyDeviceToHost));
        *train_samples = std::min(cnt, g->ts_cap);
    }
    if (steps) *steps = g->steps;
    if (last_loss) TN_HIP(hipMemcpy(last_loss, g->dloss, 4, hipMemcpyDeviceToHost));
    return TN_OK;
}

long tn_guide_get_train_set(tn_guide* g, float* out, size_t cap) {
    int rc = check_guide(g);
    if (rc) return rc;
    TN_HIP(hipDeviceSynchronize());
    uint32_t cnt = 0;
    TN_HIP(hipMemcpy(&cnt, g->ts_count, 4, hipMemcpyDeviceToHost));
    const size_t n = std::min<size_t>(std::min(cnt, g->ts_cap), cap);
    if (n && !out) return set_error(TN_ERR_INVALID, "NULL output");
    if (n) TN_HIP(hipMemcpy(out, g->ts, n * 3 * sizeof(float4), hipMemcpyDeviceToHost));
    return (long)n;
}

}  // extern "C"
