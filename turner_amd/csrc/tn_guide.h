// tn_guide.h -- learned path-guiding proposal: device-side model description
// shared by guide.hip (training / inference kernels) and render.hip (guided
// sampling).  No reference counterpart: the reference samples the hemisphere
// uniformly (lib/sampling.h:20-32).
//
// features(p, n) = [u, sin(2^k pi u_c), cos(2^k pi u_c) for c = x,y,z, k = 0..11, n]
//                  with u = (p - bmin) / (bmax - bmin)                         (78)
// MLP 78 -> 64 -> 64 -> 64 -> 40, ReLU hidden layers, BF16 weights and
// activations as MFMA operands, FP32 accumulation, FP32 master weights.
// out[5j .. 5j+4] = (logit_j, m_j, kraw_j): 8-lobe von Mises-Fisher mixture
// with pi = softmax(logit), mu = m / |m|, kappa = softplus(kraw) + 0.01.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tn {

constexpr int kGIn = 78, kGInPad = 80, kGHid = 64, kGOut = 40, kGOutPad = 48, kGLobes = 8;
constexpr int kGFreq = 12;
constexpr float kKappaMin = 0.01f, kKappaMax = 1.0e4f;
// flat FP32 parameter layout (per layer W (out x in, row major) then b)
constexpr int kGOffW1 = 0, kGOffB1 = 64 * 78;
constexpr int kGOffW2 = kGOffB1 + 64, kGOffB2 = kGOffW2 + 64 * 64;
constexpr int kGOffW3 = kGOffB2 + 64, kGOffB3 = kGOffW3 + 64 * 64;
constexpr int kGOffW4 = kGOffB3 + 64, kGOffB4 = kGOffW4 + 40 * 64;
constexpr int kGParams = kGOffB4 + 40;  // 15976
// BF16 copies of W_l (forward A operand, padded [out_pad][in_pad]) and W_l^T
// (backward A operand, [in_pad][out_pad]) in fragment order (frag_at)
constexpr int kGW1 = 0, kGW2 = kGW1 + 64 * kGInPad, kGW3 = kGW2 + 64 * 64, kGW4 = kGW3 + 64 * 64;
constexpr int kGWT2 = kGW4 + kGOutPad * 64, kGWT3 = kGWT2 + 64 * 64, kGWT4 = kGWT3 + 64 * 64;
// the training kernel's copies of W_l; these and W_l^T in fragments of K = 16
// (frag16_at)
constexpr int kGTW1 = kGWT4 + 64 * kGOutPad, kGTW2 = kGTW1 + 64 * kGInPad, kGTW3 = kGTW2 + 64 * 64,
              kGTW4 = kGTW3 + 64 * 64;
constexpr int kGBf16 = kGTW4 + kGOutPad * 64;

// Position of element (row, col) of a padded [16 out_tiles][cols] matrix in
// fragment order: for every 16-row tile the K = 32 fragments of its columns,
// 64 lanes of 8 consecutive columns each, then (cols = 32 kt32 + 16) the K = 16
// fragments of the last 16 columns, 64 lanes of 4.  A fragment load then reads
// 1 KB (512 B) in a row; row-major it touched 16 cache lines per instruction, and
// the products that read their weights from memory waited for nothing else
// (a 64 x 64 product on 16 samples: 5,000 cycles).
__host__ __device__ constexpr int frag_at(int row, int col, int kt32, int out_tiles) {
    const int mt = row / 16, r = row % 16;
    if (col < 32 * kt32) return ((mt * kt32 + col / 32) * 64 + col % 32 / 8 * 16 + r) * 8 + col % 8;
    const int c = col - 32 * kt32;
    return out_tiles * kt32 * 512 + (mt * 64 + c / 4 * 16 + r) * 4 + c % 4;
}

// The same in K = 16 fragments alone (64 lanes of 4 columns each), kt16 per row tile.
__host__ __device__ constexpr int frag16_at(int row, int col, int kt16) {
    return ((row / 16 * kt16 + col / 16) * 64 + col % 16 / 4 * 16 + row % 16) * 4 + col % 4;
}

struct GuideView {
    const uint16_t* wbf;  // BF16 weight copies (layout above)
    const float* theta;   // FP32 master parameters (biases are read from here)
    float bmin[3], inv_ext[3];
};

__host__ __device__ __forceinline__ float softplusf(float x) {
    return x > 20.f ? x : log1pf(expf(x));
}

// vMF density on the sphere, stable for small and large kappa.
__device__ __forceinline__ float vmf_pdf(float cosang, float kappa) {
    return kappa / (6.28318530717958647692f * -expm1f(-2.0f * kappa)) * expf(kappa * (cosang - 1.0f));
}

struct Mixture {
    float pi[kGLobes];
    float mu[kGLobes][3];
    float kappa[kGLobes];
};

__device__ __forceinline__ void mixture_from(const float* out, Mixture& M) {
    float mx = out[0];
    for (int j = 1; j < kGLobes; ++j) mx = fmaxf(mx, out[5 * j]);
    float sum = 0.f;
    for (int j = 0; j < kGLobes; ++j) {
        M.pi[j] = expf(out[5 * j] - mx);
        sum += M.pi[j];
        const float mx3 = out[5 * j + 1], my = out[5 * j + 2], mz = out[5 * j + 3];
        const float inv = 1.0f / fmaxf(sqrtf(mx3 * mx3 + my * my + mz * mz), 1e-12f);
        M.mu[j][0] = mx3 * inv;
        M.mu[j][1] = my * inv;
        M.mu[j][2] = mz * inv;
        M.kappa[j] = fminf(softplusf(out[5 * j + 4]) + kKappaMin, kKappaMax);
    }
    const float is = 1.0f / sum;
    for (int j = 0; j < kGLobes; ++j) M.pi[j] *= is;
}

__device__ __forceinline__ float mixture_pdf(const Mixture& M, float3 w) {
    float q = 0.f;
    for (int j = 0; j < kGLobes; ++j)
        q += M.pi[j] * vmf_pdf(M.mu[j][0] * w.x + M.mu[j][1] * w.y + M.mu[j][2] * w.z, M.kappa[j]);
    return q;
}

// Lobe by the CDF of pi (u0: the first lobe whose cumulative weight exceeds
// u0, else the last), vMF cosine by inverse CDF (u1), azimuth (u2).  The
// lobe is selected without dynamic indexing so M stays in registers.
__device__ __forceinline__ float3 mixture_sample(const Mixture& M, float u0, float u1, float u2) {
    float c = 0.f, k = M.kappa[kGLobes - 1];
    float mx = M.mu[kGLobes - 1][0], my = M.mu[kGLobes - 1][1], mz = M.mu[kGLobes - 1][2];
    bool found = false;
#pragma unroll
    for (int q = 0; q < kGLobes - 1; ++q) {
        c += M.pi[q];
        const bool take = !found && u0 < c;
        k = take ? M.kappa[q] : k;
        mx = take ? M.mu[q][0] : mx;
        my = take ? M.mu[q][1] : my;
        mz = take ? M.mu[q][2] : mz;
        found = found || take;
    }
    const float cw = fmaxf(-1.0f, fminf(1.0f, 1.0f + logf(u1 + (1.0f - u1) * expf(-2.0f * k)) / k));
    const float sw = sqrtf(fmaxf(0.f, 1.f - cw * cw));
    float sp, cp;
    __sincosf(6.28318530717958647692f * u2, &sp, &cp);
    const float sign = copysignf(1.0f, mz);
    const float a = -1.0f / (sign + mz);
    const float b = mx * my * a;
    const float3 b1 = make_float3(1.0f + sign * mx * mx * a, sign * b, -sign * mx);
    const float3 b2 = make_float3(b, sign + my * my * a, -my);
    return make_float3(cw * mx + sw * (cp * b1.x + sp * b2.x), cw * my + sw * (cp * b1.y + sp * b2.y),
                       cw * mz + sw * (cp * b1.z + sp * b2.z));
}

typedef __attribute__((ext_vector_type(4))) float g_f4;
typedef __attribute__((ext_vector_type(4))) short g_s4;

// Two FP32 values -> packed BF16 (a low, b high), round to nearest even:
// one v_cvt_pk_bf16_f32 on gfx950.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 h2;
    const h2 h = __builtin_convertvector((f2){a, b}, h2);
    uint32_t r;
    __builtin_memcpy(&r, &h, 4);
    return r;
}

// FP32 -> BF16, round to nearest even (finite x; the host form rounds the
// bits, the device form converts in hardware, with equal results).
__host__ __device__ __forceinline__ uint16_t to_bf16(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (uint16_t)pack_bf16x2(x, 0.f);
#else
    uint32_t u;
    __builtin_memcpy(&u, &x, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
#endif
}

typedef __attribute__((ext_vector_type(8))) __bf16 g_bf8;

// K = 32 tiles with gfx950's mfma_f32_16x16x32_bf16: A lane holds row
// 16mt + l%16, columns 32kt + 8(l/16) .. +7; B lane holds sample 16nt + l%16,
// features 32kt + 8(l/16) .. +7; the accumulator layout is the 16x16x16 one.
// KT32 tiles of 32 then, if TAIL, one 16x16x16 tile for columns 32 KT32 .. +15
// (A lane: row 16mt + l%16, columns 32 KT32 + 4(l/16) .. +3; B likewise).  The
// matrix is in fragment order (frag_at): lane l's part of fragment f is at
// 8 (64 f + l), of tail fragment f at 4 (64 f + l) behind the others.
template <int KT32, int OUT_TILES>
__device__ __forceinline__ g_bf8 frag32(const uint16_t* W, int mt, int kt, uint32_t l) {
    return *reinterpret_cast<const g_bf8*>(reinterpret_cast<const char*>(W) + (16u * l + 1024u * (uint32_t)(mt * KT32 + kt)));
}
template <int KT32, int OUT_TILES>
__device__ __forceinline__ g_s4 frag16(const uint16_t* W, int mt, uint32_t l) {
    return *reinterpret_cast<const g_s4*>(reinterpret_cast<const char*>(W) +
                                          (8u * l + 1024u * OUT_TILES * KT32 + 512u * (uint32_t)mt));
}
__device__ __forceinline__ g_bf8 as_bf8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const uint4 v = make_uint4(a, b, c, d);
    g_bf8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

// The network runs on 16 samples per matrix tile without LDS.  A lane (sample s =
// l % 16, group g = l / 16) computes the features of its sample that its B
// operands hold, and a layer's outputs (accumulator: outputs 16 mt + 4 g .. +3 of
// sample s) become the next layer's B operands (features 32 kt + 8 g .. +7) by two
// lane swaps.  Through LDS rows a wave wrote 78 two-byte features per lane and
// met four round trips per layer; its 20 KB also kept all but two waves off a SIMD.

// First layer operands of a tile: features 32 kt + 8 g .. +7 and 64 + 4 g .. +3.
struct GuideIn {
    g_bf8 b[2];
    g_s4 t;
};

// The lane's feature frequencies: sin / cos of 2^q pi u are those of 2 pi
// (2^(q-1) u).  A run of eight starts with the cosine at q, then sine and cosine
// at q + 1 (scale x = 2^(q-1)), then sine, cosine, sine, cosine, sine from the
// next octave (scale z), perhaps of the next axis; the last four features
// likewise.
struct GuideLane {
    int g;
    float x[2], z[2], t;
};
__device__ __forceinline__ GuideLane guide_lane() {
    const int g = (int)(threadIdx.x & 63u) >> 4;
    auto scale = [](int q) { return __uint_as_float((uint32_t)(126 + q) << 23); };
    GuideLane L;
    L.g = g;
    L.x[0] = scale(4 * g - 2);                // -, 2, 6, 10
    L.z[0] = scale(g == 3 ? 0 : 4 * g);       // 0, 4, 8, 0
    L.x[1] = scale(g == 3 ? 2 : 4 * g + 2);   // 2, 6, 10, 2
    L.z[1] = scale(g == 0 || g == 3 ? 4 : (g == 1 ? 8 : 0));
    L.t = scale(6 + 2 * g);                   // 6, 8, 10, -
    return L;
}

// The hardware sine and cosine take revolutions; the argument's fraction (exact,
// as is the power-of-two scaling) keeps them in range.  Absolute error about
// 1.3e-7 (sincospif: 5e-8), far below the BF16 step.
__device__ __forceinline__ GuideIn guide_features(const GuideView& G, const GuideLane& L, float3 p, float3 n) {
    const float ux = (p.x - G.bmin[0]) * G.inv_ext[0], uy = (p.y - G.bmin[1]) * G.inv_ext[1],
                uz = (p.z - G.bmin[2]) * G.inv_ext[2];
    auto turns = [](float a) { return __builtin_amdgcn_fractf(a); };
    auto run = [&](float x, float z, bool first) {
        const float x0 = turns(x), x1 = turns(2.0f * x), z0 = turns(z), z1 = turns(2.0f * z), z2 = turns(4.0f * z);
        float f0 = __builtin_amdgcn_cosf(x0), f1 = __builtin_amdgcn_sinf(x1), f2 = __builtin_amdgcn_cosf(x1);
        if (first) {  // features 0 .. 2
            f0 = L.g == 0 ? ux : f0;
            f1 = L.g == 0 ? uy : f1;
            f2 = L.g == 0 ? uz : f2;
        }
        return as_bf8(pack_bf16x2(f0, f1), pack_bf16x2(f2, __builtin_amdgcn_sinf(z0)),
                      pack_bf16x2(__builtin_amdgcn_cosf(z0), __builtin_amdgcn_sinf(z1)),
                      pack_bf16x2(__builtin_amdgcn_cosf(z1), __builtin_amdgcn_sinf(z2)));
    };
    GuideIn I;
    I.b[0] = run(L.x[0] * ux, L.z[0] * (L.g == 3 ? uy : ux), true);
    I.b[1] = run(L.x[1] * (L.g == 3 ? uz : uy), L.z[1] * (L.g < 2 ? uy : uz), false);
    const float x = L.t * uz, x0 = turns(x), x1 = turns(2.0f * x), x2 = turns(4.0f * x);
    float f[4] = {__builtin_amdgcn_cosf(x0), __builtin_amdgcn_sinf(x1), __builtin_amdgcn_cosf(x1),
                  __builtin_amdgcn_sinf(x2)};
    f[3] = L.g == 2 ? n.x : f[3];  // features 75 .. 77, then the padding
    f[0] = L.g == 3 ? n.y : f[0];
    f[1] = L.g == 3 ? n.z : f[1];
    f[2] = L.g == 3 ? 0.f : f[2];
    f[3] = L.g == 3 ? 0.f : f[3];
    const uint2 t = make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
    __builtin_memcpy(&I.t, &t, 8);
    return I;
}

// Y^T = W X^T for NT tiles of 16 samples: epi(mt, nt, acc).  w(mt, kt) and wt(mt)
// give the A fragments.
template <int KT32, bool TAIL, int OUT_TILES, int NT, class W, class WT, class Epi>
__device__ __forceinline__ void guide_layer(W w, WT wt, const g_bf8 (&b)[NT][2], const g_s4* bt, Epi epi) {
#pragma unroll
    for (int mt = 0; mt < OUT_TILES; ++mt) {
        g_bf8 a[KT32];
#pragma unroll
        for (int kt = 0; kt < KT32; ++kt) a[kt] = w(mt, kt);
        g_s4 at = {0, 0, 0, 0};
        if (TAIL) at = wt(mt);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            g_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < KT32; ++kt) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kt], b[nt][kt], acc, 0, 0, 0);
            if (TAIL) {  // the K = 16 tail accumulates separately: no mixed-shape accumulation chain
                g_f4 t = {0.f, 0.f, 0.f, 0.f};
                t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(at, bt[nt], t, 0, 0, 0);
                acc += t;
            }
            epi(mt, nt, acc);
        }
    }
}

// Bias, ReLU and BF16 of four outputs.
__device__ __forceinline__ uint2 guide_relu(float4 b, g_f4 v) {
    return make_uint2(pack_bf16x2(fmaxf(v[0] + b.x, 0.f), fmaxf(v[1] + b.y, 0.f)),
                      pack_bf16x2(fmaxf(v[2] + b.z, 0.f), fmaxf(v[3] + b.w, 0.f)));
}

// B operands of the next layer's K tile from the output tiles h0 (its first 16
// features) and h1: group g holds features 4 g .. +3 of both, and gets 8 g .. +7
// of the 32.  Groups 2, 3 of h0 against 0, 1 of h1, then odd groups of the one
// against even groups of the other.
__device__ __forceinline__ g_bf8 guide_operand(uint2 h0, uint2 h1) {
    const auto x = __builtin_amdgcn_permlane32_swap(h0.x, h1.x, false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(h0.y, h1.y, false, false);
    const auto u = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
    const auto v = __builtin_amdgcn_permlane16_swap(y[0], y[1], false, false);
    return as_bf8(u[0], v[0], u[1], v[1]);
}

// Weight fragments and biases of layer L (0 .. 3) from memory.
template <int L>
struct GuideMem {
    static constexpr int kW = L == 0 ? kGW1 : L == 1 ? kGW2 : L == 2 ? kGW3 : kGW4;
    static constexpr int kB = L == 0 ? kGOffB1 : L == 1 ? kGOffB2 : L == 2 ? kGOffB3 : kGOffB4;
    static constexpr int kTiles = L == 3 ? 3 : 4;
    static __device__ __forceinline__ g_bf8 w(const GuideView& G, int mt, int kt, uint32_t l) {
        return frag32<2, kTiles>(G.wbf + kW, mt, kt, l);
    }
    // padded outputs 40 .. 47 have no bias
    static __device__ __forceinline__ float4 bias(const GuideView& G, int o) {
        return *reinterpret_cast<const float4*>(G.theta + kB + (L == 3 && o >= kGOut ? 0 : o));
    }
};

// All weight fragments and biases in registers: 128 and 60 VGPRs, loaded once per
// wave and used for every tile it takes.
struct GuideRegs {
    g_bf8 a[4][4][2];
    g_s4 t[4];
    float4 b[4][4];
    template <int L>
    __device__ __forceinline__ void load(const GuideView& G, uint32_t l) {
#pragma unroll
        for (int mt = 0; mt < GuideMem<L>::kTiles; ++mt) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) a[L][mt][kt] = GuideMem<L>::w(G, mt, kt, l);
            b[L][mt] = GuideMem<L>::bias(G, 16 * mt + 4 * (int)(l >> 4));
        }
    }
    __device__ __forceinline__ explicit GuideRegs(const GuideView& G) {
        const uint32_t l = threadIdx.x & 63u;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) t[mt] = frag16<2, 4>(G.wbf + kGW1, mt, l);
        load<0>(G, l);
        load<1>(G, l);
        load<2>(G, l);
        load<3>(G, l);
    }
    template <int L>
    __device__ __forceinline__ g_bf8 w(int mt, int kt) const {
        return a[L][mt][kt];
    }
    __device__ __forceinline__ g_s4 wt(int mt) const { return t[mt]; }
    template <int L>
    __device__ __forceinline__ float4 bias(int mt) const {
        return b[L][mt];
    }
};

// The same, read layer by layer from memory (L2): for kernels that cannot spare
// the registers.
struct GuideLoads {
    const GuideView& G;
    uint32_t l;
    // The lane is opaque to the compiler, which otherwise keeps the addresses of all
    // fragments in registers across the shade kernel's loop.
    __device__ __forceinline__ explicit GuideLoads(const GuideView& g) : G(g), l(threadIdx.x & 63u) {
        asm volatile("" : "+v"(l));
    }
    template <int L>
    __device__ __forceinline__ g_bf8 w(int mt, int kt) const {
        return GuideMem<L>::w(G, mt, kt, l);
    }
    __device__ __forceinline__ g_s4 wt(int mt) const { return frag16<2, 4>(G.wbf + kGW1, mt, l); }
    template <int L>
    __device__ __forceinline__ float4 bias(int mt) const {
        return GuideMem<L>::bias(G, 16 * mt + 4 * (int)(l >> 4));
    }
};

// The network for NT tiles: out(nt, first output, four outputs) for outputs
// 0 .. 39 of the lane's sample.  Every forward evaluation of the guide (render,
// pdf, sampling, tn_guide_forward) runs this arithmetic, so a density the
// renderer sampled with is the density tn_guide_pdf reports.
template <int NT, class Net, class Out>
__device__ __forceinline__ void guide_network(const Net& N, const GuideIn (&in)[NT], Out out) {
    const int g = (int)(threadIdx.x & 63u) >> 4;
    g_bf8 b[NT][2];
    g_s4 bt[NT];
    uint2 h[NT][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        b[nt][0] = in[nt].b[0];
        b[nt][1] = in[nt].b[1];
        bt[nt] = in[nt].t;
    }
    auto operands = [&] {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            b[nt][0] = guide_operand(h[nt][0], h[nt][1]);
            b[nt][1] = guide_operand(h[nt][2], h[nt][3]);
        }
    };
    guide_layer<2, true, 4, NT>([&](int mt, int kt) { return N.template w<0>(mt, kt); }, [&](int mt) { return N.wt(mt); }, b,
                                bt, [&](int mt, int nt, g_f4 v) { h[nt][mt] = guide_relu(N.template bias<0>(mt), v); });
    operands();
    guide_layer<2, false, 4, NT>([&](int mt, int kt) { return N.template w<1>(mt, kt); }, [](int) { return g_s4{}; }, b, bt,
                                 [&](int mt, int nt, g_f4 v) { h[nt][mt] = guide_relu(N.template bias<1>(mt), v); });
    operands();
    guide_layer<2, false, 4, NT>([&](int mt, int kt) { return N.template w<2>(mt, kt); }, [](int) { return g_s4{}; }, b, bt,
                                 [&](int mt, int nt, g_f4 v) { h[nt][mt] = guide_relu(N.template bias<2>(mt), v); });
    operands();
    guide_layer<2, false, 3, NT>([&](int mt, int kt) { return N.template w<3>(mt, kt); }, [](int) { return g_s4{}; }, b, bt,
                                 [&](int mt, int nt, g_f4 v) {
                                     const int o = 16 * mt + 4 * g;
                                     if (o >= kGOut) return;  // padded rows 40 .. 47
                                     const float4 c = N.template bias<3>(mt);
                                     out(nt, o, make_float4(v[0] + c.x, v[1] + c.y, v[2] + c.z, v[3] + c.w));
                                 });
}

// Separates a wave's writes of its LDS rows from its reads of other lanes' rows:
// LDS serves a wave's accesses in order, so only the compiler has to keep them.
__device__ __forceinline__ void guide_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The network for a wave's 16 NT samples, lane l holding sample l % (16 NT): the 40
// outputs of sample k at out[k * 40 ..] (LDS).
template <int NT>
__device__ __forceinline__ void guide_forward_wave(const GuideView& G, float3 p, float3 n, bool active, float* out) {
    const int s = (int)(threadIdx.x & 15u);
    if (!active) p = n = make_float3(0.f, 0.f, 0.f);
    const GuideLoads net(G);
    const GuideLane L = guide_lane();
    GuideIn in[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int src = 16 * nt + s;
        float3 tp = p, tn = n;
        if (NT > 1) {
            tp = make_float3(__shfl(p.x, src, 64), __shfl(p.y, src, 64), __shfl(p.z, src, 64));
            tn = make_float3(__shfl(n.x, src, 64), __shfl(n.y, src, 64), __shfl(n.z, src, 64));
        }
        in[nt] = guide_features(G, L, tp, tn);
    }
    guide_network<NT>(net, in, [&](int nt, int o, float4 v) {
        *reinterpret_cast<float4*>(out + (16 * nt + s) * kGOut + o) = v;
    });
    guide_wave_sync();
}

}  // namespace tn

// Guide state behind tn_guide* (device buffers owned).
struct tn_guide {
    int device = 0;
    int cus = 256;  // compute units of the device
    float* theta = nullptr;   // FP32 master parameters
    float* adam_m = nullptr;  // Adam moments
    float* adam_v = nullptr;
    uint16_t* wbf = nullptr;  // BF16 operand copies
    float* partial = nullptr; // per-block gradient slices and sums
    uint32_t partial_blocks = 0;
    float* dloss = nullptr;   // [0] loss of the last batch, [1] its sum of weights
    float4* ts = nullptr;     // training set: 3 float4 per sample (p, c), (n, cos/pdf), (w, tag)
    uint32_t ts_cap = 0;
    uint32_t* ts_count = nullptr;
    // Deferred training (TN_RENDER_DEFER_TRAINING): the records of the last
    // render wait in ts (pending = its train_samples) and train during the
    // next render, on tstream, while that render samples from a snapshot of
    // the weights and records into the other set (ts_alt; the two swap).
    float4* ts_alt = nullptr;
    uint32_t ts_alt_cap = 0;
    uint32_t* ts_count_alt = nullptr;
    uint32_t pending = 0;
    uint16_t* wbf_snap = nullptr;
    float* theta_snap = nullptr;
    hipStream_t tstream = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    float bmin[3] = {0, 0, 0}, bmax[3] = {1, 1, 1};
    uint64_t seed = 1;
    uint32_t steps = 0;
    float lr = 1e-3f;
    uint32_t batch = 16384;
    float mis_guided = 0.5f;
    uint32_t epochs = 1;   // passes over each training pass's subset of samples
    uint32_t passes = 0;   // training passes so far
    uint32_t last_samples = 0;

    tn::GuideView view() const {
        tn::GuideView v;
        v.wbf = wbf;
        v.theta = theta;
        for (int k = 0; k < 3; ++k) {
            v.bmin[k] = bmin[k];
            const float ext = bmax[k] - bmin[k];
            v.inv_ext[k] = ext > 0 ? 1.0f / ext : 0.f;
        }
        return v;
    }
};

namespace tn {
// Grows the training set to hold `cap` samples and clears it.
int guide_reserve_set(tn_guide* g, uint32_t cap, hipStream_t stream);
// train_samples / batch Adam steps on mini-batches drawn uniformly (with
// replacement) from the training set.
int guide_train_from_set(tn_guide* g, uint32_t train_samples, hipStream_t stream);
// Trains the pending (deferred) set now, on stream.
int guide_train_pending(tn_guide* g, hipStream_t stream);
// Starts the pending set's training on the guide's stream after stream's
// current point, with a snapshot of the weights taken first on stream for
// the render to sample from; recording: the render's records go to the
// other set.  *started is false when nothing was pending.
int guide_defer_begin(tn_guide* g, hipStream_t stream, bool recording, bool* started);
}  // namespace tn
