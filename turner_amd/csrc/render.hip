// render.hip -- wavefront path tracer: the pixel loop of main.cpp:187-226 over
// trace() (pathtracer.cpp:14-102), unrolled into device queues.
//
// trace() computes  L = rho * (direct / pi + (1/m) sum_j 2 cos_j L_j)  with one
// point light (no 1/r^2, pathtracer.cpp:44-58), a uniform hemisphere per
// indirect sample (lib/sampling.h:20-32) and m samples per hit; levels
// 0..max_depth are traced and a miss returns the background.  Unrolled, a path
// segment at depth k carries the product W of the factors rho * 2 cos / m of
// its ancestors and adds W * (miss ? bg : rho * direct / pi) to its pixel.
// One chunk of primary samples is processed level by level:
//
//   raygen -> [trace -> shade -> shadow] x (max_depth + 1)
//
//   trace : closest hit for every queued segment (lane-refill traversal);
//   shade : miss / emission / next-event estimation (shadow queue) and m
//           children per hit (next queue), in slots that a block reserves for
//           all of its waves with one atomic (ballot + mbcnt prefix);
//   shadow: visibility of the shadow queue (reference predicate
//           !hit || r > dist, pathtracer.cpp:53); unoccluded contributions
//           are added to the pixel's FP32 accumulator.
//
// All counts live in device memory, so the per-chunk launch sequence needs no
// host synchronisation.  RNG: one xorshift128 (Marsaglia 2003) state per
// segment, seeded by splitmix64 from (seed, sample index) and split for the
// children.  The reference's single sequential xorshift64* stream
// (lib/sampling.h:12) cannot be reproduced by a parallel tracer; images agree
// with the reference estimator statistically.  With TN_RENDER_REF_JITTER the
// pixel jitter is the reference's exactly (xorshift64* seeded 42 per row,
// main.cpp:201-206), so primary rays are bit-identical.
//
// Guided rendering (tn_render_guided, no reference counterpart) swaps the
// hemisphere sampler in shade for one-sample MIS between the learned vMF
// mixture q and the cosine lobe: the wave runs the guide MLP on its 64 hits
// (BF16 MFMA, tn_guide.h), each child direction comes from q with
// probability a and from the cosine lobe otherwise, and carries the weight
// rho cos / (pi m (a q(w) + (1 - a) cos / pi)), so E[estimate] is unchanged.
// When training, every bounce of a path (m = 1) leaves a record (point,
// normal, direction, cos / pdf, rho f) and every segment the radiance it
// found itself (background, unoccluded next-event estimates); after the
// chunk, k_collect walks each path backwards, L_k = X_{k+1} + g_{k+1} L_{k+1},
// and appends (p, n, w, lum(L_k) cos / pdf) to the guide's training set.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

#include "tn_guide.h"
#include "tn_sample.h"
#include "tn_scene.h"

namespace tn {
namespace {

constexpr int kRBlock = 256;
// LDS short-stack entries per lane of the renderer's traversal kernels (16
// measured no faster on small or large launches than 8)
constexpr int kRStack = kStack;
constexpr uint32_t kMaxLevels = 64;
constexpr uint32_t kFixCap = 1u << 16;
constexpr uint32_t kFixHits = 4 * kMaxLevels + 2, kFixShadows = 5 * kMaxLevels + 2;
constexpr uint64_t kSceneSeedStep = 0x9E3779B97F4A7C15ull;
// scenes with at most this many emitter triangles pick one by solid angle
constexpr uint32_t kSolidAngleSelect = 4;
// concurrent render pipelines (queues + streams) that take alternate chunks;
// 3 and 4 measured slower than 2 (1920x1080: -7 %, -4 %)
constexpr int kPipes = 2;

struct Queues {
    float4* o[2];   // o.xyz, pixel (bits)
    float4* d[2];   // d.xyz, depth (bits)
    float4* w[2];   // throughput weight (RGBA)
    uint4* rng[2];  // xorshift128 state
    uint4* hit;     // id, r, s, t bits
    // shadow queues, two: level k uses [k & 1], so the shadow test of level
    // k can run (on a second stream) while level k + 1 is traced and shaded
    float4* so[2];  // shadow: origin, pixel (bits)
    float4* sd[2];  // shadow: direction, tmax
    float4* sc[2];  // shadow: contribution
    float4* sx[2];  // shadow: radiance at the segment (training records), slot (bits)
    uint32_t cap;   // capacity of each path queue (entries)
    uint32_t scap;  // capacity of the shadow queue
    // device counters: [0..4k) path and shadow counts (path_count,
    // shadow_count), [4k] overflow, [4k + 1] raycaster hits, [4k + 2..5k + 2)
    // segments and [5k + 2..6k + 2) shadow rays a refined traversal handed to
    // the reference tree (k = kMaxLevels)
    uint32_t* cnt;
    uint8_t* lit[2];  // what a level's shadow test found per queue entry (SettledChunks)
    // lists of those rays: [0] the segments of the level being traced,
    // [1 + (level & 1)] the shadow rays of a level; kFixCap entries each (a
    // list that overflows is replaced by a scan of the whole queue)
    uint32_t* fix;
    // chunk counters of the trace / shadow kernels: [kind][level][XCD], 16
    // words apart (one per 64-byte line)
    uint32_t* xwork;
    unsigned long long* totals;  // [0] segments, [1] shadow rays
    uint32_t* bar;  // grid barrier words of the persistent kernel (kBarWords)
};

// Per-scene parameters of a render: one entry per scene of a batch (one for
// a single-scene render).  Global sample j of the call belongs to the last
// scene whose sample_begin <= j; its pixel p to the last whose pixel_begin <= p.
struct SceneParams {
    float4 cam_pos;
    float cam_m[9];
    float cam_dx, cam_dy;
    uint32_t width, height, spp, nlights;
    float4 light_pos, light_col, bg;
    unsigned long long sample_begin;  // first global sample index
    uint32_t pixel_begin;             // first accumulator pixel
    uint32_t emit_begin, nemit;       // emitter range (emit_ids / emit_cdf)
    float emit_area;
};

// Chunk bounds kept on the device, so that one captured launch sequence
// serves every chunk: chunk_begin_block advances them.
struct ChunkState {
    unsigned long long next, total, first;
    unsigned long long stride;  // samples from one chunk of this pipeline to its next
    uint32_t chunk, count;
};

struct RenderArgs {
    SceneView sv;        // the tree the traversal kernels walk (refined tree of a TN_SCENE_REFINED scene)
    SceneView sv_exact;  // the reference tree behind a refined one (rays the refined traversal marks)
    bool refined;        // sv is a refined tree
    const float* normals;  // 9 per triangle
    const float4* albedo;
    const float4* emission;
    const float4* trirec;  // device triangle records (geometric normal in rec[1])
    const uint32_t* emit_ids;
    const float* emit_cdf;  // per scene: inclusive prefix of its emitters' areas
    const SceneParams* sp;
    uint32_t nscenes;
    ChunkState* cs;
    uint32_t* status;  // [2]: traversals abandoned as incomplete
    int32_t max_depth, mc;
    uint32_t flags;
    uint64_t seed;
    const float* jitter;  // 2 * width * spp (REF_JITTER, single scene) or null
    float4* accum;
    uint64_t seed_pass;  // seed of this call's sample range (sample_offset)
    // guided sampling
    GuideView gv;
    float mis;  // probability of drawing from the guide
    // training records, slot = path * rstride + level (null unless training)
    float4* rec_p;  // hit point, cos / pdf
    float4* rec_n;  // shading normal, valid (1) when the bounce spawned its child
    float4* rec_w;  // direction
    float4* rec_g;  // rho * f: the child's weight relative to its parent
    float4* rec_x;  // radiance found by the segment itself (its level), local units
    uint32_t rstride;
    float4* ts;  // guide training set (3 float4 per sample)
    uint32_t* ts_count;
    uint32_t ts_cap;
    float accept;  // probability that a record enters the training set
    // raycaster / raytracer
    float max_vis;    // raycaster max_visibility
    float shadow_si;  // raytracer shadow_intensity
    const float4* reflective;   // raytracer: reflective colour per triangle
    const float* reflectivity;  // raytracer: null = no reflection
};

__device__ __forceinline__ uint32_t scene_of_pixel(const RenderArgs& A, uint32_t pixel) {
    if (A.nscenes <= 1) return 0;
    uint32_t lo = 0, hi = A.nscenes - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (A.sp[mid].pixel_begin <= pixel) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ uint32_t scene_of_sample(const RenderArgs& A, unsigned long long j) {
    if (A.nscenes <= 1) return 0;
    uint32_t lo = 0, hi = A.nscenes - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (A.sp[mid].sample_begin <= j) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ uint4 rng_seed(uint64_t a, uint64_t b) {
    const uint64_t h1 = splitmix64(a ^ splitmix64(b));
    const uint64_t h2 = splitmix64(h1 + 0x632BE59BD9B4E019ull);
    uint4 s = make_uint4((uint32_t)h1, (uint32_t)(h1 >> 32), (uint32_t)h2, (uint32_t)(h2 >> 32));
    if ((s.x | s.y | s.z | s.w) == 0) s.x = 1;
    return s;
}

// xorshift128 (Marsaglia 2003)
__device__ __forceinline__ uint32_t rng_next(uint4& s) {
    uint32_t t = s.x ^ (s.x << 11);
    s.x = s.y;
    s.y = s.z;
    s.z = s.w;
    s.w = s.w ^ (s.w >> 19) ^ (t ^ (t >> 8));
    return s.w;
}
__device__ __forceinline__ float rng_uniform(uint4& s) { return (float)(rng_next(s) >> 8) * 0x1p-24f; }

// Stream of child c: two words of the parent's stream, high word first (named
// locals fix the order, which an expression with two calls would leave open).
__device__ __forceinline__ uint4 child_seed(uint4& parent, uint32_t c) {
    const uint64_t hi = rng_next(parent);
    const uint64_t lo = rng_next(parent);
    return rng_seed((hi << 32) | lo, c);
}

__device__ __forceinline__ float4 mul4(float4 a, float4 b) {
    return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}
__device__ __forceinline__ float4 scale4(float s, float4 a) {
    return make_float4(s * a.x, s * a.y, s * a.z, s * a.w);
}
__device__ __forceinline__ void accumulate(float4* acc, uint32_t pixel, float4 c) {
    float* p = reinterpret_cast<float*>(acc + pixel);
    if (c.x != 0.f) atomicAdd(p + 0, c.x);
    if (c.y != 0.f) atomicAdd(p + 1, c.y);
    if (c.z != 0.f) atomicAdd(p + 2, c.z);
    if (c.w != 0.f) atomicAdd(p + 3, c.w);
}

// Adds one contribution per lane (those with `on`) to the pixels, called by all
// lanes of the wave.  Queue neighbours often share a pixel (its samples, their
// children), and an atomic on memory costs far more than the wave's own
// additions: runs of lanes with the same pixel are summed by a segmented scan
// (six DPP steps) and the last lane of a run adds the sum.
__device__ __forceinline__ void accumulate_wave(float4* acc, uint32_t pixel, float4 c, bool on) {
    if (!__ballot(on)) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t key = on ? pixel : ~0u;  // no pixel: images hold fewer than 2^32 - 1 of them
    if (!on) c = make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t prev = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane - 1u) << 2, (int)key);
    const uint64_t heads = __ballot(lane == 0 || prev != key);
    bool last = true;
    if (heads != ~0ull) {
        const uint32_t start = 63u - (uint32_t)__clzll(heads & (~0ull >> (63u - lane)));  // first lane of the run
#define TN_RUN_STEP(ctrl, rows, bound, cond)                                                                    \
    {                                                                                                           \
        const bool take = cond;                                                                                 \
        auto add = [&](float& x) {                                                                              \
            const float y =                                                                                     \
                __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, rows, 0xf, bound));      \
            x += take ? y : 0.f;                                                                                \
        };                                                                                                      \
        add(c.x);                                                                                               \
        add(c.y);                                                                                               \
        add(c.z);                                                                                               \
        add(c.w);                                                                                               \
    }
        TN_RUN_STEP(0x111, 0xf, true, lane - start >= 1u)              // row_shr:1
        TN_RUN_STEP(0x112, 0xf, true, lane - start >= 2u)              // row_shr:2
        TN_RUN_STEP(0x114, 0xf, true, lane - start >= 4u)              // row_shr:4
        TN_RUN_STEP(0x118, 0xf, true, lane - start >= 8u)              // row_shr:8
        TN_RUN_STEP(0x142, 0xa, false, (lane & 16u) && start < (lane & ~15u))  // row_bcast:15 into rows 1, 3
        TN_RUN_STEP(0x143, 0xc, false, lane >= 32u && start <= 31u)    // row_bcast:31 into rows 2, 3
#undef TN_RUN_STEP
        last = lane == 63u || ((heads >> (lane + 1u)) & 1ull);
    }
    if (last && key != ~0u) accumulate(acc, key, c);
}

// Paths queued at a level and shadow rays queued by shading it.  What shading
// level k pushes -- paths of level k + 1 and shadow rays of level k -- is
// counted in the two halves of one 64-bit word, so one atomic reserves both.
__host__ __device__ __forceinline__ uint32_t path_count(int level) { return 2u * (uint32_t)level; }
__host__ __device__ __forceinline__ uint32_t shadow_count(int level) { return 2u * (uint32_t)level + 3u; }

// Queue slots of one block iteration of the shade kernels.  The counters of a
// level are one address that every XCD's L2 takes in turn; an atomic per wave
// and queue bound the shade kernels (about 10 ns each: 819,200 segments of the
// Cornell box took 181 us at level 0), so a block reserves for all of its
// waves at once: 54 us; 1080p m 4 pass 134.7 -> 121.2 ms, raytracer
// 961x541x4 2.06 -> 1.82 ms, a batch of six small scenes 1.17 -> 0.96 ms,
// 512^2 one-sample pass 2.22 -> 2.07 ms; guided 512^2x8 4.52 -> 4.37 ms
// (a wave per block as before, on the packed word: 4.86).  Called by all
// threads of the block; the two sets of words alternate by `turn`, so that a
// wave may run ahead into the next iteration's counts.
struct BlockSlots {
    uint32_t n[2][2][kRBlock / 64];  // [turn][paths, shadow rays][wave]
    unsigned long long base[2];
};
__device__ __forceinline__ void reserve_slots(BlockSlots& S, uint32_t turn, uint32_t* cnt, int level, uint32_t paths,
                                              uint32_t shadows, uint32_t& pbase, uint32_t& sbase) {
    const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    if ((threadIdx.x & 63u) == 0) {
        S.n[turn][0][wave] = paths;
        S.n[turn][1][wave] = shadows;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t p = 0, q = 0;
        for (uint32_t w = 0; w < waves; ++w) {
            p += S.n[turn][0][w];
            q += S.n[turn][1][w];
        }
        S.base[turn] = (p | q) ? atomicAdd(reinterpret_cast<unsigned long long*>(cnt + path_count(level + 1)),
                                           (unsigned long long)q << 32 | p)
                               : 0ull;
    }
    __syncthreads();
    pbase = (uint32_t)S.base[turn];
    sbase = (uint32_t)(S.base[turn] >> 32);
    for (uint32_t w = 0; w < wave; ++w) {
        pbase += S.n[turn][0][w];
        sbase += S.n[turn][1][w];
    }
}

// Words of the persistent kernel's grid barrier (grid_sync).
constexpr uint32_t kBarGen = 0, kBarOut = 32, kBarGroups = 64, kBarGroup = 96;
constexpr uint32_t kBarWords = kBarGroup + 32 * kXcds;

// Starts the pipeline's next chunk (one block of any size): its bounds, and its
// counters zeroed but for the overflow word, which lives for the whole render.
__device__ __forceinline__ void chunk_begin_block(uint32_t* cnt, uint32_t* xwork, ChunkState* cs) {
    const unsigned long long first = cs->next;
    const unsigned long long left = cs->total > first ? cs->total - first : 0ull;
    const uint32_t count = (uint32_t)(left < cs->chunk ? left : cs->chunk);
    for (uint32_t i = threadIdx.x; i < 6 * kMaxLevels + 2; i += blockDim.x)
        if (i != 4 * kMaxLevels) cnt[i] = (i == 0) ? count : 0u;
    for (uint32_t k = threadIdx.x; k < 2 * kMaxLevels * kXcds; k += blockDim.x) xwork[16 * k] = 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
        cs->first = first;
        cs->count = count;
        cs->next = first + cs->stride;
    }
}

// What a render reports, in pinned host memory (or, where there is none, in the
// pipeline's own memory, copied back at the end): each pipeline writes its own
// after every chunk, so that the call ends with a stream synchronisation alone.
struct RenderReport {
    unsigned long long rays, shadow_rays;
    uint32_t overflow, incomplete, barrier_out;
};

// One wave.  Adds a chunk's rays to the pipeline's totals.  levels < 0: the
// raycaster, whose rays are its hits (cnt[4 kMaxLevels + 1]).
__device__ __forceinline__ void chunk_totals(const uint32_t* cnt, unsigned long long* totals, int levels) {
    static_assert(kMaxLevels <= 64, "a lane per level");
    const int k = (int)(threadIdx.x & 63u);
    unsigned long long a = k < levels ? cnt[path_count(k)] : 0u, b = k < levels ? cnt[shadow_count(k)] : 0u;
    if (k == 0 && levels < 0) a = cnt[4 * kMaxLevels + 1];
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
    }
    if (k == 0) {
        totals[0] += a;
        totals[1] += b;
    }
}

// One thread.  `incomplete` counts both pipelines' abandoned traversals.
__device__ __forceinline__ void write_report(const Queues& Q, const uint32_t* incomplete, bool barriers,
                                             RenderReport* out) {
    out->rays = Q.totals[0];
    out->shadow_rays = Q.totals[1];
    out->overflow = Q.cnt[4 * kMaxLevels];
    out->incomplete = *incomplete;
    out->barrier_out = barriers ? Q.bar[kBarOut] : 0u;
}

// End of a chunk: its counts are added up and reported, then the next begins.
__global__ __launch_bounds__(512) void k_chunk_end(Queues Q, ChunkState* cs, const uint32_t* incomplete, int levels,
                                                   RenderReport* out) {
    if (threadIdx.x < 64) chunk_totals(Q.cnt, Q.totals, levels);
    if (threadIdx.x == 0) write_report(Q, incomplete, false, out);
    __syncthreads();
    chunk_begin_block(Q.cnt, Q.xwork, cs);
}

__global__ void k_persist_end(Queues Q, const uint32_t* incomplete, RenderReport* out) {
    if (threadIdx.x == 0) write_report(Q, incomplete, true, out);
}

// Primary samples: within a scene, j = (y * width + x) * spp + i
// (main.cpp:193-215 order); scenes follow each other in the sample space.
__device__ __forceinline__ void raygen_one(const RenderArgs& A, const Queues& Q, uint32_t i) {
    const unsigned long long j = A.cs->first + i;
    const uint32_t si = scene_of_sample(A, j);
    const SceneParams& S = A.sp[si];
    const unsigned long long local = j - S.sample_begin;
    const uint32_t sample = (uint32_t)(local % S.spp);
    const uint64_t pix = local / S.spp;
    const uint32_t x = (uint32_t)(pix % S.width), y = (uint32_t)(pix / S.width);
    // scene s of a batch draws the streams of a single render seeded seed + s * kSceneSeedStep
    uint4 rng = rng_seed(A.seed_pass + si * kSceneSeedStep, local);
    float dx, dy;
    if (A.jitter) {
        const size_t k = 2 * ((size_t)x * S.spp + sample);
        dx = A.jitter[k];
        dy = A.jitter[k + 1];
    } else {
        dx = rng_uniform(rng);
        dy = rng_uniform(rng);
    }
    // lib/types.h:119-123
    const float px = (float)x + dx, py = (float)y + dy;
    const float w = (float)S.width, h = (float)S.height;
    const float cx = -S.cam_dx * (1 - 2 * px / w);
    const float cy = S.cam_dy * (1 - 2 * py / h);
    const float cz = -1;
    const float* m = S.cam_m;
    const float3 d = make_float3(m[0] * cx + m[1] * cy + m[2] * cz, m[3] * cx + m[4] * cy + m[5] * cz,
                                 m[6] * cx + m[7] * cy + m[8] * cz);
    Q.o[0][i] = make_float4(S.cam_pos.x, S.cam_pos.y, S.cam_pos.z, __uint_as_float(S.pixel_begin + (uint32_t)pix));
    Q.d[0][i] = make_float4(d.x, d.y, d.z, __uint_as_float(i));  // .w: path within the chunk
    Q.w[0][i] = make_float4(1.f, 1.f, 1.f, 1.f);
    Q.rng[0][i] = rng;
}

__global__ __launch_bounds__(kRBlock) void k_raygen(RenderArgs A, Queues Q) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.cs->count) return;
    raygen_one(A, Q, i);
}

// Caller rays (tn_trace): ray j accumulates into accum[j]; seeds from (seed, j).
__global__ __launch_bounds__(kRBlock) void k_raygen_rays(RenderArgs A, Queues Q, const float* o3,
                                                         const float* d3) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.cs->count) return;
    const uint64_t j = A.cs->first + i;
    Q.o[0][i] = make_float4(o3[3 * j], o3[3 * j + 1], o3[3 * j + 2], __uint_as_float((uint32_t)j));
    Q.d[0][i] = make_float4(d3[3 * j], d3[3 * j + 1], d3[3 * j + 2], __uint_as_float(i));
    Q.w[0][i] = make_float4(1.f, 1.f, 1.f, 1.f);
    Q.rng[0][i] = rng_seed(A.seed_pass, j);
}

// coop_loop's `whole`.
__device__ __forceinline__ bool a_ray_per_lane(uint32_t n) { return n <= gridDim.x * blockDim.x; }

// Per-wave chunks of a device-counted queue.  The chunk shrinks with the
// queue (a sixteenth of a wave's share, at least 64; queues of less than 64
// paths for every fourth wave by small_share: a shadow launch and the other
// pipeline usually share the chip) to keep every wave busy on short queues.
// Guided 512x512x8 / raytracer 961x541x4 / one-sample 512^2 pass: 4.60 / 2.26 /
// 2.24 ms with 64 at least, 4.67 / 2.04 / 2.23 for every second wave, 4.20 /
// 2.04 / 2.21 for every fourth, 4.54 / 2.06 / 2.25 for every eighth.  A queue of at
// most one chunk per wave is dealt statically (wave w takes chunk w) with no
// atomics: every wave hitting one device-wide counter at once serialises,
// and on 1-spp passes (262 k paths) dropping those atomics made a pass 21 %
// faster.  Longer queues hand out chunks by atomic counters, one per XCD
// (blocks are dealt to the XCDs round-robin): XCD x takes chunks x, x + 8,
// x + 16, ... so neighbouring chunks still spread over the XCDs.  (A static
// first chunk per wave measured 5 % slower on long queues.)
struct DynamicChunks {
    uint32_t n;
    uint32_t* xw;  // this queue's eight counters, 16 words apart
    uint32_t size, nchunks, nwaves, wave;
    bool first;
    __device__ DynamicChunks(uint32_t n_, uint32_t* xw_) : n(n_), xw(xw_), first(true) {
        nwaves = (gridDim.x * blockDim.x) >> 6;
        wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
        uint32_t c = (uint32_t)(((uint64_t)n + 16ull * nwaves - 1) / (16ull * nwaves));
        c = (c + 63u) & ~63u;
        size = c <= 64u ? small_share(n, max(nwaves / 4u, 1u), nwaves) : (c > (uint32_t)kChunk ? (uint32_t)kChunk : c);
        nchunks = (n + size - 1) / size;
    }
    __device__ bool operator()(uint32_t& b, uint32_t& e) {
        uint32_t idx;
        if (nchunks <= nwaves) {
            if (!first) return false;
            first = false;
            idx = wave;
        } else {
            const uint32_t groups = gridDim.x >= kXcds ? kXcds : 1u;  // every group has waves
            const uint32_t x = blockIdx.x % groups;
            uint32_t k = 0;
            if ((threadIdx.x & 63u) == 0) k = atomicAdd(xw + 16 * x, 1u);
            idx = x + groups * __shfl(k, 0, 64);
        }
        if (idx >= nchunks) return false;
        b = idx * size;
        e = min(b + size, n);
        return true;
    }
};

// An unoccluded shadow ray's radiance goes to the segment's record (training).
__device__ __forceinline__ void record_lit(const RenderArgs& A, const Queues& Q, int sb, uint32_t k) {
    if (!A.rec_x) return;
    const float4 x = Q.sx[sb][k];
    float* dst = reinterpret_cast<float*>(A.rec_x + __float_as_uint(x.w));
    atomicAdd(dst + 0, x.x);
    atomicAdd(dst + 1, x.y);
    atomicAdd(dst + 2, x.z);
}

// An unoccluded shadow ray: its contribution goes to the pixel (and, when
// training, its radiance to the segment's record).
__device__ __forceinline__ void shadow_lit(const RenderArgs& A, const Queues& Q, int sb, uint32_t k) {
    accumulate(A.accum, __float_as_uint(Q.so[sb][k].w), Q.sc[sb][k]);
    record_lit(A, Q, sb, k);
}

// The chunks of the shadow queue a wave has taken.  Rays finish in any order,
// so what the test found is only noted per entry (Q.lit), and when the wave has
// no rays left it goes through its chunks in queue order, where neighbours share
// pixels (accumulate_wave): the atomics of the shadow test fall by the length
// of the runs.  With accumulate_wave in the shade kernels too: Cornell box, 8
// samples per pixel, 1.32 -> 0.96 ms (level 0's shadow test 330 -> 187 us, level
// 1's shade 212 -> 79 us); 1080p m 4 pass 121.0 -> 100.8 ms; raytracer
// 961x541x4 1.82 -> 1.49 ms; one sample per pixel, no runs: 2.07 -> 2.09 ms.
// A wave that takes more than 64 chunks adds the rays that
// finish from then on directly.
struct SettledChunks {
    DynamicChunks from;
    uint32_t begins = 0, count = 0;  // begins: lane i holds the start of chunk i
    bool direct = false;
    __device__ SettledChunks(uint32_t n, uint32_t* xw) : from(n, xw) {}
    __device__ bool operator()(uint32_t& b, uint32_t& e) {
        if (!from(b, e)) return false;
        if (count < 64u) {
            if ((threadIdx.x & 63u) == count) begins = b;
            ++count;
        } else {
            direct = true;
        }
        return true;
    }
    // visit(k, in) by all lanes for every entry of the chunks, 64 at a time
    template <class Visit>
    __device__ void settle(Visit visit) {
        // the notes of this wave's other lanes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        for (uint32_t i = 0; i < count; ++i) {
            const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)begins, (int)i), e = min(b + from.size, from.n);
            for (uint32_t k = b; k < e; k += 64u) {
                const uint32_t mine = k + (threadIdx.x & 63u);
                visit(mine, mine < e);
            }
        }
    }
};

// REF: the refined tree of a TN_SCENE_REFINED scene; rays tied at their
// closest distance and rays with a zero direction component get the hit
// record kFixId, which k_fix_hits replaces before anything reads it, and go
// on the level's fix list.
template <bool EXH, bool REF>
__device__ __forceinline__ void trace_body(const RenderArgs& A, const Queues& Q, int level, int buf, uint2* stk,
                                           CoopLds* wl) {
    const uint32_t n = min(Q.cnt[path_count(level)], Q.cap);  // overflow is reported, never read
    const float4* qo = Q.o[buf];
    const float4* qd = Q.d[buf];
    uint4* hit = Q.hit;
    TraversalCounters cnt;
    coop_loop<kRStack, EXH, false, false, false, REF>(
        A.sv, stk + threadIdx.x, kRBlock, wl + threadIdx.x / 64, !REF && a_ray_per_lane(n),
        DynamicChunks{n, Q.xwork + 16 * kXcds * level},
        [&](uint32_t k, float3& o, float3& d, float&, uint32_t& scene) {
            const float4 a = qo[k], b = qd[k];
            o = make_float3(a.x, a.y, a.z);
            d = make_float3(b.x, b.y, b.z);
            scene = scene_of_pixel(A, __float_as_uint(a.w));
        },
        [&](uint32_t k, const CoopHit& T) {
            if (REF && (T.tie || needs_reference(T.d))) {
                hit[k] = make_uint4(kFixId, 0u, 0u, 0u);
                const uint32_t slot = atomicAdd(Q.cnt + kFixHits + level, 1u);
                if (slot < kFixCap) Q.fix[slot] = k;
                return;
            }
            hit[k] = make_uint4(T.id, __float_as_uint(T.r), __float_as_uint(T.s), __float_as_uint(T.t));
        },
        cnt);
    if (cnt.incomplete) atomicAdd(A.status + 2, 1u);
}

template <bool EXH, bool REF>
__global__ __launch_bounds__(kRBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_trace(
    RenderArgs A, Queues Q, int level, int buf) {
    __shared__ uint2 stk[kRStack * kRBlock];
    __shared__ CoopLds wl[kRBlock / 64];
    trace_body<EXH, REF>(A, Q, level, buf, stk, wl);
}

// The segments of one level that k_trace<..., true> marked, traced one per
// lane on the reference tree (the reference's leaves and order decide them):
// the entries of the fix list, or every marked entry of the queue when the
// list overflowed.
template <bool EXH>
__global__ __launch_bounds__(kRBlock) void k_fix_hits(RenderArgs A, Queues Q, int level, int buf) {
    __shared__ uint2 stk[kRStack * kRBlock];
    const uint32_t m = Q.cnt[kFixHits + level];
    if (m == 0) return;
    const bool scan = m > kFixCap;
    const uint32_t n = scan ? min(Q.cnt[path_count(level)], Q.cap) : m;
    TraversalCounters cnt;
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t i = scan ? j : Q.fix[j];
        if (scan && Q.hit[i].x != kFixId) continue;
        const float4 a = Q.o[buf][i], b = Q.d[buf][i];
        float r = FLT_MAX, s = 0.f, t = 0.f;
        const uint32_t id = traverse<kRStack, EXH, false, false, false>(
            A.sv_exact, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), 0.f, r, s, t, stk + threadIdx.x,
            kRBlock, cnt);
        const bool h = id != kInvalidId;
        Q.hit[i] = make_uint4(h ? id : kInvalidId, __float_as_uint(h ? r : FLT_MAX), __float_as_uint(h ? s : 0.f),
                              __float_as_uint(h ? t : 0.f));
    }
    if (cnt.incomplete) atomicAdd(A.status + 2, 1u);
}

// Shadow rays (any hit up to tmax).  REF: the refined tree; a ray with a zero
// direction component is marked (lit 2) and listed for k_fix_shadows.
template <bool EXH, bool REF>
__device__ __forceinline__ void shadow_body(const RenderArgs& A, const Queues& Q, int level, uint2* stk,
                                            CoopLds* wl) {
    const uint32_t n = min(Q.cnt[shadow_count(level)], Q.scap);
    const int sb = level & 1;
    TraversalCounters cnt;
    SettledChunks chunks(n, Q.xwork + 16 * kXcds * (kMaxLevels + level));
    coop_loop<kRStack, EXH, false, true, false>(
        A.sv, stk + threadIdx.x, kRBlock, wl + threadIdx.x / 64, !REF && a_ray_per_lane(n),
        [&](uint32_t& b, uint32_t& e) { return chunks(b, e); },
        [&](uint32_t k, float3& o, float3& d, float& tmax, uint32_t& scene) {
            const float4 a = Q.so[sb][k], b = Q.sd[sb][k];
            o = make_float3(a.x, a.y, a.z);
            d = make_float3(b.x, b.y, b.z);
            tmax = b.w;
            scene = scene_of_pixel(A, __float_as_uint(a.w));
        },
        [&](uint32_t k, const CoopHit& T) {
            uint8_t lit = T.id == kInvalidId ? 1 : 0;
            if (REF && needs_reference(T.d)) {
                lit = 2;
                const uint32_t slot = atomicAdd(Q.cnt + kFixShadows + level, 1u);
                if (slot < kFixCap) Q.fix[(1 + sb) * kFixCap + slot] = k;
            } else if (chunks.direct && lit) {
                shadow_lit(A, Q, sb, k);
                lit = 0;
            }
            Q.lit[sb][k] = lit;
        },
        cnt);
    chunks.settle([&](uint32_t k, bool in) {
        const bool lit = in && Q.lit[sb][k] == 1;
        uint32_t pixel = 0;
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        if (lit) {
            pixel = __float_as_uint(Q.so[sb][k].w);
            c = Q.sc[sb][k];
            record_lit(A, Q, sb, k);
        }
        accumulate_wave(A.accum, pixel, c, lit);
    });
    if (cnt.incomplete) atomicAdd(A.status + 2, 1u);
}

template <bool EXH, bool REF>
__global__ __launch_bounds__(kRBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_shadow(
    RenderArgs A, Queues Q, int level) {
    __shared__ uint2 stk[kRStack * kRBlock];
    __shared__ CoopLds wl[kRBlock / 64];
    shadow_body<EXH, REF>(A, Q, level, stk, wl);
}

// The shadow rays of one level that k_shadow<..., true> marked, tested one
// per lane on the reference tree: the fix list's entries, or every marked
// entry of the queue when the list overflowed.
template <bool EXH>
__global__ __launch_bounds__(kRBlock) void k_fix_shadows(RenderArgs A, Queues Q, int level) {
    __shared__ uint2 stk[kRStack * kRBlock];
    const uint32_t m = Q.cnt[kFixShadows + level];
    if (m == 0) return;
    const bool scan = m > kFixCap;
    const int sb = level & 1;
    const uint32_t n = scan ? min(Q.cnt[shadow_count(level)], Q.scap) : m;
    TraversalCounters cnt;
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const uint32_t i = scan ? j : Q.fix[(1 + sb) * kFixCap + j];
        if (scan && Q.lit[sb][i] != 2) continue;
        const float4 a = Q.so[sb][i], b = Q.sd[sb][i];
        float r = FLT_MAX, s = 0.f, t = 0.f;
        const uint32_t id = traverse<kRStack, EXH, false, true, false>(
            A.sv_exact, make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), b.w, r, s, t, stk + threadIdx.x,
            kRBlock, cnt);
        if (id == kInvalidId) shadow_lit(A, Q, sb, i);
    }
    if (cnt.incomplete) atomicAdd(A.status + 2, 1u);
}

// Orthonormal basis around n (Duff et al. 2017, "Building an Orthonormal
// Basis, Revisited").
__device__ __forceinline__ void onb(float3 n, float3& b1, float3& b2) {
    const float sign = copysignf(1.0f, n.z);
    const float a = -1.0f / (sign + n.z);
    const float b = n.x * n.y * a;
    b1 = make_float3(1.0f + sign * n.x * n.x * a, sign * b, -sign * n.x);
    b2 = make_float3(b, sign + n.y * n.y * a, -n.y);
}

__device__ __forceinline__ void push_shadow(const Queues& Q, int sb, uint32_t k, float3 o, uint32_t pixel,
                                            float3 dir, float tmax, float4 contrib, float4 local, uint32_t slot,
                                            bool records) {
    Q.so[sb][k] = make_float4(o.x, o.y, o.z, __uint_as_float(pixel));
    Q.sd[sb][k] = make_float4(dir.x, dir.y, dir.z, tmax);
    Q.sc[sb][k] = contrib;
    if (records) Q.sx[sb][k] = make_float4(local.x, local.y, local.z, __uint_as_float(slot));
}

// ------------------------------------------------ raycaster and raytracer
// The reference's other two trace() plugins on the same queues and traversal.

// Raycaster shade (raycaster.cpp:7-24), level 0 only: a miss gives the
// background; a hit the triangle's diffuse colour with alpha
// clamp(1 - r / max_visibility, 0, 1).  Hits are counted in cnt[4 kMaxLevels + 1]
// (the reference counts num_rays on hits only).
__global__ __launch_bounds__(kRBlock) void k_cast(RenderArgs A, Queues Q, int level, int buf) {
    const uint32_t n = min(Q.cnt[path_count(level)], Q.cap);
    uint32_t hits = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        uint32_t pixel = 0;
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n) {
            pixel = __float_as_uint(Q.o[buf][i].w);
            const uint4 h = Q.hit[i];
            if (h.x == kInvalidId) {
                c = A.sp[scene_of_pixel(A, pixel)].bg;
            } else {
                ++hits;
                c = A.albedo[h.x];
                const float a = 1.f - __uint_as_float(h.y) / A.max_vis;
                c.w = a < 0.f ? 0.f : (a > 1.f ? 1.f : a);  // clamp of src/turner.h:28-36
            }
            c = mul4(Q.w[buf][i], c);
        }
        accumulate_wave(A.accum, pixel, c, i < n);
    }
    for (int off = 32; off > 0; off >>= 1) hits += __shfl_xor(hits, off, 64);
    if ((threadIdx.x & 63u) == 0 && hits) atomicAdd(Q.cnt + 4 * kMaxLevels + 1, hits);
}

// Raytracer shade (raytracer.cpp:6-67) of one level.  A segment carries the
// product W of the factors reflectivity * reflective (and shadow darkening)
// of its ancestors.  A hit contributes W * colour, colour = Lambert
// max(0, L.n) diffuse light (lib/lambertian.h:15-19), times (1 - reflectivity)
// when it reflects, and spawns the mirror ray d - 2 (n.d) n from p2 with
// weight W * reflectivity * reflective.  The contribution waits in the shadow
// queue with the child's index: k_rt_shadow darkens both by the shadow
// intensity when the light is blocked (raytracer.cpp:57-64).  Children beyond
// max_depth are counted (the reference counts the call that returns {})
// but not queued.
__global__ __launch_bounds__(kRBlock) void k_rt_shade(RenderArgs A, Queues Q, int level, int buf) {
    const uint32_t n = min(Q.cnt[path_count(level)], Q.cap);
    __shared__ BlockSlots slots;
    const int ob = buf ^ 1;
    uint32_t turn = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x, turn ^= 1u) {
        const uint32_t i = base + threadIdx.x;
        bool spawn = false, shadow = false;
        float3 p2 = make_float3(0, 0, 0), rdir = p2, sdir = p2;
        float sdist = 0.f;
        float4 contrib = make_float4(0, 0, 0, 0), cw = contrib;
        uint32_t pixel = 0;
        float pathbits = 0.f;
        if (i < n) {
            const float4 qo = Q.o[buf][i], qd = Q.d[buf][i];
            const float4 w = Q.w[buf][i];
            pixel = __float_as_uint(qo.w);
            pathbits = qd.w;
            const SceneParams& S = A.sp[scene_of_pixel(A, pixel)];
            const uint4 h = Q.hit[i];
            if (h.x == kInvalidId) {
                contrib = mul4(w, S.bg);  // raytracer.cpp:19-21
            } else {
                const uint32_t id = h.x;
                const float r = __uint_as_float(h.y), s = __uint_as_float(h.z), t = __uint_as_float(h.w);
                const float3 p = make_float3(qo.x + r * qd.x, qo.y + r * qd.y, qo.z + r * qd.z);
                // raytracer.cpp:24-26: light direction from p
                const float3 l = make_float3(S.light_pos.x - p.x, S.light_pos.y - p.y, S.light_pos.z - p.z);
                const float il = 1.0f / sqrtf(l.x * l.x + l.y * l.y + l.z * l.z);
                const float3 ld = make_float3(il * l.x, il * l.y, il * l.z);
                // raytracer.cpp:29-30 (lib/triangle.h:54-56)
                const float* nv = A.normals + 9 * (size_t)id;
                const float b0 = 1.f - s - t;
                const float3 ni = make_float3(b0 * nv[0] + s * nv[3] + t * nv[6], b0 * nv[1] + s * nv[4] + t * nv[7],
                                              b0 * nv[2] + s * nv[5] + t * nv[8]);
                const float inv = 1.0f / sqrtf(ni.x * ni.x + ni.y * ni.y + ni.z * ni.z);
                const float3 nn = make_float3(inv * ni.x, inv * ni.y, inv * ni.z);
                // raytracer.cpp:33-34
                const float cosa = fmaxf(0.f, ld.x * nn.x + ld.y * nn.y + ld.z * nn.z);
                const float4 direct = mul4(scale4(cosa, A.albedo[id]), S.light_col);
                // raytracer.cpp:37
                p2 = make_float3(p.x + nn.x * 0.0001f, p.y + nn.y * 0.0001f, p.z + nn.z * 0.0001f);
                float4 color = direct;
                const float refl = A.reflectivity ? A.reflectivity[id] : 0.f;
                if (refl > 0) {  // raytracer.cpp:42-52
                    const float dn = 2.f * (nn.x * qd.x + nn.y * qd.y + nn.z * qd.z);
                    rdir = make_float3(qd.x - dn * nn.x, qd.y - dn * nn.y, qd.z - dn * nn.z);
                    color = scale4(1.f - refl, direct);
                    cw = mul4(w, scale4(refl, A.reflective[id]));
                    spawn = true;
                }
                contrib = mul4(w, color);
                // raytracer.cpp:55-60: shadow ray from p2 toward the light
                const float3 l2 = make_float3(S.light_pos.x - p2.x, S.light_pos.y - p2.y, S.light_pos.z - p2.z);
                sdist = sqrtf(l2.x * l2.x + l2.y * l2.y + l2.z * l2.z);
                const float il2 = 1.0f / sdist;
                sdir = make_float3(il2 * l2.x, il2 * l2.y, il2 * l2.z);
                shadow = sdist > 0.f;
            }
        }
        // children (mirror rays) and shadow rays
        const uint64_t mc = __ballot(spawn), ms = __ballot(shadow);
        uint32_t cbase, sbase;
        reserve_slots(slots, turn, Q.cnt, level, (uint32_t)__popcll(mc), (uint32_t)__popcll(ms), cbase, sbase);
        uint32_t child = ~0u;
        if (spawn && level < A.max_depth) {
            const uint32_t k = cbase + lanes_below(mc);
            if (k < Q.cap) {
                Q.o[ob][k] = make_float4(p2.x, p2.y, p2.z, __uint_as_float(pixel));
                Q.d[ob][k] = make_float4(rdir.x, rdir.y, rdir.z, pathbits);
                Q.w[ob][k] = cw;
                child = k;
            } else {
                atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
            }
        }
        // misses, and hits whose light sits at p2 itself (lit), are final
        accumulate_wave(A.accum, pixel, contrib, i < n && !shadow);
        if (shadow) {
            const uint32_t k = sbase + lanes_below(ms);
            if (k < Q.scap) {
                // shadowed iff the closest hit is nearer than the light
                // (strict): any hit with r <= the float below sdist
                const float tmax = __uint_as_float(__float_as_uint(sdist) - 1u);
                const int sb = level & 1;
                Q.so[sb][k] = make_float4(p2.x, p2.y, p2.z, __uint_as_float(pixel));
                Q.sd[sb][k] = make_float4(sdir.x, sdir.y, sdir.z, tmax);
                Q.sc[sb][k] = contrib;
                Q.sx[sb][k] = make_float4(__uint_as_float(child), 0.f, 0.f, 0.f);
            } else {
                atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
            }
        }
    }
}

// Raytracer shadow test (raytracer.cpp:55-64): a blocked light darkens the
// segment's colour, and so the weight of its mirror child, by
// c -= c * shadow_intensity.
template <bool EXH>
__global__ __launch_bounds__(kRBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_rt_shadow(
    RenderArgs A, Queues Q, int level, int buf) {
    __shared__ uint2 stk[kRStack * kRBlock];
    __shared__ CoopLds wl[kRBlock / 64];
    const uint32_t n = min(Q.cnt[shadow_count(level)], Q.scap);
    const int ob = buf ^ 1;
    const int sb = level & 1;
    TraversalCounters cnt;
    // the raytracer's shadow test darkens the mirror child too: it runs on the
    // reference tree itself (no marks to resolve afterwards)
    const SceneView& sv = A.refined ? A.sv_exact : A.sv;
    const float si = A.shadow_si;
    auto darken = [&](float4 c) { return make_float4(c.x - c.x * si, c.y - c.y * si, c.z - c.z * si, c.w - c.w * si); };
    SettledChunks chunks(n, Q.xwork + 16 * kXcds * (kMaxLevels + level));
    coop_loop<kRStack, EXH, false, true, false>(
        sv, stk + threadIdx.x, kRBlock, wl + threadIdx.x / 64, a_ray_per_lane(n),
        [&](uint32_t& b, uint32_t& e) { return chunks(b, e); },
        [&](uint32_t k, float3& o, float3& d, float& tmax, uint32_t& scene) {
            const float4 a = Q.so[sb][k], b = Q.sd[sb][k];
            o = make_float3(a.x, a.y, a.z);
            d = make_float3(b.x, b.y, b.z);
            tmax = b.w;
            scene = scene_of_pixel(A, __float_as_uint(a.w));
        },
        [&](uint32_t k, const CoopHit& T) {
            uint8_t lit = T.id == kInvalidId ? 1 : 0;
            if (!lit) {
                const uint32_t child = __float_as_uint(Q.sx[sb][k].x);
                if (child != ~0u) Q.w[ob][child] = darken(Q.w[ob][child]);
            }
            if (chunks.direct) {
                const float4 c = Q.sc[sb][k];
                accumulate(A.accum, __float_as_uint(Q.so[sb][k].w), lit ? c : darken(c));
                lit = 2;
            }
            Q.lit[sb][k] = lit;
        },
        cnt);
    chunks.settle([&](uint32_t k, bool in) {
        const uint8_t lit = in ? Q.lit[sb][k] : 2;
        uint32_t pixel = 0;
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        if (lit != 2) {
            pixel = __float_as_uint(Q.so[sb][k].w);
            c = Q.sc[sb][k];
            if (!lit) c = darken(c);
        }
        accumulate_wave(A.accum, pixel, c, lit != 2);
    });
    if (cnt.incomplete) atomicAdd(A.status + 2, 1u);
}

// Shade one level: the block's waves take 64 segments each per iteration.
// gout: the calling wave's outputs of the guide's network (GUIDED).
template <bool GUIDED>
__device__ __forceinline__ void shade_body(const RenderArgs& A, const Queues& Q, int level, int buf,
                                           float* gout, BlockSlots& slots) {
    const uint32_t n = min(Q.cnt[path_count(level)], Q.cap);
    const uint32_t lane = threadIdx.x & 63u;
    const bool spawn = level < A.max_depth && A.mc > 0;
    const uint32_t m = (uint32_t)max(A.mc, 0);
    const bool cosine = A.flags & TN_RENDER_COSINE;
    const bool area_flag = (A.flags & TN_RENDER_AREA_LIGHTS) != 0;
    const bool records = GUIDED && A.rec_p != nullptr;
    const float inv_pi = 0.318309886183790671538f;
    uint32_t turn = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        const bool active = i < n;
        bool has_hit = false, has_point = false, has_area = false;
        float4 w = make_float4(0, 0, 0, 0), rho = w;
        float3 p = make_float3(0, 0, 0), p2 = p, nn = p, ldir = p, adir = p;
        float ldist = 0.f, adist = 0.f;
        float4 lcontrib = w, acontrib = w, llocal = w, alocal = w;
        uint32_t pixel = 0, slot = 0;
        uint4 rng = make_uint4(1, 0, 0, 0);
        const uint4 h = active ? Q.hit[i] : make_uint4(kInvalidId, 0, 0, 0);
        has_hit = h.x != kInvalidId;
        // what the segment brings itself: the background (pathtracer.cpp:26-28)
        // or, seen by the camera, an emitter's front
        {
            float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
            bool has_own = active && !has_hit;
            if (active) {
                w = Q.w[buf][i];
                pixel = __float_as_uint(Q.o[buf][i].w);
                if (!has_hit) {
                    own = A.sp[scene_of_pixel(A, pixel)].bg;
                } else if (level == 0 && area_flag) {
                    own = A.emission[h.x];
                    const float4 g = A.trirec[4 * (size_t)h.x + 1], qd = Q.d[buf][i];  // geometric normal
                    has_own = A.sp[scene_of_pixel(A, pixel)].nemit > 0 && (own.x > 0 || own.y > 0 || own.z > 0) &&
                              g.x * qd.x + g.y * qd.y + g.z * qd.z < 0;
                }
            }
            accumulate_wave(A.accum, pixel, mul4(w, own), has_own);
            if (records && active && !has_hit) A.rec_x[__float_as_uint(Q.d[buf][i].w) * A.rstride + (uint32_t)level] = own;
        }
        if (active) {
            const float4 qo = Q.o[buf][i], qd = Q.d[buf][i];
            rng = Q.rng[buf][i];
            slot = __float_as_uint(qd.w) * A.rstride + (uint32_t)level;
            const SceneParams& S = A.sp[scene_of_pixel(A, pixel)];
            if (has_hit) {
                const uint32_t id = h.x;
                const float r = __uint_as_float(h.y), s = __uint_as_float(h.z), t = __uint_as_float(h.w);
                // pathtracer.cpp:30-36
                p = make_float3(qo.x + r * qd.x, qo.y + r * qd.y, qo.z + r * qd.z);
                const float* nv = A.normals + 9 * (size_t)id;
                const float b0 = 1.f - s - t;
                float3 ni = make_float3(b0 * nv[0] + s * nv[3] + t * nv[6], b0 * nv[1] + s * nv[4] + t * nv[7],
                                        b0 * nv[2] + s * nv[5] + t * nv[8]);
                const float inv = 1.0f / sqrtf(ni.x * ni.x + ni.y * ni.y + ni.z * ni.z);
                nn = make_float3(inv * ni.x, inv * ni.y, inv * ni.z);
                p2 = make_float3(p.x + 0.0001f * nn.x, p.y + 0.0001f * nn.y, p.z + 0.0001f * nn.z);
                rho = A.albedo[id];
                const float4 wr = mul4(w, rho);
                if (S.nlights) {  // pathtracer.cpp:44-58
                    float3 l = make_float3(S.light_pos.x - p.x, S.light_pos.y - p.y, S.light_pos.z - p.z);
                    const float il = 1.0f / sqrtf(l.x * l.x + l.y * l.y + l.z * l.z);
                    ldir = make_float3(il * l.x, il * l.y, il * l.z);
                    const float3 l2 = make_float3(S.light_pos.x - p2.x, S.light_pos.y - p2.y, S.light_pos.z - p2.z);
                    ldist = sqrtf(l2.x * l2.x + l2.y * l2.y + l2.z * l2.z);
                    const float c = fmaxf(0.f, ldir.x * nn.x + ldir.y * nn.y + ldir.z * nn.z);
                    lcontrib = scale4(inv_pi, mul4(wr, scale4(c, S.light_col)));
                    if (records) llocal = scale4(inv_pi, mul4(rho, scale4(c, S.light_col)));
                    has_point = true;
                }
                if (area_flag && S.nemit > 0) {
                    const float u0 = rng_uniform(rng), u1 = rng_uniform(rng), u2 = rng_uniform(rng);
                    // one emitter k with probability pk: by solid angle among
                    // the front-facing ones of a scene with few emitters, else
                    // by area
                    uint32_t k = 0;
                    float pk = 0.f;
                    if (S.nemit <= kSolidAngleSelect) {
                        float wk[kSolidAngleSelect];
                        float wsum = 0.f;
#pragma unroll
                        for (uint32_t j = 0; j < kSolidAngleSelect; ++j) {
                            wk[j] = 0.f;
                            if (j < S.nemit) {
                                const uint32_t kj = A.emit_ids[S.emit_begin + j];
                                const float4 r0 = A.trirec[4 * (size_t)kj], rn = A.trirec[4 * (size_t)kj + 1],
                                             ru = A.trirec[4 * (size_t)kj + 2], rv = A.trirec[4 * (size_t)kj + 3];
                                const float3 a = make_float3(r0.x - p.x, r0.y - p.y, r0.z - p.z);
                                if (-(a.x * rn.x + a.y * rn.y + a.z * rn.z) > 0.f)  // p in front of the emitter
                                    wk[j] = tri_solid_angle(a, v3axpy(1.f, make_float3(ru.x, ru.y, ru.z), a),
                                                            v3axpy(1.f, make_float3(rv.x, rv.y, rv.z), a));
                            }
                            wsum += wk[j];
                        }
                        const float x = u0 * wsum;
                        float run = 0.f;
                        bool picked = false;
#pragma unroll
                        for (uint32_t j = 0; j < kSolidAngleSelect; ++j) {
                            run += wk[j];
                            if (!picked && wk[j] > 0.f && (x < run || run >= wsum)) {
                                picked = true;
                                k = A.emit_ids[S.emit_begin + j];
                                pk = wk[j] / wsum;
                            }
                        }
                    } else {
                        const float x = u0 * S.emit_area;
                        const float* cdf = A.emit_cdf + S.emit_begin;
                        uint32_t lo = 0, hi = S.nemit - 1;
                        while (lo < hi) {
                            const uint32_t mid = (lo + hi) >> 1;
                            if (cdf[mid] <= x) lo = mid + 1;
                            else hi = mid;
                        }
                        k = A.emit_ids[S.emit_begin + lo];
                        const float cprev = lo ? cdf[lo - 1] : 0.f;
                        pk = (cdf[lo] - cprev) / S.emit_area;
                    }
                    if (pk > 0.f) {
                        const float4 e0 = A.trirec[4 * (size_t)k], en = A.trirec[4 * (size_t)k + 1],
                                     eu = A.trirec[4 * (size_t)k + 2], ev = A.trirec[4 * (size_t)k + 3];
                        const float3 a = make_float3(e0.x - p.x, e0.y - p.y, e0.z - p.z);
                        const float3 n3 = make_float3(en.x, en.y, en.z);
                        const float3 eu3 = make_float3(eu.x, eu.y, eu.z), ev3 = make_float3(ev.x, ev.y, ev.z);
                        // direction and inverse density per steradian
                        float inv_pdf = 0.f;
                        float3 q;
                        SphTri st;
                        if (sph_tri_setup(a, v3axpy(1.f, eu3, a), v3axpy(1.f, ev3, a), st) &&
                            st.omega >= kMinSolidAngle) {
                            adir = sph_tri_sample(st, u1, u2);
                            const float dn = v3dot(adir, n3);  // = -cos_l
                            const float tq = dn < 0.f ? v3dot(a, n3) / dn : 0.f;
                            q = v3axpy(tq, adir, p);
                            inv_pdf = dn < 0.f ? st.omega : 0.f;
                        } else {  // uniform point by area: density d^2 / (cos_l area)
                            const float su = sqrtf(u1);
                            const float bu = su * (1.0f - u2), bv = su * u2;
                            q = make_float3(e0.x + bu * eu.x + bv * ev.x, e0.y + bu * eu.y + bv * ev.y,
                                            e0.z + bu * eu.z + bv * ev.z);
                            const float3 dl = v3sub(q, p);
                            const float d2 = v3dot(dl, dl);
                            adir = v3scale(1.0f / sqrtf(d2), dl);
                            const float cl = -v3dot(adir, n3);
                            const float3 cr = v3cross(eu3, ev3);
                            inv_pdf = cl > 0.f ? cl * 0.5f * sqrtf(v3dot(cr, cr)) / d2 : 0.f;
                        }
                        const float cosx = v3dot(adir, nn);
                        if (cosx > 0 && inv_pdf > 0) {
                            const float3 q2 = v3sub(q, p2);
                            adist = sqrtf(v3dot(q2, q2)) * (1.0f - 1e-4f);
                            const float4 lek = A.emission[k];
                            const float gterm = cosx * inv_pdf / pk;
                            acontrib = scale4(inv_pi, mul4(wr, scale4(gterm, lek)));
                            if (records) alocal = scale4(inv_pi, mul4(rho, scale4(gterm, lek)));
                            has_area = true;
                        }
                    }
                }
            }
        }
        // shadow rays and unguided children (guided ones are drawn later)
        const uint64_t mp = __ballot(has_point), ma = __ballot(has_area);
        const uint64_t mh = spawn && !GUIDED ? __ballot(has_hit) : 0ull;
        const uint32_t tot = (uint32_t)(__popcll(mp) + __popcll(ma));
        uint32_t hbase = 0, sbase = 0;
        reserve_slots(slots, turn, Q.cnt, level, (uint32_t)__popcll(mh) * m, tot, hbase, sbase);
        turn ^= 1u;
        if (tot) {
            if (has_point) {
                const uint32_t k = sbase + lanes_below(mp);
                if (k < Q.scap) push_shadow(Q, level & 1, k, p2, pixel, ldir, ldist, lcontrib, llocal, slot, records);
                else atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
            }
            if (has_area) {
                const uint32_t k = sbase + (uint32_t)__popcll(mp) + lanes_below(ma);
                if (k < Q.scap) push_shadow(Q, level & 1, k, p2, pixel, adir, adist, acontrib, alocal, slot, records);
                else atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
            }
        }
        if (!spawn) continue;
        const int ob = buf ^ 1;
        const float invm = 1.0f / (float)m;
        const float4 wr = mul4(w, rho);
        const float pathbits = Q.d[buf][active ? i : 0].w;
        float3 b1, b2;
        onb(nn, b1, b2);
        if (!GUIDED) {
            // children: m per hit (pathtracer.cpp:72-85)
            if (!has_hit) continue;
            const uint32_t first = hbase + lanes_below(mh) * m;
            for (uint32_t c = 0; c < m; ++c) {
                const float u1 = rng_uniform(rng), u2 = rng_uniform(rng);
                float lx, ly, lz, f;
                const float phi = 6.28318530717958647692f * u2;
                float sp, cp;
                __sincosf(phi, &sp, &cp);
                if (cosine) {
                    const float rr = sqrtf(u1);
                    lx = rr * cp;
                    ly = rr * sp;
                    lz = sqrtf(fmaxf(0.f, 1.f - u1));
                    f = invm;
                } else {  // lib/sampling.h:20-32
                    lz = u1;
                    const float rr = sqrtf(fmaxf(0.f, 1.f - lz * lz));
                    lx = rr * cp;
                    ly = rr * sp;
                    f = 2.f * u1 * invm;
                }
                const float3 dir = make_float3(lx * b1.x + ly * b2.x + lz * nn.x, lx * b1.y + ly * b2.y + lz * nn.y,
                                               lx * b1.z + ly * b2.z + lz * nn.z);
                const uint32_t k = first + c;
                if (k < Q.cap) {
                    Q.o[ob][k] = make_float4(p2.x, p2.y, p2.z, __uint_as_float(pixel));
                    Q.d[ob][k] = make_float4(dir.x, dir.y, dir.z, pathbits);
                    Q.w[ob][k] = scale4(f, wr);
                    Q.rng[ob][k] = child_seed(rng, c);
                } else {
                    atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
                }
            }
        } else {
            // guided: the wave's 64 hits through the guide MLP
            guide_forward_wave<4>(A.gv, p, nn, has_hit, gout);
            Mixture M;
            mixture_from(gout + lane * kGOut, M);
            guide_wave_sync();  // gout is overwritten by the next iteration's forward pass
            for (uint32_t c = 0; c < m; ++c) {
                const float us = rng_uniform(rng), u0 = rng_uniform(rng), u1 = rng_uniform(rng),
                            u2 = rng_uniform(rng);
                float3 dir;
                if (us < A.mis) {
                    dir = mixture_sample(M, u0, u1, u2);
                } else {
                    const float rr = sqrtf(u1);
                    float sp, cp;
                    __sincosf(6.28318530717958647692f * u2, &sp, &cp);
                    const float lx = rr * cp, ly = rr * sp, lz = sqrtf(fmaxf(0.f, 1.f - u1));
                    dir = make_float3(lx * b1.x + ly * b2.x + lz * nn.x, lx * b1.y + ly * b2.y + lz * nn.y,
                                      lx * b1.z + ly * b2.z + lz * nn.z);
                }
                const float cosn = dir.x * nn.x + dir.y * nn.y + dir.z * nn.z;
                const bool ok = has_hit && cosn > 0.f;
                float f = 0.f, cos_pdf = 0.f;
                if (ok) {
                    const float pdf = A.mis * mixture_pdf(M, dir) + (1.0f - A.mis) * cosn * inv_pi;
                    cos_pdf = cosn / pdf;
                    f = inv_pi * cos_pdf * invm;
                }
                const uint64_t mc = __ballot(ok);
                uint32_t cbase, none;
                reserve_slots(slots, turn, Q.cnt, level, (uint32_t)__popcll(mc), 0u, cbase, none);
                turn ^= 1u;
                if (records && has_hit) {
                    A.rec_p[slot] = make_float4(p.x, p.y, p.z, cos_pdf);
                    A.rec_n[slot] = make_float4(nn.x, nn.y, nn.z, ok ? 1.f : 0.f);
                    A.rec_w[slot] = make_float4(dir.x, dir.y, dir.z, 0.f);
                    A.rec_g[slot] = scale4(f, rho);
                }
                if (!ok) continue;
                const uint32_t k = cbase + lanes_below(mc);
                if (k < Q.cap) {
                    Q.o[ob][k] = make_float4(p2.x, p2.y, p2.z, __uint_as_float(pixel));
                    Q.d[ob][k] = make_float4(dir.x, dir.y, dir.z, pathbits);
                    Q.w[ob][k] = scale4(f, wr);
                    Q.rng[ob][k] = child_seed(rng, c);
                } else {
                    atomicOr(&Q.cnt[4 * kMaxLevels], 1u);
                }
            }
        }
    }
}

// Two waves per block, each with 10 KB for the outputs of the guide's network:
// guided 512^2x8 at depth 6 4.21 ms with its features and activations in LDS rows
// (20 KB), 4.06 without; three or four waves per SIMD (16 or 32 samples at a time)
// 4.07 to 4.14.
constexpr int kGuidedBlock = 128;
__global__ __launch_bounds__(kGuidedBlock) void k_shade_guided(RenderArgs A, Queues Q, int level, int buf) {
    __shared__ __align__(16) float gout[kGuidedBlock / 64][64 * kGOut];
    __shared__ BlockSlots slots;
    shade_body<true>(A, Q, level, buf, gout[threadIdx.x >> 6], slots);
}

// The unguided shade capped at 72 VGPRs (7 waves per SIMD, 68 bytes of
// spill) instead of its natural 99 (5 waves): at 1920x1080, depth 3, m 4
// the render went 1151 -> 1191 Mrays/s on the rendering tree (6 waves, 80
// VGPRs: 1157).
__global__ __launch_bounds__(kRBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_shade_plain(
    RenderArgs A, Queues Q, int level, int buf) {
    __shared__ BlockSlots slots;
    shade_body<false>(A, Q, level, buf, nullptr, slots);
}

// ---------------------------------------------------------- persistent
// Grid barrier of the persistent kernel (all blocks resident: cooperative
// launch), two-level so that no counter sees more than a few hundred
// atomics: the blocks count in at one of eight group counters (block b in
// group b % 8, the XCD it is dealt to), the last of a group at the group
// total, and the last group publishes the next generation, which the others
// poll.  Words, each on its own 128-byte line: [0] generation, [32] set when
// a wait ran out, [64] groups arrived, [96 + 32 g] arrivals in group g.  A
// wait is bounded (2^22 polls of about 64 cycles): then [32] is set, and
// every block stops at its next barrier (grid_sync returns false).
constexpr uint32_t kBarrierPolls = 1u << 22;

__device__ __forceinline__ bool grid_sync(uint32_t* bar, uint32_t& gen) {
    __shared__ uint32_t ok;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t good = __hip_atomic_load(bar + kBarOut, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u;
        if (good) {
            __threadfence();
            const uint32_t target = gen + 1u;
            const uint32_t groups = gridDim.x < kXcds ? gridDim.x : kXcds;
            const uint32_t g = blockIdx.x % groups;
            const uint32_t members = gridDim.x / groups + (g < gridDim.x % groups ? 1u : 0u);
            bool released = false;
            if (atomicAdd(bar + kBarGroup + 32 * g, 1u) == members - 1u) {
                atomicExch(bar + kBarGroup + 32 * g, 0u);  // reset before the group counts in
                __threadfence();
                if (atomicAdd(bar + kBarGroups, 1u) == groups - 1u) {
                    atomicExch(bar + kBarGroups, 0u);
                    __threadfence();
                    atomicExch(bar + kBarGen, target);
                    released = true;
                }
            }
            if (!released) {
                for (uint32_t polls = 0;
                     __hip_atomic_load(bar + kBarGen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != target; ++polls) {
                    if (polls >= kBarrierPolls) {
                        atomicExch(bar + kBarOut, 1u);
                        good = 0u;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            __threadfence();
        }
        ok = good;
    }
    __syncthreads();
    ++gen;
    return ok != 0u;
}

// Plain path tracing (no guide, no training records, no refined tree) of
// every chunk of a call in one cooperative launch: per chunk, raygen, then
// per level the same trace, shade and shadow stages as the wavefront
// kernels, separated by grid barriers instead of kernel boundaries.  One
// pipeline; the shadow test of a level no longer overlaps the next level's
// tracing.  The chunk loop ends when a chunk is empty; every barrier wait is
// bounded.
template <bool EXH>
__global__ __launch_bounds__(kRBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_persist(RenderArgs A, Queues Q, int levels) {
    __shared__ uint2 stk[kRStack * kRBlock];
    __shared__ CoopLds wl[kRBlock / 64];
    __shared__ BlockSlots slots;
    uint32_t gen = 0;
    for (;;) {
        if (blockIdx.x == 0) chunk_begin_block(Q.cnt, Q.xwork, A.cs);
        if (!grid_sync(Q.bar, gen)) return;
        const uint32_t count = __hip_atomic_load(&A.cs->count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (count == 0u) return;
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x)
            raygen_one(A, Q, i);
        if (!grid_sync(Q.bar, gen)) return;
        int buf = 0;
        for (int lv = 0; lv < levels; ++lv) {
            trace_body<EXH, false>(A, Q, lv, buf, stk, wl);
            if (!grid_sync(Q.bar, gen)) return;
            shade_body<false>(A, Q, lv, buf, nullptr, slots);
            if (!grid_sync(Q.bar, gen)) return;
            shadow_body<EXH, false>(A, Q, lv, stk, wl);
            if (!grid_sync(Q.bar, gen)) return;
            buf ^= 1;
        }
        if (blockIdx.x == 0 && threadIdx.x < 64) chunk_totals(Q.cnt, Q.totals, levels);
        __syncthreads();  // the counts are read before block 0 clears them for the next chunk
    }
}

// Clears the training records of a chunk: valid flags and found radiance.
__global__ void k_rec_clear(RenderArgs A) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= A.cs->count * A.rstride) return;
    A.rec_n[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    A.rec_x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Walks each path of the chunk backwards (L_k = X_{k+1} + g_{k+1} L_{k+1})
// and appends (p, n, w, lum(L_k) cos / pdf) of every bounce that brought
// light back to the training set (kept with probability A.accept).  Sample
// layout: (p, c), (n, cos / pdf), (w, sample << 6 | level as bits), sample =
// the path's sample index within the call modulo 2^26.
__global__ __launch_bounds__(kRBlock) void k_collect(RenderArgs A, int levels_with_records) {
    const uint32_t npaths = A.cs->count;
    const uint64_t salt = A.seed_pass ^ (A.cs->first * 0x9E3779B97F4A7C15ull);
    const uint32_t pid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const bool act = pid < npaths;
    float3 L = make_float3(0.f, 0.f, 0.f), gprev = L;
    bool have = false;
    for (int k = levels_with_records - 1; k >= 0; --k) {
        const uint32_t slot = (act ? pid : 0u) * A.rstride + (uint32_t)k;
        bool emit = false;
        float4 rp, rn, rw;
        float c = 0.f;
        if (act) {
            rn = A.rec_n[slot];
            if (rn.w == 0.f) {
                have = false;
            } else {
                const float4 x = A.rec_x[slot + 1];
                float3 Lk = make_float3(x.x, x.y, x.z);
                if (have) {
                    Lk.x += gprev.x * L.x;
                    Lk.y += gprev.y * L.y;
                    Lk.z += gprev.z * L.z;
                }
                const float4 g = A.rec_g[slot];
                rp = A.rec_p[slot];
                rw = A.rec_w[slot];
                L = Lk;
                gprev = make_float3(g.x, g.y, g.z);
                have = true;
                c = (0.2126f * Lk.x + 0.7152f * Lk.y + 0.0722f * Lk.z) * rp.w;
                if (c > 0.f && isfinite(c)) {
                    const uint64_t h = splitmix64(salt ^ ((uint64_t)pid << 8) ^ (uint64_t)k);
                    emit = (float)(h >> 40) * 0x1p-24f < A.accept;
                }
            }
        }
        const uint64_t me = __ballot(emit);
        if (!me) continue;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(A.ts_count, (uint32_t)__popcll(me));
        base = __shfl(base, 0);
        if (!emit) continue;
        const uint32_t t = base + lanes_below(me);
        if (t < A.ts_cap) {
            A.ts[3 * (size_t)t] = make_float4(rp.x, rp.y, rp.z, c);
            A.ts[3 * (size_t)t + 1] = make_float4(rn.x, rn.y, rn.z, rp.w);
            const uint32_t sample = (uint32_t)(A.cs->first + pid) & ((1u << 26) - 1u);
            A.ts[3 * (size_t)t + 2] = make_float4(rw.x, rw.y, rw.z, __uint_as_float((sample << 6) | (uint32_t)k));
        }
    }
}

// The reference jitter sequence of one row: xorshift64* seeded 42,
// float = low 24 bits * 2^-24 (lib/xorshift.h:36-62, main.cpp:201-206).
std::vector<float> reference_jitter(uint32_t width, uint32_t spp) {
    std::vector<float> j(2 * (size_t)width * spp);
    uint64_t s = 42;
    for (float& v : j) {
        s ^= s >> 12;
        s ^= s << 25;
        s ^= s >> 27;
        const uint64_t out = s * 2685821657736338717ull;
        v = (float)(out & 0xFFFFFFull) * 0x1p-24f;
    }
    return j;
}

// Queue entries a pipeline's deepest level may take by default (404 bytes each):
// larger chunks are fewer launches, and fewer levels that only part of the chip
// works on.  1920 x 1080 x 2, depth 3, m 4 at 2^23 entries 100.3 ms, 2^24 90.8,
// 2^25 85.8, 2^26 83.7; m 2 18.1, 16.6, 16.5, 16.5; m 1 (8 samples) at 2^22 paths
// per chunk 19.0, 2^23 17.7, 2^24 17.6.  2^25 entries are 13.6 GB a pipeline;
// where that is more than a share of the free memory, half, down to the least.
constexpr uint32_t kQueueEntries = 1u << 25, kLeastQueueEntries = 1u << 23;

// Entries of a first allocation (1.7 GB), so that small renders of growing sizes
// share it; not when the caller sizes the chunks, nor from scarce memory.
constexpr uint32_t kLeastQueueAlloc = 1u << 22;

struct RenderBuffers {
    Queues q{};
    size_t bytes = 0;
    char* base = nullptr;
    ChunkState* cs = nullptr;
    RenderReport* rep = nullptr;  // where no memory is pinned
    SceneParams* sp = nullptr;
    uint32_t sp_cap = 0;
    // the shadow tests run on a second stream (default priority), ordered
    // against the main stream by one event per level and kind
    hipStream_t side = nullptr;
    hipEvent_t ev_shade[kMaxLevels] = {};
    hipEvent_t ev_shadow[kMaxLevels] = {};
};

int ensure_side_stream(RenderBuffers& rb) {
    if (rb.side) return TN_OK;
    TN_HIP(hipStreamCreateWithFlags(&rb.side, hipStreamNonBlocking));
    for (uint32_t k = 0; k < kMaxLevels; ++k) {
        TN_HIP(hipEventCreateWithFlags(&rb.ev_shade[k], hipEventDisableTiming));
        TN_HIP(hipEventCreateWithFlags(&rb.ev_shadow[k], hipEventDisableTiming));
    }
    return TN_OK;
}

// Queues, streams and events of the renders on one device.  A render call
// holds the context's lock from its first enqueued operation until its
// streams have drained, so concurrent calls on one device take turns; the
// buffers grow (no allocation once a call of the same size has run); large ones go
// back with the last scene and batch of the device (release_owner).
constexpr int kMaxDevices = 64;

// Carves the queue buffers out of one allocation; with base == nullptr it
// only measures (every piece is rounded up to 256 bytes).
size_t carve(Queues& q, ChunkState** cs, RenderReport** rep, char* base, uint32_t cap) {
    size_t off = 0;
    auto take = [&](size_t b) {
        char* r = base ? base + off : nullptr;
        off += (b + 255) & ~(size_t)255;
        return r;
    };
    for (int k = 0; k < 2; ++k) {
        q.o[k] = (float4*)take((size_t)cap * 16);
        q.d[k] = (float4*)take((size_t)cap * 16);
        q.w[k] = (float4*)take((size_t)cap * 16);
        q.rng[k] = (uint4*)take((size_t)cap * 16);
    }
    q.hit = (uint4*)take((size_t)cap * 16);
    q.scap = 2 * cap;
    for (int k = 0; k < 2; ++k) {
        q.so[k] = (float4*)take((size_t)q.scap * 16);
        q.sd[k] = (float4*)take((size_t)q.scap * 16);
        q.sc[k] = (float4*)take((size_t)q.scap * 16);
        q.sx[k] = (float4*)take((size_t)q.scap * 16);
        q.lit[k] = (uint8_t*)take(q.scap);
    }
    q.cnt = (uint32_t*)take((6 * kMaxLevels + 2) * sizeof(uint32_t));
    q.fix = (uint32_t*)take(3 * (size_t)kFixCap * sizeof(uint32_t));
    q.xwork = (uint32_t*)take(2 * kMaxLevels * kXcds * 16 * sizeof(uint32_t));
    q.totals = (unsigned long long*)take(2 * sizeof(unsigned long long));
    q.bar = (uint32_t*)take(kBarWords * sizeof(uint32_t));
    *cs = (ChunkState*)take(sizeof(ChunkState));
    *rep = (RenderReport*)take(sizeof(RenderReport));
    q.cap = cap;
    return off;
}

int reserve_scenes(RenderBuffers& rb, uint32_t nscenes) {
    if (rb.sp && rb.sp_cap >= nscenes) return TN_OK;
    if (rb.sp) (void)hipFree(rb.sp);
    rb.sp = nullptr;
    rb.sp_cap = 0;
    const uint32_t want = std::max(nscenes, 64u);
    TN_HIP(hipMalloc(&rb.sp, (size_t)want * sizeof(SceneParams)));
    rb.sp_cap = want;
    return TN_OK;
}

size_t queue_bytes(uint32_t cap) {
    Queues probe{};
    ChunkState* pcs = nullptr;
    RenderReport* prep = nullptr;
    return carve(probe, &pcs, &prep, nullptr, cap);
}

constexpr size_t kFreeShare = 4;  // new queues take at most a quarter of the free memory

// Queues of `cap` entries for the first npipes pipelines, of kLeastQueueAlloc
// unless `exact` or those exceed 1/kFreeShare of the memory that is free or held by
// the queues they replace.  limited: TN_ERR_OOM, before anything is touched, if
// `cap` entries exceed it.
int reserve_queues(RenderBuffers* rbs, int npipes, uint32_t cap, bool exact, bool limited) {
    size_t lacking = 0, held = 0;  // pipelines to allocate for, and what they hold
    for (int p = 0; p < npipes; ++p)
        if (!rbs[p].base || rbs[p].q.cap < cap) {
            ++lacking;
            held += rbs[p].bytes;
        }
    if (!lacking) return TN_OK;
    size_t free_bytes = 0, all = 0;
    TN_HIP(hipMemGetInfo(&free_bytes, &all));
    const size_t share = (free_bytes + held) / kFreeShare;
    uint32_t least = exact ? cap : std::max(cap, kLeastQueueAlloc);
    if (least > cap && lacking * queue_bytes(least) > share) least = cap;
    if (limited && lacking * queue_bytes(least) > share)
        return set_error(TN_ERR_OOM, "queues of %zu bytes, %zu are free", lacking * queue_bytes(least), free_bytes);
    for (int p = 0; p < npipes; ++p) {
        RenderBuffers& rb = rbs[p];
        if (rb.base && rb.q.cap >= cap) continue;
        if (rb.base) (void)hipFree(rb.base);
        rb.base = nullptr;
        rb.bytes = 0;
        uint32_t take = least;
        size_t need = queue_bytes(take);
        hipError_t e = hipMalloc(&rb.base, need);
        if (e != hipSuccess && take > cap) {  // no room for more than this call needs
            (void)hipGetLastError();
            take = cap;
            need = queue_bytes(take);
            e = hipMalloc(&rb.base, need);
        }
        if (e != hipSuccess) {
            rb.base = nullptr;
            (void)hipGetLastError();  // reported here
            return hip_error(e, "hipMalloc(ray queues)");
        }
        rb.bytes = need;
        carve(rb.q, &rb.cs, &rb.rep, rb.base, take);
    }
    return TN_OK;
}

struct RecordBuffers {
    float4* base = nullptr;
    size_t slots = 0;
};

int alloc_records(RecordBuffers& rb, size_t slots) {
    if (rb.base && rb.slots >= slots) return TN_OK;
    if (rb.base) (void)hipFree(rb.base);
    rb.base = nullptr;
    rb.slots = 0;
    TN_HIP(hipMalloc(&rb.base, slots * 5 * sizeof(float4)));
    rb.slots = slots;
    return TN_OK;
}

struct RenderContext {
    std::mutex mu;
    std::atomic<int> owners{0};  // scenes and batches of the device
    RenderBuffers rbs[kPipes];
    RecordBuffers recs[kPipes];
    // main streams of pipelines 1.. (pipeline 0 runs on the caller's stream)
    hipStream_t pipe_stream[kPipes] = {};
    hipEvent_t ev_fork = nullptr, ev_join[kPipes] = {};
    float* jitter = nullptr;  // reference pixel jitter (TN_RENDER_REF_JITTER)
    size_t jitter_cap = 0;
    // pinned: the pipelines' reports, then scene table and jitter on their way to
    // the device (free again when the call that wrote them returns; null where no
    // pinned memory is to be had)
    char* host = nullptr;
    size_t host_cap = 0;
    // graph replay (TN_RENDER_GRAPH): the capture stream and the executable
    // graph of the last captured chunk sequence, updated in place while the
    // topology stays the same
    hipStream_t cap_stream = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t graph_instantiations = 0, graph_updates = 0;
};

// A pinned scene table or jitter is at most this; a longer one takes a copy of its own.
constexpr size_t kPinnedTable = 1u << 20;

bool reserve_host(RenderContext& C, size_t bytes) {
    if (C.host && C.host_cap >= bytes) return true;
    if (C.host) (void)hipHostFree(C.host);
    C.host = nullptr;
    C.host_cap = 0;
    bytes = std::max<size_t>(bytes, 1u << 16);
    if (hipHostMalloc((void**)&C.host, bytes, hipHostMallocDefault) != hipSuccess) {
        C.host = nullptr;
        (void)hipGetLastError();  // the caller does without
        return false;
    }
    C.host_cap = bytes;
    return true;
}

RenderContext& render_context(int device) {
    static RenderContext ctx[kMaxDevices];
    return ctx[device];
}

// Gives back the context's device memory and pinned tables (its lock held, no render
// under way) if that is more than the least default queues of all pipelines (6.8 GB).
// A program that makes a scene, renders it and destroys it, again and again, thus
// keeps the memory of small renders: 64 x 64 Cornell box 0.34 ms a turn, 0.84 with all
// memory given back each time.  Large renders outweigh that (0.4 ms to allocate 27 GB,
// 0.7 to free them).
void release_memory(RenderContext& C) {
    size_t held = C.jitter_cap * sizeof(float);
    for (int p = 0; p < kPipes; ++p) held += C.rbs[p].bytes + C.recs[p].slots * 5 * sizeof(float4);
    if (held <= kPipes * queue_bytes(kLeastQueueEntries)) return;
    for (RenderBuffers& rb : C.rbs) {
        (void)hipFree(rb.base);
        (void)hipFree(rb.sp);
        rb.base = nullptr;
        rb.bytes = 0;
        rb.sp = nullptr;
        rb.sp_cap = 0;
    }
    for (RecordBuffers& r : C.recs) {
        (void)hipFree(r.base);
        r = RecordBuffers{};
    }
    (void)hipFree(C.jitter);
    C.jitter = nullptr;
    C.jitter_cap = 0;
    if (C.host) (void)hipHostFree(C.host);
    C.host = nullptr;
    C.host_cap = 0;
}

__global__ void k_scale(const float4* __restrict__ a, float4* __restrict__ out, uint32_t n, float f) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = a[i];
    out[i] = make_float4(v.x * f, v.y * f, v.z * f, v.w * f);
}

// Start of a render in one launch.  Block 0: counters and totals of every
// pipeline (pipeline p of n renders chunks p, p + n, p + 2n, ...) and, unless the
// persistent kernel does that itself, their first chunks; all blocks: scene table
// and jitter from pinned host memory.  With separate launches and copies here,
// and a blocking copy per counter at the end, a 320 x 320 Cornell render took
// 966 us (now 875), 512 x 512 x 1 at depth 6 2075 (2030), a batch of six small
// scenes 900 (850).
struct RenderStart {
    Queues q[kPipes];
    ChunkState* cs[kPipes];
    uint32_t pipes, chunk;
    unsigned long long total;
    bool persistent;
    uint32_t* incomplete;
    const uint32_t* src[2];
    uint32_t* dst[2];
    uint32_t words[2];
};
__global__ __launch_bounds__(512) void k_render_start(RenderStart R) {
    for (int k = 0; k < 2; ++k)
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < R.words[k]; i += gridDim.x * blockDim.x)
            R.dst[k][i] = R.src[k][i];
    if (blockIdx.x != 0) return;
    if (threadIdx.x == 0) *R.incomplete = 0;
    for (uint32_t p = 0; p < R.pipes; ++p) {
        const Queues& Q = R.q[p];
        if (threadIdx.x == 0) {
            Q.totals[0] = Q.totals[1] = 0;
            Q.cnt[4 * kMaxLevels] = 0;  // queue overflow
            ChunkState c{};
            c.next = (unsigned long long)p * R.chunk;
            c.total = R.total;
            c.stride = (unsigned long long)R.pipes * R.chunk;
            c.chunk = R.chunk;
            *R.cs[p] = c;
        }
        if (R.persistent) {
            for (uint32_t i = threadIdx.x; i < kBarWords; i += blockDim.x) Q.bar[i] = 0u;
            continue;
        }
        __syncthreads();
        chunk_begin_block(Q.cnt, Q.xwork, R.cs[p]);
    }
}

// The geometry a render traverses and shades: one scene, or the packed
// forest of a batch.
struct RenderGeom {
    SceneView sv;
    SceneView exact;       // TN_SCENE_REFINED: the reference tree behind the refined sv
    bool refined = false;
    const float* normals;
    const float4* albedo;
    const float4* emission;
    const float4* trirec;
    const uint32_t* emit_ids;
    const float* emit_cdf;
    const float4* reflective = nullptr;
    const float* reflectivity = nullptr;
    int device;
    int cus;
    uint32_t* status;  // 4 words; [2] counts incomplete render traversals
};

RenderGeom geom_of(const tn_scene* sc) {
    RenderGeom g;
    g.sv = sc->refined ? sc->fview() : sc->view();
    g.exact = sc->view();
    g.refined = sc->refined;
    g.normals = sc->d_normals;
    g.albedo = sc->d_albedo;
    g.emission = sc->d_emission;
    g.trirec = sc->d_tris;
    g.emit_ids = sc->d_emit_ids;
    g.emit_cdf = sc->d_emit_cdf;
    g.reflective = sc->d_reflective;
    g.reflectivity = sc->d_reflectivity;
    g.device = sc->device;
    g.cus = sc->cus;
    g.status = sc->d_status;
    return g;
}

SceneParams scene_params(const tn_camera* cam, const tn_light* lights, uint32_t nl, uint32_t width,
                         uint32_t height, uint32_t spp, const float bg[4], uint32_t emit_begin, uint32_t nemit,
                         float emit_area) {
    SceneParams S{};
    if (cam) {
        S.cam_pos = make_float4(cam->pos[0], cam->pos[1], cam->pos[2], 0);
        std::memcpy(S.cam_m, cam->trafo, sizeof S.cam_m);
        S.cam_dx = cam->delta_x;
        S.cam_dy = cam->delta_y;
    }
    S.width = width;
    S.height = height;
    S.spp = spp;
    S.nlights = nl;
    if (nl) {
        S.light_pos = make_float4(lights[0].pos[0], lights[0].pos[1], lights[0].pos[2], 0);
        S.light_col = make_float4(lights[0].color[0], lights[0].color[1], lights[0].color[2], lights[0].color[3]);
    }
    S.bg = make_float4(bg[0], bg[1], bg[2], bg[3]);
    S.emit_begin = emit_begin;
    S.nemit = nemit;
    S.emit_area = emit_area;
    return S;
}

}  // namespace

// Launch shape of the wavefront loop: primary samples per chunk (0: from the
// queue budget), blocks per CU of the persistent trace / shade / shadow
// kernels, and whether the per-chunk launch sequence is captured once in a
// hipGraph and replayed for every chunk.
struct LaunchShape {
    uint32_t chunk = 0;
    uint32_t blocks_per_cu = 8;
    bool graph = false;
    bool persistent = false;  // one cooperative launch walks every chunk and level (k_persist)
};

int check_render_params(const tn_render_params* P) {
    if (P->max_depth < 0 || P->mc_samples < 0) return set_error(TN_ERR_INVALID, "invalid render parameters");
    if ((uint32_t)P->max_depth + 2 > kMaxLevels) return set_error(TN_ERR_LIMIT, "max_depth too large");
    return TN_OK;
}

double path_fan(const tn_render_params* P) {
    double fan = 1;
    for (int k = 0; k < P->max_depth; ++k) fan *= std::max(1u, (uint32_t)P->mc_samples);
    return fan;
}

// Chunk size for a render: the queue of a chunk's deepest level holds
// chunk * m^max_depth segments, by default `entries` at most.
int chunk_size(const tn_render_params* P, uint32_t requested, uint32_t entries, uint32_t& chunk, uint32_t& cap) {
    const double fan = path_fan(P);
    chunk = requested ? requested : P->chunk_paths;
    if (chunk == 0)
        chunk = (uint32_t)std::max(1.0, std::min((double)entries / fan, (double)std::max(entries / 4, 1u << 22)));
    if (fan * chunk > 2147483647.0) return set_error(TN_ERR_LIMIT, "queue would exceed 2^31 entries");
    cap = (uint32_t)std::max(1.0, fan * chunk);
    return TN_OK;
}

// Chunks of a call: samples per chunk, queue entries of a pipeline, pipelines.
struct ChunkPlan {
    uint32_t chunk = 0, cap = 0;
    int npipes = 1;
};

// Two pipelines, each with its own queues and streams, render alternate chunks
// concurrently, so that one's launch tails (the slowest rays of a level) overlap
// the other's work.  A render of one chunk is split evenly between them when the
// halves still fill the chip.  With the path tracer that is from 2^19 samples or
// 2^23 segments at the deepest level, from where on it paid in every render
// measured, batches too (milliseconds whole / split: Cornell box 819,200 samples
// 0.87 / 0.81; m 1, depth 6, 524,176 samples 2.43 / 2.34; m 4, depth 3, 259,200
// samples 7.2 / 6.6; batches of six small scenes, depth 3: m 1, 529,056 samples 1.04 /
// 0.98, 993,408 1.47 / 1.42, m 2, 529,056 2.17 / 2.14, m 4, 239,760 4.42 / 4.15).
// Below it depends on the scene: m 1, 262,144 samples 2.02 / 1.98, but a batch of
// 280,000 0.85 / 0.88; m 2, 131,044 samples 1.74 / 1.67; m 4, 36,864 samples 1.94 /
// 1.88, but 65,536 2.48 / 2.56.  With the raytracer, whose levels thin out, it is from
// 2^20 (262,144 samples 0.68 / 0.73, 524,176 0.78 / 0.82, 2,079,604 1.33 with two).
// Several chunks are made equal so that both pipelines end together.  Chunks that
// the caller sizes and those of training renders (`plain` false; which records
// these keep depends on their chunks) are not made equal, and a single one is
// split from 2^20 samples on.
constexpr uint64_t kSplitPaths = 1u << 19, kSplitOther = 1u << 20;
constexpr double kSplitEntries = 8388608.0;
int plan_chunks(const tn_render_params* P, uint32_t requested, uint32_t entries, uint64_t total, int npipes,
                bool plain, ChunkPlan& plan) {
    int rc = chunk_size(P, requested, entries, plan.chunk, plan.cap);
    if (rc) return rc;
    const bool even = plain && !requested && P->chunk_paths == 0;
    const bool paths = even && P->renderer == TN_RENDERER_PATHTRACER;
    uint64_t parts = 0;
    if (npipes > 1 && total <= plan.chunk) {
        if (total >= (paths ? kSplitPaths : kSplitOther) || (paths && path_fan(P) * (double)total >= kSplitEntries))
            parts = npipes;
        else npipes = 1;
    } else if (npipes > 1 && even) {
        const uint64_t round = (uint64_t)npipes * plan.chunk;
        parts = (total + round - 1) / round * npipes;
    }
    plan.npipes = npipes;
    if (parts) {
        const uint64_t part = std::min<uint64_t>(plan.chunk, ((total + parts - 1) / parts + 255) & ~255ull);
        return chunk_size(P, (uint32_t)part, entries, plan.chunk, plan.cap);
    }
    // a call of less than one chunk needs no more queue than its samples do
    if (total && total < plan.chunk) return chunk_size(P, (uint32_t)total, entries, plan.chunk, plan.cap);
    return TN_OK;
}

// The wavefront loop over `total` samples of the scenes in `table` (sample
// and pixel ranges filled in by the caller), adding per-pixel radiance sums
// into accum.  Caller rays (ray_o/ray_d) replace the camera for tn_trace.
int render_core(const RenderGeom& G, const std::vector<SceneParams>& table, uint64_t total,
                const tn_render_params* P, const LaunchShape& shape, float* accum, tn_render_stats* st,
                hipStream_t stream, const float* ray_o, const float* ray_d, const float* jitter_host,
                size_t jitter_len, tn_guide* guide, uint32_t train_samples) {
    const bool rays = ray_o != nullptr;
    const bool guided = guide != nullptr;
    const bool training = guided && train_samples > 0;
    int rc = check_render_params(P);
    if (rc) return rc;
    if ((P->flags & TN_RENDER_GUIDED) && !guided)
        return set_error(TN_ERR_INVALID, "TN_RENDER_GUIDED needs a guide (tn_render_guided)");
    if (training && P->mc_samples != 1)
        return set_error(TN_ERR_INVALID, "training records need mc_samples == 1 (one path per sample)");
    if (guided && guide->device != G.device)
        return set_error(TN_ERR_INVALID, "guide and scene live on different devices");
    const uint32_t renderer = P->renderer;
    if (renderer > TN_RENDERER_RAYTRACER) return set_error(TN_ERR_INVALID, "unknown renderer %u", renderer);
    if (renderer != TN_RENDERER_PATHTRACER && guided)
        return set_error(TN_ERR_INVALID, "guided rendering needs the path tracer");
    if (renderer == TN_RENDERER_RAYTRACER)
        for (const SceneParams& S : table)
            if (S.nlights != 1)
                return set_error(TN_ERR_INVALID, "the raytracer needs one point light (raytracer.cpp:14)");
    // queue sizing: the raycaster traces one level, the raytracer spawns at
    // most one (mirror) child per hit
    tn_render_params q = *P;
    if (renderer == TN_RENDERER_RAYCASTER) q.max_depth = 0;
    if (renderer != TN_RENDERER_PATHTRACER) q.mc_samples = 1;
    // the persistent kernel serves plain path tracing of camera samples
    const bool persistent = shape.persistent && renderer == TN_RENDERER_PATHTRACER && !guided && !rays && !G.refined;
    // A graph-replayed render uses one pipeline: capturing the second
    // pipeline's stream, which itself forks its shadow stream, crashed the host
    // process, so that combination stays off.
    const int most_pipes = (shape.graph || persistent) ? 1 : kPipes;
    // a training render's chunks stay as small as their five records per bounce
    // make advisable
    uint32_t entries = training ? kLeastQueueEntries : kQueueEntries;
    ChunkPlan plan;
    if ((rc = plan_chunks(&q, shape.chunk, entries, total, most_pipes, !training, plan))) return rc;
    if (st) *st = tn_render_stats{};
    if (total == 0) return TN_OK;

    if (G.device < 0 || G.device >= kMaxDevices) return set_error(TN_ERR_LIMIT, "device %d", G.device);
    RenderContext& C = render_context(G.device);
    std::lock_guard<std::mutex> lock(C.mu);
    RenderBuffers* rbs = C.rbs;
    hipStream_t* pipe_stream = C.pipe_stream;
    // Every exit after the first enqueued operation drains the streams this
    // call used, so that no later call (once the lock is released) reuses
    // queues or records that kernels of this one may still read.
    bool enqueued = false;
    bool deferred = false;  // a deferred training set trains on the guide's stream during this call
    auto fail = [&](int code) {
        if (deferred) (void)hipStreamSynchronize(guide->tstream);
        if (enqueued) {
            (void)hipStreamSynchronize(stream);
            for (int p = 0; p < kPipes; ++p) {
                if (pipe_stream[p]) (void)hipStreamSynchronize(pipe_stream[p]);
                if (rbs[p].side) (void)hipStreamSynchronize(rbs[p].side);
            }
        }
        return code;
    };
#define TN_RHIP(call)                                                    \
    do {                                                                 \
        hipError_t e_ = (call);                                          \
        if (e_ != hipSuccess) return fail(::tn::hip_error(e_, #call));   \
    } while (0)
    const bool sized = shape.chunk || q.chunk_paths;  // by the caller
    while ((rc = reserve_queues(rbs, plan.npipes, plan.cap, sized, entries > kLeastQueueEntries))) {
        if (rc != TN_ERR_OOM || entries <= kLeastQueueEntries) return rc;
        entries /= 2;
        if ((rc = plan_chunks(&q, shape.chunk, entries, total, most_pipes, !training, plan))) return rc;
    }
    const uint32_t chunk = plan.chunk;
    const int npipes = plan.npipes;
    for (int p = 0; p < npipes; ++p) {
        if ((rc = reserve_scenes(rbs[p], (uint32_t)table.size()))) return rc;
        if ((rc = ensure_side_stream(rbs[p]))) return rc;
    }
    if (!C.ev_fork) {
        TN_HIP(hipEventCreateWithFlags(&C.ev_fork, hipEventDisableTiming));
        for (int p = 1; p < kPipes; ++p) {
            TN_HIP(hipStreamCreateWithFlags(&pipe_stream[p], hipStreamNonBlocking));
            TN_HIP(hipEventCreateWithFlags(&C.ev_join[p], hipEventDisableTiming));
        }
    }
    if (jitter_host && C.jitter_cap < jitter_len) {
        if (C.jitter) (void)hipFree(C.jitter);
        C.jitter = nullptr;
        C.jitter_cap = 0;
        TN_HIP(hipMalloc(&C.jitter, jitter_len * sizeof(float)));
        C.jitter_cap = jitter_len;
    }
    for (int p = 0; p < npipes && training; ++p)
        if ((rc = alloc_records(C.recs[p], (size_t)chunk * ((uint32_t)P->max_depth + 1)))) return rc;
    const size_t table_bytes = table.size() * sizeof(SceneParams);
    const size_t jitter_bytes = jitter_host ? jitter_len * sizeof(float) : 0;
    bool pin_table = table_bytes <= kPinnedTable, pin_jitter = jitter_bytes <= kPinnedTable;
    static_assert(sizeof(RenderReport) * kPipes <= 256 && sizeof(SceneParams) % 4 == 0, "layout of the pinned memory");
    const size_t jitter_at = 256 + (pin_table ? table_bytes : 0);
    const bool pinned = reserve_host(C, jitter_at + (pin_jitter ? jitter_bytes : 0));
    if (!pinned) pin_table = pin_jitter = false;
    if (pin_table) std::memcpy(C.host + 256, table.data(), table_bytes);
    if (pin_jitter && jitter_bytes) std::memcpy(C.host + jitter_at, jitter_host, jitter_bytes);
    RenderReport* report[kPipes];
    for (int p = 0; p < npipes; ++p) report[p] = pinned ? (RenderReport*)C.host + p : rbs[p].rep;
    enqueued = true;
    if (!pin_table)
        TN_RHIP(hipMemcpyAsync(rbs[0].sp, table.data(), table_bytes, hipMemcpyHostToDevice, stream));

    RenderArgs A0{};
    A0.sv = G.sv;
    A0.sv_exact = G.exact;
    A0.refined = G.refined;
    A0.normals = G.normals;
    A0.albedo = G.albedo;
    A0.emission = G.emission;
    A0.trirec = G.trirec;
    A0.emit_ids = G.emit_ids;
    A0.emit_cdf = G.emit_cdf;
    A0.sp = rbs[0].sp;
    A0.nscenes = (uint32_t)table.size();
    A0.status = G.status;
    A0.max_depth = q.max_depth;
    A0.mc = P->mc_samples;
    A0.max_vis = P->max_visibility;
    A0.shadow_si = P->shadow_intensity;
    A0.reflective = G.reflective;
    A0.reflectivity = G.reflectivity;
    A0.flags = P->flags;
    A0.seed = P->seed;
    A0.accum = (float4*)accum;
    A0.seed_pass = P->seed + (uint64_t)P->sample_offset * 0xD1B54A32D192ED03ull;
    // deferred training: the records of the last render train on the
    // guide's stream while this one renders from a snapshot of the weights
    const bool defer = guided && (P->flags & TN_RENDER_DEFER_TRAINING);
    if (guided && guide->pending) {
        if (defer) rc = guide_defer_begin(guide, stream, training, &deferred);
        else rc = guide_train_pending(guide, stream);
        if (rc) return fail(rc);
    }
    if (guided) {
        A0.gv = guide->view();
        if (deferred) {
            A0.gv.wbf = guide->wbf_snap;
            A0.gv.theta = guide->theta_snap;
        }
        A0.mis = guide->mis_guided;
    }
    if (training) {
        A0.rstride = (uint32_t)P->max_depth + 1;
        // every bounce of every path is a candidate; keep about kTrainSet of them
        constexpr uint32_t kTrainSet = 1u << 21;
        if ((rc = guide_reserve_set(guide, kTrainSet, stream))) return fail(rc);
        const double candidates = (double)total * std::max(1, P->max_depth);
        A0.accept = (float)std::min(1.0, 0.95 * kTrainSet / std::max(1.0, candidates));
        A0.ts = guide->ts;
        A0.ts_count = guide->ts_count;
        A0.ts_cap = guide->ts_cap;
    }
    if (jitter_host) {
        if (!pin_jitter)
            TN_RHIP(hipMemcpyAsync(C.jitter, jitter_host, jitter_bytes, hipMemcpyHostToDevice, stream));
        A0.jitter = C.jitter;
    }
    RecordBuffers* recs = C.recs;
    RenderArgs A[kPipes];
    Queues Q[kPipes];
    RenderStart R{};
    for (int p = 0; p < npipes; ++p) {
        A[p] = A0;
        A[p].cs = rbs[p].cs;
        Q[p] = rbs[p].q;
        if (training) {
            const size_t ns = recs[p].slots;
            A[p].rec_p = recs[p].base;
            A[p].rec_n = recs[p].base + ns;
            A[p].rec_w = recs[p].base + 2 * ns;
            A[p].rec_g = recs[p].base + 3 * ns;
            A[p].rec_x = recs[p].base + 4 * ns;
        }
        R.q[p] = Q[p];
        R.cs[p] = rbs[p].cs;
    }
    R.pipes = (uint32_t)npipes;
    R.chunk = chunk;
    R.total = total;
    R.persistent = persistent;
    R.incomplete = G.status + 2;
    R.src[0] = pin_table ? (const uint32_t*)(C.host + 256) : nullptr;
    R.dst[0] = (uint32_t*)rbs[0].sp;
    R.words[0] = pin_table ? (uint32_t)(table_bytes / 4) : 0u;
    R.src[1] = pin_jitter ? (const uint32_t*)(C.host + jitter_at) : nullptr;
    R.dst[1] = (uint32_t*)C.jitter;
    R.words[1] = pin_jitter ? (uint32_t)(jitter_bytes / 4) : 0u;
    const uint32_t start_blocks = std::min<uint32_t>(64u, 1u + (R.words[0] + R.words[1]) / 512u);
    k_render_start<<<start_blocks, 512, 0, stream>>>(R);
    const bool exh = P->flags & TN_RENDER_EXHAUSTIVE;
    const int levels = q.max_depth + 1;
    const uint32_t bpc = std::max(1u, shape.blocks_per_cu);
    const dim3 tgrid((uint32_t)G.cus * bpc), tblock(kRBlock);
    const uint32_t rgrid = (chunk + kRBlock - 1) / kRBlock;
    // One chunk of pipeline p: raygen, then per level trace and shade on the
    // main stream s and the level's shadow test on the pipeline's side
    // stream, so that the shadow test of level k overlaps the tracing of
    // level k + 1.  Shade of level k writes shadow queue k & 1, so it waits
    // for the shadow test of level k - 2; the raytracer's shade also reads
    // the child weights the shadow test of level k - 1 darkens, so it waits
    // for that one.
    const bool shadows = renderer != TN_RENDERER_RAYCASTER;
    auto chunk_start = [&](int p, hipStream_t s) {
        const RenderArgs& Ap = A[p];
        const Queues& Qp = Q[p];
        if (training) k_rec_clear<<<(uint32_t)(((size_t)chunk * Ap.rstride + 255) / 256), 256, 0, s>>>(Ap);
        if (rays) k_raygen_rays<<<rgrid, kRBlock, 0, s>>>(Ap, Qp, ray_o, ray_d);
        else k_raygen<<<rgrid, kRBlock, 0, s>>>(Ap, Qp);
    };
    auto chunk_level = [&](int p, hipStream_t s, int lv) -> hipError_t {
        hipError_t e = hipSuccess;
        auto chk = [&](hipError_t x) {
            if (e == hipSuccess) e = x;
        };
        RenderBuffers& rb = rbs[p];
        const RenderArgs& Ap = A[p];
        const Queues& Qp = Q[p];
        const hipStream_t side = rb.side;
        const int buf = lv & 1;
        const bool refd = G.refined;
        const dim3 fgrid(32u);  // fix lists are short (a scan after an overflow is rare)
        if (refd) {
            if (exh) k_trace<true, true><<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
            else k_trace<false, true><<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
            if (exh) k_fix_hits<true><<<fgrid, kRBlock, 0, s>>>(Ap, Qp, lv, buf);
            else k_fix_hits<false><<<fgrid, kRBlock, 0, s>>>(Ap, Qp, lv, buf);
        } else {
            if (exh) k_trace<true, false><<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
            else k_trace<false, false><<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
        }
        if (renderer == TN_RENDERER_RAYCASTER) {
            k_cast<<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
            return e;
        }
        const int dep = renderer == TN_RENDERER_RAYTRACER ? lv - 1 : lv - 2;
        if (dep >= 0) chk(hipStreamWaitEvent(s, rb.ev_shadow[dep], 0));
        if (renderer == TN_RENDERER_RAYTRACER) k_rt_shade<<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
        else if (guided) k_shade_guided<<<tgrid.x * (kRBlock / kGuidedBlock), kGuidedBlock, 0, s>>>(Ap, Qp, lv, buf);
        else k_shade_plain<<<tgrid, tblock, 0, s>>>(Ap, Qp, lv, buf);
        chk(hipEventRecord(rb.ev_shade[lv], s));
        chk(hipStreamWaitEvent(side, rb.ev_shade[lv], 0));
        if (renderer == TN_RENDERER_RAYTRACER) {
            if (exh) k_rt_shadow<true><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv, buf);
            else k_rt_shadow<false><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv, buf);
        } else if (refd) {
            if (exh) k_shadow<true, true><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv);
            else k_shadow<false, true><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv);
            if (exh) k_fix_shadows<true><<<fgrid, kRBlock, 0, side>>>(Ap, Qp, lv);
            else k_fix_shadows<false><<<fgrid, kRBlock, 0, side>>>(Ap, Qp, lv);
        } else {
            if (exh) k_shadow<true, false><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv);
            else k_shadow<false, false><<<tgrid, tblock, 0, side>>>(Ap, Qp, lv);
        }
        chk(hipEventRecord(rb.ev_shadow[lv], side));
        return e;
    };
    auto chunk_finish = [&](int p, hipStream_t s) -> hipError_t {
        RenderBuffers& rb = rbs[p];
        const RenderArgs& Ap = A[p];
        const Queues& Qp = Q[p];
        // every shadow test is done before the counts are read (the side
        // stream runs in order, so its last event covers all of them)
        hipError_t e = hipSuccess;
        if (shadows) e = hipStreamWaitEvent(s, rb.ev_shadow[levels - 1], 0);
        // the raytracer also counts the mirror rays of its last level
        // (trace() is entered and returns {} beyond max_depth)
        if (training) k_collect<<<rgrid, kRBlock, 0, s>>>(Ap, P->max_depth);
        k_chunk_end<<<1, 512, 0, s>>>(Qp, rb.cs, Ap.status + 2,
                                      renderer == TN_RENDERER_RAYCASTER   ? -1
                                      : renderer == TN_RENDERER_RAYTRACER ? levels + 1
                                                                          : levels,
                                      report[p]);
        return e;
    };
    // One chunk of each of n pipelines on its stream, enqueued level by level, so
    // that the second starts when the first does and not when the host has
    // launched all of the first's kernels.
    auto round = [&](const hipStream_t* s, int n) -> hipError_t {
        hipError_t e = hipSuccess;
        for (int p = 0; p < n; ++p) chunk_start(p, s[p]);
        for (int lv = 0; lv < levels; ++lv)
            for (int p = 0; p < n && e == hipSuccess; ++p) e = chunk_level(p, s[p], lv);
        for (int p = 0; p < n && e == hipSuccess; ++p) e = chunk_finish(p, s[p]);
        return e;
    };
    // All rounds: pipeline 0 on `stream`, pipeline 1 forked onto its own stream and
    // joined back after its last chunk.  The pipelines share nothing but the
    // accumulator's atomics, and joined after every round the one waited for the
    // other's last shadow test.
    auto all_rounds = [&](uint64_t rounds) -> hipError_t {
        hipError_t e = hipSuccess;
        hipStream_t s[kPipes] = {stream};
        if (npipes > 1) e = hipEventRecord(C.ev_fork, stream);
        for (int p = 1; p < npipes && e == hipSuccess; ++p) {
            s[p] = pipe_stream[p];
            e = hipStreamWaitEvent(s[p], C.ev_fork, 0);
        }
        for (uint64_t c = 0; c < rounds && e == hipSuccess; ++c) e = round(s, npipes);
        for (int p = 1; p < npipes && e == hipSuccess; ++p) {
            e = hipEventRecord(C.ev_join[p], s[p]);
            if (e == hipSuccess) e = hipStreamWaitEvent(stream, C.ev_join[p], 0);
        }
        return e;
    };
    const uint64_t nchunks = (total + chunk - 1) / chunk;
    const uint64_t rounds = (nchunks + npipes - 1) / npipes;
    auto t0 = std::chrono::steady_clock::now();
    if (persistent) {
        // every block resident at once: the occupancy the kernel allows, at
        // most the shape's blocks per CU
        const void* kfn = exh ? (const void*)k_persist<true> : (const void*)k_persist<false>;
        int per_cu = 0;
        TN_RHIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, kRBlock, 0));
        if (per_cu < 1) return fail(set_error(TN_ERR_LIMIT, "the persistent kernel does not fit a CU"));
        const dim3 pgrid((uint32_t)G.cus * std::min<uint32_t>((uint32_t)per_cu, bpc));
        TN_RHIP(hipGetLastError());
        RenderArgs pa = A[0];
        Queues pq = Q[0];
        int plevels = levels;
        void* args[] = {&pa, &pq, &plevels};
        TN_RHIP(hipLaunchCooperativeKernel(kfn, pgrid, dim3(kRBlock), args, 0, stream));
        k_persist_end<<<1, 64, 0, stream>>>(Q[0], G.status + 2, report[0]);
    } else if (shape.graph && rounds > 1) {
        // The chunk sequence is captured on every call (host-side recording;
        // its kernel arguments change from call to call) and applied to the
        // executable graph kept from the last call by hipGraphExecUpdate,
        // which needs the same topology; only a changed topology (levels,
        // renderer, guided or training work) instantiates a new one.
        if (!C.cap_stream) TN_RHIP(hipStreamCreateWithFlags(&C.cap_stream, hipStreamNonBlocking));
        hipGraph_t graph = nullptr;
        hipError_t e = hipStreamBeginCapture(C.cap_stream, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            const hipError_t es = round(&C.cap_stream, 1);  // its shadow stream joins and leaves the capture
            e = hipStreamEndCapture(C.cap_stream, &graph);
            if (e == hipSuccess) e = es;
        }
        if (e == hipSuccess && C.exec) {
            hipGraphNode_t bad = nullptr;
            hipGraphExecUpdateResult why = hipGraphExecUpdateSuccess;
            if (hipGraphExecUpdate(C.exec, graph, &bad, &why) != hipSuccess || why != hipGraphExecUpdateSuccess) {
                (void)hipGetLastError();
                (void)hipGraphExecDestroy(C.exec);
                C.exec = nullptr;
            } else {
                ++C.graph_updates;
            }
        }
        if (e == hipSuccess && !C.exec) {
            e = hipGraphInstantiate(&C.exec, graph, nullptr, nullptr, 0);
            if (e == hipSuccess) ++C.graph_instantiations;
            else C.exec = nullptr;
        }
        for (uint64_t c = 0; e == hipSuccess && c < rounds; ++c) e = hipGraphLaunch(C.exec, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (graph) (void)hipGraphDestroy(graph);
        if (e != hipSuccess) return fail(hip_error(e, "captured chunk sequence"));
    } else {
        const hipError_t e = all_rounds(rounds);
        if (e != hipSuccess) return fail(hip_error(e, "chunk sequence"));
    }
    TN_RHIP(hipGetLastError());
    if (training) {
        if (defer) guide->pending = train_samples;  // trains during the next deferred call (or tn_guide_flush)
        else if ((rc = guide_train_from_set(guide, train_samples, stream))) return fail(rc);
    }
    if (deferred) TN_RHIP(hipStreamWaitEvent(stream, guide->ev_join, 0));
    TN_RHIP(hipStreamSynchronize(stream));
    RenderReport seen[kPipes];
    for (int p = 0; p < npipes; ++p) {
        if (pinned) seen[p] = *report[p];
        else TN_RHIP(hipMemcpy(&seen[p], report[p], sizeof(RenderReport), hipMemcpyDeviceToHost));
    }
#undef TN_RHIP
    const double ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    for (int p = 0; p < npipes; ++p)
        if (seen[p].overflow) return set_error(TN_ERR_QUEUE, "a ray queue overflowed");
    if (seen[0].barrier_out) return set_error(TN_ERR_INCOMPLETE, "a grid barrier wait of the persistent kernel ran out");
    // counted by both pipelines in one word: the later report has them all
    uint32_t incomplete = 0;
    for (int p = 0; p < npipes; ++p) incomplete = std::max(incomplete, seen[p].incomplete);
    if (incomplete) return set_error(TN_ERR_INCOMPLETE, "%u render traversals hit the visit cap", incomplete);
    if (st) {
        st->rays = st->shadow_rays = 0;
        for (int p = 0; p < npipes; ++p) {
            st->rays += seen[p].rays;
            st->shadow_rays += seen[p].shadow_rays;
        }
        st->primary_rays = rays ? 0 : total;
        st->ms = ms;
    }
    return TN_OK;
}

// Renders params->width x height x spp samples of one scene, adding the
// per-pixel SUM of sample radiance into accum (device, RGBA).
int render_into(tn_scene* sc, const tn_camera* cam, const tn_light* lights, uint32_t nl,
                const tn_render_params* P, float* accum, tn_render_stats* st, hipStream_t stream,
                const float* ray_o = nullptr, const float* ray_d = nullptr, uint64_t nrays = 0,
                tn_guide* guide = nullptr, uint32_t train_samples = 0) {
    const bool rays = ray_o != nullptr;
    if ((!rays && (P->width == 0 || P->height == 0 || P->pixel_samples < 1)) || P->max_depth < 0 ||
        P->mc_samples < 0)
        return set_error(TN_ERR_INVALID, "invalid render parameters");
    if (nl > 1) return set_error(TN_ERR_LIMIT, "at most one point light (main.cpp:123)");
    if (!rays && (size_t)P->width * P->height >= (1ull << 32))
        return set_error(TN_ERR_LIMIT, "image too large");
    if (rays && nrays >= (1ull << 32)) return set_error(TN_ERR_LIMIT, "too many rays");
    const uint32_t spp = rays ? 1u : (uint32_t)P->pixel_samples;
    std::vector<SceneParams> table(1, scene_params(cam, lights, nl, rays ? 1u : P->width, rays ? 1u : P->height,
                                                   spp, P->bg, 0, sc->nemit, sc->emit_area));
    const uint64_t total = rays ? nrays : (uint64_t)P->width * P->height * spp;
    std::vector<float> jit;
    if (!rays && (P->flags & TN_RENDER_REF_JITTER)) jit = reference_jitter(P->width, spp);
    LaunchShape shape;
    shape.graph = (P->flags & TN_RENDER_GRAPH) != 0;
    shape.persistent = (P->flags & TN_RENDER_PERSISTENT) != 0;
    return render_core(geom_of(sc), table, total, P, shape, accum, st, stream, ray_o, ray_d,
                       jit.empty() ? nullptr : jit.data(), jit.size(), guide, train_samples);
}

// ---------------------------------------------------------------- batches
namespace {

}  // namespace
}  // namespace tn

// Scenes packed into one forest: node, reference, triangle and shading arrays
// concatenated (indices rebased), one root per scene.
struct tn_batch {
    int device = 0, cus = 256;
    uint32_t nscenes = 0;
    uint4* treelets = nullptr;
    uint32_t* refs = nullptr;
    float4* tris = nullptr;
    float4* lrec = nullptr;  // records per reference (first halves, then second halves)
    size_t nrefs = 0;
    float* normals = nullptr;
    float4* albedo = nullptr;
    float4* emission = nullptr;
    uint32_t* emit_ids = nullptr;
    float* emit_cdf = nullptr;
    tn::SceneRoot* roots = nullptr;
    uint32_t* status = nullptr;
    std::vector<uint32_t> emit_begin, nemit;
    std::vector<float> emit_area;
    struct Tuned {
        int32_t depth, mc;
        uint32_t flags;
        int total_log2;
        tn::LaunchShape shape;
        tn_batch_tuning info;
    };
    std::vector<Tuned> tuned;
    tn_batch_tuning last{};

    tn::RenderGeom geom() const {
        tn::RenderGeom g;
        g.sv.nodes = nullptr;
        g.sv.treelets = treelets;
        g.sv.refs = refs;
        g.sv.tris = tris;
        g.sv.lra = lrec;
        g.sv.lrb = lrec + 2 * nrefs;
        for (int k = 0; k < 3; ++k) g.sv.bmin[k] = g.sv.bmax[k] = 0.f;
        g.sv.roots = roots;
        g.normals = normals;
        g.albedo = albedo;
        g.emission = emission;
        g.trirec = tris;
        g.emit_ids = emit_ids;
        g.emit_cdf = emit_cdf;
        g.device = device;
        g.cus = cus;
        g.status = status;
        return g;
    }
};

namespace tn {
namespace {

void free_batch(tn_batch* b) {
    for (void* p : {(void*)b->treelets, (void*)b->refs, (void*)b->tris, (void*)b->lrec, (void*)b->normals,
                    (void*)b->albedo,
                    (void*)b->emission, (void*)b->emit_ids, (void*)b->emit_cdf, (void*)b->roots,
                    (void*)b->status})
        if (p) (void)hipFree(p);
}

// Copies a scene's n treelets to a forest that already holds `first` treelets and
// ref_base references: child indices and leaf offsets move by these.  (A batch of 60
// scenes of 332 to 20,492 triangles is made in 3.0 ms; with its treelets built on the host,
// 4.4 to 5.5.)
__global__ void k_pack_treelets(const uint4* __restrict__ src, uint32_t n, uint32_t first, uint32_t ref_base,
                                uint4* __restrict__ dst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 a = src[2 * (size_t)i], b = src[2 * (size_t)i + 1];  // root_x, left_x, right_x, root_y; left_y, right_y
    if ((a.w & 3u) == 3u) a.x += ref_base;
    if ((b.x & 3u) == 3u) a.y += ref_base;
    else b.x += first << 2;
    if ((b.y & 3u) == 3u) a.z += ref_base;
    else b.y += first << 2;
    dst[2 * (size_t)i] = a;
    dst[2 * (size_t)i + 1] = b;
}

// Packs n scenes (of one device, current) into b; what it allocated is freed by the
// caller, also after an error.
int fill_batch(tn_scene* const* scenes, uint32_t n, tn_batch* b) {
    std::vector<uint32_t> refs, eids;
    std::vector<float> ecdf;
    std::vector<SceneRoot> roots(n);
    b->device = scenes[0]->device;
    b->cus = scenes[0]->cus;
    b->nscenes = n;
    uint64_t ntri = 0, nnodes = 0, nrefs = 0, ntreelets = 0;
    std::vector<uint64_t> tri_base(n), ref_base(n);
    for (uint32_t s = 0; s < n; ++s) {
        const tn_scene* sc = scenes[s];
        tri_base[s] = ntri;
        ref_base[s] = nrefs;
        roots[s].treelet = (uint32_t)ntreelets;  // below 2^30, as the nodes
        ntri += sc->ntris;
        nnodes += sc->tree.nodes.size();
        nrefs += sc->tree.refs.size();
        ntreelets += sc->ntreelets;
        if (ntri >= TN_INVALID_ID || nnodes >= (1ull << 30) || nrefs >= (1ull << 32))
            return set_error(TN_ERR_LIMIT, "batch exceeds 2^30 triangles or nodes");
    }
    refs.reserve(nrefs);
    for (uint32_t s = 0; s < n; ++s) {
        const tn_scene* sc = scenes[s];
        for (int k = 0; k < 3; ++k) {
            roots[s].bmin[k] = sc->tree.box[k];
            roots[s].bmax[k] = sc->tree.box[3 + k];
        }
        for (uint32_t r : sc->tree.refs) refs.push_back(r + (uint32_t)tri_base[s]);
        b->emit_begin.push_back((uint32_t)eids.size());
        b->nemit.push_back(sc->nemit);
        b->emit_area.push_back(sc->emit_area);
        if (sc->nemit) {
            std::vector<uint32_t> ids(sc->nemit);
            std::vector<float> cdf(sc->nemit);
            hipError_t e = hipMemcpy(ids.data(), sc->d_emit_ids, sc->nemit * 4, hipMemcpyDeviceToHost);
            if (e == hipSuccess) e = hipMemcpy(cdf.data(), sc->d_emit_cdf, sc->nemit * 4, hipMemcpyDeviceToHost);
            if (e != hipSuccess) return hip_error(e, "hipMemcpy");
            for (uint32_t& i : ids) i += (uint32_t)tri_base[s];
            eids.insert(eids.end(), ids.begin(), ids.end());
            ecdf.insert(ecdf.end(), cdf.begin(), cdf.end());
        }
    }
    hipError_t e;
    const size_t nt = std::max<uint64_t>(ntri, 1);
    if ((e = hipMalloc(&b->treelets, ntreelets * sizeof(Treelet))) != hipSuccess ||
        (e = hipMalloc(&b->refs, std::max<size_t>(refs.size(), 1) * 4)) != hipSuccess ||
        (e = hipMalloc(&b->tris, nt * 64)) != hipSuccess || (e = hipMalloc(&b->normals, nt * 36)) != hipSuccess ||
        (e = hipMalloc(&b->albedo, nt * 16)) != hipSuccess || (e = hipMalloc(&b->emission, nt * 16)) != hipSuccess ||
        (e = hipMalloc(&b->emit_ids, std::max<size_t>(eids.size(), 1) * 4)) != hipSuccess ||
        (e = hipMalloc(&b->emit_cdf, std::max<size_t>(ecdf.size(), 1) * 4)) != hipSuccess ||
        (e = hipMalloc(&b->roots, n * sizeof(SceneRoot))) != hipSuccess ||
        (e = hipMalloc(&b->status, 4 * sizeof(uint32_t))) != hipSuccess)
        return hip_error(e, "hipMalloc");
    if ((e = hipMemset(b->status, 0, 4 * sizeof(uint32_t))) != hipSuccess) return hip_error(e, "hipMemset");
    if ((e = hipMemcpy(b->refs, refs.data(), refs.size() * 4, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemcpy(b->roots, roots.data(), n * sizeof(SceneRoot), hipMemcpyHostToDevice)) != hipSuccess ||
        (!eids.empty() &&
         (e = hipMemcpy(b->emit_ids, eids.data(), eids.size() * 4, hipMemcpyHostToDevice)) != hipSuccess) ||
        (!ecdf.empty() &&
         (e = hipMemcpy(b->emit_cdf, ecdf.data(), ecdf.size() * 4, hipMemcpyHostToDevice)) != hipSuccess))
        return hip_error(e, "hipMemcpy");
    for (uint32_t s = 0; s < n; ++s) {
        const tn_scene* sc = scenes[s];
        const size_t t0 = tri_base[s], k = sc->ntris;
        const uint32_t first = roots[s].treelet;
        k_pack_treelets<<<(sc->ntreelets + 255) / 256, 256, 0, nullptr>>>(sc->d_treelets, sc->ntreelets, first,
                                                                          (uint32_t)ref_base[s], b->treelets + 2 * (size_t)first);
        if ((e = hipGetLastError()) != hipSuccess) return hip_error(e, "k_pack_treelets");
        if ((e = hipMemcpy(b->tris + 4 * t0, sc->d_tris, k * 64, hipMemcpyDeviceToDevice)) != hipSuccess ||
            (e = hipMemcpy(b->normals + 9 * t0, sc->d_normals, k * 36, hipMemcpyDeviceToDevice)) != hipSuccess ||
            (e = hipMemcpy(b->albedo + t0, sc->d_albedo, k * 16, hipMemcpyDeviceToDevice)) != hipSuccess ||
            (e = hipMemcpy(b->emission + t0, sc->d_emission, k * 16, hipMemcpyDeviceToDevice)) != hipSuccess)
            return hip_error(e, "hipMemcpy");
    }
    b->nrefs = refs.size();
    if ((e = hipMalloc(&b->lrec, std::max<size_t>(b->nrefs, 1) * 64)) != hipSuccess) return hip_error(e, "hipMalloc");
    return gather_leaf_records(b->tris, b->refs, b->nrefs, b->lrec);
}

int batch_table(const tn_batch* b, const tn_batch_job* jobs, std::vector<SceneParams>& table, uint64_t& total,
                uint64_t& pixels) {
    table.resize(b->nscenes);
    total = 0;
    pixels = 0;
    for (uint32_t s = 0; s < b->nscenes; ++s) {
        const tn_batch_job& J = jobs[s];
        if (J.width == 0 || J.height == 0 || J.pixel_samples < 1 || J.num_lights > 1)
            return set_error(TN_ERR_INVALID, "invalid job %u", s);
        table[s] = scene_params(&J.cam, &J.light, J.num_lights, J.width, J.height, (uint32_t)J.pixel_samples,
                                J.bg, b->emit_begin[s], b->nemit[s], b->emit_area[s]);
        table[s].sample_begin = total;
        table[s].pixel_begin = (uint32_t)pixels;
        total += (uint64_t)J.width * J.height * (uint32_t)J.pixel_samples;
        pixels += (uint64_t)J.width * J.height;
        if (pixels >= (1ull << 32)) return set_error(TN_ERR_LIMIT, "batch images exceed 2^32 pixels");
    }
    return TN_OK;
}

// Times candidate launch shapes on the first samples of the batch (into a
// scratch accumulator) and returns the fastest.
int autotune(tn_batch* b, const std::vector<SceneParams>& table, uint64_t total, uint64_t pixels,
             const tn_render_params* P, hipStream_t stream, LaunchShape& best, tn_batch_tuning& info) {
    // the probe spans at least two of the largest chunks, so both pipelines
    // of a direct-launch shape are busy as in the full render
    const uint64_t probe = std::min<uint64_t>(total, 1ull << 23);
    float* scratch = nullptr;
    TN_HIP(hipMalloc(&scratch, (size_t)pixels * 16));
    const uint32_t chunks[] = {1u << 18, 1u << 20, 1u << 22};
    const uint32_t grids[] = {4, 8, 16};
    double best_rate = -1;
    info = tn_batch_tuning{};
    auto t0 = std::chrono::steady_clock::now();
    int rc = TN_OK;
    for (uint32_t c : chunks) {
        uint32_t ch = 0, cap = 0;
        if (chunk_size(P, c, kLeastQueueEntries, ch, cap) != TN_OK || cap > (1u << 24)) continue;  // queue budget
        if (c > 2 * probe && c != chunks[0]) continue;
        for (uint32_t g : grids) {
            // graph replay (one pipeline) or direct launches (two
            // pipelines); the persistent launch is no candidate (slower than
            // both on every batch measured)
            for (const bool graph : {true, false}) {
                LaunchShape sh;
                sh.chunk = c;
                sh.blocks_per_cu = g;
                sh.graph = graph;
                tn_render_stats st{};
                rc = render_core(b->geom(), table, probe, P, sh, scratch, &st, stream, nullptr, nullptr, nullptr,
                                 0, nullptr, 0);
                if (rc) break;
                const double rate = (double)probe / std::max(st.ms, 1e-3);
                ++info.candidates;
                if (rate > best_rate) {
                    best_rate = rate;
                    best = sh;
                }
            }
            if (rc) break;
        }
        if (rc) break;
    }
    (void)hipFree(scratch);
    if (rc) return rc;
    if (best_rate < 0) return set_error(TN_ERR_LIMIT, "no launch shape fits the queue budget");
    info.chunk_paths = best.chunk;
    info.blocks_per_cu = best.blocks_per_cu;
    info.graph = best.graph ? 1u : 0u;
    info.best_rate = best_rate;
    info.probe_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return TN_OK;
}

}  // namespace
}  // namespace tn

namespace tn {

void add_owner(int device) {
    if (device >= 0 && device < kMaxDevices) ++render_context(device).owners;
}

void release_owner(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    RenderContext& C = render_context(device);
    if (--C.owners != 0) return;  // without the lock: renders of the others may be under way
    std::lock_guard<std::mutex> lock(C.mu);
    if (C.owners == 0) release_memory(C);
}

}  // namespace tn

using namespace tn;

extern "C" {

int tn_sample_triangle_host(const float* p3, const float* tri9, const float* u2, uint32_t n, float* dir3,
                            float* omega, float* omega_vos) {
    if (!p3 || !tri9 || (n && (!u2 || !dir3)) || !omega || !omega_vos)
        return set_error(TN_ERR_INVALID, "NULL argument");
    const float3 p = make_float3(p3[0], p3[1], p3[2]);
    const float3 a = v3sub(make_float3(tri9[0], tri9[1], tri9[2]), p),
                 b = v3sub(make_float3(tri9[3], tri9[4], tri9[5]), p),
                 c = v3sub(make_float3(tri9[6], tri9[7], tri9[8]), p);
    SphTri st;
    if (!sph_tri_setup(a, b, c, st)) return set_error(TN_ERR_INVALID, "degenerate spherical triangle");
    *omega = st.omega;
    *omega_vos = tri_solid_angle(a, b, c);
    for (uint32_t i = 0; i < n; ++i) {
        const float3 d = sph_tri_sample(st, u2[2 * i], u2[2 * i + 1]);
        dir3[3 * i] = d.x;
        dir3[3 * i + 1] = d.y;
        dir3[3 * i + 2] = d.z;
    }
    return TN_OK;
}

int tn_render_accumulate(tn_scene* sc, const tn_camera* cam, const tn_light* lights, uint32_t nl,
                         const tn_render_params* P, float* accum, tn_render_stats* st, void* stream) {
    if (!sc || !cam || !P || !accum || (nl && !lights))
        return set_error(TN_ERR_INVALID, "NULL argument");
    return render_into(sc, cam, lights, nl, P, accum, st, (hipStream_t)stream);
}

int tn_render_guided(tn_scene* sc, const tn_camera* cam, const tn_light* lights, uint32_t nl,
                     const tn_render_params* P, tn_guide* guide, uint32_t train_samples, float* accum,
                     tn_render_stats* st, void* stream) {
    if (!sc || !cam || !P || !guide || !accum || (nl && !lights))
        return set_error(TN_ERR_INVALID, "NULL argument");
    tn_render_params q = *P;
    q.flags |= TN_RENDER_GUIDED;
    return render_into(sc, cam, lights, nl, &q, accum, st, (hipStream_t)stream, nullptr, nullptr, 0, guide,
                       train_samples);
}

int tn_trace(tn_scene* sc, const float* o3, const float* d3, uint32_t n, int32_t depth,
             const tn_light* lights, uint32_t nl, const tn_render_params* P, float* rgba,
             tn_render_stats* st, void* stream) {
    if (!sc || !P || (n && (!o3 || !d3 || !rgba)) || (nl && !lights) || depth < 0)
        return set_error(TN_ERR_INVALID, "NULL or invalid argument");
    if (st) *st = tn_render_stats{};
    if (n == 0) return TN_OK;
    tn_render_params q = *P;
    if (P->renderer == TN_RENDERER_RAYCASTER) {
        q.max_depth = 0;  // raycaster.cpp:7-24 ignores the depth
    } else if (depth > P->max_depth) {  // pathtracer.cpp:17-19, raytracer.cpp:9-13
        if (st && P->renderer == TN_RENDERER_RAYTRACER) st->rays = n;  // counted before the return
        return TN_OK;
    } else {
        q.max_depth = P->max_depth - depth;  // levels depth..max_depth remain
    }
    return render_into(sc, nullptr, lights, nl, &q, rgba, st, (hipStream_t)stream, o3, d3, n);
}

int tn_render(tn_scene* sc, const tn_camera* cam, const tn_light* lights, uint32_t nl,
              const tn_render_params* P, float* linear, float* display, tn_render_stats* st) {
    if (!sc || !cam || !P || (nl && !lights)) return set_error(TN_ERR_INVALID, "NULL argument");
    if (P->width == 0 || P->height == 0 || P->pixel_samples < 1)
        return set_error(TN_ERR_INVALID, "invalid render parameters");
    const size_t np = (size_t)P->width * P->height;
    TN_HIP(hipSetDevice(sc->device));
    std::lock_guard<std::mutex> lock(sc->stage_mu);
    if (int rc = sc->reserve_stage(np * 16 * 2)) return rc;
    float* acc = (float*)sc->d_stage;
    float* out = acc + np * 4;
    int rc = TN_OK;
    hipError_t e = hipMemsetAsync(acc, 0, np * 16, nullptr);
    if (e != hipSuccess) rc = hip_error(e, "hipMemsetAsync");
    if (!rc) rc = render_into(sc, cam, lights, nl, P, acc, st, nullptr);
    const float inv = 1.0f / (float)P->pixel_samples;
    if (!rc && linear) {  // mean over pixel samples (main.cpp:216)
        k_scale<<<(uint32_t)((np + 255) / 256), 256, 0, nullptr>>>((const float4*)acc, (float4*)out, (uint32_t)np, inv);
        if ((e = hipGetLastError()) != hipSuccess) rc = hip_error(e, "k_scale");
        if (!rc && (e = hipMemcpy(linear, out, np * 16, hipMemcpyDeviceToHost)) != hipSuccess)
            rc = hip_error(e, "hipMemcpy");
    }
    if (!rc && display) {
        rc = tn_tonemap(acc, out, (uint32_t)np, inv, P->exposure, P->inverse_gamma, P->gamma_enabled,
                        nullptr);
        if (!rc && (e = hipMemcpy(display, out, np * 16, hipMemcpyDeviceToHost)) != hipSuccess)
            rc = hip_error(e, "hipMemcpy");
    }
    if (rc) (void)hipDeviceSynchronize();  // no kernel of this call still uses the staging memory
    return rc;
}

int tn_batch_create(tn_scene* const* scenes, uint32_t n, tn_batch** out) {
    if (!scenes || !out || n == 0) return set_error(TN_ERR_INVALID, "NULL argument or empty batch");
    *out = nullptr;
    for (uint32_t s = 0; s < n; ++s)
        if (!scenes[s]) return set_error(TN_ERR_INVALID, "NULL scene %u", s);
    const int dev = scenes[0]->device;
    for (uint32_t s = 0; s < n; ++s)
        if (scenes[s]->device != dev) return set_error(TN_ERR_INVALID, "scenes live on different devices");
    TN_HIP(hipSetDevice(dev));
    std::unique_ptr<tn_batch> b(new (std::nothrow) tn_batch());
    if (!b) return set_error(TN_ERR_OOM, "host allocation failed");
    int rc;
    try {
        rc = fill_batch(scenes, n, b.get());
    } catch (const std::bad_alloc&) {
        rc = set_error(TN_ERR_OOM, "host allocation failed");
    }
    if (rc) {
        free_batch(b.get());
        return rc;
    }
    add_owner(dev);
    *out = b.release();
    return TN_OK;
}

int tn_batch_destroy(tn_batch* b) {
    if (!b) return TN_OK;
    (void)hipSetDevice(b->device);
    (void)hipDeviceSynchronize();
    free_batch(b);
    release_owner(b->device);
    delete b;
    return TN_OK;
}

int tn_batch_render(tn_batch* b, const tn_batch_job* jobs, const tn_render_params* P, float* accum,
                    tn_render_stats* st, void* stream) {
    if (!b || !jobs || !P || !accum) return set_error(TN_ERR_INVALID, "NULL argument");
    if (P->flags & (TN_RENDER_GUIDED | TN_RENDER_REF_JITTER))
        return set_error(TN_ERR_INVALID, "batches render without guide or reference jitter");
    if (P->renderer != TN_RENDERER_PATHTRACER) return set_error(TN_ERR_INVALID, "batches render with the path tracer");
    int rc = check_render_params(P);
    if (rc) return rc;
    TN_HIP(hipSetDevice(b->device));
    std::vector<SceneParams> table;
    uint64_t total = 0, pixels = 0;
    if ((rc = batch_table(b, jobs, table, total, pixels))) return rc;
    hipStream_t s = (hipStream_t)stream;
    LaunchShape shape;
    shape.graph = (P->flags & TN_RENDER_GRAPH) != 0;
    shape.persistent = (P->flags & TN_RENDER_PERSISTENT) != 0;
    if ((P->flags & TN_RENDER_AUTOTUNE) && P->chunk_paths == 0) {
        const uint32_t key_flags = P->flags & ~(TN_RENDER_GRAPH | TN_RENDER_AUTOTUNE | TN_RENDER_PERSISTENT);
        int lg = 0;
        while ((1ull << lg) < total) ++lg;
        const tn_batch::Tuned* hit = nullptr;
        for (const auto& t : b->tuned)
            if (t.depth == P->max_depth && t.mc == P->mc_samples && t.flags == key_flags && t.total_log2 == lg)
                hit = &t;
        if (hit) {
            shape = hit->shape;
            b->last = hit->info;
        } else {
            tn_batch_tuning info{};
            if ((rc = autotune(b, table, total, pixels, P, s, shape, info))) return rc;
            b->tuned.push_back({P->max_depth, P->mc_samples, key_flags, lg, shape, info});
            b->last = info;
        }
    }
    return render_core(b->geom(), table, total, P, shape, accum, st, s, nullptr, nullptr, nullptr, 0, nullptr, 0);
}

int tn_batch_get_tuning(const tn_batch* b, tn_batch_tuning* out) {
    if (!b || !out) return set_error(TN_ERR_INVALID, "NULL argument");
    *out = b->last;
    return TN_OK;
}

}  // extern "C"
