// Wavefront transient path tracer for gfx950 (MI355X) and the C ABI declared in include/tr_api.h.
//
// Per wavefront of `wave` paths:
//   camera_kernel                 camera ray + per-path PCG32 streams       (TransientRenderer.h:130-163,
//                                                                            StratifiedSampler.h:47-89,
//                                                                            PinholeCamera.h:82-108)
//   for each bounce:
//     extend_kernel               closest hit of every queued ray           (World::first_intersection)
//     shade_kernel                free-flight correction, vertex, NEE light
//                                 sample -> shadow queue, roulette, next
//                                 direction -> next ray queue               (BidirectionalPathTracing.h:486-692)
//     shadow_kernel               occlusion of every shadow ray             (World::intersects)
//     film_kernel                 visible contributions binned into the
//                                 film's compensated FP32 (sum, comp) pairs (StreakCameraFilm.h:139-192)
// A wavefront of few paths runs camera, bounces and shadow rays in one launch (path_kernel), then film_kernel.
//
// Path state lives in HBM as structure-of-arrays float4/uint4 records in two buffers: the rays of
// bounce k are records [0, count) of buffer k & 1, and shade writes the paths that continue,
// compacted in queue order, into the other buffer, so every kernel reads and writes its records
// densely. Queue counters live in device memory so no host round trip is needed between kernels.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "tr_api.h"
#include "tr_device.h"
#include "tr_guide.h"
#include "tr_guide_host.h"
#include "tr_internal.h"
#include "tr_readback.h"

using namespace trd;

namespace {

constexpr int kTraceBlock = 128;   // traversal kernels: 128 threads, STACK ints of LDS each
constexpr int kBlock = 256;        // other kernels
constexpr int kShadeBlock = 1024;  // shade: one queue atomic per 1024 paths
// Paths per wavefront: the launches of a wavefront's last bounces hold few rays each and run at the
// length of their longest query (100-190 us on the 82k-triangle scene), so fewer, larger wavefronts are
// faster: a 67 M-path frame takes 20.7 ms in one wavefront, 22.2 in two, 24.0 in four, 27.2 in eight.
constexpr uint32_t kDefaultWave = 1u << 26;
// Shadow records a wavefront may collect before they are traced and deposited, for the same reason:
// with room for them, the shadow rays of several bounces share one shadow and one film launch. All of
// a media scanline's 16 bounces together: shadow 0.33 -> 0.15 ms, film 0.44 -> 0.23 ms per pass (1.75 ->
// 1.41 ms in all); a 67 M-path frame in wavefronts of 2^25: 24.3 ms with one bounce per launch,
// 23.3 with two, 22.6 with four, 22.1 with all eight.
constexpr uint32_t kShadowRecords = 1u << 28;
// Device memory of the two, up to 25 GB: see WaveBuffers::fit. Wavefronts of kSmallWave paths and one
// bounce (6.7 GB) are always tried, and smaller ones down to kLeastWave where memory has run out.
constexpr uint32_t kSmallWave = 1u << 25;
constexpr uint32_t kLeastWave = 1u << 18;
// Largest wavefronts whose bounces run in one launch (path_kernel) instead of two per bounce. A render of
// 2^10 paths through the two: 163 and 84 us (22 triangles), 642 and 266 (81,930 triangles), 370 and 161 (a
// medium, 16 bounces); of 2^18 paths 200 and 100, 1,074 and 586, 540 and 224. Where the line lies, in us through
// the queues and in one launch, without and with a medium (16 bounces):
//   4-wide nodes (triangles)   2^19              2^20                      2^21                      2^23
//        4 (22)                                  578, 391   1,090,   665     839,   627  1,545, 1,102  2,277, 2,016  4,525, 3,628
//       11 (58)                                  666, 461   1,170,   760     942,   752  1,638, 1,245  2,488, 2,423  4,538, 4,028
//       16 (82)                                  738, 609   1,310,   907   1,040, 1,019  1,807, 1,569  2,746, 3,285  4,954, 5,044
//       22 (90)                                  771, 686   1,403, 1,018   1,062, 1,127  1,917, 1,723  2,878, 3,752  5,366, 5,835
//      287 (1,290)                               977, 1,013 1,697, 1,334   1,286, 1,651  2,244, 2,281  3,495, 5,506  5,900, 7,816
//   18,388 (81,930)       1,381, 1,037         1,825, 1,604 2,812, 2,016   1,983, 2,717  3,269, 3,474
//   73,614 (327,690)      1,800, 1,762         2,395, 2,861 3,503, 3,346   3,400, 4,689  4,923, 5,752
// (the last with 32-bit stack entries, whose LDS leaves room for fewer wavefronts).
constexpr uint32_t kPathWave = 1u << 20;
constexpr uint32_t kPathWave32 = 1u << 19;       // with 32-bit stack entries
constexpr uint32_t kPathWaveShallow = 1u << 23;
constexpr uint32_t kShallowNodes = 11;  // 4-wide nodes of a shallow tree
constexpr uint32_t kPathSegs = 1u << 15;  // GPU wavefronts of a path launch, at most
constexpr int kPathRefill = 8;  // idle lanes that begin new paths (24: 2 % slower in a medium)
constexpr uint32_t kFetchMax = 512;  // rays per work fetch of a traversal wavefront (upper bound)
constexpr uint32_t kTraceRaysPerThread = 8;   // lower bound on a full wavefront's rays per traversal thread
constexpr uint32_t kTraceMinPerCu = 4;        // traversal blocks per CU below which that bound yields

// Rays per work fetch: large enough that same-address fetch atomics stay rare, small enough that
// every wavefront of the grid still gets several fetches when the queue is short.
__device__ __forceinline__ uint32_t fetch_chunk(uint32_t count)
{
    uint32_t waves = gridDim.x * (blockDim.x >> 6);
    uint32_t c = count / (waves * 4u);
    c = c < 64u ? 64u : (c > kFetchMax ? kFetchMax : c);
    return c & ~63u;
}
constexpr float kPi = 3.14159265358979323846f;
constexpr float kInvPi = 0.318309886183790671538f;
constexpr float kInv4Pi = 0.0795774715459476678844f;  // .25 * M_1_PI (IsotropicPhaseFunction.h:43-47)
constexpr float kSigmaVisibility = 1e-5f;             // _SIGMA_VISIBILITY_ (bunnykiller.h:76-78)
// material bits of a scene triangle: index | two-sided material | smooth (per-corner normals)
constexpr int32_t kMatTwoSided = 1 << 30;
constexpr int32_t kMatSmooth = 1 << 29;
constexpr int32_t kMatIndex = kMatSmooth - 1;
// multibounce films: bits of a shadow record's tag that hold its layer (at most 32 layers)
constexpr uint32_t kMaxLayersTagBits = kMbLayerTagBits;

// counters[] layout (uint32 words): queue lengths and per-launch statistics in the first 256 bytes,
// then kParts partitions of 256 bytes each holding the work-fetch cursors of the persistent
// traversal grids and the visible-contribution count. Atomics to one address are serialised, and
// the wavefronts of a launch fetch work all the time: blocks are dealt to the 8 XCDs in turn, so
// partition blockIdx.x % kParts takes the fetches of one XCD's blocks on its own 256-byte line.
constexpr uint32_t kParts = 8;
constexpr uint32_t kPartBase = 64;
constexpr uint32_t kPartWords = 64;
// Queue lengths come in two 64-bit pairs, one per record buffer k: (rays of buffer k, shadow
// records: those carried over from earlier bounces and those made from the paths of the other
// buffer), so that shade appends to both of its output queues with one atomic.
enum {
    C_Q0 = 0,                                            // pairs: words 2k (rays), 2k + 1 (shadow rays)
    C_STAT_EXT = 4, C_STAT_SHADOW = 6,                   // 64-bit statistics
    C_WORDS = kPartBase + kParts * kPartWords
};
__host__ __device__ constexpr uint32_t qword(int k) { return uint32_t(2 * k); }
__host__ __device__ constexpr uint32_t shword(int k) { return uint32_t(2 * k + 1); }
enum { P_FETCH_EXT = 0, P_FETCH_SHADOW = 1, P_STAT_CONTRIB = 2, P_STAT_EXT = 4, P_STAT_SHADOW = 6 };  // words of a partition (P_STAT_*: 64-bit)
__host__ __device__ constexpr uint32_t part_word(uint32_t part, uint32_t w) { return kPartBase + part * kPartWords + w; }

struct SceneDev {
    const float4* nodes;       // binary BVH (4 float4 per node)
    const float4* nodes4;      // quantized 4-wide BVH (4 x 16 bytes per node, Bvh4DevNode)
    const float4* tris;        // rotated triangle records in slot order (4 float4 each, see TriRot)
    const float4* tri_normal;  // per slot: geometric normal xyz, w = material bits (int)
    const float4* tri_vn;      // smooth triangles: p0, e1, e2, n0, n1, n2 (null if none)
    const float4* mats;        // Kd xyz, w = mean albedo used by the roulette
    const LightHost* lights;
    int32_t n_lights;
    int32_t has_medium;
    float3 sigma_s, sigma_t;
    float lambda;              // mean extinction (HomogeneousMedium.h:50-51)
    float medium_albedo;       // mean of sigma_s / sigma_t
    float plane_bound;         // largest |plane| of the quantized BVH (qbvh_plane_bound)
};

struct RenderDev {
    // film
    float* film;               // compensated sums [rows][W][T][3]: sum ...
    float* film_comp;          // ... and the rounding errors of its additions (film_add3)
    int32_t W, H, T, row0, spp, spp2, n_inc;
    float exposure, offset, total_time, inv_inc;
    int32_t unwarp, max_bounces;
    // camera
    float3 cpos, nv, uv, vv;
    float fd, xw2, yw2, ratio, inv_spp;
    uint64_t seed;
    // MultibounceStreakFilm: `layers` bounce films of layer_stride bins each (0 = plain film)
    int32_t layers;
    uint32_t layer_stride;
    float* steady;             // [rows][W][3] every sample, any time (multibounce films) ...
    float* steady_comp;        // ... and its compensation
    float* layer_w;            // [layers][rows][W] camera samples with samples of each layer
    uint32_t* cs_bits;         // per camera sample of the wavefront: layers that received samples
    // Transient sampling mode (-time-sampling): free-flight rate 4 / (T * exposure); 0 = steady state
    float ts_lambda;
    int32_t time_sampling;
    uint64_t pid0;             // path id of the job's first path (row0 * W * spp2 * n_inc)
};

struct WaveDev {
    // path records of the current ([cur]) and the next ([cur ^ 1]) bounce. The camera kernel writes
    // the direction alone (and the job of batched renders): every camera ray starts at the camera
    // with unit throughput at time 0 and its streams at their seeds, so the first bounce makes the
    // rest from the path's index. All paths of a wavefront are at the same level. A path id follows
    // from the index and the light stream's state from its number of draws (pcg_at): 64 bytes per
    // continuing path instead of 80, 16 instead of 48 for a camera ray (33.5 M camera rays 253 ->
    // 179 us, shading of the 67 M-path frame 4.64 -> 4.32 ms, of the media scanline 0.59 -> 0.55 ms).
    float4* ray_o[2]; // origin xyz, w = sampled free-flight distance of this segment (inf without medium)
    float4* ray_d[2]; // direction xyz, w = the path's index in its wavefront (uint bits)
    float4* thr[2];   // throughput xyz (with the pending BSDF/phase weight and roulette), w = time
    uint4* st[2];     // x = film pixel, y = light-stream draws so far | job << 16, z/w = path-stream PCG32 state
    float* uw[2];     // unwarp distance (renders with camera unwarp only)
    float2* hit;      // per record of the current bounce: x = distance, y = triangle slot (int bits) or -1
    float4* sh_o;     // light point xyz, w = distance
    float4* sh_d;     // direction xyz, w = film element index (uint bits)
    float4* sh_c;     // contribution rgb, w = film pixel (uint bits)
    uint8_t* sh_vis;  // 1 if the shadow ray is unoccluded
    uint32_t* sh_tag; // guided renders: training record of the contribution (or ~0)
    uint32_t* sh_job; // batched renders: job of each shadow record
    // path launches: GPU wavefront w runs seg_paths paths, from w * seg_paths on, and their shadow records are
    // w * seg_cap + j for j below seg_n[w] (seg_cap = 0: the records are one queue, whose length is a counter)
    uint32_t* seg_n;
    uint32_t seg_cap, seg_paths;
    struct WaveCtl* ctl;
    uint32_t* counters;
    float3 cpos;      // single-job renders: camera position (batched renders: their job's R.cpos)
};

// One render job of a batched launch: its scene, film/camera set-up and first global path index.
struct JobDev {
    SceneDev S;
    RenderDev R;
    uint64_t path_begin;
};

// Paths of the current wavefront: [base, base + n) of the launch's global path range. Kept in
// device memory so that the bounce loop of a wavefront can be replayed from a captured graph.
struct WaveCtl {
    uint64_t base;
    uint32_t n;
    uint32_t pad;
};

// (the first wavefront of a render also clears the counters)
__global__ void __launch_bounds__(kBlock) set_wave_kernel(WaveCtl* ctl, uint64_t base, uint32_t n, uint32_t* counters)
{
    if (threadIdx.x == 0) {
        ctl->base = base;
        ctl->n = n;
        ctl->pad = 0u;
    }
    if (base == 0)
        for (uint32_t k = threadIdx.x; k < C_WORDS; k += kBlock) counters[k] = 0u;
}
// the counters of a finished render, to pinned host memory
__global__ void __launch_bounds__(kBlock) read_counters_kernel(const uint32_t* __restrict__ counters, uint32_t* __restrict__ out)
{
    for (uint32_t k = threadIdx.x; k < C_WORDS; k += kBlock) out[k] = counters[k];
}

__device__ __forceinline__ uint64_t u64(uint32_t lo, uint32_t hi) { return uint64_t(lo) | (uint64_t(hi) << 32); }

// Free-flight distance -log(eps) / lambda (BidirectionalPathTracing.h:258-259, float log): the
// log is taken in double and rounded, which gives the correctly rounded float log that host libms
// return, so that a path's distances match the host's bit for bit in all but rare cases.
__device__ __forceinline__ float free_flight(float eps, float lambda)
{
    return -float(log(double(eps))) / lambda;
}

// o + d * t rounded as two operations (no fused multiply-add), as the reference computes vertex
// positions (Ray::get_position): the time-angular sampler's geometry is ill-conditioned near
// backward scattering, so positions must match the host's to the last bit there.
__device__ __forceinline__ f3 point_on_ray(f3 o, f3 d, float t)
{
#pragma clang fp contract(off)
    return mk(o.x + d.x * t, o.y + d.y * t, o.z + d.z * t);
}

// the last job whose first path is <= the global path index
__device__ __forceinline__ uint32_t job_of(const JobDev* __restrict__ jobs, uint32_t n_jobs, uint64_t gidx)
{
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1u) {
        uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].path_begin <= gidx) lo = mid;
        else hi = mid;
    }
    return lo;
}

// direction of the camera ray of a job's path (fewer than 2^32: 32-bit index arithmetic) and its film pixel
__device__ __forceinline__ f3 camera_ray(const RenderDev& R, uint32_t pid_local, uint32_t& pix_local)
{
    uint32_t cs_local = pid_local / uint32_t(R.n_inc);
    pix_local = cs_local / uint32_t(R.spp2);   // film pixel (row relative)
    uint32_t sub = cs_local - pix_local * uint32_t(R.spp2);
    uint32_t rowl = pix_local / uint32_t(R.W);
    uint32_t xr = pix_local - rowl * uint32_t(R.W);
    uint32_t y = rowl + uint32_t(R.row0);
    uint32_t sy = sub / uint32_t(R.spp);
    uint32_t sx = sub - sy * uint32_t(R.spp);
    uint64_t cs = (uint64_t(y) * uint64_t(R.W) + xr) * uint64_t(R.spp2) + sub;

    // StratifiedSampler::get_next_sample: jittered position clamped inside the pixel
    uint64_t cinc = pcg_inc((1ull << 62) | cs);
    uint64_t cst = pcg_seed(R.seed, (1ull << 62) | cs);
    float jx = pcg_float(cst, cinc), jy = pcg_float(cst, cinc);
    float px = fminf(float(xr) + (float(sx) + jx) * R.inv_spp, __uint_as_float(__float_as_uint(float(xr + 1)) - 1u));
    float py = fminf(float(y) + (float(sy) + jy) * R.inv_spp, __uint_as_float(__float_as_uint(float(y + 1)) - 1u));
    // Film::window_coords2image_coords + PinholeCamera::get_ray_direction
    float ic0 = (px - R.xw2) / float(R.W);
    float ic1 = (py - R.yw2) / float(R.H) / R.ratio;
    f3 nv = mk(R.nv.x, R.nv.y, R.nv.z), uv = mk(R.uv.x, R.uv.y, R.uv.z), vv = mk(R.vv.x, R.vv.y, R.vv.z);
    f3 dir = nv * R.fd + uv * (2.0f * ic0) - vv * (2.0f * ic1);
    return normalize(normalize(dir));  // get_ray_direction normalises, Ray3D normalises again
}

// ---------------------------------------------------------------------------------------------
// camera: one thread per path of the wavefront
template <bool BATCH>
__global__ void __launch_bounds__(kBlock) camera_kernel(SceneDev S0, RenderDev R0, const JobDev* __restrict__ jobs,
                                                        uint32_t n_jobs, WaveDev Wv)
{
    const WaveCtl ctl = *Wv.ctl;
    const uint32_t n = ctl.n;
    uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot == 0) Wv.counters[C_Q0] = n;
    if (slot < kParts) Wv.counters[part_word(slot, P_FETCH_EXT)] = 0;
    if (slot >= n) return;
    const uint64_t gidx = ctl.base + slot;
    const uint32_t jid = BATCH ? job_of(jobs, n_jobs, gidx) : 0u;
    const uint32_t pid_local = BATCH ? uint32_t(gidx - jobs[jid].path_begin) : uint32_t(gidx);
    uint32_t pix_local;
    const f3 dir = camera_ray(BATCH ? jobs[jid].R : R0, pid_local, pix_local);
    Wv.ray_d[0][slot] = make_float4(dir.x, dir.y, dir.z, __uint_as_float(slot));
    if constexpr (BATCH) Wv.st[0][slot] = make_uint4(pix_local, jid << 16, 0u, 0u);
}

// ---------------------------------------------------------------------------------------------
// Traversal variants: the binary BVH, or the 4-wide BVH with 32-bit, 16-bit or keyed 16-bit stack
// entries (trd::kStack*). Any-hit queries of a keyed launch use the 16-bit format.
enum { kTravBinary = 0, kTravWide = 1, kTravWide16 = 2, kTravWideKeyed = 3 };

// LDS words per thread of a traversal block for a stack of STACK entries
template <int TRAV, int STACK>
constexpr int stack_words() { return TRAV == kTravWide16 ? (STACK + 1) / 2 : STACK; }

// one query to its end (public queries, whose tnear may be any number unless POS, and the binary BVH)
template <bool ANY, int TRAV, bool POS = false>
__device__ __forceinline__ int32_t trace_scene(const SceneDev& S, const RayPre& r, float tnear, float& tfar,
                                               uint32_t* stack)
{
    static_assert(TRAV != kTravWideKeyed, "keyed entries need a positive tnear");
    if constexpr (TRAV == kTravBinary)
        return trace<ANY>(S.nodes, S.tris, r, tnear, tfar, reinterpret_cast<int32_t*>(stack) + threadIdx.x, kTraceBlock);
    else
        return trace4<ANY, TRAV == kTravWide ? kStack32 : kStack16, POS>(S.nodes4, S.tris, r, tnear, tfar, stack,
                                                                           threadIdx.x, kTraceBlock);
}

template <int TRAV>
constexpr int stack_kind() { return TRAV == kTravWide ? kStack32 : TRAV == kTravWide16 ? kStack16 : kStackKeyed; }

// Per-lane ray refill for the persistent 4-wide traversal kernels: a lane whose query is complete
// takes the next ray at once instead of waiting for the wavefront's slowest ray. The wavefront
// claims `chunk` queue entries at a time (its static share first, then through its partition's
// fetch cursor) and hands them to its idle lanes in lane order. Call with every lane of the
// wavefront; `rec` is the queue entry of the lane's query, kIdle if it has none.
constexpr uint32_t kIdle = 0xFFFFFFFFu;
// lanes of `mask` below this one
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}
// idle lanes that trigger a refill (unless the whole wavefront is idle): closest-hit and any-hit launches
// (with camera rays in their own packet kernel, 16 and 32 for either were 0.2-0.7 % slower than 24)
constexpr int kRefillMinExtend = 24;
constexpr int kRefillMinShadow = 24;
// Share of its even split of the queue that each wavefront takes without an atomic, in quarters
// (0: one fetch chunk). Larger static shares measured slower on the 82k-triangle scene, whose rays'
// costs vary across the image, and faster on the 22-triangle media scene, whose launches the
// fetch atomics dominated before the partitioned cursors.
constexpr uint32_t kStaticQuarters = 0;

struct RayRefill {
    uint32_t pos = 0, end = 0;  // the wavefront's claimed range of queue entries (uniform)
    uint32_t dyn_base = 0;      // first queue entry handed out through the fetch cursors
    uint32_t parts = 1, part = 0;
    bool drained = false;       // the queue has no entries left for this wavefront (uniform)

    // Every wavefront starts on its own contiguous static share of the queue (entries
    // [wave * share, (wave + 1) * share), at least one chunk) without an atomic. The entries after
    // all static shares are dealt in chunks, in queue order, through per-partition cursors: chunk
    // g = k * parts + p is the k-th fetch of partition p = blockIdx.x % parts, so the partitions'
    // wavefronts work through interleaved chunks (every partition sees the same mix of cheap and
    // costly rays) while their fetch atomics go to `parts` different lines. A launch with no
    // entries beyond the static shares takes no atomic at all (the last bounces of a render, whose
    // few rays otherwise waited on one failing fetch per wavefront of the grid). Handing chunks out
    // in queue order keeps the wavefronts on neighbouring rays (and so on the same part of the BVH
    // in cache).
    __device__ __forceinline__ RayRefill(uint32_t count, uint32_t chunk)
    {
        const uint32_t waves = gridDim.x * (blockDim.x >> 6);
        const uint32_t wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
        uint32_t share = (count / waves) * kStaticQuarters / 4u;
        share = share < chunk ? chunk : share - share % chunk;
        const uint64_t first = uint64_t(wave) * share, all = uint64_t(waves) * share;
        pos = first < count ? uint32_t(first) : count;
        end = first + share < count ? uint32_t(first + share) : count;
        dyn_base = all < count ? uint32_t(all) : count;
        parts = gridDim.x < kParts ? gridDim.x : kParts;
        part = blockIdx.x % parts;
    }

    // Assigns queue entries to idle lanes (their `rec`) and begins their queries with `start(i)`.
    // `cursor` is the partition word (P_FETCH_EXT / P_FETCH_SHADOW) of the launch's queue.
    template <int kRefillMin = kRefillMinExtend, class Start>
    __device__ __forceinline__ void run(uint32_t count, uint32_t chunk, uint32_t* counters, uint32_t cursor,
                                        uint32_t& rec, Start start)
    {
        uint64_t idle = __ballot(rec == kIdle);
        // refill in bulk: ray set-up runs once for many idle lanes instead of once per finished ray
        // (24 idle lanes measured best on the 82k-triangle scene: 1-2 % faster than 16 or 32, 4 % than 48,
        // and 13 % faster than refilling each lane at once)
        if (drained || (__popcll(idle) < kRefillMin && idle != ~0ull)) return;
        uint32_t take = kIdle;
        do {
            if (pos >= end) {
                if (dyn_base >= count) {  // nothing beyond the static shares
                    drained = true;
                    break;
                }
                uint32_t k = 0;
                if (__lane_id() == 0) k = atomicAdd(counters + part_word(part, cursor), 1u);
                k = uint32_t(__builtin_amdgcn_readfirstlane(int(k)));
                const uint64_t b = uint64_t(dyn_base) + (uint64_t(k) * parts + part) * chunk;
                if (b >= count) {
                    drained = true;
                    break;
                }
                pos = uint32_t(b);
                end = uint32_t(min(b + chunk, uint64_t(count)));
            }
            const uint32_t avail = end - pos;
            const uint32_t rank = lanes_below(idle);
            if (rec == kIdle && take == kIdle && rank < avail) take = pos + rank;
            pos += min(uint32_t(__popcll(idle)), avail);
            idle = __ballot(rec == kIdle && take == kIdle);
        } while (idle);
        if (take != kIdle) {
            rec = take;
            start(take);
        }
    }
};

// ---------------------------------------------------------------------------------------------
// extend: closest hit for each queued ray (7 wavefronts per SIMD: the batched variant's per-lane
// scene pointers fit the 72-VGPR budget without spills)
template <int TRAV, int STACK, bool BATCH>
__global__ void __launch_bounds__(kTraceBlock, 7) extend_kernel(SceneDev S0, const JobDev* __restrict__ jobs, WaveDev Wv,
                                                             int cur_first)
{
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const int cur = cur_first & 1;
    const bool first = (cur_first & 2) != 0;  // camera rays: the origin is the camera's
    const bool carry = (cur_first & 4) != 0;  // earlier bounces' shadow records are still in the queue
    const uint32_t count = Wv.counters[qword(cur)];
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid == 0) {
        Wv.counters[qword(cur ^ 1)] = 0;
        Wv.counters[shword(cur ^ 1)] = carry ? Wv.counters[shword(cur)] : 0u;
        atomicAdd(reinterpret_cast<unsigned long long*>(Wv.counters + C_STAT_EXT), (unsigned long long)count);
    }
    if (gid < kParts) Wv.counters[part_word(gid, P_FETCH_SHADOW)] = 0;
    const uint32_t chunk = fetch_chunk(count);
    if constexpr (TRAV != kTravBinary) {
        // persistent grid with per-lane refill: every lane steps its own query one node at a time
        RayRefill rf(count, chunk);
        uint32_t rec = kIdle;
        RayPre r;
        Trav4 st;
        const float4 *nodes = S0.nodes4, *tris = S0.tris;
        for (;;) {
            rf.run(count, chunk, Wv.counters, P_FETCH_EXT, rec, [&](uint32_t i) {
                const float4 d = Wv.ray_d[cur][i];
                float3 c = Wv.cpos;
                float pb = S0.plane_bound;
                if constexpr (BATCH) {
                    const JobDev& J = jobs[Wv.st[cur][i].y >> 16];
                    nodes = J.S.nodes4;
                    tris = J.S.tris;
                    c = J.R.cpos;
                    pb = J.S.plane_bound;
                }
                f3 o = mk(c.x, c.y, c.z);
                // (in registers: otherwise the compiler selects between two addresses and uses flat loads)
                asm("" : "+v"(o.x), "+v"(o.y), "+v"(o.z));
                if (!first) o = mk(Wv.ray_o[cur][i]);
                r = ray_pre(o, mk(d), pb);
                trav4_begin(st, __int_as_float(0x7f800000), threadIdx.x);
            });
            if (__ballot(rec != kIdle) == 0ull) break;  // the queue is drained and every query complete
            if (rec != kIdle && trace4_step<false, stack_kind<TRAV>(), true>(nodes, tris, r, kSigmaVisibility, st, stack,
                                                                             threadIdx.x, kTraceBlock)) {
                Wv.hit[rec] = make_float2(st.hit >= 0 ? st.tfar : -1.0f, __int_as_float(st.hit));
                rec = kIdle;
            }
        }
    } else {
        // persistent grid: each wavefront fetches `chunk` queue entries at a time until the queue
        // is drained (one fetch atomic per `chunk` rays)
        const uint32_t lane = __lane_id();
        for (;;) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(Wv.counters + part_word(0, P_FETCH_EXT), chunk);
            base = __shfl(base, 0);
            if (base >= count) break;
            for (uint32_t j = 0; j < chunk; j += 64) {
                const uint32_t i = base + j + lane;
                if (i < count) {
                    const float4 d = Wv.ray_d[cur][i];
                    const uint32_t jid = BATCH ? Wv.st[cur][i].y >> 16 : 0u;
                    const SceneDev& S = BATCH ? jobs[jid].S : S0;
                    const float3 c = BATCH ? jobs[jid].R.cpos : Wv.cpos;
                    const float4 o = first ? make_float4(c.x, c.y, c.z, 0.0f) : Wv.ray_o[cur][i];
                    RayPre r = ray_pre(mk(o), mk(d), S.plane_bound);
                    float tfar = __int_as_float(0x7f800000);
                    int32_t tri = trace_scene<false, TRAV>(S, r, kSigmaVisibility, tfar, stack);
                    Wv.hit[i] = make_float2(tri >= 0 ? tfar : -1.0f, __int_as_float(tri));
                }
            }
        }
    }
}

// extend for the camera rays of single-job renders (the first bounce): the queue holds them in path
// order, so a wavefront's 64 consecutive entries are samples of one pixel, traced as one packet
// (trace4_packet); the lanes finish together and the refill hands them the next 64 entries. The
// hits are those of extend_kernel (the flag TR_RENDER_NO_CAMERA_PACKETS selects it instead).
template <int TRAV, int STACK>
__global__ void __launch_bounds__(kTraceBlock, 7) extend_camera_kernel(SceneDev S0, WaveDev Wv, int cur)
{
    static_assert(TRAV == kTravWide || TRAV == kTravWide16 || TRAV == kTravWideKeyed, "4-wide stacks");
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const uint32_t count = Wv.counters[qword(cur)];
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid == 0) {
        Wv.counters[qword(cur ^ 1)] = 0;
        Wv.counters[shword(cur ^ 1)] = 0;
        atomicAdd(reinterpret_cast<unsigned long long*>(Wv.counters + C_STAT_EXT), (unsigned long long)count);
    }
    if (gid < kParts) Wv.counters[part_word(gid, P_FETCH_SHADOW)] = 0;
    const uint32_t chunk = fetch_chunk(count);
    RayRefill rf(count, chunk);
    uint32_t rec = kIdle;
    RayPre r;
    const int col = int(threadIdx.x & ~63u);
    const f3 cam = mk(Wv.cpos.x, Wv.cpos.y, Wv.cpos.z);
    for (;;) {
        rf.run(count, chunk, Wv.counters, P_FETCH_EXT, rec,
               [&](uint32_t i) { r = ray_pre(cam, mk(Wv.ray_d[cur][i]), S0.plane_bound); });
        if (__ballot(rec != kIdle) == 0ull) break;  // the queue is drained
        float tfar = __int_as_float(0x7f800000);
        int32_t hit = -1;
        trace4_packet<stack_kind<TRAV>()>(S0.nodes4, S0.tris, r, kSigmaVisibility, rec != kIdle, tfar, hit, stack, col,
                                          kTraceBlock);
        if (rec != kIdle) {
            Wv.hit[rec] = make_float2(hit >= 0 ? tfar : -1.0f, __int_as_float(hit));
            rec = kIdle;
        }
    }
}

// Lambertian cosine-weighted direction in the reference's shading frame
// (Sampling.h:131-143, Intersection.h:167-178, Lambertian.h:107-122).
__device__ __forceinline__ f3 sample_lambert(f3 n, float e1, float e2, float* cos_sampled)
{
    float phi = 2.0f * kPi * e1;
    float ct = sqrtf(e2);
    float st = sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
    float sp, cp;
    sincosf(phi, &sp, &cp);
    f3 l = mk(cp * st, ct, sp * st);
    f3 aux = (fabsf(n.x) > fabsf(n.z)) ? mk(-n.y, n.x, n.z) : mk(0.0f, -n.z, n.y);
    f3 tv = normalize(aux);
    f3 tu = cross(n, tv);
    *cos_sampled = ct;
    return normalize(tu * l.x + n * l.y + tv * l.z);
}

// Cosine-weighted direction in an orthonormal frame around n (Duff et al. 2017); the density is
// exactly cos/pi, which one-sample MIS with the guiding mixture needs.
__device__ __forceinline__ f3 sample_lambert_onb(f3 n, float e1, float e2, float* cos_sampled)
{
    float phi = 2.0f * kPi * e1;
    float ct = sqrtf(e2);
    float st = sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
    float sp, cp;
    sincosf(phi, &sp, &cp);
    float sign = copysignf(1.0f, n.z);
    float a = -1.0f / (sign + n.z);
    float b = n.x * n.y * a;
    f3 t = mk(1.0f + sign * n.x * n.x * a, sign * b, -sign * n.x);
    f3 bt = mk(b, sign + n.y * n.y * a, -n.y);
    *cos_sampled = ct;
    return normalize(t * (cp * st) + bt * (sp * st) + n * ct);
}

// Interpolated shading normal of a smooth triangle at point p (per-corner normals n0, n1, n2 with
// the barycentrics of p), not renormalised, as the reference uses it (World.h:589-598,
// Triangle.h:155-159).
__device__ __forceinline__ f3 smooth_normal(const float4* V, f3 p)
{
    f3 p0 = mk(V[0]), e1 = mk(V[1]), e2 = mk(V[2]), q = p - p0;
    float d00 = dot(e1, e1), d01 = dot(e1, e2), d11 = dot(e2, e2), d20 = dot(q, e1), d21 = dot(q, e2);
    float inv = 1.0f / (d00 * d11 - d01 * d01);
    float u = (d11 * d20 - d01 * d21) * inv, v = (d00 * d21 - d01 * d20) * inv;
    return mk(V[3]) * (1.0f - u - v) + mk(V[4]) * u + mk(V[5]) * v;
}

// tVectorN::transform_matrix_to(from = (0,1,0), to) applied to v (VectorN.h:429-523): the
// rotation taking +y onto `to`, built from `to` as given (the time-angular sampler passes an
// unnormalised vector, as the reference does), result normalised.
__device__ __forceinline__ f3 rotate_from_y(f3 v, f3 wi)
{
    f3 from = mk(0.0f, 1.0f, 0.0f);
    f3 vx = cross(from, wi);
    float e = wi.y;
    float f = fabsf(e);
    float m[3][3];
    if (double(f) > 1.0 - double(1.e-4f)) {
        f3 x = mk(1.0f, 0.0f, 0.0f);  // smallest |component| of (0,1,0) with the reference's tie order
        f3 u = x - from, w = x - wi;
        float c1 = 2.0f / dot(u, u), c2 = 2.0f / dot(w, w), c3 = c1 * c2 * dot(u, w);
        float ua[3] = {u.x, u.y, u.z}, wa[3] = {w.x, w.y, w.z};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < 3; ++j) m[i][j] = -c1 * ua[i] * ua[j] - c2 * wa[i] * wa[j] + c3 * wa[i] * ua[j];
            m[i][i] += 1.0f;
        }
    } else {
        float h = 1.0f / (1.0f + e);
        float hvx = h * vx.x, hvz = h * vx.z;
        float hvxy = hvx * vx.y, hvxz = hvx * vx.z, hvyz = hvz * vx.y;
        m[0][0] = e + hvx * vx.x;
        m[0][1] = hvxy - vx.z;
        m[0][2] = hvxz + vx.y;
        m[1][0] = hvxy + vx.z;
        m[1][1] = e + h * vx.y * vx.y;
        m[1][2] = hvyz - vx.x;
        m[2][0] = hvxz - vx.y;
        m[2][1] = hvyz + vx.x;
        m[2][2] = e + hvz * vx.z;
    }
    f3 s = mk(m[0][0] * v.x + m[0][1] * v.y + m[0][2] * v.z, m[1][0] * v.x + m[1][1] * v.y + m[1][2] * v.z,
              m[2][0] * v.x + m[2][1] * v.y + m[2][2] * v.z);
    return normalize(s);
}

// Isotropic phase-function direction: uniform sphere rotated so that +y maps onto wi
// (Sampling.h:80-94, IsotropicPhaseFunction.h:54-60); the new Ray normalises it again.
__device__ __forceinline__ f3 sample_isotropic(f3 wi, float e1, float e2)
{
    float phi = 2.0f * kPi * e1;
    float ct = 1.0f - 2.0f * e2;
    float st = sqrtf(fmaxf(0.0f, 1.0f - ct * ct));
    float sp, cp;
    sincosf(phi, &sp, &cp);
    return normalize(rotate_from_y(mk(cp * st, ct, sp * st), wi));
}

// Time-angular direction sampling at a medium vertex (AngularSampling::ShortestTime,
// BidirectionalPathTracing.h:357-398 with Probability::TimeAngular, SamplingTechniques.h:170-250;
// eta = 1, c = 1/time_of_flight(1) = 1): the angle theta to the direction of the light point `l`
// is drawn so that a free flight of r followed by the straight line to the light arrives
// uniformly in the time window [ta, tb] (clipped to what the geometry allows), ta being the
// straight-line arrival time. The caller first checks time_angular_window (no draw): when the window
// left after this flight is shorter than one exposure it samples the phase function. Returns false
// when the density falls below 1e-5 (the caller then samples the phase function with two more
// draws). pdf is per (theta, phi), as the reference uses it.
__device__ __forceinline__ bool time_angular_window(float modl, float time, float r, float tb, float exposure)
{
#pragma clang fp contract(off)
    const float ta = modl * 1.0f + time;
    return !((tb - (ta + r * 1.0f)) < exposure);
}

__device__ __forceinline__ bool sample_time_angular(f3 l, float modl, float time, float r, float tb, float e_theta,
                                                    float e_phi, f3* dir, float* pdf)
{
#pragma clang fp contract(off)
    const float ta = modl * 1.0f + time;
    // set_temporal_boundaries with ec = 1
    float t_a = r > modl ? fmaxf(ta, 2.0f * r - modl) : fmaxf(ta, modl);
    float t_b = fminf(tb, 2.0f * r + modl);
    float t = e_theta * (t_b - t_a) + t_a;
    float cos_t = float((double(modl * modl) + 2.0 * double(t) * double(r) - double(t * t)) /
                        (2.0 * double(r) * double(modl)));
    cos_t = fmaxf(-1.0f, fminf(cos_t, 1.0f));
    const float theta = float(acos(double(cos_t)));  // correctly rounded, as the host's acosf
    const float phi = float(2.0 * 3.14159265358979323846 * double(e_phi));
    float sp, cp, st, ct;
    sincosf(phi, &sp, &cp);
    sincosf(theta, &st, &ct);
    *dir = normalize(rotate_from_y(mk(cp * st, ct, sp * st), l));  // the new Ray normalises
    const double den = sqrt(double(r * r + modl * modl) - 2.0 * double(r) * double(modl) * double(ct));
    const float dtdtheta = float(double(modl * r * st) / den);
    *pdf = float(double(dtdtheta / (t_b - t_a)) / (2.0 * 3.14159265358979323846));
    return !(double(*pdf) < 1e-5);
}

// The light point a path aims at in the Transient sampling mode: the reference draws it per
// incoming sample with World::sample_light + LightSource::sample(ls, pdf)
// (BidirectionalPathTracing.h:1115-1118; PointLightSource.h:173-183, RectangularAreaLightSource.h:
// 250-271); here it comes from the path's own stream seq = 3 * 2^61 | path id.
__device__ __forceinline__ f3 light_target(const SceneDev& S, uint64_t seed, uint64_t pid)
{
#pragma clang fp contract(off)
    const uint64_t seq = (3ull << 61) | pid;
    uint64_t tinc = pcg_inc(seq), tst = pcg_seed(seed, seq);
    float u = pcg_float(tst, tinc);
    int li = min(int(u * float(S.n_lights)), S.n_lights - 1);
    const LightHost& L = S.lights[li];
    f3 p = mk(L.pos[0], L.pos[1], L.pos[2]);
    if (int(L.I[3]) != kLightPoint) {
        float a = pcg_float(tst, tinc), b = pcg_float(tst, tinc);
        p = mk((p.x + L.left[0] * a) + L.up[0] * b, (p.y + L.left[1] * a) + L.up[1] * b,
               (p.z + L.left[2] * a) + L.up[2] * b);
    }
    return p;
}

// A path's vertex: what sampling its next direction needs.
struct Vertex {
    f3 f, pos, n;   // throughput up to here, position, shading normal
    bool medium_event, two_sided;
    bool want;      // the path goes on
    int32_t mat;
    float pi, time, nsampled;  // roulette probability, time of arrival, next free flight
};
// Its connection to a light, if it has one (`emit`): a shadow record.
struct Connection {
    float4 o, d, c;
    uint32_t tag;
    bool emit;
};

__device__ __forceinline__ float flight_rate(const SceneDev& S, const RenderDev& R)
{
    return R.time_sampling ? R.ts_lambda : S.lambda;  // NextEventSampling::Time / MeanFreePath
}

// The vertex at the end of the ray (o, d), whose closest hit is `h`: the free flight's correction, the
// connection to a light and the decision to go on. thr: throughput and time of the path before it,
// sampled: its free flight, pst / pinc: the path's stream, nee: light-stream draws so far. LAYERS: the
// film may be a multibounce one.
template <bool LAYERS>
__device__ __forceinline__ void path_vertex(const SceneDev& S, const RenderDev& R, uint32_t level, uint32_t slot, uint64_t pid,
                                            uint64_t pinc, uint32_t pix, float2 h, f3 o, f3 d, float4 thr, float sampled,
                                            float uw, uint64_t& pst, uint32_t& nee, Vertex& vx, Connection& sh)
{
    const int32_t tri = __float_as_int(h.y);
    const float lam = flight_rate(S, R);
    f3 &f = vx.f, &pos = vx.pos, &n = vx.n;
    bool &medium_event = vx.medium_event, &two_sided = vx.two_sided;
    int32_t& mat = vx.mat;
    float &pi = vx.pi, &time = vx.time, &nsampled = vx.nsampled;
    // correct_next_event_distance (BidirectionalPathTracing.h:275-307)
    float dist, pd = 1.0f;
    bool alive = true;
    if (!S.has_medium) {
        alive = tri >= 0;
        dist = h.x;
    } else if (tri >= 0 && h.x < sampled) {
        dist = h.x;
        pd = expf(-dist * lam);
    } else {
        dist = sampled;
        medium_event = true;
        pd = expf(-dist * lam) * lam;
    }
    if (alive) {
        f = mk(thr);
        if (S.has_medium) {
            f = mk(f.x * expf(-dist * S.sigma_t.x), f.y * expf(-dist * S.sigma_t.y), f.z * expf(-dist * S.sigma_t.z));
            f = f * (1.0f / pd);
        }
        time = thr.w + dist;
        pos = point_on_ray(o, d, dist);
        n = mk(0.0f, 0.0f, 0.0f);
        if (!medium_event) {
            float4 nn = S.tri_normal[tri];
            n = mk(nn);
            mat = __float_as_int(nn.w);
            two_sided = (mat & kMatTwoSided) != 0;
            if (mat & kMatSmooth) n = smooth_normal(S.tri_vn + 6 * size_t(tri), pos);
            mat &= kMatIndex;
        }
        // the light stream (sequence 2 pid + 1) after `nee` draws
        const uint64_t ninc = pcg_inc(2 * pid + 1);
        uint64_t nst = pcg_at(R.seed, ninc, nee);
        // ---- next-event estimation at this vertex (connect_paths :976-1045,
        //      connect_vertex_with_light :650-692)
        if (int(level) + 1 <= R.max_bounces && time <= R.total_time) {
            float u = pcg_float(nst, ninc);
            ++nee;
            int li = min(int(u * float(S.n_lights)), S.n_lights - 1);
            const LightHost& L = S.lights[li];
            int type = int(L.I[3]);
            f3 lp, ldir;
            float ldist, pl2 = 1.0f;
            f3 irr;
            bool ok = true;
            if (type == kLightPoint) {
                lp = mk(L.pos[0], L.pos[1], L.pos[2]);
                f3 v = pos - lp;
                float d2 = dot(v, v);
                ldist = sqrtf(d2);
                ldir = v * (1.0f / ldist);
                float att = 1.0f / d2;
                irr = mk(L.I[0] * att, L.I[1] * att, L.I[2] * att);
            } else {
                float uu = pcg_float(nst, ninc), vv = pcg_float(nst, ninc);
                nee += 2;
                lp = mk(L.pos[0], L.pos[1], L.pos[2]) + mk(L.left[0], L.left[1], L.left[2]) * uu +
                     mk(L.up[0], L.up[1], L.up[2]) * vv;
                f3 v = pos - lp;
                ldist = sqrtf(dot(v, v));
                ldir = v * (1.0f / ldist);
                float dl = dot(ldir, mk(L.normal[0], L.normal[1], L.normal[2]));
                ok = dl > 0.0f;
                float a = L.I[0] * dl / (ldist * ldist);
                irr = mk(a, a, a);
                pl2 = L.normal[3];
                ldir = normalize(ldir);
            }
            if (ok) {
                f3 fe;
                if (medium_event) {
                    fe = mk(S.sigma_s.x, S.sigma_s.y, S.sigma_s.z) * kInv4Pi;
                } else {
                    float4 kd = S.mats[mat];
                    // dot_clamped, or dot_abs for a two-sided material (Path.h:188-193)
                    float cd = -dot(ldir, n);
                    float c = two_sided ? fabsf(cd) : fmaxf(cd, 0.0f);
                    fe = mk(kd.x, kd.y, kd.z) * (kInvPi * c);
                }
                f3 att = mk(1.0f, 1.0f, 1.0f);
                if (S.has_medium)
                    att = mk(expf(-S.sigma_t.x * ldist), expf(-S.sigma_t.y * ldist), expf(-S.sigma_t.z * ldist));
                float scale = R.inv_inc / (pl2 / float(S.n_lights));
                f3 val = mul(mul(f, fe), mul(irr, att)) * scale;
                float ts = ldist + time;
                float cam_time = R.unwarp ? ts - uw : ts;
                float sensor = (cam_time - R.offset) / R.exposure;
                bool finite = isfinite(val.x) && isfinite(val.y) && isfinite(val.z);
                bool nonzero = val.x != 0.0f || val.y != 0.0f || val.z != 0.0f;
                const bool in_window = sensor >= 0.0f && sensor < float(R.T);
                if (LAYERS && R.layers > 0) {
                    // multibounce film: every connected sample counts for its layer's
                    // weight and the steady image, in the time window or not
                    // (MultibounceStreakCameraFilm.h:137-157, Film.h:263-283)
                    const uint32_t layer = min(level, uint32_t(R.layers - 1));
                    uint32_t fidx = 0xFFFFFFFFu;
                    if (in_window)
                        fidx = layer * R.layer_stride + pix * uint32_t(R.T) +
                               min(uint32_t(floorf(sensor)), uint32_t(R.T - 1));
                    if (!finite) val = mk(0.0f, 0.0f, 0.0f);  // TransientRenderer.h:167-171
                    sh.emit = true;
                    sh.o = make_float4(lp.x, lp.y, lp.z, ldist);
                    sh.d = make_float4(ldir.x, ldir.y, ldir.z, __uint_as_float(fidx));
                    sh.c = make_float4(val.x, val.y, val.z, __uint_as_float(pix));
                    sh.tag = ((slot / uint32_t(R.n_inc)) << kMaxLayersTagBits) | layer;
                } else if (in_window && finite && nonzero) {
                    uint32_t bin = min(uint32_t(floorf(sensor)), uint32_t(R.T - 1));
                    uint32_t fidx = pix * uint32_t(R.T) + bin;
                    sh.emit = true;
                    sh.o = make_float4(lp.x, lp.y, lp.z, ldist);
                    sh.d = make_float4(ldir.x, ldir.y, ldir.z, __uint_as_float(fidx));
                    sh.c = make_float4(val.x, val.y, val.z, __uint_as_float(pix));
                }
            }
        }
        // ---- termination: later vertices cannot contribute past the bounce cap or the
        //      film window; otherwise Russian roulette on the mean albedo, or in the
        //      Transient mode the film's time length alone (TotalTime) (:447-481)
        if (int(level) + 1 < R.max_bounces && time <= R.total_time) {
            float albedo = medium_event ? S.medium_albedo : S.mats[mat].w;
            float eps = R.time_sampling ? 0.0f : pcg_float(pst, pinc);
            if (!(eps > albedo)) {
                pi = R.time_sampling ? 1.0f : albedo;
                nsampled = __int_as_float(0x7f800000);
                if (S.has_medium) nsampled = free_flight(pcg_float(pst, pinc), lam);
                vx.want = true;
            }
        }
    }
}

// The direction that an unguided path goes on in, its BSDF (with the cosine) or phase function and its
// density. onb: orthonormal shading frame.
__device__ __forceinline__ void path_direction(const SceneDev& S, const RenderDev& R, bool onb, uint64_t pid, uint64_t pinc, f3 d,
                                               const Vertex& vx, uint64_t& pst, f3& nd, f3& fa, float& pa)
{
    const f3 pos = vx.pos, n = vx.n;
    const float time = vx.time, nsampled = vx.nsampled;
    if (vx.medium_event) {
        bool timed = false;
        if (R.time_sampling) {
            const f3 tg = light_target(S, R.seed, pid);
            f3 l;
            float modl;
            {
#pragma clang fp contract(off)
                l = mk(tg.x - pos.x, tg.y - pos.y, tg.z - pos.z);
                modl = sqrtf((l.x * l.x + l.y * l.y) + l.z * l.z);
            }
            if (time_angular_window(modl, time, nsampled, R.total_time, R.exposure)) {
                float e1 = pcg_float(pst, pinc), e2 = pcg_float(pst, pinc);
                timed = sample_time_angular(l, modl, time, nsampled, R.total_time, e1, e2, &nd, &pa);
            }
        }
        if (!timed) {
            float e1 = pcg_float(pst, pinc), e2 = pcg_float(pst, pinc);
            nd = sample_isotropic(d, e1, e2);
            pa = kInv4Pi;
        }
        fa = mk(S.sigma_s.x, S.sigma_s.y, S.sigma_s.z) * kInv4Pi;
    } else {
        (void)pcg_float(pst, pinc);  // BSDF pick of a single-BSDF UberMaterial
        float e1 = pcg_float(pst, pinc), e2 = pcg_float(pst, pinc);
        float ct;
        nd = onb ? sample_lambert_onb(n, e1, e2, &ct) : sample_lambert(n, e1, e2, &ct);
        // a two-sided material hit from behind samples in its inverted frame
        // (TwoSided.h:80-88, Intersection.h:180-185)
        if (vx.two_sided && dot(d, n) > 0.0f) nd = nd * -1.0f;
        float4 kd = S.mats[vx.mat];
        fa = mk(kd.x, kd.y, kd.z) * (kInvPi * fabsf(dot(n, nd)));
        pa = ct * kInvPi;
    }
}

// ---------------------------------------------------------------------------------------------
// shade: one thread per queued path whose ray has just been traced
// Shading modes: the reference's shading frame (default), an orthonormal frame (same estimator
// without the frame quirk), and guided sampling (orthonormal frame + one-sample MIS of the BSDF /
// phase function with the network's vMF mixture).
enum { kShadeRef = 0, kShadeOnb = 1, kShadeGuided = 2 };
constexpr int kShadeBlockGuided = 256;  // 4 wavefronts x 10 KiB of LDS for the network

__device__ __forceinline__ float mean3(f3 v) { return (v.x + v.y + v.z) * (1.0f / 3.0f); }

template <int MODE, bool BATCH>
__global__ void __launch_bounds__(MODE == kShadeGuided ? kShadeBlockGuided : kShadeBlock)
    shade_kernel(SceneDev S0, RenderDev R0, const JobDev* __restrict__ jobs, WaveDev Wv, int cur_level, trg::GuideView G)
{
    static_assert(!(BATCH && MODE == kShadeGuided), "guided renders take one job");
    constexpr bool GUIDED = MODE == kShadeGuided;
    __shared__ uint32_t scan[kShadeBlock / 64 + 2];
    __shared__ float glds[GUIDED ? (kShadeBlockGuided / 64) * 64 * trg::kRow : 1];
    __shared__ uint4 gfrag[GUIDED ? trg::kFwdFrags * 64 : 1];
    const int cur = cur_level & 1;
    const uint32_t level = uint32_t(cur_level >> 1);  // of every path of the launch
    const uint64_t wave_base = Wv.ctl->base;
    const uint32_t count = Wv.counters[qword(cur)];
    if (blockIdx.x == 0 && threadIdx.x < kParts) Wv.counters[part_word(threadIdx.x, P_FETCH_EXT)] = 0;  // for the next extend
    if (blockIdx.x * blockDim.x >= count) return;  // no paths for this block (the last bounces' launches)
    if constexpr (GUIDED) {
        // the network's weight fragments stay in LDS for the whole block (38 KiB; with the rows of
        // four wavefronts 80.3 KB, two blocks per CU); the biases are read from global memory
        for (uint32_t k = threadIdx.x; k < uint32_t(trg::kFwdFrags * 64); k += blockDim.x) gfrag[k] = G.frag[k];
        __syncthreads();
    }
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x; base < count; base += stride) {
        const uint32_t i = base + threadIdx.x;
        bool live = i < count;
        const float4 d4 = live ? Wv.ray_d[cur][i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const uint32_t slot = __float_as_uint(d4.w);  // the path's index in its wavefront
        uint4 st = {};
        if (live && (BATCH || level > 0)) st = Wv.st[cur][i];
        const uint32_t jid = BATCH ? st.y >> 16 : 0u;
        const SceneDev& S = BATCH ? jobs[jid].S : S0;
        const RenderDev& R = BATCH ? jobs[jid].R : R0;
        bool cont = false;
        float4 n_o = {}, n_d = {}, n_thr = {};
        uint32_t tag = 0xFFFFFFFFu;  // guided: training record of this vertex
        Vertex vx = {};              // a vertex that goes on to sample a direction
        vx.mat = -1;
        vx.pi = 1.0f;
        Connection sh = {};
        sh.tag = 0xFFFFFFFFu;
        f3 d = {};
        uint64_t pst = 0, pinc = 0, pid = 0;
        uint32_t nee = 0;    // light-stream draws
        float uw = 0.0f;     // unwarp distance
        if (live) {
            const float2 h = Wv.hit[i];
            const uint32_t pid_local = uint32_t(wave_base + slot - (BATCH ? jobs[jid].path_begin : 0ull));
            pid = R.pid0 + pid_local;
            pinc = pcg_inc(2 * pid);
            f3 o = mk(R.cpos.x, R.cpos.y, R.cpos.z);
            float4 thr = make_float4(1.0f, 1.0f, 1.0f, 0.0f);
            float sampled = __int_as_float(0x7f800000);
            if (level == 0) {
                // a camera ray: unit throughput, the path stream at its seed
                pst = pcg_seed(R.seed, 2 * pid);
                if (S.has_medium) sampled = free_flight(pcg_float(pst, pinc), flight_rate(S, R));
                if (!BATCH) st.x = pid_local / (uint32_t(R.n_inc) * uint32_t(R.spp2));
                if (R.unwarp) uw = __float_as_int(h.y) >= 0 ? h.x : 3.402823466e+38f;
            } else {
                const float4 o4 = Wv.ray_o[cur][i];
                o = mk(o4);
                sampled = o4.w;
                thr = Wv.thr[cur][i];
                pst = u64(st.z, st.w);
                nee = st.y & 0xFFFFu;
                if (R.unwarp) uw = Wv.uw[cur][i];
            }
            d = mk(d4);
            path_vertex<!BATCH && !GUIDED>(S, R, level, slot, pid, pinc, st.x, h, o, d, thr, sampled, uw, pst, nee, vx, sh);
            if constexpr (GUIDED) {
                if (slot % G.stride == 0u && slot / G.stride < G.train_paths) sh.tag = tag = (slot / G.stride) * G.max_levels + level;
            }
        }
        if (!vx.want) tag = 0xFFFFFFFFu;
        // ---- guided: the network's mixture for every vertex of this wavefront that samples a
        //      direction (all 64 lanes take part in the matrix-core evaluation)
        float raw[GUIDED ? trg::kRaw : 1];
        float* mine = glds + (GUIDED ? (threadIdx.x >> 6) * 64 * trg::kRow : 0);
        if constexpr (GUIDED) {
            const f3 pn = mk((vx.pos.x - G.bb_lo.x) * G.bb_inv.x, (vx.pos.y - G.bb_lo.y) * G.bb_inv.y,
                             (vx.pos.z - G.bb_lo.z) * G.bb_inv.z);
            raw[0] = pn.x, raw[1] = pn.y, raw[2] = pn.z;
            raw[3] = -d.x, raw[4] = -d.y, raw[5] = -d.z;
            raw[6] = vx.n.x, raw[7] = vx.n.y, raw[8] = vx.n.z;
            raw[9] = fminf(fmaxf(vx.time / R.total_time, 0.0f), 1.0f);
            raw[10] = vx.medium_event ? 1.0f : 0.0f;
            raw[11] = 0.0f;
            if (__ballot(vx.want) != 0ull) {
                const int lane = int(__lane_id());
                float feat[trg::kFeat];
                trg::encode_features(raw, feat);
                trg::store_feature_row(reinterpret_cast<uint32_t*>(mine) + lane * trg::kRow, feat);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                trg::mlp_forward_wave<1>(mine, gfrag, G.bias, nullptr);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
        if (vx.want) {
            const f3 f = vx.f, pos = vx.pos, n = vx.n;
            const bool medium_event = vx.medium_event, two_sided = vx.two_sided;
            const int32_t mat = vx.mat;
            const float pi = vx.pi;
            f3 nd, fa;
            float pa;
            bool ok = true;
            if constexpr (!GUIDED) {
                path_direction(S, R, MODE == kShadeOnb, pid, pinc, d, vx, pst, nd, fa, pa);
            } else {
                const float alpha = G.alpha;
                const f3 nside = (two_sided && dot(d, n) > 0.0f) ? n * -1.0f : n;  // side the path arrives on
                float usel = pcg_float(pst, pinc);
                float e1, e2;
                if (usel < alpha) {
                    e1 = pcg_float(pst, pinc), e2 = pcg_float(pst, pinc);
                    float ct;
                    nd = medium_event ? sample_isotropic(d, e1, e2) : sample_lambert_onb(nside, e1, e2, &ct);
                }
                trg::Mixture mix;
                trg::mixture_decode(mine + __lane_id() * trg::kRow, mix);
                if (!(usel < alpha)) {
                    float ul = pcg_float(pst, pinc);
                    e1 = pcg_float(pst, pinc), e2 = pcg_float(pst, pinc);
                    trg::Lobe L = trg::pick_lobe(mix, ul);
                    trg::vmf_sample(L, e1, e2, &nd.x, &nd.y, &nd.z);
                }
                float q = trg::mixture_pdf(mix, nd.x, nd.y, nd.z);
                if (medium_event) {
                    fa = mk(S.sigma_s.x, S.sigma_s.y, S.sigma_s.z) * kInv4Pi;
                    pa = alpha * kInv4Pi + (1.0f - alpha) * q;
                } else {
                    float c = dot(nside, nd);
                    ok = c > 0.0f;  // below the surface the one-sided Lambertian reflects nothing
                    float4 kd = S.mats[mat];
                    fa = mk(kd.x, kd.y, kd.z) * (kInvPi * fmaxf(c, 0.0f));
                    pa = alpha * fmaxf(c, 0.0f) * kInvPi + (1.0f - alpha) * q;
                }
                ok = ok && pa > 0.0f;
                if (ok && tag != 0xFFFFFFFFu) {
                    // training record: inputs, sampled direction and pi / throughput (the later
                    // contributions along this direction, divided by the throughput after this
                    // vertex, times BSDF x cosine / density)
                    float mf = mean3(f);
                    float4* rec = G.rec + size_t(tag) * 4;
                    rec[0] = make_float4(raw[0], raw[1], raw[2], raw[9]);
                    rec[1] = make_float4(raw[3], raw[4], raw[5], raw[10]);
                    rec[2] = make_float4(raw[6], raw[7], raw[8], mf > 0.0f ? pi / mf : 0.0f);
                    rec[3] = make_float4(nd.x, nd.y, nd.z, 0.0f);
                    G.n_rec[tag / G.max_levels] = tag % G.max_levels + 1u;
                }
            }
            if (ok) {
                f3 nf = mul(f, fa) * (1.0f / (pi * pa));
                cont = true;
                n_o = make_float4(pos.x, pos.y, pos.z, vx.nsampled);
                n_d = make_float4(nd.x, nd.y, nd.z, d4.w);
                n_thr = make_float4(nf.x, nf.y, nf.z, vx.time);
                st = make_uint4(st.x, nee | (jid << 16), uint32_t(pst), uint32_t(pst >> 32));
            }
        }
        uint32_t q_pos, sh_pos;
        block_append2(Wv.counters + qword(cur ^ 1), cont ? 1u : 0u, sh.emit ? 1u : 0u, scan, &q_pos, &sh_pos);
        if (sh.emit) {
            Wv.sh_o[sh_pos] = sh.o;
            Wv.sh_d[sh_pos] = sh.d;
            Wv.sh_c[sh_pos] = sh.c;
            if (GUIDED || (!BATCH && R.layers > 0)) Wv.sh_tag[sh_pos] = sh.tag;
            if constexpr (BATCH) Wv.sh_job[sh_pos] = jid;
        }
        if (cont) {
            Wv.ray_o[cur ^ 1][q_pos] = n_o;
            Wv.ray_d[cur ^ 1][q_pos] = n_d;
            Wv.thr[cur ^ 1][q_pos] = n_thr;
            Wv.st[cur ^ 1][q_pos] = st;
            if (R.unwarp) Wv.uw[cur ^ 1][q_pos] = uw;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// path: all bounces of a small wavefront's paths in one launch, a path per lane, and then their shadow rays,
// in place of the camera launch, an extend and a shade launch per bounce and the shadow launch. Those take
// 10-20 us each however few paths there are (a launch, and a ray's chain of node reads), and each waits for
// the longest ray of the one before it; here a GPU wavefront waits for its own rays only. It loses lanes as
// paths end, which the queues' compaction avoids, so it begins new paths in them: it takes 128 paths from 2^20 on,
// 256 from 2^21 and 512 of 2^23 (22 triangles, 2^21 paths: 796 us with 64 paths per wavefront, 627 with 256, in a
// medium 1,347 and 1,102; 2^23: 2,920 and, with 512, 2,016, in a medium 4,850 and 3,628; 20,490 triangles,
// 2^20: 1,417 and, with 128, 1,300), and large wavefronts keep the queues (kPathWave). Where there are
// fewer than two GPU wavefronts of 64 per SIMD, each takes 32 or 16 paths: fewer lanes wait for the longest
// ray and for each other's branches (1,290 triangles, 2^14 paths: 267, 227, 207 us with 64, 32, 16;
// 81,930 triangles 444, 366, 343; a medium 169, 162, 158; 22 triangles, 2^10 paths of 8 bounces: 73.4 and
// 68.5 with 64 and 16, of 4 bounces 71.3 and 67.4, of 2 57.3 and 58.9). Its shadow
// records are a segment of its own: appending each bounce's to one queue took 12 ns per atomic, 2.2 ms of a
// 2^20-path medium render that takes 0.6. Lanes and order aside, every path is computed as by the queue's
// kernels.
template <int TRAV, int STACK, bool BATCH>
__global__ void __launch_bounds__(kTraceBlock, 4) path_kernel(SceneDev S0, RenderDev R0, const JobDev* __restrict__ jobs,
                                                             uint32_t n_jobs, WaveDev Wv, bool onb)
{
    static_assert(TRAV == kTravWide || TRAV == kTravWide16, "4-wide BVH, plain stacks");
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const WaveCtl ctl = *Wv.ctl;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, rec0 = wave * Wv.seg_cap;
    const uint32_t end = min(ctl.n, (wave + 1u) * Wv.seg_paths);
    uint32_t fresh = wave * Wv.seg_paths;  // the wavefront's next path to begin
    if (fresh >= ctl.n) return;
    uint32_t traced = 0, n_rec = 0;
    bool live = false;
    uint32_t slot = 0, jid = 0, level = 0, pix = 0, nee = 0;
    uint64_t pid = 0, pst = 0;
    f3 o = {}, d = {};
    float4 thr = {};
    float sampled = 0.0f, uw = 0.0f;
    for (;;) {
        const uint64_t idle = __ballot(!live);
        if (fresh < end && (__popcll(idle) >= kPathRefill || idle == ~0ull)) {
            const uint32_t i = fresh + lanes_below(idle);
            if (!live && i < end) {
                const uint64_t gidx = ctl.base + i;
                slot = i;
                if constexpr (BATCH) jid = job_of(jobs, n_jobs, gidx);
                const SceneDev& S = BATCH ? jobs[jid].S : S0;
                const RenderDev& R = BATCH ? jobs[jid].R : R0;
                const uint32_t pid_local = BATCH ? uint32_t(gidx - jobs[jid].path_begin) : uint32_t(gidx);
                pid = R.pid0 + pid_local;
                o = mk(R.cpos.x, R.cpos.y, R.cpos.z);
                d = camera_ray(R, pid_local, pix);
                thr = make_float4(1.0f, 1.0f, 1.0f, 0.0f);
                sampled = __int_as_float(0x7f800000);
                pst = pcg_seed(R.seed, 2 * pid);
                if (S.has_medium) sampled = free_flight(pcg_float(pst, pcg_inc(2 * pid)), flight_rate(S, R));
                level = nee = 0;
                live = true;
            }
            fresh += uint32_t(__popcll(idle));
        }
        const uint64_t active = __ballot(live);
        if (active == 0ull) break;  // every path of the wavefront is done
        traced += uint32_t(__popcll(active));
        Connection sh = {};
        if (live) {
            const SceneDev& S = BATCH ? jobs[jid].S : S0;
            const RenderDev& R = BATCH ? jobs[jid].R : R0;
            const uint64_t pinc = pcg_inc(2 * pid);
            float tfar = __int_as_float(0x7f800000);
            const int32_t hit = trace4<false, stack_kind<TRAV>(), true>(S.nodes4, S.tris, ray_pre(o, d, S.plane_bound),
                                                                        kSigmaVisibility, tfar, stack, threadIdx.x, kTraceBlock);
            const float2 h = make_float2(hit >= 0 ? tfar : -1.0f, __int_as_float(hit));
            if (level == 0 && R.unwarp) uw = hit >= 0 ? tfar : 3.402823466e+38f;
            Vertex vx = {};
            vx.mat = -1;
            vx.pi = 1.0f;
            path_vertex<!BATCH>(S, R, level, slot, pid, pinc, pix, h, o, d, thr, sampled, uw, pst, nee, vx, sh);
            live = vx.want;
            if (live) {
                f3 nd, fa;
                float pa;
                path_direction(S, R, onb, pid, pinc, d, vx, pst, nd, fa, pa);
                const f3 nf = mul(vx.f, fa) * (1.0f / (vx.pi * pa));
                o = vx.pos;
                d = nd;
                sampled = vx.nsampled;
                thr = make_float4(nf.x, nf.y, nf.z, vx.time);
                ++level;
            }
        }
        const uint64_t emitted = __ballot(sh.emit);
        if (sh.emit) {
            const uint32_t at = rec0 + n_rec + lanes_below(emitted);
            Wv.sh_o[at] = sh.o;
            Wv.sh_d[at] = sh.d;
            Wv.sh_c[at] = sh.c;
            if (!BATCH && R0.layers > 0) Wv.sh_tag[at] = sh.tag;
            if constexpr (BATCH) Wv.sh_job[at] = jid;
        }
        n_rec += uint32_t(__popcll(emitted));
    }
    // the wavefront's shadow rays, handed to idle lanes as in shadow_kernel
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    uint32_t next = 0, rec = kIdle, visible = 0;
    RayPre r;
    Trav4 st;
    const float4 *nodes = S0.nodes4, *tris = S0.tris;
    for (;;) {
        const uint64_t idle = __ballot(rec == kIdle);
        if (next < n_rec && (__popcll(idle) >= kRefillMinShadow || idle == ~0ull)) {
            const uint32_t i = next + lanes_below(idle);
            if (rec == kIdle && i < n_rec) {
                rec = i;
                float pb = S0.plane_bound;
                if constexpr (BATCH) {
                    const SceneDev& J = jobs[Wv.sh_job[rec0 + i]].S;
                    nodes = J.nodes4;
                    tris = J.tris;
                    pb = J.plane_bound;
                }
                const float4 so = Wv.sh_o[rec0 + i], sd = Wv.sh_d[rec0 + i];
                r = ray_pre(mk(so), mk(sd), pb);
                trav4_begin(st, so.w - kSigmaVisibility, threadIdx.x);
            }
            next += uint32_t(__popcll(idle));
        }
        if (__ballot(rec != kIdle) == 0ull) break;  // none left
        if (rec != kIdle && trace4_step<true, stack_kind<TRAV>(), true>(nodes, tris, r, kSigmaVisibility, st, stack, threadIdx.x,
                                                                        kTraceBlock)) {
            const bool vis = st.hit < 0;
            Wv.sh_vis[rec0 + rec] = vis ? 1 : 0;
            visible += vis ? 1u : 0u;
            rec = kIdle;
        }
    }
    visible = wave_sum(visible);
    if (__lane_id() == 0) {
        Wv.seg_n[wave] = n_rec;
        uint32_t* part = Wv.counters + part_word(blockIdx.x % kParts, 0);
        if (traced) atomicAdd(reinterpret_cast<unsigned long long*>(part + P_STAT_EXT), (unsigned long long)traced);
        if (n_rec) atomicAdd(reinterpret_cast<unsigned long long*>(part + P_STAT_SHADOW), (unsigned long long)n_rec);
        if (visible) atomicAdd(reinterpret_cast<unsigned long long*>(part + P_STAT_CONTRIB), (unsigned long long)visible);
    }
}

// calls f(r, visible) for the shadow records of the launch, 64 neighbours at a time with all lanes of a
// wavefront: those of the queue `sh`, or, of path launches, those of every wavefront's segment
template <class F>
__device__ __forceinline__ void each_record(const WaveDev& Wv, int sh, F f)
{
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, waves = (gridDim.x * blockDim.x) >> 6;
    const bool queue = Wv.seg_cap == 0u;
    const uint32_t count = queue ? Wv.counters[shword(sh)] : 0u;
    const uint32_t segs = queue ? (count + 63u) / 64u : (Wv.ctl->n + Wv.seg_paths - 1u) / Wv.seg_paths;
    for (uint32_t w = wave; w < segs; w += waves) {
        const uint32_t r0 = w * (queue ? 64u : Wv.seg_cap), n = queue ? min(count - r0, 64u) : Wv.seg_n[w];
        for (uint32_t j = 0; j < n; j += 64u) {
            const uint32_t r = r0 + j + __lane_id();
            f(r, j + __lane_id() < n && Wv.sh_vis[r]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// shadow: occlusion test light -> vertex in (eps, dist - eps]; visible contributions go to the film
// (7 wavefronts per SIMD: the any-hit leaf mode's state fits 72 VGPRs without spills; at 64 VGPRs
// it spilled and ran 2 % slower)
template <int TRAV, int STACK, bool BATCH>
__global__ void __launch_bounds__(kTraceBlock, 7) shadow_kernel(SceneDev S0, const JobDev* __restrict__ jobs, WaveDev Wv,
                                                                             int sh)
{
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const uint32_t count = Wv.counters[shword(sh)];
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid == 0)
        atomicAdd(reinterpret_cast<unsigned long long*>(Wv.counters + C_STAT_SHADOW), (unsigned long long)count);
    const uint32_t lane = __lane_id();
    uint32_t visible = 0;
    const uint32_t chunk = fetch_chunk(count);
    if constexpr (TRAV != kTravBinary) {
        // persistent grid with per-lane refill (see extend_kernel)
        RayRefill rf(count, chunk);
        uint32_t rec = kIdle;
        RayPre r;
        Trav4 st;
        const float4 *nodes = S0.nodes4, *tris = S0.tris;
        for (;;) {
            rf.run<kRefillMinShadow>(count, chunk, Wv.counters, P_FETCH_SHADOW, rec, [&](uint32_t i) {
                float pb = S0.plane_bound;
                if constexpr (BATCH) {
                    const SceneDev& S = jobs[Wv.sh_job[i]].S;
                    nodes = S.nodes4;
                    tris = S.tris;
                    pb = S.plane_bound;
                }
                const float4 o = Wv.sh_o[i], d = Wv.sh_d[i];
                r = ray_pre(mk(o), mk(d), pb);
                trav4_begin(st, o.w - kSigmaVisibility, threadIdx.x);
            });
            if (__ballot(rec != kIdle) == 0ull) break;
            // any hit: a keyed launch uses the 16-bit format (its LDS holds either)
            constexpr int SK = stack_kind<TRAV>() == kStackKeyed ? kStack16 : stack_kind<TRAV>();
            if (rec != kIdle && trace4_step<true, SK, true>(nodes, tris, r, kSigmaVisibility, st, stack, threadIdx.x,
                                                            kTraceBlock)) {
                const bool vis = st.hit < 0;
                Wv.sh_vis[rec] = vis ? 1 : 0;
                visible += vis ? 1u : 0u;
                rec = kIdle;
            }
        }
    } else {
        for (;;) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(Wv.counters + part_word(0, P_FETCH_SHADOW), chunk);
            base = __shfl(base, 0);
            if (base >= count) break;
            for (uint32_t j = 0; j < chunk; j += 64) {
                const uint32_t i = base + j + lane;
                if (i < count) {
                    const SceneDev& S = BATCH ? jobs[Wv.sh_job[i]].S : S0;
                    float4 o = Wv.sh_o[i], d = Wv.sh_d[i];
                    RayPre r = ray_pre(mk(o), mk(d), S.plane_bound);
                    float tfar = o.w - kSigmaVisibility;
                    bool vis = trace_scene<true, TRAV>(S, r, kSigmaVisibility, tfar, stack) < 0;
                    Wv.sh_vis[i] = vis ? 1 : 0;
                    visible += vis ? 1u : 0u;
                }
            }
        }
    }
    visible = wave_sum(visible);
    if (lane == 0 && visible)
        atomicAdd(reinterpret_cast<unsigned long long*>(Wv.counters + part_word(blockIdx.x % kParts, P_STAT_CONTRIB)),
                  (unsigned long long)visible);
}

// ---------------------------------------------------------------------------------------------
// film accumulation with compensated sums. Every film element is a pair of FP32 accumulators
// (sum, comp). An addition of x is an atomic add that returns the old value a; the rounding error
// of the stored a + x is then recovered exactly with Knuth's TwoSum and added to comp, so after
// any number n of additions in any order sum + comp equals the exact total up to the rounding of
// the additions into comp: within (2u + O(n u^2)) sum|x| (u = 2^-24), against n u sum|x| for a plain
// FP32 running sum. The hardware atomic rounds to nearest-even like the vector ALU, which is what
// makes the recovered error exact.
__device__ __forceinline__ float two_sum_err(float a, float b, float s)
{
    // s = fl(a + b); returns (a + b) - s exactly
    const float bb = s - a;
    return (a - (s - bb)) + (b - bb);
}

// an RGB contribution into elements i, i + 1, i + 2 of the compensated pair (sum, comp) held in
// global memory: the three returning atomics are issued before the first result is awaited (one
// round trip instead of three)
__device__ __forceinline__ void film_add3(float* __restrict__ sum, float* __restrict__ comp, size_t i, float x,
                                          float y, float z)
{
    const float a0 = unsafeAtomicAdd(sum + i, x);
    const float a1 = unsafeAtomicAdd(sum + i + 1, y);
    const float a2 = unsafeAtomicAdd(sum + i + 2, z);
    const float e0 = two_sum_err(a0, x, a0 + x), e1 = two_sum_err(a1, y, a1 + y), e2 = two_sum_err(a2, z, a2 + z);
    if (e0 != 0.0f) unsafeAtomicAdd(comp + i, e0);
    if (e1 != 0.0f) unsafeAtomicAdd(comp + i + 1, e1);
    if (e2 != 0.0f) unsafeAtomicAdd(comp + i + 2, e2);
}

// a compensated partial (s, c) into the pair (sum[i], comp[i])
__device__ __forceinline__ void film_add_partial(float* __restrict__ sum, float* __restrict__ comp, size_t i, float s,
                                                 float c)
{
    if (s != 0.0f) {
        const float a = unsafeAtomicAdd(sum + i, s);
        c += two_sum_err(a, s, a + s);
    }
    if (c != 0.0f) unsafeAtomicAdd(comp + i, c);
}

// film: bins the visible contributions of this bounce into the film. A block takes ranges of
// kFilmRange consecutive shadow records; their pixels are few (paths are enumerated pixel-major
// and queue compaction keeps runs of neighbouring paths together), so each block accumulates into
// LDS histograms of up to `pix_slots` pixels x T bins x RGB and flushes each non-zero bin with one
// compensated add. A block takes kFilmRun ranges in a row, or the segments of 512 or more paths, and
// flushes at their end or when a range's pixels find no slot; the records left out then try again, and only
// those left after kFilmRounds rounds go straight to HBM (a range's records come from a few append chunks of
// the shading kernel, each holding paths of one or two pixels). Flushing after every range instead made up
// to three times as many returning atomics as bins: media scanline 164 -> 78 us, guided 366 -> 327, 67 M-path
// icosphere frame 2.20 -> 2.04 ms (runs of 1, 4, 16 ranges: 2.36, 2.04, 2.13).
// The LDS histograms hold FP64 partials (non-returning LDS atomic adds): a partial of n float
// contributions is exact to within n 2^-53 of their magnitude sum (2^-36 for the 130,000 of a group of
// 4,096 paths with 32 vertices), far inside the film's compensated FP32 bound, and is flushed as the float
// pair (hi, lo) = (float(p), float(p - hi)). The kernel waits on its loads
// and returning atomics: 1024-thread blocks (two per CU, 32 wavefronts) ran it 12-16 % faster than
// 256-thread blocks (three per CU, 12 wavefronts), and 72 KB of LDS per block (three 1024-bin
// pixels instead of two, still two blocks per CU) 10-14 % faster again.
// (StreakCameraFilm::add_samples / add_temporal_sample, StreakCameraFilm.h:139-192, 280-297)
constexpr int kFilmBlock = 1024;
constexpr uint32_t kFilmRange = 512;
constexpr uint32_t kFilmLdsBytes = 72 * 1024;  // FP64 histograms: pix_slots * T * 3 * 8 bytes (3 pixels of 1024 bins)
constexpr uint32_t kFilmMaxSlots = 8;
constexpr int kFilmRounds = 3;
constexpr uint32_t kFilmRun = 4;
constexpr uint32_t kFilmSegs = 32;  // segments of a path launch that a block takes at a time, at most
static_assert(kFilmRange <= uint32_t(kFilmBlock), "one record of a range per thread");

// Where the contributions come from: a render's queue of shadow records, that of a guided render (whose
// contributions are also credited to training records), samples that the caller made, or the shadow
// records of a path launch, of which a block takes those of 512 paths, or of 8 segments, in turn.
enum { kFilmRender = 0, kFilmGuided = 1, kFilmSamples = 2, kFilmPath = 3 };
struct SamplesDev {
    const tr_film_sample* samples;
    uint32_t n;
    const uint32_t* bad;  // index of the first sample outside the film (~0: none): then nothing is added;
                          // null if the host has checked them
};

template <int SRC>
__global__ void __launch_bounds__(kFilmBlock) film_kernel(RenderDev R, WaveDev Wv, int sh, uint32_t pix_slots,
                                                          float* contrib, SamplesDev Q)
{
    constexpr bool GUIDED = SRC == kFilmGuided;
    extern __shared__ double hist[];         // pix_slots * T * 3 partials
    __shared__ uint32_t slot_pix[kFilmMaxSlots];
    constexpr bool SEGS = SRC == kFilmPath;
    __shared__ uint32_t seg_end[SEGS ? kFilmSegs : 1];  // records of the block's segments up to and with each
    const uint32_t per_group = SEGS ? min(max(kFilmRange / Wv.seg_paths, 8u), kFilmSegs) : 1u;
    const uint32_t segs = SEGS ? (Wv.ctl->n + Wv.seg_paths - 1u) / Wv.seg_paths : 0u;
    const uint32_t count = SRC == kFilmSamples ? Q.n : SEGS ? 0u : Wv.counters[shword(sh)];
    if (SRC == kFilmSamples && Q.bad && *Q.bad != 0xFFFFFFFFu) return;
    // records that a block takes in a row: a path launch's group of segments, or kFilmRun ranges (fewer where
    // blocks would go without)
    const uint32_t run = min(max((count + kFilmRange - 1) / kFilmRange / gridDim.x, 1u), kFilmRun) * kFilmRange;
    const uint32_t groups = SEGS ? (segs + per_group - 1) / per_group : (count + run - 1) / run;
    if (blockIdx.x >= groups) return;  // no range for this block (the last bounces' launches)
    const uint32_t T = uint32_t(R.T), T3 = 3u * T, hsize = pix_slots * T3;
    const int rounds = pix_slots ? kFilmRounds : 1;
    // the histograms start at zero; each flush reads and clears only the slots that were used
    for (uint32_t i = threadIdx.x; i < hsize; i += blockDim.x) hist[i] = 0.0;
    if (threadIdx.x < kFilmMaxSlots) slot_pix[threadIdx.x] = 0xFFFFFFFFu;
    __syncthreads();
    auto flush = [&]() {
        for (uint32_t i = threadIdx.x; i < hsize; i += blockDim.x) {
            const uint32_t k = i / T3;
            if (slot_pix[k] == 0xFFFFFFFFu) continue;
            const double v = hist[i];
            if (v != 0.0) {
                const float hi = float(v), lo = float(v - double(hi));
                film_add_partial(R.film, R.film_comp, size_t(slot_pix[k]) * T3 + (i - k * T3), hi, lo);
                hist[i] = 0.0;
            }
        }
        __syncthreads();
        if (threadIdx.x < kFilmMaxSlots) slot_pix[threadIdx.x] = 0xFFFFFFFFu;
        __syncthreads();
    };
    uint32_t group = blockIdx.x, start = 0;  // the range's group of records and first record in it
    while (group < groups) {
        uint32_t total = SEGS ? 0u : min(run, count - group * run);
        if constexpr (SEGS) {
            if (start == 0) {
                if (threadIdx.x < 64) {
                    const uint32_t w = group * per_group + threadIdx.x;
                    uint32_t x = threadIdx.x < per_group && w < segs ? Wv.seg_n[w] : 0u;
                    for (uint32_t off = 1; off < kFilmSegs; off <<= 1) {
                        const uint32_t y = __shfl_up(x, off);
                        if (threadIdx.x >= off) x += y;
                    }
                    if (threadIdx.x < kFilmSegs) seg_end[threadIdx.x] = x;
                }
                __syncthreads();
            }
            total = seg_end[kFilmSegs - 1];
        }
        // this thread's record of the range, if it is a visible contribution
        const uint32_t j = start + threadIdx.x;
        const bool mine = threadIdx.x < kFilmRange && j < total;
        uint32_t r = group * run + j;
        if (SEGS && mine) {
            uint32_t k = 0;
            while (j >= seg_end[k]) ++k;
            r = (group * per_group + k) * Wv.seg_cap + j - (k ? seg_end[k - 1] : 0u);
        }
        start += kFilmRange;
        const bool last = start >= total;  // of its group
        if (last) {
            start = 0;
            group += gridDim.x;
        }
        bool pending = false;
        float4 c = {};
        uint32_t pix = 0, bin = 0;
        if constexpr (SRC == kFilmSamples) {
            if (mine) {
                const tr_film_sample q = Q.samples[r];
                const float sensor = (q.time - R.offset) / R.exposure;
                c = make_float4(q.rgb[0], q.rgb[1], q.rgb[2], 0.0f);
                pix = uint32_t(q.y - R.row0) * uint32_t(R.W) + uint32_t(q.x);
                pending = sensor < float(T) && sensor >= 0.0f;
                bin = pending ? min(uint32_t(floorf(sensor)), T - 1u) : 0u;
            }
        } else if (mine && Wv.sh_vis[r]) {
            c = Wv.sh_c[r];
            if constexpr (GUIDED) {
                // luminance of the contribution, credited to the training record of its vertex
                uint32_t tag = Wv.sh_tag[r];
                if (tag != 0xFFFFFFFFu) atomicAdd(contrib + tag, (c.x + c.y + c.z) * (1.0f / 3.0f));
            }
            pix = __float_as_uint(c.w);
            bin = __float_as_uint(Wv.sh_d[r].w) - pix * T;
            pending = true;
        }
        for (int round = 0; round < rounds; ++round) {
            if (pending) {
                // neighbouring pixels begin at different slots, so the first one tried is mostly the right one
                int slot = -1;
                uint32_t k = pix_slots ? pix % pix_slots : 0u;
                for (uint32_t t = 0; t < pix_slots; ++t) {
                    uint32_t v = *static_cast<volatile uint32_t*>(&slot_pix[k]);
                    if (v == 0xFFFFFFFFu) v = atomicCAS(&slot_pix[k], 0xFFFFFFFFu, pix);
                    if (v == 0xFFFFFFFFu || v == pix) {
                        slot = int(k);
                        break;
                    }
                    k = k + 1 == pix_slots ? 0u : k + 1;
                }
                if (slot >= 0) {
                    double* h = hist + uint32_t(slot) * T3 + bin * 3u;
                    atomicAdd(h + 0, double(c.x));
                    atomicAdd(h + 1, double(c.y));
                    atomicAdd(h + 2, double(c.z));
                    pending = false;
                } else if (round == rounds - 1) {
                    film_add3(R.film, R.film_comp, (size_t(pix) * T + bin) * 3, c.x, c.y, c.z);
                    pending = false;
                }
            }
            if (!__syncthreads_or(pending)) break;
            flush();
        }
        if (last) flush();
    }
}

// index of the first caller-made sample outside the film (of `rows` rows), before they are deposited
__global__ void samples_begin_kernel(uint32_t* bad) { *bad = 0xFFFFFFFFu; }
__global__ void __launch_bounds__(kBlock) samples_check_kernel(const tr_film_sample* __restrict__ samples, uint32_t n,
                                                               int32_t W, int32_t row0, int32_t rows, uint32_t* bad)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int2 at = *reinterpret_cast<const int2*>(samples + i);
        const int32_t row = int32_t(uint32_t(at.y) - uint32_t(row0));
        if (at.x < 0 || at.x >= W || row < 0 || row >= rows) atomicMin(bad, i);
    }
}

// multibounce films: visible connections mark their layer for the camera sample, add to the
// steady image, and (inside the time window) to their layer's film. The steady image is summed in double
// by each lane for the wavefront's current pixel (neighbouring records are mostly of one) and added once
// per pixel and wavefront: adds to one address take 12 ns each, and 64 lanes added to one pixel's sums in turn
// (168,000 paths of 2,600 pixels: this kernel 254 -> 91 us, mb_weight_kernel 56 -> 6).
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}
__global__ void __launch_bounds__(kBlock) film_mb_kernel(RenderDev R, WaveDev Wv, int sh)
{
    uint32_t at = 0xFFFFFFFFu;  // the wavefront's pixel
    double acc[3] = {0.0, 0.0, 0.0};
    auto flush = [&]() {
        if (at != 0xFFFFFFFFu) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double v = wave_sum(acc[k]);
                const float hi = float(v), lo = float(v - double(hi));
                if (__lane_id() == 0) film_add_partial(R.steady, R.steady_comp, size_t(at) * 3 + k, hi, lo);
            }
        }
        acc[0] = acc[1] = acc[2] = 0.0;
    };
    each_record(Wv, sh, [&](uint32_t r, bool visible) {
        float4 c = {};
        uint32_t pix = 0;
        if (visible) {
            c = Wv.sh_c[r];
            const uint32_t tag = Wv.sh_tag[r];
            pix = __float_as_uint(c.w);
            atomicOr(R.cs_bits + (tag >> kMaxLayersTagBits), 1u << (tag & ((1u << kMaxLayersTagBits) - 1u)));
        }
        bool pending = visible && (c.x != 0.0f || c.y != 0.0f || c.z != 0.0f);
        if (pending) {
            const uint32_t fidx = __float_as_uint(Wv.sh_d[r].w);
            if (fidx != 0xFFFFFFFFu) film_add3(R.film, R.film_comp, size_t(fidx) * 3, c.x, c.y, c.z);
        }
        for (;;) {
            const uint64_t left = __ballot(pending);
            if (left == 0ull) break;
            const uint32_t p = uint32_t(__builtin_amdgcn_readlane(int(pix), int(__builtin_ctzll(left))));
            if (p != at) {
                flush();
                at = p;
            }
            if (pending && pix == p) {
                acc[0] += double(c.x);
                acc[1] += double(c.y);
                acc[2] += double(c.z);
                pending = false;
            }
        }
    });
    flush();
}

// multibounce films, after a wavefront: each camera sample adds 1 to the weight of every layer it
// sent samples to (a bounce film only sees those camera samples), then its marks are cleared
__global__ void __launch_bounds__(kBlock) mb_weight_kernel(RenderDev R, WaveDev Wv)
{
    const WaveCtl ctl = *Wv.ctl;
    const uint32_t n_cs = ctl.n / uint32_t(R.n_inc);
    const uint32_t cs0 = uint32_t(ctl.base / uint64_t(R.n_inc));
    const uint32_t pixels = R.layer_stride / uint32_t(R.T);
    // (one add per pixel, layer and wavefront; whole numbers, so their order does not matter)
    for (uint32_t i0 = (blockIdx.x * blockDim.x + threadIdx.x) & ~63u; i0 < n_cs; i0 += gridDim.x * blockDim.x) {
        const uint32_t i = i0 + __lane_id();
        const uint32_t bits = i < n_cs ? R.cs_bits[i] : 0u;
        if (bits) R.cs_bits[i] = 0u;
        const uint32_t pix = (cs0 + i) / uint32_t(R.spp2);
        for (uint64_t left = __ballot(bits != 0u); left != 0ull;) {
            const uint32_t p = uint32_t(__builtin_amdgcn_readlane(int(pix), int(__builtin_ctzll(left))));
            const bool here = bits != 0u && pix == p;
            for (int b = 0; b < R.layers; ++b) {
                const uint32_t n = uint32_t(__popcll(__ballot(here && (bits & (1u << b)))));
                if (n && __lane_id() == 0) atomicAdd(R.layer_w + size_t(b) * pixels + p, float(n));
            }
            left &= ~__ballot(here);
        }
    }
}

// batched renders: visible contributions go straight to their job's film, one compensated add each
__global__ void __launch_bounds__(kBlock) film_batch_kernel(const JobDev* __restrict__ jobs, WaveDev Wv, int sh)
{
    each_record(Wv, sh, [&](uint32_t r, bool visible) {
        if (!visible) return;
        const RenderDev& R = jobs[Wv.sh_job[r]].R;
        float4 c = Wv.sh_c[r];
        uint32_t pix = __float_as_uint(c.w);
        uint32_t bin = __float_as_uint(Wv.sh_d[r].w) - pix * uint32_t(R.T);
        film_add3(R.film, R.film_comp, (size_t(pix) * uint32_t(R.T) + bin) * 3, c.x, c.y, c.z);
    });
}

// ---------------------------------------------------------------------------------------------
// film read-back. The weight of a pixel: one for all of them (films that only renders added to), one
// per pixel, or one per pixel of each bounce film.
struct FilmWeight {
    double same;
    const double* pixel;
    const float* layer;
    __device__ __forceinline__ double at(size_t p) const { return pixel ? pixel[p] : layer ? double(layer[p]) : same; }
};
// (sum + comp) / weight (0/0 -> 0, ImageRow::weight, Image.h:153-162) in double precision, rounded
// (StreakCameraFilm.h:369-397)
__device__ __forceinline__ void film_value(float s, float c, double w, float* o)
{
    const double v = (double(s) + double(c)) / w;
    *o = isfinite(v) ? float(v) : 0.0f;
}
// or the compensated sum itself
__device__ __forceinline__ void film_value(float s, float c, double, double* o) { *o = double(s) + double(c); }

// `n` values from element 0 of `sum` / `comp` (at bin `j0` of pixel `p0`) on, written to pinned host memory;
// bound by PCIe (50 GB/s). Four values per thread (16-byte stores); `vec`: sum and comp are 16-byte
// aligned and can be read so.
constexpr uint32_t kValuesPerBlock = 1024;
template <class Out>
__global__ void __launch_bounds__(kValuesPerBlock / 4) film_values_kernel(const float* __restrict__ sum,
                                                                          const float* __restrict__ comp, FilmWeight weight,
                                                                          size_t p0, uint32_t j0, uint32_t T3, uint32_t n,
                                                                          bool vec, Out* __restrict__ out)
{
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * 4u;
    if (i < n) {
        const uint64_t q = uint64_t(j0) + i;
        size_t p = p0 + q / T3;
        uint32_t j = uint32_t(q % T3);
        float s[4], c[4];
        if (vec && i + 4u <= n) {
            const float4 a = *reinterpret_cast<const float4*>(sum + i), b = *reinterpret_cast<const float4*>(comp + i);
            s[0] = a.x, s[1] = a.y, s[2] = a.z, s[3] = a.w;
            c[0] = b.x, c[1] = b.y, c[2] = b.z, c[3] = b.w;
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                s[k] = i + k < n ? sum[i + k] : 0.0f;
                c[k] = i + k < n ? comp[i + k] : 0.0f;
            }
        }
        double w = weight.at(p);
        struct alignas(16) Four {
            Out v[4];
        } r;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            film_value(s[k], c[k], w, &r.v[k]);
            if (++j == T3) {
                j = 0;
                ++p;
                if (k < 3 && i + k + 1 < n) w = weight.at(p);
            }
        }
        Out* o = out + i;
        if (i + 4u <= n) {
            *reinterpret_cast<Four*>(o) = r;
        } else {
            for (uint32_t k = 0; i + k < n; ++k) o[k] = r.v[k];
        }
    }
}

// the steady image (StreakCameraFilm.h:369-397): one block per pixel sums its T x RGB values
constexpr int kNormBlock = 256;
__global__ void __launch_bounds__(kNormBlock) film_steady_kernel(const float* __restrict__ sum,
                                                                const float* __restrict__ comp, FilmWeight weight,
                                                                size_t p0, uint32_t T3, float* __restrict__ steady)
{
    __shared__ double part[kNormBlock / 64][3];
    const size_t p = blockIdx.x;
    const double w = weight.at(p0 + p);
    double acc[3] = {0.0, 0.0, 0.0};
    for (uint32_t j = threadIdx.x; j < T3; j += kNormBlock) {
        const size_t i = p * T3 + j;
        double v = (double(sum[i]) + double(comp[i])) / w;
        if (!isfinite(v)) v = 0.0;
        const uint32_t k = j % 3u;
        acc[0] += k == 0 ? v : 0.0;
        acc[1] += k == 1 ? v : 0.0;
        acc[2] += k == 2 ? v : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        for (int off = 32; off > 0; off >>= 1) acc[k] += __shfl_xor(acc[k], off);
    if (__lane_id() == 0)
        for (int k = 0; k < 3; ++k) part[threadIdx.x >> 6][k] = acc[k];
    __syncthreads();
    if (threadIdx.x < 3) {
        double t = 0.0;
        for (int q = 0; q < kNormBlock / 64; ++q) t += part[q][threadIdx.x];
        steady[p * 3 + threadIdx.x] = float(t);
    }
}

// batch closest hit for the public query entry point
template <int TRAV, int STACK>
__global__ void __launch_bounds__(kTraceBlock) intersect_kernel(SceneDev S, const tr_ray* __restrict__ rays,
                                                                tr_hit* __restrict__ hits, const uint4* __restrict__ ids,
                                                                uint32_t n)
{
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        tr_ray q = rays[i];
        RayPre r = ray_pre(mk(q.org[0], q.org[1], q.org[2]), mk(q.dir[0], q.dir[1], q.dir[2]), S.plane_bound);
        float tfar = q.tfar;
        const int32_t slot = trace_scene<false, TRAV>(S, r, q.tnear, tfar, stack);
        tr_hit h;
        if (slot >= 0) {
            const uint4 id = ids[slot];
            h.t = tfar;
            h.geom_id = id.x;
            h.prim_id = id.y;
            h.tri = id.z;
        } else {
            h.t = -1.0f;
            h.geom_id = 0xFFFFFFFFu;
            h.prim_id = 0xFFFFFFFFu;
            h.tri = 0xFFFFFFFFu;
        }
        hits[i] = h;
    }
}

// any hit in (tnear, tfar] for each ray (the shadow kernel's query)
template <int TRAV, int STACK>
__global__ void __launch_bounds__(kTraceBlock) occluded_kernel(SceneDev S, const tr_ray* __restrict__ rays,
                                                               uint8_t* __restrict__ occluded, uint32_t n)
{
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        tr_ray q = rays[i];
        RayPre r = ray_pre(mk(q.org[0], q.org[1], q.org[2]), mk(q.dir[0], q.dir[1], q.dir[2]), S.plane_bound);
        float tfar = q.tfar;
        occluded[i] = trace_scene<true, TRAV>(S, r, q.tnear, tfar, stack) >= 0 ? 1 : 0;
    }
}

// Queries of host rays, read from and answered into pinned host memory by the kernel itself: no copy, no
// device buffer. A ray is words of four arrays, each at its own stride (0: the same for every ray), so
// that records and separate arrays are read alike.
struct RayArrays {
    const uint32_t *org, *dir, *tnear, *tfar;
    uint32_t so, sd, sn, sf;  // words from ray to ray
    double shorten;           // taken off tfar in double
};
struct HitArrays {
    uint32_t *t, *geom, *prim, *tri;
    uint32_t stride;
    uint8_t* occluded;
};
constexpr uint32_t kQueryRayWords = 8;  // words of a ray at most

// `per_wave` rays per wavefront: the kernel is bound by each ray's chain of node reads, and lanes wait for the
// longest of their wavefront and for each other's branches, so calls are spread over the chip: one ray per
// wavefront up to 2,048 rays, then as many as make 2,048 wavefronts, at most 16 (81,930 triangles, closest
// hits: 1,000 rays 116, 81, 65 us with 64, 8, 1 per wavefront; 16,384 rays 139, 100, 154; 262,144 rays 562
// with 8, 460 with 16). Host memory is
// read coalesced, each word once, by way of the LDS: lanes that read their own ray's words (12 or 32 bytes
// apart) fetch every line over PCIe several times. POS: tnear is positive.
template <bool ANY, int TRAV, int STACK, bool POS>
__global__ void __launch_bounds__(kTraceBlock) query_kernel(SceneDev S, RayArrays in, HitArrays out,
                                                           const uint4* __restrict__ ids, uint32_t n, uint32_t per_wave)
{
    __shared__ uint32_t stack[stack_words<TRAV, STACK>() * kTraceBlock];
    __shared__ uint32_t words[kTraceBlock * kQueryRayWords];
    const uint32_t per_block = per_wave * (kTraceBlock / 64), first = blockIdx.x * per_block;
    const uint32_t rays = min(per_block, n - first);
    // words [first * stride, (first + rays) * stride) of each array; arrays inside another's records are not copied again
    auto stage = [&](const uint32_t* a, uint32_t stride, uint32_t at) {
        for (uint32_t k = threadIdx.x; k < rays * stride; k += kTraceBlock) words[at + k] = a[size_t(first) * stride + k];
    };
    const bool records = in.so == kQueryRayWords;
    const uint32_t at_d = records ? 4u : 3u * per_block, at_n = records ? 3u : 6u * per_block, at_f = records ? 7u : 7u * per_block;
    stage(in.org, in.so, 0u);
    if (!records) {
        stage(in.dir, in.sd, at_d);
        if (in.sn) stage(in.tnear, in.sn, at_n);
        if (in.sf) stage(in.tfar, in.sf, at_f);
    }
    const float near0 = __uint_as_float(in.sn ? 0u : *in.tnear), far0 = __uint_as_float(in.sf ? 0u : *in.tfar);
    __syncthreads();
    const uint32_t j = (threadIdx.x >> 6) * per_wave + (threadIdx.x & 63u);
    if ((threadIdx.x & 63u) >= per_wave || j >= rays) return;
    const uint32_t i = first + j;
    auto word = [&](uint32_t at, uint32_t stride, uint32_t k) { return __uint_as_float(words[at + j * stride + k]); };
    const f3 o = mk(word(0, in.so, 0), word(0, in.so, 1), word(0, in.so, 2));
    const f3 d = mk(word(at_d, in.sd, 0), word(at_d, in.sd, 1), word(at_d, in.sd, 2));
    const float tnear = in.sn ? word(at_n, in.sn, 0) : near0;
    float tfar = float(double(in.sf ? word(at_f, in.sf, 0) : far0) - in.shorten);
    int32_t slot = -1;
    if (tfar > tnear)  // (nothing to hit otherwise, also where either is NaN)
        slot = trace_scene<ANY, TRAV, POS>(S, ray_pre(o, d, S.plane_bound), tnear, tfar, stack);
    if (ANY) {
        out.occluded[i] = slot >= 0 ? 1 : 0;
        return;
    }
    const uint4 id = slot >= 0 ? ids[slot] : make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u);
    const uint32_t t = __float_as_uint(slot >= 0 ? tfar : -1.0f);
    if (out.stride == 4u) {
        reinterpret_cast<uint4*>(out.t)[i] = make_uint4(t, id.x, id.y, id.z);
    } else {
        out.t[i] = t;
        out.geom[i] = id.x;
        out.prim[i] = id.y;
        out.tri[i] = id.z;
    }
}

// The traversal stack holds at most one entry per BVH level; the smallest instantiation that
// covers the scene's depth keeps LDS per block (and so occupancy) in check.
// `bound` = entries that wait on the traversal stack at most (binary: depth; 4-wide: Bvh4::stack_bound). An
// any-hit step pushes one more before it pops it, so a stack holds at least bound + 1 (tr_scene_commit refuses
// trees with bound >= kBvhStack).
// Launches kernel k on `s`; with a start event, through hipExtLaunchKernelGGL, which stamps the
// start and stop events as part of the dispatch itself instead of as marker packets around it (a
// marker pair between two launches drains the GPU: 3 % of a media-workload render timed this way).
template <class... P, class... A>
void launch_timed(void (*k)(P...), uint32_t grid, uint32_t block, hipStream_t s, hipEvent_t e0, hipEvent_t e1, A... a)
{
    if (e0) hipExtLaunchKernelGGL(k, dim3(grid), dim3(block), 0u, s, e0, e1, 0u, P(a)...);
    else k<<<grid, block, 0, s>>>(a...);
}
// (the extend / shadow dispatch macros below run inside LaunchSet, whose ev_start / ev_stop are
// the current launch's events, or null)
#define TR_STACK_DISPATCH3(T, bound, B, KERNEL, GRID, BLOCK, STREAM, ...)                                   \
    do {                                                                                                    \
        if ((bound) < 16) launch_timed(KERNEL<T, 16, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 24) launch_timed(KERNEL<T, 24, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 32) launch_timed(KERNEL<T, 32, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else launch_timed(KERNEL<T, kBvhStack, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__);      \
    } while (0)
#define TR_STACK_DISPATCH3B(T, bound, batch, KERNEL, GRID, BLOCK, STREAM, ...)                             \
    do {                                                                                                   \
        if (batch) TR_STACK_DISPATCH3(T, bound, true, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__);           \
        else TR_STACK_DISPATCH3(T, bound, false, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__);                \
    } while (0)
// extend / shadow launches: `trav` = kTrav* chosen on the host (trav_for)
#define TR_TRACE_DISPATCH(trav, bound, batch, KERNEL, GRID, BLOCK, STREAM, ...)                             \
    do {                                                                                                    \
        switch (trav) {                                                                                     \
        case kTravBinary: TR_STACK_DISPATCH3B(kTravBinary, bound, batch, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break; \
        case kTravWide: TR_STACK_DISPATCH3B(kTravWide, bound, batch, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break;     \
        case kTravWide16: TR_STACK_DISPATCH3B(kTravWide16, bound, batch, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break; \
        default: TR_STACK_DISPATCH3B(kTravWideKeyed, bound, batch, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break;       \
        }                                                                                                   \
    } while (0)
// camera-ray packets (extend_camera_kernel), timed like the other extend launches
#define TR_CAMERA_DISPATCH_T(T, bound, GRID, BLOCK, STREAM, ...)                                                      \
    do {                                                                                                             \
        if ((bound) < 16) launch_timed(extend_camera_kernel<T, 16>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 24) launch_timed(extend_camera_kernel<T, 24>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 32) launch_timed(extend_camera_kernel<T, 32>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else launch_timed(extend_camera_kernel<T, kBvhStack>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__);      \
    } while (0)
// path launches (path_kernel), timed like them
#define TR_PATH_DISPATCH_T(T, bound, B, GRID, BLOCK, STREAM, ...)                                                    \
    do {                                                                                                            \
        if ((bound) < 16) launch_timed(path_kernel<T, 16, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 24) launch_timed(path_kernel<T, 24, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else if ((bound) < 32) launch_timed(path_kernel<T, 32, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__); \
        else launch_timed(path_kernel<T, kBvhStack, B>, GRID, BLOCK, STREAM, ev_start, ev_stop, __VA_ARGS__);        \
    } while (0)
#define TR_STACK_DISPATCH_T(T, bound, KERNEL, GRID, BLOCK, STREAM, ...)                   \
    do {                                                                                   \
        if ((bound) < 16) KERNEL<T, 16><<<GRID, BLOCK, 0, STREAM>>>(__VA_ARGS__);          \
        else if ((bound) < 24) KERNEL<T, 24><<<GRID, BLOCK, 0, STREAM>>>(__VA_ARGS__);     \
        else if ((bound) < 32) KERNEL<T, 32><<<GRID, BLOCK, 0, STREAM>>>(__VA_ARGS__);     \
        else KERNEL<T, kBvhStack><<<GRID, BLOCK, 0, STREAM>>>(__VA_ARGS__);                \
    } while (0)
// public closest-hit queries: the scene's own traversal choice
#define TR_STACK_DISPATCH(trav, bound, KERNEL, GRID, BLOCK, STREAM, ...)                                  \
    do {                                                                                                  \
        switch (trav) {                                                                                   \
        case kTravBinary: TR_STACK_DISPATCH_T(kTravBinary, bound, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break; \
        case kTravWide: TR_STACK_DISPATCH_T(kTravWide, bound, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break;     \
        default: TR_STACK_DISPATCH_T(kTravWide16, bound, KERNEL, GRID, BLOCK, STREAM, __VA_ARGS__); break;          \
        }                                                                                                 \
    } while (0)

}  // namespace

// =============================================================================================
// host side

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                            \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return fail(TR_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));       \
    } while (0)

int check_device()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(TR_ERR_DEVICE, "no HIP device available");
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t p;
    HIP_TRY(hipGetDeviceProperties(&p, dev));
    if (std::strncmp(p.gcnArchName, "gfx950", 6) != 0)
        return fail(TR_ERR_DEVICE, std::string("device is ") + p.gcnArchName + ", the library is built for gfx950");
    return TR_OK;
}

bool release_idle_buffers();

template <class T>
int dev_alloc(T** p, size_t count, uint64_t* bytes = nullptr)
{
    *p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(p), count * sizeof(T));
    if (e == hipErrorOutOfMemory && release_idle_buffers()) {
        (void)hipGetLastError();  // (the next launch would report it)
        e = hipMalloc(reinterpret_cast<void**>(p), count * sizeof(T));
    }
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return fail(TR_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    if (bytes) *bytes += count * sizeof(T);
    return TR_OK;
}

template <class T>
void dev_free(T*& p)
{
    if (p) (void)hipFree(p);
    p = nullptr;
}

// Launch shape and scheduling choices of a render (the autotuner searches over these).
struct LaunchCfg {
    uint32_t wave = kDefaultWave;   // paths per wavefront
    uint32_t trace_per_cu = 24;     // persistent traversal blocks per compute unit (24: 1 % faster than 16 on 2^25-path wavefronts)
    uint32_t shade_per_cu = 2;      // shade blocks (1024 threads) per compute unit
    bool wide = true;               // 4-wide BVH
    bool graph = false;             // replay each wavefront's bounce loop from a captured hipGraph
    bool prof = false;              // per-kernel HIP events
    bool prof_extend = false;       // ... around the extend launches only
    int mode = kShadeRef;
    // 4-wide traversal stack entries: 0 = 16-bit when the BVH has at most 65,536 nodes (else
    // 32-bit); 1 = always 32-bit; 2 = keyed 16-bit for closest hits (16-bit for any hits)
    int stack_fmt = 0;
    // batches: render the jobs one after another (single-job kernels, LDS-privatised film) instead of
    // in one shared sequence of wavefronts
    bool per_job = false;
    // single-job renders: camera rays traced as per-pixel packets (extend_camera_kernel)
    bool camera_packets = true;
    bool path_launch = true;  // small wavefronts: all bounces in one launch (path_kernel)
    uint32_t group = 0;       // bounces whose shadow rays are traced together, at most (0: as the buffers hold)
};

// launch flags -> stack format
static int stack_fmt_of(uint32_t flags)
{
    if (flags & TR_RENDER_POSTPONE_LEAVES) return 2;
    return (flags & TR_RENDER_STACK32) ? 1 : (flags & TR_RENDER_STACK_KEYED) ? 2 : 0;
}
static uint32_t stack_flags_of(int fmt)
{
    return fmt == 1 ? TR_RENDER_STACK32 : fmt == 2 ? TR_RENDER_STACK_KEYED : 0u;
}

struct WaveBuffers;

// The wavefront buffers of every scene and batch: those that no render uses are given back when device
// memory runs out, and what they hold bounds what another may take (WaveBuffers::fit).
class BufferList {
public:
    static BufferList& get()
    {
        static BufferList* l = new BufferList;  // (outlives the scenes)
        return *l;
    }
    void add(WaveBuffers* b);
    void remove(WaveBuffers* b);
    void use(WaveBuffers* b, int by);
    bool release_idle();
    uint64_t others(const WaveBuffers* b);

private:
    std::mutex mutex_;
    WaveBuffers* first_ = nullptr;
};

struct WaveBuffers {
    // renders at work in these buffers, the device they are on and their bytes (changed and read under the
    // list's lock)
    int users = 0, device = 0;
    uint64_t held = 0;
    WaveBuffers *prev = nullptr, *next = nullptr;
    uint32_t cap = 0, sh_cap = 0;  // path records, shadow records
    float4 *ray_o[2] = {}, *ray_d[2] = {}, *thr[2] = {};
    uint4* st[2] = {};
    float* uw[2] = {};  // allocated by the first render with camera unwarp
    float2* hit = nullptr;
    float4 *sh_o = nullptr, *sh_d = nullptr, *sh_c = nullptr;
    uint8_t* sh_vis = nullptr;
    uint32_t* sh_tag = nullptr;  // allocated by the first guided render
    uint32_t* sh_job = nullptr;  // allocated by the first batched render
    uint32_t* seg_n = nullptr;   // shadow records per wavefront of a path launch
    WaveCtl* ctl = nullptr;
    JobDev* d_jobs = nullptr;
    // pinned host staging of the job table: the upload is asynchronous, so its source must stay
    // valid until the copy has run (every render ends with a stream synchronisation; a pageable
    // vector freed right after hipMemcpyAsync may still be read by the runtime's copy)
    JobDev* h_jobs = nullptr;
    uint32_t jobs_cap = 0;
    uint32_t* cs_bits = nullptr;  // multibounce films: layer marks per camera sample of a wavefront
    uint32_t cs_cap = 0;
    uint32_t* counters = nullptr;

    WaveBuffers() { BufferList::get().add(this); }
    ~WaveBuffers()
    {
        BufferList::get().remove(this);
        release();
    }
    WaveBuffers(const WaveBuffers&) = delete;
    WaveBuffers& operator=(const WaveBuffers&) = delete;

    void release()
    {
        for (int b = 0; b < 2; ++b) {
            dev_free(ray_o[b]); dev_free(ray_d[b]); dev_free(thr[b]); dev_free(st[b]); dev_free(uw[b]);
        }
        dev_free(hit); dev_free(sh_o); dev_free(sh_d); dev_free(sh_c); dev_free(sh_vis); dev_free(counters);
        dev_free(sh_tag); dev_free(sh_job); dev_free(seg_n); dev_free(ctl); dev_free(d_jobs); dev_free(cs_bits);
        if (h_jobs) (void)hipHostFree(h_jobs);
        h_jobs = nullptr;
        cap = 0;
        sh_cap = 0;
        jobs_cap = 0;
        cs_cap = 0;
    }
    int ensure_cs(uint32_t n)
    {
        if (n <= cs_cap) return TR_OK;
        dev_free(cs_bits);
        cs_cap = 0;
        int rc = dev_alloc(&cs_bits, n);
        if (rc) return rc;
        cs_cap = n;
        return TR_OK;
    }
    int ensure_batch(uint32_t n_jobs)
    {
        int rc;
        if (!sh_job && sh_cap && (rc = dev_alloc(&sh_job, sh_cap))) return rc;
        if (n_jobs + 1 > jobs_cap) {
            // an earlier upload from the pinned table may still be queued (a render that failed
            // before its final synchronisation): drain the device before freeing it
            if (h_jobs) {
                (void)hipDeviceSynchronize();
                (void)hipHostFree(h_jobs);
                h_jobs = nullptr;
            }
            dev_free(d_jobs);
            jobs_cap = 0;
            if ((rc = dev_alloc(&d_jobs, n_jobs + 1))) return rc;
            if (hipHostMalloc(reinterpret_cast<void**>(&h_jobs), size_t(n_jobs + 1) * sizeof(JobDev), hipHostMallocDefault) !=
                hipSuccess) {
                h_jobs = nullptr;
                dev_free(d_jobs);
                (void)hipGetLastError();
                return fail(TR_ERR_NOMEM, "hipHostMalloc: job table");
            }
            jobs_cap = n_jobs + 1;
        }
        return TR_OK;
    }
    int ensure_unwarp()
    {
        int rc;
        for (int b = 0; b < 2; ++b)
            if (!uw[b] && cap && (rc = dev_alloc(&uw[b], cap))) return rc;
        return TR_OK;
    }
    int ensure_tags()
    {
        if (sh_tag || sh_cap == 0) return TR_OK;
        return dev_alloc(&sh_tag, sh_cap);
    }
    // device bytes of n path records and n_sh shadow records (with every optional array)
    static uint64_t bytes(uint64_t n, uint64_t n_sh)
    {
        return n * (2 * (3 * sizeof(float4) + sizeof(uint4) + sizeof(float)) + sizeof(float2)) +
               n_sh * (3 * sizeof(float4) + sizeof(uint8_t) + 2 * sizeof(uint32_t));
    }
    // Makes `group` bounces per shadow launch and then `wave` (whole units of paths) smaller until their
    // buffers fit a quarter of the device memory that is free or held by this object, and with those of other
    // scenes and batches a quarter of all memory: a process with many scenes keeps a few of the large
    // shapes, and 6.7 GB for each further one (a 67 M-path frame 24.3 ms instead of 20.7).
    void fit(uint32_t& wave, uint32_t& group, uint32_t unit) const
    {
        if (wave <= cap && uint64_t(wave) * group <= sh_cap) return;
        size_t free_bytes = 0, total_bytes = 0;
        if (hipMemGetInfo(&free_bytes, &total_bytes) != hipSuccess) return;
        const uint64_t other = BufferList::get().others(this), quarter = uint64_t(total_bytes) / 4;
        const uint64_t room = std::max(bytes(kSmallWave, kSmallWave), std::min((uint64_t(free_bytes) + bytes(cap, sh_cap)) / 4,
                                                                              quarter > other ? quarter - other : 0));
        while (group > 1 && bytes(wave, uint64_t(wave) * group) > room) group = (group + 1) / 2;
        while (wave > kSmallWave && bytes(wave, wave) > room && smaller(wave, group, unit)) {}
    }
    // the next smaller shape: fewer bounces per group, then fewer paths (whole units of them)
    static bool smaller(uint32_t& wave, uint32_t& group, uint32_t unit)
    {
        if (group > 1) {
            group = (group + 1) / 2;
            return true;
        }
        if (wave / 2 < std::max(kLeastWave, unit)) return false;
        wave = wave / 2 / unit * unit;
        return true;
    }
    int ensure(uint32_t n, uint32_t n_sh)
    {
        if (n <= cap && n_sh <= sh_cap) return TR_OK;
        n = std::max(n, cap);
        n_sh = std::max(n_sh, sh_cap);
        release();
        int rc;
        for (int b = 0; b < 2; ++b)
            if ((rc = dev_alloc(&ray_o[b], n)) || (rc = dev_alloc(&ray_d[b], n)) || (rc = dev_alloc(&thr[b], n)) ||
                (rc = dev_alloc(&st[b], n))) {
                release();
                return rc;
            }
        if ((rc = dev_alloc(&hit, n)) || (rc = dev_alloc(&sh_o, n_sh)) ||
            (rc = dev_alloc(&sh_d, n_sh)) || (rc = dev_alloc(&sh_c, n_sh)) || (rc = dev_alloc(&sh_vis, n_sh)) ||
            (rc = dev_alloc(&counters, C_WORDS)) || (rc = dev_alloc(&ctl, 1)) ||
            (rc = dev_alloc(&seg_n, kPathSegs))) {
            release();
            return rc;
        }
        cap = n;
        sh_cap = n_sh;
        return TR_OK;
    }
    // everything that a render of wavefronts of `wave` paths needs
    int ensure_all(uint32_t wave, uint32_t group, bool unwarp, bool tags, uint32_t camera_samples, uint32_t jobs)
    {
        int rc = ensure(wave, wave * group);
        if (!rc && unwarp) rc = ensure_unwarp();
        if (!rc && tags) rc = ensure_tags();
        if (!rc && camera_samples) rc = ensure_cs(camera_samples);
        if (!rc && jobs) rc = ensure_batch(jobs);
        if (rc) release();
        return rc;
    }
    WaveDev view() const
    {
        WaveDev w;
        for (int b = 0; b < 2; ++b) {
            w.ray_o[b] = ray_o[b]; w.ray_d[b] = ray_d[b]; w.thr[b] = thr[b]; w.st[b] = st[b]; w.uw[b] = uw[b];
        }
        w.hit = hit;
        w.sh_o = sh_o; w.sh_d = sh_d; w.sh_c = sh_c; w.sh_vis = sh_vis; w.sh_tag = sh_tag;
        w.sh_job = sh_job; w.ctl = ctl;
        w.seg_n = seg_n;
        w.seg_cap = w.seg_paths = 0u;
        w.counters = counters;
        return w;
    }
};

void BufferList::add(WaveBuffers* b)
{
    std::lock_guard<std::mutex> lock(mutex_);
    b->next = first_;
    if (first_) first_->prev = b;
    first_ = b;
}
void BufferList::remove(WaveBuffers* b)
{
    std::lock_guard<std::mutex> lock(mutex_);
    (b->prev ? b->prev->next : first_) = b->next;
    if (b->next) b->next->prev = b->prev;
}
// a render begins (1) or ends (-1) in `b`
void BufferList::use(WaveBuffers* b, int by)
{
    int device = 0;
    (void)hipGetDevice(&device);
    std::lock_guard<std::mutex> lock(mutex_);
    b->users += by;
    b->device = device;
    b->held = WaveBuffers::bytes(b->cap, b->sh_cap);
}
// gives back the buffers on the current device that no render uses; false if there are none
bool BufferList::release_idle()
{
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return false;
    bool any = false;
    std::lock_guard<std::mutex> lock(mutex_);
    for (WaveBuffers* b = first_; b; b = b->next)
        if (b->users == 0 && b->held != 0 && b->device == device) {
            b->release();
            b->held = 0;
            any = true;
        }
    return any;
}
// bytes that all but `b` hold on the current device
uint64_t BufferList::others(const WaveBuffers* b)
{
    int device = 0;
    (void)hipGetDevice(&device);
    uint64_t sum = 0;
    std::lock_guard<std::mutex> lock(mutex_);
    for (const WaveBuffers* o = first_; o; o = o->next)
        if (o != b && o->device == device) sum += o->held;
    return sum;
}
bool release_idle_buffers() { return BufferList::get().release_idle(); }

}  // namespace

namespace tri {
int fail(int code, const std::string& msg) { return ::fail(code, msg); }
bool release_idle_buffers() { return ::release_idle_buffers(); }
int check_device() { return ::check_device(); }
int compute_units()
{
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) return 256;
    return cu;
}
}  // namespace tri

struct tr_scene_s {
    std::vector<float> tris;        // n*9
    std::vector<int32_t> tri_mat;   // material index | kMatTwoSided | kMatSmooth
    std::vector<uint32_t> tri_geom, tri_prim;
    std::vector<float> tri_vn;      // per triangle corner shading normals (9 floats), once a mesh has some
    std::vector<float> mats;        // n_mat*4
    std::vector<LightHost> lights;
    uint32_t n_geoms = 0;
    bool has_medium = false;
    float sa[3] = {0, 0, 0}, ss[3] = {0, 0, 0};
    bool committed = false;
    hipStream_t stream = nullptr;
    float4 *d_nodes = nullptr, *d_nodes4 = nullptr, *d_tris = nullptr, *d_tri_normal = nullptr, *d_mats = nullptr;
    float4* d_tri_vn = nullptr;  // smooth triangles: p0, e1, e2, n0, n1, n2 (6 float4 per triangle)
    LightHost* d_lights = nullptr;
    uint4* d_ids = nullptr;     // per triangle slot: geometry, primitive, scene triangle
    uint32_t n_nodes = 0, n_nodes4 = 0;
    int depth = 0, depth4 = 0, stack4 = 0;
    bool wide = true;   // the 4-wide BVH can be traversed (its scaled grid steps are finite; otherwise the binary one is)
    float bb_lo[3] = {0, 0, 0}, bb_hi[3] = {1, 1, 1};  // bounds of the triangles (set at commit)
    float plane_bound = 1.0f;  // largest |plane| of the quantized BVH (set at commit)
    LaunchCfg tune;     // launch shape used by renders of this scene (tr_autotune sets it)
    double build_ms = 0.0;
    uint64_t dev_bytes = 0;
    WaveBuffers wave;
    hipEvent_t ev[2 * 256] = {};
    bool ev_made = false;
    int compute_units = 256;

    void release_device()
    {
        dev_free(d_nodes); dev_free(d_nodes4); dev_free(d_tris); dev_free(d_tri_normal); dev_free(d_mats); dev_free(d_lights);
        dev_free(d_tri_vn);
        dev_free(d_ids);
        dev_bytes = 0;
    }
    SceneDev view() const
    {
        SceneDev s;
        s.nodes = d_nodes;
        s.nodes4 = d_nodes4;
        s.tris = d_tris;
        s.tri_normal = d_tri_normal;
        s.tri_vn = d_tri_vn;
        s.mats = d_mats;
        s.lights = d_lights;
        s.n_lights = int32_t(lights.size());
        s.has_medium = has_medium ? 1 : 0;
        s.sigma_s = make_float3(ss[0], ss[1], ss[2]);
        s.sigma_t = make_float3(sa[0] + ss[0], sa[1] + ss[1], sa[2] + ss[2]);
        s.lambda = (s.sigma_t.x + s.sigma_t.y + s.sigma_t.z) / 3.0f;
        s.medium_albedo = has_medium ? (ss[0] / s.sigma_t.x + ss[1] / s.sigma_t.y + ss[2] / s.sigma_t.z) / 3.0f : 0.f;
        s.plane_bound = plane_bound;
        return s;
    }
};

struct tr_film_s {
    tr_film_desc desc{};
    int rows = 0;
    int layers = 0;      // multibounce bounce films (0: one streak film)
    size_t n_elems = 0;  // max(layers, 1) * rows*W*T*3
    // one allocation, cleared as a whole: compensated sums (sum + comp = film) and, of multibounce films, the
    // layers' weights and the steady image (sums, then comps)
    float *d_sum = nullptr, *d_comp = nullptr;
    float *d_layer_w = nullptr, *d_steady = nullptr;
    size_t device_floats = 0;
    float* d_read_steady = nullptr;  // steady image on its way to the host (allocated by the first read of one)
    double* d_read_w = nullptr;      // per-pixel weights, uploaded by reads of films with caller-made samples
    tr_film_sample* d_samples = nullptr;  // caller-made samples being added, behind a 256-byte head (first bad index)
    size_t samples_cap = 0;
    std::vector<double> weight;      // rows*W
    bool same_weight = true;         // every pixel has the same weight (no caller-made samples)
    std::vector<double> added;       // weights of the samples being added, per pixel (zeros between calls)
    hipStream_t stream = nullptr;
};

extern "C" {

const char* tr_last_error(void) { return g_err.c_str(); }

int tr_device_info(char* name, int name_len, int* compute_units, uint64_t* global_mem)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(TR_ERR_DEVICE, "no HIP device available");
    hipDeviceProp_t p;
    HIP_TRY(hipGetDeviceProperties(&p, 0));
    if (name && name_len > 0) {
        std::snprintf(name, size_t(name_len), "%s (%s)", p.name, p.gcnArchName);
    }
    if (compute_units) *compute_units = p.multiProcessorCount;
    if (global_mem) *global_mem = p.totalGlobalMem;
    return TR_OK;
}

int tr_scene_create(tr_scene* out)
{
    if (!out) return fail(TR_ERR_INVALID, "tr_scene_create: null output");
    *out = nullptr;
    int rc = check_device();
    if (rc) return rc;
    tr_scene s = new (std::nothrow) tr_scene_s();
    if (!s) return fail(TR_ERR_NOMEM, "tr_scene_create: host allocation");
    if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess) {
        delete s;
        return fail(TR_ERR_DEVICE, "tr_scene_create: hipStreamCreate failed");
    }
    {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess)
            s->compute_units = p.multiProcessorCount;
    }
    *out = s;
    return TR_OK;
}

int tr_scene_destroy(tr_scene s)
{
    if (!s) return TR_OK;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    s->release_device();
    if (s->ev_made)
        for (auto& e : s->ev) (void)hipEventDestroy(e);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
    return TR_OK;
}

int tr_scene_add_mesh(tr_scene s, const float* xyz, uint32_t nv, const uint32_t* idx, uint32_t nt,
                      const tr_material* m, uint32_t* geom_id)
{
    return tr_scene_add_mesh_ex(s, xyz, nv, idx, nt, nullptr, m, 0u, geom_id);
}

int tr_scene_add_obj(tr_scene s, const char* path, const tr_material* m, uint32_t flags, uint32_t* geom_id)
{
    if (!s || !path || !m) return fail(TR_ERR_INVALID, "tr_scene_add_obj: null argument");
    tri::ObjMesh mesh;
    int rc = tri::load_obj(path, &mesh);
    if (rc) return rc;
    return tr_scene_add_mesh_ex(s, mesh.xyz.data(), uint32_t(mesh.xyz.size() / 3), mesh.idx.data(),
                                uint32_t(mesh.idx.size() / 3), mesh.has_normals ? mesh.normals.data() : nullptr, m,
                                flags, geom_id);
}

int tr_scene_add_mesh_ex(tr_scene s, const float* xyz, uint32_t nv, const uint32_t* idx, uint32_t nt,
                         const float* normals, const tr_material* m, uint32_t flags, uint32_t* geom_id)
{
    if (!s || (nt > 0 && (!xyz || !idx)) || !m) return fail(TR_ERR_INVALID, "tr_scene_add_mesh: null argument");
    if (flags & ~uint32_t(TR_MATERIAL_TWO_SIDED)) return fail(TR_ERR_INVALID, "tr_scene_add_mesh: unknown flags");
    for (uint32_t i = 0; i < 3 * nt; ++i)
        if (idx[i] >= nv) return fail(TR_ERR_INVALID, "tr_scene_add_mesh: vertex index out of range");
    for (int k = 0; k < 3; ++k)
        if (!(m->kd[k] >= 0.f && m->kd[k] <= 1.f)) return fail(TR_ERR_INVALID, "tr_scene_add_mesh: Kd outside [0,1]");
    if (s->tris.size() / 9 + nt > 0x7FFFFFFFu) return fail(TR_ERR_INVALID, "tr_scene_add_mesh: too many triangles");
    int32_t mat = int32_t(s->mats.size() / 4);
    // mean albedo used by the roulette: mean of 1 - (1 - Kd) (BidirectionalPathTracing.h:632-638)
    float alb = ((1.f - (1.f - m->kd[0])) + (1.f - (1.f - m->kd[1])) + (1.f - (1.f - m->kd[2]))) / 3.0f;
    s->mats.insert(s->mats.end(), {m->kd[0], m->kd[1], m->kd[2], alb});
    uint32_t g = s->n_geoms++;
    // material index with the two-sided flag (bit 30) and, per triangle, the smooth flag (bit 29)
    const int32_t mat_bits = mat | ((flags & TR_MATERIAL_TWO_SIDED) ? kMatTwoSided : 0);
    // corner normals: none in the scene, or those of every triangle (zeros for meshes without)
    const bool any_normals = normals || !s->tri_vn.empty();
    if (normals) s->tri_vn.resize(s->tri_mat.size() * 9, 0.f);
    for (uint32_t t = 0; t < nt; ++t) {
        for (int k = 0; k < 3; ++k) {
            const float* p = xyz + 3 * size_t(idx[3 * t + k]);
            s->tris.insert(s->tris.end(), {p[0], p[1], p[2]});
        }
        bool smooth = false;  // all-zero corner normals mean a flat triangle
        if (normals)
            for (int k = 0; k < 9; ++k) smooth = smooth || normals[9 * size_t(t) + k] != 0.f;
        s->tri_mat.push_back(smooth ? (mat_bits | kMatSmooth) : mat_bits);
        s->tri_geom.push_back(g);
        s->tri_prim.push_back(t);
        if (any_normals) {
            if (normals) s->tri_vn.insert(s->tri_vn.end(), normals + 9 * size_t(t), normals + 9 * size_t(t) + 9);
            else s->tri_vn.insert(s->tri_vn.end(), 9, 0.f);
        }
    }
    if (geom_id) *geom_id = g;
    s->committed = false;
    return TR_OK;
}

int tr_scene_add_point_light(tr_scene s, const float position[3], const float intensity[3])
{
    if (!s || !position || !intensity) return fail(TR_ERR_INVALID, "tr_scene_add_point_light: null argument");
    LightHost L{};
    std::memcpy(L.pos, position, 12);
    std::memcpy(L.I, intensity, 12);
    L.I[3] = float(kLightPoint);
    s->lights.push_back(L);
    s->committed = false;
    return TR_OK;
}

int tr_scene_add_rect_light(tr_scene s, const float corner[3], const float target[3], const float size[2],
                            float intensity)
{
    if (!s || !corner || !target || !size) return fail(TR_ERR_INVALID, "tr_scene_add_rect_light: null argument");
    if (!(size[0] > 0.f && size[1] > 0.f)) return fail(TR_ERR_INVALID, "tr_scene_add_rect_light: non-positive size");
    // RectangularAreaLightSource::setup (RectangularAreaLightSource.h:66-80)
    double n[3] = {double(target[0]) - corner[0], double(target[1]) - corner[1], double(target[2]) - corner[2]};
    float nf[3] = {float(target[0] - corner[0]), float(target[1] - corner[1]), float(target[2] - corner[2])};
    float len = std::sqrt(nf[0] * nf[0] + nf[1] * nf[1] + nf[2] * nf[2]);
    if (!(len > 0.f)) return fail(TR_ERR_INVALID, "tr_scene_add_rect_light: target equals corner");
    (void)n;
    float inv = float(1. / double(len));
    float N[3] = {nf[0] * inv, nf[1] * inv, nf[2] * inv};
    float up[3] = {0.f, 1.f, 0.f};
    if (!(std::fabs(double(N[1])) < 0.9999)) {
        up[1] = 0.f;
        up[2] = 1.f;
    }
    auto crs = [](const float* a, const float* b, float* o) {
        o[0] = a[1] * b[2] - a[2] * b[1];
        o[1] = a[2] * b[0] - a[0] * b[2];
        o[2] = a[0] * b[1] - a[1] * b[0];
    };
    float left[3], up2[3];
    crs(N, up, left);
    crs(N, left, up2);
    LightHost L{};
    std::memcpy(L.pos, corner, 12);
    for (int k = 0; k < 3; ++k) {
        L.left[k] = left[k] * size[0];
        L.up[k] = up2[k] * size[1];
        L.normal[k] = N[k];
        L.I[k] = intensity;
    }
    L.normal[3] = float(1. / double(size[0] * size[1]));
    L.I[3] = float(kLightRect);
    s->lights.push_back(L);
    s->committed = false;
    return TR_OK;
}

int tr_scene_set_medium(tr_scene s, const float sigma_a[3], const float sigma_s[3])
{
    if (!s) return fail(TR_ERR_INVALID, "tr_scene_set_medium: null scene");
    if (!sigma_a || !sigma_s) {
        s->has_medium = false;
        return TR_OK;
    }
    for (int k = 0; k < 3; ++k)
        if (!(sigma_a[k] >= 0.f && sigma_s[k] >= 0.f && sigma_a[k] + sigma_s[k] > 0.f))
            return fail(TR_ERR_INVALID, "tr_scene_set_medium: coefficients must be >= 0 with positive extinction");
    std::memcpy(s->sa, sigma_a, 12);
    std::memcpy(s->ss, sigma_s, 12);
    s->has_medium = true;
    s->committed = false;
    return TR_OK;
}

int tr_scene_commit(tr_scene s)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_scene_commit: null scene");
    uint32_t n = uint32_t(s->tri_mat.size());
    BvhBuildResult b = build_bvh(s->tris.data(), s->tri_mat.data(), n);
    if (b.depth >= kBvhStack) return fail(TR_ERR_INVALID, "tr_scene_commit: BVH deeper than the traversal stack");
    Bvh4 b4 = collapse_bvh4(b);
    if (b4.stack_bound >= kBvhStack) return fail(TR_ERR_INVALID, "tr_scene_commit: 4-wide BVH deeper than the traversal stack");
    if (b4.nodes.size() >= (size_t(1) << 29) || b.tris.size() >= (size_t(1) << 29))
        return fail(TR_ERR_INVALID, "tr_scene_commit: more than 2^29 nodes or triangles");
    const std::vector<Bvh4QNodeHost> q4 = quantize_bvh4(b4);
    const Bvh4Device dev4 = device_bvh4(q4, b.tris.size());
    // the binary BVH's leaves refer to the same triangle slots
    for (BvhNodeHost& nd : b.nodes)
        for (int side = 0; side < 2; ++side)
            if (nd.d[2 + side] > 0) nd.d[side] = int32_t(dev4.tri_slot[size_t(nd.d[side])]);
    HIP_TRY(hipStreamSynchronize(s->stream));
    s->release_device();
    // per-triangle arrays, in slot order, from the builder's copies of the triangles (whose order is close to
    // the slots': gathering the scene's own arrays instead took 2 of the 37 ms after the build of 81,930 triangles)
    const size_t nt = b.tris.size();
    std::vector<uint32_t> slot_tri(n);  // scene triangle of each slot
    std::vector<float4> normals(n > 0 ? n : 1);
    std::vector<uint4> ids(n > 0 ? n : 1);
    // rotated triangle records (TriRot): per vertex x y z x y, then the scene triangle index
    std::vector<float> trot(16 * std::max<size_t>(1, nt));
    for (uint32_t i = 0; i < n; ++i) {
        const TriHost& t = b.tris[dev4.tri_order[i]];
        // ng = normalize(cross(p2 - p0, p1 - p0)) (World.h:449)
        float e2[3] = {t.p2[0] - t.p0[0], t.p2[1] - t.p0[1], t.p2[2] - t.p0[2]};
        float e1[3] = {t.p1[0] - t.p0[0], t.p1[1] - t.p0[1], t.p1[2] - t.p0[2]};
        float c[3] = {e2[1] * e1[2] - e2[2] * e1[1], e2[2] * e1[0] - e2[0] * e1[2], e2[0] * e1[1] - e2[1] * e1[0]};
        float l = std::sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
        float inv = l > 0.f ? float(1. / double(l)) : 0.f;
        normals[i] = make_float4(c[0] * inv, c[1] * inv, c[2] * inv, t.p1[3]);  // w: material bits
        uint32_t tri;
        std::memcpy(&tri, &t.p0[3], 4);
        slot_tri[i] = tri;
        ids[i] = make_uint4(s->tri_geom[tri], s->tri_prim[tri], tri, 0u);
        const float* P[3] = {t.p0, t.p1, t.p2};
        float* o = &trot[16 * size_t(i)];
        for (int v = 0; v < 3; ++v) {
            o[5 * v + 0] = P[v][0];
            o[5 * v + 1] = P[v][1];
            o[5 * v + 2] = P[v][2];
            o[5 * v + 3] = P[v][0];
            o[5 * v + 4] = P[v][1];
        }
        o[15] = t.p0[3];  // scene triangle index bits
    }
    for (int k = 0; k < 3; ++k) {
        s->bb_lo[k] = n ? 3.4e38f : 0.0f;
        s->bb_hi[k] = n ? -3.4e38f : 1.0f;
    }
    for (size_t v = 0; v < size_t(n) * 3; ++v)
        for (int k = 0; k < 3; ++k) {
            s->bb_lo[k] = std::min(s->bb_lo[k], s->tris[3 * v + size_t(k)]);
            s->bb_hi[k] = std::max(s->bb_hi[k], s->tris[3 * v + size_t(k)]);
        }
    size_t nn = b.nodes.size(), nm = std::max<size_t>(1, s->mats.size() / 4),
           nl = std::max<size_t>(1, s->lights.size());
    int rc;
    if ((rc = dev_alloc(&s->d_nodes, 4 * nn, &s->dev_bytes)) || (rc = dev_alloc(&s->d_nodes4, 4 * q4.size(), &s->dev_bytes)) || (rc = dev_alloc(&s->d_tris, 4 * std::max<size_t>(1, nt), &s->dev_bytes)) ||
        (rc = dev_alloc(&s->d_tri_normal, normals.size(), &s->dev_bytes)) || (rc = dev_alloc(&s->d_mats, nm, &s->dev_bytes)) ||
        (rc = dev_alloc(&s->d_lights, nl, &s->dev_bytes)) || (rc = dev_alloc(&s->d_ids, ids.size(), &s->dev_bytes))) {
        s->release_device();
        return rc;
    }
    HIP_TRY(hipMemcpyAsync(s->d_nodes, b.nodes.data(), nn * sizeof(BvhNodeHost), hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_nodes4, dev4.nodes.data(), dev4.nodes.size() * sizeof(Bvh4DevNode), hipMemcpyHostToDevice, s->stream));
    if (nt) HIP_TRY(hipMemcpyAsync(s->d_tris, trot.data(), nt * 16 * sizeof(float), hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_tri_normal, normals.data(), normals.size() * sizeof(float4), hipMemcpyHostToDevice, s->stream));
    if (!s->mats.empty())
        HIP_TRY(hipMemcpyAsync(s->d_mats, s->mats.data(), s->mats.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
    if (!s->lights.empty())
        HIP_TRY(hipMemcpyAsync(s->d_lights, s->lights.data(), s->lights.size() * sizeof(LightHost), hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->d_ids, ids.data(), ids.size() * sizeof(uint4), hipMemcpyHostToDevice, s->stream));
    std::vector<float4> vn;
    if (!s->tri_vn.empty()) {
        // smooth triangles: the plane frame for barycentrics from a hit point, and corner normals
        vn.resize(size_t(n) * 6);
        for (uint32_t i = 0; i < n; ++i) {
            const float* t = &s->tris[9 * size_t(slot_tri[i])];
            const float* q = &s->tri_vn[9 * size_t(slot_tri[i])];
            vn[6 * size_t(i) + 0] = make_float4(t[0], t[1], t[2], 0.f);
            vn[6 * size_t(i) + 1] = make_float4(t[3] - t[0], t[4] - t[1], t[5] - t[2], 0.f);
            vn[6 * size_t(i) + 2] = make_float4(t[6] - t[0], t[7] - t[1], t[8] - t[2], 0.f);
            for (int k = 0; k < 3; ++k) vn[6 * size_t(i) + 3 + k] = make_float4(q[3 * k], q[3 * k + 1], q[3 * k + 2], 0.f);
        }
        if ((rc = dev_alloc(&s->d_tri_vn, vn.size(), &s->dev_bytes))) {
            s->release_device();
            return rc;
        }
        HIP_TRY(hipMemcpyAsync(s->d_tri_vn, vn.data(), vn.size() * sizeof(float4), hipMemcpyHostToDevice, s->stream));
    }
    HIP_TRY(hipStreamSynchronize(s->stream));
    s->n_nodes = uint32_t(nn);
    s->depth = b.depth;
    s->n_nodes4 = uint32_t(b4.nodes.size());
    s->depth4 = b4.depth;
    s->stack4 = b4.stack_bound;
    s->plane_bound = qbvh_plane_bound(q4);
    s->wide = dev4.scaled;
    s->build_ms = b.build_ms;
    s->committed = true;
    return TR_OK;
}

int tr_scene_info_get(tr_scene s, tr_scene_info* info)
{
    if (!s || !info) return fail(TR_ERR_INVALID, "tr_scene_info_get: null argument");
    info->n_tris = uint32_t(s->tri_mat.size());
    info->n_bvh_nodes = s->n_nodes;
    info->bvh_depth = uint32_t(s->depth);
    info->n_lights = uint32_t(s->lights.size());
    info->device_bytes = s->dev_bytes;
    info->build_ms = s->build_ms;
    return TR_OK;
}

static uint32_t trace_grid(uint32_t n)
{
    uint32_t blocks = (n + kTraceBlock - 1) / kTraceBlock;
    return std::max(1u, std::min(blocks, 256u * 40u));
}

// Persistent traversal grids: enough blocks to fill every CU (each wavefront then keeps fetching
// queue entries), never more blocks than the wavefront has rays.
static uint32_t persistent_grid(uint32_t n, int compute_units)
{
    uint32_t blocks = (n + kTraceBlock - 1) / kTraceBlock;
    return std::max(1u, std::min(blocks, uint32_t(std::max(compute_units, 1)) * 16u));
}

int tr_intersect_batch_device(tr_scene s, const tr_ray* d_rays, uint32_t n, tr_hit* d_hits, void* stream)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_intersect_batch_device: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_intersect_batch_device: scene not committed");
    if (n == 0) return TR_OK;
    if (!d_rays || !d_hits) return fail(TR_ERR_INVALID, "tr_intersect_batch_device: null buffer");
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : s->stream;
    const int trav = !s->wide ? kTravBinary : s->n_nodes4 <= 65536u ? kTravWide16 : kTravWide;
    TR_STACK_DISPATCH(trav, s->wide ? s->stack4 : s->depth, intersect_kernel, trace_grid(n), kTraceBlock, st, s->view(),
                      d_rays, d_hits, s->d_ids, n);
    HIP_TRY(hipGetLastError());
    return TR_OK;
}

}  // extern "C"

namespace {

template <bool ANY, int TRAV, bool POS>
void launch_query(int bound, uint32_t grid, hipStream_t q, const SceneDev& S, const RayArrays& in, const HitArrays& out,
                  const uint4* ids, uint32_t n, uint32_t per_wave)
{
    if (bound < 16) query_kernel<ANY, TRAV, 16, POS><<<grid, kTraceBlock, 0, q>>>(S, in, out, ids, n, per_wave);
    else if (bound < 24) query_kernel<ANY, TRAV, 24, POS><<<grid, kTraceBlock, 0, q>>>(S, in, out, ids, n, per_wave);
    else if (bound < 32) query_kernel<ANY, TRAV, 32, POS><<<grid, kTraceBlock, 0, q>>>(S, in, out, ids, n, per_wave);
    else query_kernel<ANY, TRAV, kBvhStack, POS><<<grid, kTraceBlock, 0, q>>>(S, in, out, ids, n, per_wave);
}

// Host rays of a call: records (tr_ray), or separate arrays with one or a per-ray tnear and tfar.
struct HostRays {
    const float *org, *dir, *tnear, *tfar;
    bool records, many_near, many_far;
    double shorten;
};
struct HostHits {
    tr_hit* records;
    float* t;
    uint32_t *geom, *prim, *tri;
    uint8_t* occluded;
};

// Rays of a launch. Several threads each copy a launch's rays into pinned memory, wait for it and copy the
// answers out, so that copies and launches overlap. A launch lasts as long as its longest ray, 50-80 us over
// 81,930 triangles however many rays it has: 262,144 rays took 885 us with 4 threads and launches of 8,192
// rays, 625 with 16,384, 562 with 32,768. One thread per launch, up to a call's eight chunks: with 4, 6 and 8
// threads 262,144 rays take 550, 510 and 525 us, 524,288 take 960, 900 and 885, 1,000,000 take 1.80, 1.64 and
// 1.56 ms; visibility of 1,000,000 records 1.35, 1.21 and 1.16 ms, where a copy, a kernel and a copy
// take 1.18 (up to 131,072 rays all are alike). In all, with buffers made for each call, the runtime's copies
// and records packed by the caller, 262,144 rays took 2,700 us; 1,000 took 74 and take 50.
constexpr uint32_t kQueryChunk = 32768;
constexpr uint32_t kMaxQueryThreads = trb::kSlots;
constexpr uint32_t kQueryPerWave = 16;
static_assert(kQueryChunk * (sizeof(tr_ray) + sizeof(tr_hit)) + 64 <= trb::kChunk, "a launch's rays and answers fit a chunk");

template <bool ANY>
int query_host(tr_scene s, const HostRays& in, uint32_t n, const HostHits& out, const char* who)
{
    const int trav = !s->wide ? kTravBinary : s->n_nodes4 <= 65536u ? kTravWide16 : kTravWide;
    const int bound = s->wide ? s->stack4 : s->depth;
    const bool pos = !in.records && !in.many_near && *in.tnear > 0.0f;
    uint32_t per_wave = 1;
    while (per_wave < kQueryPerWave && per_wave * 2048u < n) per_wave *= 2u;
    const SceneDev S = s->view();
    const uint32_t threads = uint32_t(std::min<uint64_t>(kMaxQueryThreads, (uint64_t(n) + kQueryChunk - 1) / kQueryChunk));
    const hipError_t e = trb::run_chunks(n, kQueryChunk, threads, [&](const trb::Chunk& chunk, size_t first, size_t m) {
        const hipStream_t q = chunk.stream;
        char* const host = chunk.host;
        // in: the rays; then, 16-byte aligned, the answers
        RayArrays r{};
        r.shorten = in.shorten;
        uint32_t* w = reinterpret_cast<uint32_t*>(host);
        auto put = [&](const float* from, size_t count) {
            uint32_t* at = w;
            std::memcpy(at, from, count * sizeof(float));
            w += count;
            return static_cast<const uint32_t*>(at);
        };
        if (in.records) {
            r.org = put(in.org + first * kQueryRayWords, m * kQueryRayWords);
            r.dir = r.tnear = r.tfar = r.org;
            r.so = r.sd = r.sn = r.sf = kQueryRayWords;
        } else {
            r.org = put(in.org + 3 * first, 3 * m);
            r.dir = put(in.dir + 3 * first, 3 * m);
            r.tnear = put(in.tnear + (in.many_near ? first : 0), in.many_near ? m : 1);
            r.tfar = put(in.tfar + (in.many_far ? first : 0), in.many_far ? m : 1);
            r.so = r.sd = 3u;
            r.sn = in.many_near ? 1u : 0u;
            r.sf = in.many_far ? 1u : 0u;
        }
        w += (4 - (w - reinterpret_cast<uint32_t*>(host)) % 4) % 4;
        HitArrays h{};
        h.occluded = reinterpret_cast<uint8_t*>(w);
        h.stride = out.records ? 4u : 1u;
        h.t = w;
        h.geom = w + m;
        h.prim = w + 2 * m;
        h.tri = w + 3 * m;
        const uint32_t per_block = per_wave * (kTraceBlock / 64), grid = uint32_t((m + per_block - 1) / per_block);
        if (trav == kTravBinary) launch_query<ANY, kTravBinary, false>(bound, grid, q, S, r, h, s->d_ids, uint32_t(m), per_wave);
        else if (!ANY && pos && trav == kTravWide16)
            launch_query<ANY, kTravWide16, !ANY>(bound, grid, q, S, r, h, s->d_ids, uint32_t(m), per_wave);
        else if (trav == kTravWide16)
            launch_query<ANY, kTravWide16, false>(bound, grid, q, S, r, h, s->d_ids, uint32_t(m), per_wave);
        else launch_query<ANY, kTravWide, false>(bound, grid, q, S, r, h, s->d_ids, uint32_t(m), per_wave);
        hipError_t err = hipGetLastError();
        if (err == hipSuccess) err = hipEventRecord(chunk.done, q);
        if (err == hipSuccess) err = hipEventSynchronize(chunk.done);
        if (err != hipSuccess) return err;
        if (ANY) {
            std::memcpy(out.occluded + first, h.occluded, m);
        } else if (out.records) {
            std::memcpy(out.records + first, h.t, m * sizeof(tr_hit));
        } else {
            std::memcpy(out.t + first, h.t, m * 4);
            std::memcpy(out.geom + first, h.geom, m * 4);
            std::memcpy(out.prim + first, h.prim, m * 4);
            std::memcpy(out.tri + first, h.tri, m * 4);
        }
        return hipSuccess;
    });
    if (e == hipErrorOutOfMemory) return fail(TR_ERR_NOMEM, std::string(who) + ": " + hipGetErrorString(e));
    if (e != hipSuccess) return fail(TR_ERR_DEVICE, std::string(who) + ": " + hipGetErrorString(e));
    return TR_OK;
}

HostRays host_records(const tr_ray* rays)
{
    const float* w = reinterpret_cast<const float*>(rays);
    return HostRays{w, w, w, w, true, true, true, 0.0};
}

}  // namespace

extern "C" {

int tr_intersect_batch(tr_scene s, const tr_ray* rays, uint32_t n, tr_hit* hits)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_intersect_batch: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_intersect_batch: scene not committed");
    if (n == 0) return TR_OK;
    if (!rays || !hits) return fail(TR_ERR_INVALID, "tr_intersect_batch: null buffer");
    return query_host<false>(s, host_records(rays), n, HostHits{hits, nullptr, nullptr, nullptr, nullptr, nullptr},
                             "tr_intersect_batch");
}

int tr_intersect_arrays(tr_scene s, const float* org, const float* dir, const float* tnear, uint32_t n_tnear, const float* tfar,
                        uint32_t n_tfar, uint32_t n, float* t, uint32_t* geom_id, uint32_t* prim_id, uint32_t* tri)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_intersect_arrays: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_intersect_arrays: scene not committed");
    if (n == 0) return TR_OK;
    if (!org || !dir || !tnear || !tfar || !t || !geom_id || !prim_id || !tri)
        return fail(TR_ERR_INVALID, "tr_intersect_arrays: null buffer");
    if ((n_tnear != 1 && n_tnear != n) || (n_tfar != 1 && n_tfar != n))
        return fail(TR_ERR_INVALID, "tr_intersect_arrays: tnear and tfar hold one value or one per ray");
    return query_host<false>(s, HostRays{org, dir, tnear, tfar, false, n_tnear > 1, n_tfar > 1, 0.0}, n,
                             HostHits{nullptr, t, geom_id, prim_id, tri, nullptr}, "tr_intersect_arrays");
}

}  // extern "C"

// ---- closest-hit queries without allocation ---------------------------------------------------
// Staging for tr_intersect_batch_noalloc: rays, then hits, of at most TR_NOALLOC_MAX_RAYS rays, in
// one static device array per GPU (held until the process ends). Host code never passes the
// array's name to a kernel or a copy: it takes the device address from hipGetSymbolAddress once
// per device and uses that.
namespace {
constexpr size_t kNoAllocRayBytes = size_t(TR_NOALLOC_MAX_RAYS) * sizeof(tr_ray);
constexpr size_t kNoAllocBytes = kNoAllocRayBytes + size_t(TR_NOALLOC_MAX_RAYS) * sizeof(tr_hit);
static_assert(kNoAllocRayBytes % 256 == 0, "hits start 256-byte aligned");
__device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// device address of this device's scratch array (looked up on the first call on each device)
int scratch_on_current_device(void** out)
{
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(TR_ERR_DEVICE, "tr_intersect_batch_noalloc: device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(TR_ERR_DEVICE, std::string("tr_intersect_batch_noalloc: hipGetSymbolAddress: ") +
                                           hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return TR_OK;
}
}  // namespace

extern "C" {

int tr_intersect_batch_noalloc(tr_scene s, const tr_ray* rays, uint32_t n, tr_hit* hits)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_intersect_batch_noalloc: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_intersect_batch_noalloc: scene not committed");
    if (n == 0) return TR_OK;
    if (!rays || !hits) return fail(TR_ERR_INVALID, "tr_intersect_batch_noalloc: null buffer");
    if (n > TR_NOALLOC_MAX_RAYS)
        return fail(TR_ERR_INVALID, "tr_intersect_batch_noalloc: " + std::to_string(n) + " rays exceed the limit of " +
                                        std::to_string(TR_NOALLOC_MAX_RAYS) + " per call");
    void* base = nullptr;
    int rc = scratch_on_current_device(&base);
    if (rc) return rc;
    tr_ray* dr = static_cast<tr_ray*>(base);
    tr_hit* dh = reinterpret_cast<tr_hit*>(static_cast<unsigned char*>(base) + kNoAllocRayBytes);
    int out = TR_OK;
    if (hipMemcpyAsync(dr, rays, size_t(n) * sizeof(tr_ray), hipMemcpyHostToDevice, s->stream) != hipSuccess)
        out = fail(TR_ERR_DEVICE, "tr_intersect_batch_noalloc: upload failed");
    if (!out) out = tr_intersect_batch_device(s, dr, n, dh, s->stream);
    if (!out && hipMemcpyAsync(hits, dh, size_t(n) * sizeof(tr_hit), hipMemcpyDeviceToHost, s->stream) != hipSuccess)
        out = fail(TR_ERR_DEVICE, "tr_intersect_batch_noalloc: download failed");
    // also on failure: the queued copies read and write the caller's buffers
    if (hipStreamSynchronize(s->stream) != hipSuccess && !out)
        out = fail(TR_ERR_DEVICE, "tr_intersect_batch_noalloc: kernel failed");
    return out;
}

int tr_occluded_batch_device(tr_scene s, const tr_ray* d_rays, uint32_t n, uint8_t* d_occ, void* stream)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_occluded_batch_device: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_occluded_batch_device: scene not committed");
    if (n == 0) return TR_OK;
    if (!d_rays || !d_occ) return fail(TR_ERR_INVALID, "tr_occluded_batch_device: null buffer");
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : s->stream;
    const int trav = !s->wide ? kTravBinary : s->n_nodes4 <= 65536u ? kTravWide16 : kTravWide;
    TR_STACK_DISPATCH(trav, s->wide ? s->stack4 : s->depth, occluded_kernel, trace_grid(n), kTraceBlock, st, s->view(),
                      d_rays, d_occ, n);
    HIP_TRY(hipGetLastError());
    return TR_OK;
}

int tr_occluded_batch(tr_scene s, const tr_ray* rays, uint32_t n, uint8_t* occluded)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_occluded_batch: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_occluded_batch: scene not committed");
    if (n == 0) return TR_OK;
    if (!rays || !occluded) return fail(TR_ERR_INVALID, "tr_occluded_batch: null buffer");
    return query_host<true>(s, host_records(rays), n, HostHits{nullptr, nullptr, nullptr, nullptr, nullptr, occluded},
                            "tr_occluded_batch");
}

int tr_occluded_arrays(tr_scene s, const float* org, const float* dir, const float* tnear, uint32_t n_tnear, const float* tfar,
                       uint32_t n_tfar, double shorten, uint32_t n, uint8_t* occluded)
{
    if (!s) return fail(TR_ERR_INVALID, "tr_occluded_arrays: null scene");
    if (!s->committed) return fail(TR_ERR_STATE, "tr_occluded_arrays: scene not committed");
    if (n == 0) return TR_OK;
    if (!org || !dir || !tnear || !tfar || !occluded) return fail(TR_ERR_INVALID, "tr_occluded_arrays: null buffer");
    if ((n_tnear != 1 && n_tnear != n) || (n_tfar != 1 && n_tfar != n))
        return fail(TR_ERR_INVALID, "tr_occluded_arrays: tnear and tfar hold one value or one per ray");
    return query_host<true>(s, HostRays{org, dir, tnear, tfar, false, n_tnear > 1, n_tfar > 1, shorten}, n,
                            HostHits{nullptr, nullptr, nullptr, nullptr, nullptr, occluded}, "tr_occluded_arrays");
}

int tr_film_create(tr_film* out, const tr_film_desc* d)
{
    if (!out || !d) return fail(TR_ERR_INVALID, "tr_film_create: null argument");
    *out = nullptr;
    if (d->width <= 0 || d->height <= 0 || d->time_bins <= 0 || !(d->exposure > 0.f) ||
        d->scanline >= d->height || d->scanline < -1)
        return fail(TR_ERR_INVALID, "tr_film_create: bad film geometry");
    if (d->bounce_layers < 0 || d->bounce_layers > 32)
        return fail(TR_ERR_INVALID, "tr_film_create: bounce_layers must be in [0, 32]");
    int rc = check_device();
    if (rc) return rc;
    int rows = d->scanline >= 0 ? 1 : d->height;
    const int layers = d->bounce_layers;
    size_t n = size_t(std::max(layers, 1)) * size_t(rows) * size_t(d->width) * size_t(d->time_bins) * 3;
    if (n / 3 >= 0xFFFFFFFFull) return fail(TR_ERR_INVALID, "tr_film_create: film larger than 2^32 bins");
    tr_film f = new (std::nothrow) tr_film_s();
    if (!f) return fail(TR_ERR_NOMEM, "tr_film_create: host allocation");
    f->desc = *d;
    f->rows = rows;
    f->layers = layers;
    f->n_elems = n;
    auto part = [&](size_t count) {  // 256-byte aligned
        const size_t at = f->device_floats;
        f->device_floats += (count + 63) / 64 * 64;
        return at;
    };
    const size_t px = size_t(rows) * size_t(d->width);
    part(n);
    const size_t comp = part(n), layer_w = part(size_t(layers) * px), steady = part(layers ? px * 6 : 0);
    if ((rc = dev_alloc(&f->d_sum, f->device_floats))) {
        delete f;
        return rc;
    }
    f->d_comp = f->d_sum + comp;
    if (layers) {
        f->d_layer_w = f->d_sum + layer_w;
        f->d_steady = f->d_sum + steady;
    }
    if (hipStreamCreateWithFlags(&f->stream, hipStreamNonBlocking) != hipSuccess) {
        dev_free(f->d_sum);
        delete f;
        return fail(TR_ERR_DEVICE, "tr_film_create: hipStreamCreate failed");
    }
    f->weight.assign(size_t(rows) * size_t(d->width), 0.0);
    *out = f;
    rc = tr_film_clear(f);
    if (rc) {
        tr_film_destroy(f);
        *out = nullptr;
    }
    return rc;
}

int tr_film_destroy(tr_film f)
{
    if (!f) return TR_OK;
    if (f->stream) (void)hipStreamSynchronize(f->stream);
    dev_free(f->d_sum);
    dev_free(f->d_samples); dev_free(f->d_read_steady); dev_free(f->d_read_w);
    if (f->stream) (void)hipStreamDestroy(f->stream);
    delete f;
    return TR_OK;
}

int tr_film_clear(tr_film f)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_clear: null film");
    HIP_TRY(hipMemsetAsync(f->d_sum, 0, f->device_floats * sizeof(float), f->stream));
    HIP_TRY(hipStreamSynchronize(f->stream));
    std::fill(f->weight.begin(), f->weight.end(), 0.0);
    f->same_weight = true;
    return TR_OK;
}

}  // extern "C"

namespace {

// values of the film's elements [first, first + n) (n > 0) into the host array `out`: normalised (float) or
// the compensated sums (double). Every entry point that writes a film returns after its work has completed,
// so the staging's streams can read it.
template <class Out>
int film_values(tr_film f, size_t first, size_t n, const FilmWeight& w, Out* out, hipStream_t own = nullptr)
{
    static_assert(trb::kChunk % (4 * sizeof(Out)) == 0, "chunks hold whole groups of four values");
    const uint32_t T3 = 3u * uint32_t(f->desc.time_bins);
    const hipError_t e = trb::read_back(out, n * sizeof(Out), [&](hipStream_t stream, void* dst, size_t at, size_t size) {
        const size_t i = first + at / sizeof(Out);
        const uint32_t m = uint32_t(size / sizeof(Out));
        film_values_kernel<Out><<<(m + kValuesPerBlock - 1) / kValuesPerBlock, kValuesPerBlock / 4, 0, stream>>>(
            f->d_sum + i, f->d_comp + i, w, i / T3, uint32_t(i % T3), T3, m, i % 4 == 0, static_cast<Out*>(dst));
        return hipGetLastError();
    }, own);
    if (e != hipSuccess)
        return fail(e == hipErrorOutOfMemory ? TR_ERR_NOMEM : TR_ERR_DEVICE, std::string("tr_film_read: ") + hipGetErrorString(e));
    return TR_OK;
}

}  // namespace

extern "C" {

int tr_film_read_sums(tr_film f, double* sums, double* weights)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_read_sums: null film");
    if (sums) {
        const int rc = film_values(f, 0, f->n_elems, FilmWeight{}, sums);
        if (rc) return rc;
    }
    if (weights) {
        if (f->layers) {
            const size_t n = size_t(f->layers) * f->weight.size();
            std::vector<float> lw(n);
            HIP_TRY(hipMemcpyAsync(lw.data(), f->d_layer_w, n * sizeof(float), hipMemcpyDeviceToHost, f->stream));
            HIP_TRY(hipStreamSynchronize(f->stream));
            for (size_t i = 0; i < n; ++i) weights[i] = double(lw[i]);
        } else {
            std::copy(f->weight.begin(), f->weight.end(), weights);
        }
    }
    return TR_OK;
}

int tr_film_read_rows(tr_film f, int32_t row_begin, int32_t row_count, float* out, float* steady)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_read_rows: null film");
    if (f->layers) return fail(TR_ERR_INVALID, "tr_film_read_rows: multibounce films are read whole (tr_film_read)");
    if (row_begin < 0 || row_count < 0 || row_begin + int64_t(row_count) > f->rows)
        return fail(TR_ERR_INVALID, "tr_film_read_rows: rows outside the film");
    if ((!out && !steady) || row_count == 0) return TR_OK;
    const size_t W = size_t(f->desc.width), T3 = size_t(f->desc.time_bins) * 3, P = size_t(f->rows) * W;
    const size_t p0 = size_t(row_begin) * W, np = size_t(row_count) * W;
    int rc;
    if (steady && !f->d_read_steady && (rc = dev_alloc(&f->d_read_steady, P * 3))) return rc;
    FilmWeight w{f->weight[0], nullptr, nullptr};
    hipStream_t own = nullptr;  // a read of one chunk follows the upload of its weights on the film's stream
    if (!f->same_weight) {
        if (!f->d_read_w && (rc = dev_alloc(&f->d_read_w, P))) return rc;
        HIP_TRY(hipMemcpyAsync(f->d_read_w, f->weight.data(), P * sizeof(double), hipMemcpyHostToDevice, f->stream));
        w.pixel = f->d_read_w;
        // (the upload reads f->weight, which stays as it is until this call returns)
        if (out && np * T3 * sizeof(float) <= trb::kChunk) own = f->stream;
        else HIP_TRY(hipStreamSynchronize(f->stream));
    }
    if (out && (rc = film_values(f, p0 * T3, np * T3, w, out, own))) return rc;
    if (steady) {
        film_steady_kernel<<<uint32_t(np), kNormBlock, 0, f->stream>>>(f->d_sum + p0 * T3, f->d_comp + p0 * T3, w, p0,
                                                                      uint32_t(T3), f->d_read_steady);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(steady, f->d_read_steady, np * 3 * sizeof(float), hipMemcpyDeviceToHost, f->stream));
        HIP_TRY(hipStreamSynchronize(f->stream));
    }
    return TR_OK;
}

int tr_film_read(tr_film f, float* out, float* steady)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_read: null film");
    if (!out && !steady) return TR_OK;
    if (!f->layers) return tr_film_read_rows(f, 0, f->rows, out, steady);
    // multibounce films: each bounce film divided by its own weights; the steady image holds every
    // sample
    int rc;
    if (out && (rc = film_values(f, 0, f->n_elems, FilmWeight{0.0, nullptr, f->d_layer_w}, out))) return rc;
    if (steady) {
        const size_t P = f->weight.size();
        std::vector<float> st(P * 6);
        HIP_TRY(hipMemcpyAsync(st.data(), f->d_steady, st.size() * sizeof(float), hipMemcpyDeviceToHost, f->stream));
        HIP_TRY(hipStreamSynchronize(f->stream));
        for (size_t p = 0; p < P; ++p)
            for (size_t k = 0; k < 3; ++k) {
                const double v = (double(st[p * 3 + k]) + double(st[(P + p) * 3 + k])) / f->weight[p];
                steady[p * 3 + k] = std::isfinite(v) ? float(v) : 0.0f;
            }
    }
    return TR_OK;
}

int tr_film_write(tr_film f, const char* name, const char* ext)
{
    if (!f || !name || !*name) return fail(TR_ERR_INVALID, "tr_film_write: null film or name");
    const std::string e = ext ? ext : "hdr";
    if (e != "hdr" && e != "raw")
        return fail(TR_ERR_INVALID, "Error: unsupported output file format: \"" + e + "\"");
    const int W = f->desc.width, T = f->desc.time_bins, H = f->desc.height;
    std::vector<float> img(f->n_elems), steady(size_t(f->rows) * size_t(W) * 3);
    int rc = tr_film_read(f, img.data(), steady.data());
    if (rc) return rc;
    const size_t slice = size_t(W) * size_t(T) * 3;
    std::vector<float> tr;
    char path[4096];
    // multibounce films: bounce film b is "<name>_b%02d" (b + 1) (MultibounceStreakCameraFilm.h:127-135)
    for (int l = 0; l < std::max(f->layers, 1); ++l)
    for (int r = 0; r < f->rows; ++r) {
        const int y = f->desc.scanline >= 0 ? f->desc.scanline : r;
        // a slice is an image T wide and W high; below 8 columns it is stored transposed
        const float* data = img.data() + (size_t(l) * f->rows + size_t(r)) * slice;
        int width = T, height = W;
        if (T < 8) {
            tr.resize(slice);
            for (int x = 0; x < W; ++x)
                for (int t = 0; t < T; ++t)
                    for (int c = 0; c < 3; ++c) tr[(size_t(t) * W + x) * 3 + c] = data[(size_t(x) * T + t) * 3 + c];
            data = tr.data();
            width = W, height = T;
        }
        if (f->layers) std::snprintf(path, sizeof path, "%s_b%02d_%04d.%s", name, l + 1, y, e.c_str());
        else std::snprintf(path, sizeof path, "%s_%04d.%s", name, y, e.c_str());
        rc = e == "hdr" ? tri::write_rgbe(path, data, width, height) : tri::write_raw(path, data, slice);
        if (rc) return rc;
    }
    // steady image: W x H, time-integrated radiance (only the streak row in scanline mode)
    std::vector<float> full(size_t(W) * size_t(H) * 3, 0.0f);
    for (int r = 0; r < f->rows; ++r) {
        const int y = f->desc.scanline >= 0 ? f->desc.scanline : r;
        std::copy(steady.begin() + size_t(r) * W * 3, steady.begin() + size_t(r + 1) * W * 3,
                  full.begin() + size_t(y) * W * 3);
    }
    std::snprintf(path, sizeof path, "%s.hdr", name);
    return tri::write_rgbe(path, full.data(), W, H);
}

int tr_film_device_buffers(tr_film f, float** d_sum, float** d_comp)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_device_buffers: null film");
    if (d_sum) *d_sum = f->d_sum;
    if (d_comp) *d_comp = f->d_comp;
    return TR_OK;
}

// StreakCameraFilm::add_samples for caller-made samples: checked, binned as the reference bins
// (pos_sensor = (time - offset) / exposure, kept if 0 <= pos_sensor < T; StreakCameraFilm.h:165-171) and
// deposited on the device, by the renders' own film kernel. (Binned on the host into shadow-record
// arrays, 500,000 samples took 1.5 ms on one thread and 0.6 ms of allocations and extra copies.) The
// weights are summed by the host, per pixel in the order of the samples, so that the same calls give the
// same bits: 1-2 ns each. Up to kHostSamples they are checked by the host too, as the device's two launches take
// longer; larger calls sum while the device works, and calls of kThreadSamples or more already while the
// runtime copies the samples (500,000: 480 us on one thread), by a second thread where there are at least as
// many samples as pixels (fewer are scattered over lines of another core's cache: 17,000 over 256 x 256
// pixels took 300 us, and take 66). Nothing that follows the deposit needs memory.
int tr_film_add_samples(tr_film f, const tr_film_sample* samples, uint32_t n)
{
    if (!f) return fail(TR_ERR_INVALID, "tr_film_add_samples: null film");
    if (f->layers) return fail(TR_ERR_INVALID, "tr_film_add_samples: multibounce films take samples from renders only");
    if (n == 0) return TR_OK;
    if (!samples) return fail(TR_ERR_INVALID, "tr_film_add_samples: null samples");
    if (n > (1u << 31)) return fail(TR_ERR_INVALID, "tr_film_add_samples: more than 2^31 samples in one call");
    const tr_film_desc& fd = f->desc;
    const uint32_t T = uint32_t(fd.time_bins), P = uint32_t(f->weight.size());
    const int32_t row0 = fd.scanline >= 0 ? fd.scanline : 0;
    constexpr size_t kHead = 256 / sizeof(tr_film_sample), kKept = size_t(32) << 20;  // samples buffers up to 32 MiB are kept
    constexpr uint32_t kHostSamples = 16384, kThreadSamples = 131072;
    const bool on_host = n <= kHostSamples;
    try {
        f->added.resize(P, 0.0);
    } catch (const std::bad_alloc&) {
        return fail(TR_ERR_NOMEM, "tr_film_add_samples: host allocation");
    }
    // sums the weights into f->added; stops at the first sample outside the film
    uint32_t first_bad = 0xFFFFFFFFu;
    auto pixel = [&](uint32_t i) {
        const uint32_t x = uint32_t(samples[i].x), row = uint32_t(samples[i].y) - uint32_t(row0);
        return x < uint32_t(fd.width) && row < uint32_t(f->rows) ? row * uint32_t(fd.width) + x : 0xFFFFFFFFu;
    };
    auto sum_weights = [&]() {
        uint32_t at = 0xFFFFFFFFu;  // a run of samples of one pixel
        double sum = 0.0;
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t p = pixel(i);
            if (p == 0xFFFFFFFFu) {
                first_bad = i;
                break;
            }
            if (p != at) {
                if (at != 0xFFFFFFFFu) f->added[at] = sum;
                at = p;
                sum = f->added[p];
            }
            sum += double(samples[i].weight);
        }
        if (at != 0xFFFFFFFFu) f->added[at] = sum;
    };
    // calls use(p) at least once for each pixel that sum_weights has added to
    auto each_pixel = [&](auto use) {
        const uint32_t m = std::min(n, first_bad);
        if (m < P / 16)
            for (uint32_t i = 0; i < m; ++i) use(pixel(i));
        else
            for (uint32_t p = 0; p < P; ++p) use(p);
    };
    auto outside = [&]() {
        each_pixel([&](uint32_t p) { f->added[p] = 0.0; });
        return fail(TR_ERR_INVALID, "tr_film_add_samples: sample " + std::to_string(first_bad) + " lies outside the film");
    };
    int rc;
    if (f->samples_cap < n) {
        dev_free(f->d_samples);
        f->samples_cap = 0;
        if ((rc = dev_alloc(&f->d_samples, kHead + n))) return rc;
        f->samples_cap = n;
    }
    std::thread summing;
    if (on_host) {
        sum_weights();
        if (first_bad != 0xFFFFFFFFu) return outside();
    } else if (n >= kThreadSamples && n >= P) {
        try {
            summing = std::thread(sum_weights);
        } catch (...) {  // no more threads: below
        }
    }
    uint32_t* bad = reinterpret_cast<uint32_t*>(f->d_samples);
    tr_film_sample* d = f->d_samples + kHead;
    RenderDev R{};
    R.film = f->d_sum;
    R.film_comp = f->d_comp;
    R.W = fd.width;
    R.H = fd.height;
    R.T = fd.time_bins;
    R.row0 = row0;
    R.offset = fd.offset;
    R.exposure = fd.exposure;
    const uint32_t pix_slots = std::min<uint32_t>(kFilmMaxSlots, kFilmLdsBytes / (T * 24u));
    const size_t lds = size_t(pix_slots) * size_t(T) * 24u;
    const uint32_t cu = uint32_t(tri::compute_units());
    const uint32_t fg = std::max(1u, std::min((n + kFilmRange - 1) / kFilmRange, cu * 4u));
    hipError_t e = hipMemcpyAsync(d, samples, size_t(n) * sizeof(tr_film_sample), hipMemcpyHostToDevice, f->stream);
    if (e == hipSuccess && !on_host) {
        samples_begin_kernel<<<1, 1, 0, f->stream>>>(bad);
        samples_check_kernel<<<std::min((n + kBlock - 1) / kBlock, cu * 16u), kBlock, 0, f->stream>>>(
            d, n, fd.width, row0, f->rows, bad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        film_kernel<kFilmSamples><<<fg, kFilmBlock, lds, f->stream>>>(R, WaveDev{}, 0, pix_slots, nullptr,
                                                                     SamplesDev{d, n, on_host ? nullptr : bad});
        e = hipGetLastError();
    }
    if (summing.joinable()) summing.join();
    else if (!on_host) sum_weights();
    // the copy reads the caller's samples: wait in any case
    const hipError_t se = hipStreamSynchronize(f->stream);
    if (e == hipSuccess) e = se;
    if (f->samples_cap * sizeof(tr_film_sample) > kKept) {
        dev_free(f->d_samples);
        f->samples_cap = 0;
    }
    if (first_bad != 0xFFFFFFFFu) return outside();
    if (e != hipSuccess) {
        each_pixel([&](uint32_t p) { f->added[p] = 0.0; });
        return fail(TR_ERR_DEVICE, std::string("tr_film_add_samples: ") + hipGetErrorString(e));
    }
    f->same_weight = false;
    each_pixel([&](uint32_t p) {
        f->weight[p] += f->added[p];
        f->added[p] = 0.0;
    });
    return TR_OK;
}

}  // extern "C"

namespace {

// A render job as the host prepares it.
struct HostJob {
    tr_scene scene;
    tr_film film;
    JobDev dev;          // scene view, film/camera set-up, first global path index
    uint64_t paths;
    uint32_t spp2;
    int max_bounces;
};

// Camera and film set-up of one job (PinholeCamera.h:56-80; bunnykiller.cpp:1156-1160).
int make_job(tr_scene s, const tr_camera* cam, tr_film f, const tr_render_desc* d, HostJob* out, const char* who)
{
    if (!s || !cam || !f || !d) return fail(TR_ERR_INVALID, std::string(who) + ": null argument");
    if (!s->committed) return fail(TR_ERR_STATE, std::string(who) + ": scene not committed");
    if (s->lights.empty()) return fail(TR_ERR_INVALID, std::string(who) + ": scene has no light");
    if (d->sqrt_spp <= 0 || d->n_incoming <= 0 || d->max_bounces < 0)
        return fail(TR_ERR_INVALID, std::string(who) + ": bad sampling parameters");
    const tr_film_desc& fd = f->desc;
    const uint64_t spp2 = uint64_t(d->sqrt_spp) * uint64_t(d->sqrt_spp);
    const uint64_t total = uint64_t(f->rows) * uint64_t(fd.width) * spp2 * uint64_t(d->n_incoming);
    if ((uint64_t(fd.height) * fd.width * spp2 * uint64_t(d->n_incoming)) >= (1ull << 61))
        return fail(TR_ERR_INVALID, std::string(who) + ": too many paths for the RNG stream ids");
    if (total >= (1ull << 32))
        return fail(TR_ERR_INVALID, std::string(who) + ": more than 2^32 - 1 paths in one job; split into passes");
    if (uint64_t(f->rows) * uint64_t(fd.width) >= (1ull << 24))
        return fail(TR_ERR_INVALID, std::string(who) + ": film has more than 2^24 pixels");
    if (d->max_bounces > 255) return fail(TR_ERR_INVALID, std::string(who) + ": max_bounces above 255");
    auto nrm = [](float* v) {
        float l = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        float inv = float(1. / double(l));
        for (int k = 0; k < 3; ++k) v[k] *= inv;
    };
    auto crs = [](const float* a, const float* b, float* o) {
        o[0] = a[1] * b[2] - a[2] * b[1];
        o[1] = a[2] * b[0] - a[0] * b[2];
        o[2] = a[0] * b[1] - a[1] * b[0];
    };
    float up[3] = {cam->up[0], cam->up[1], cam->up[2]};
    nrm(up);
    float nv[3] = {cam->focus[0] - cam->position[0], cam->focus[1] - cam->position[1], cam->focus[2] - cam->position[2]};
    nrm(nv);
    float uv[3], vv[3];
    crs(nv, up, uv);
    nrm(uv);
    crs(uv, nv, vv);
    nrm(vv);
    float fov = float(M_PI / 180. * double(cam->fov_deg) / 2);
    RenderDev R{};
    R.film = f->d_sum;
    R.film_comp = f->d_comp;
    R.W = fd.width;
    R.H = fd.height;
    R.T = fd.time_bins;
    R.row0 = fd.scanline >= 0 ? fd.scanline : 0;
    R.spp = d->sqrt_spp;
    R.spp2 = int32_t(spp2);
    R.n_inc = d->n_incoming;
    R.exposure = fd.exposure;
    R.offset = fd.offset;
    R.total_time = float(fd.time_bins) * fd.exposure + fd.offset;
    // NextEventSampling::Time: m_avg_nb_vertices_path (4) / (T * exposure / time_of_flight(1) / ior)
    // (BidirectionalPathTracing.h:131, 246-252; World.h:776-786: time_of_flight(d) = d, ior = 1)
    R.time_sampling = (d->flags & TR_RENDER_TIME_SAMPLING) ? 1 : 0;
    R.ts_lambda = 4.0f / (float(fd.time_bins) * fd.exposure / 1.0f / 1.0f);
    R.inv_inc = float(1. / double(float(d->n_incoming)));
    R.unwarp = fd.camera_unwarp ? 1 : 0;
    R.pid0 = uint64_t(R.row0) * uint64_t(R.W) * spp2 * uint64_t(R.n_inc);
    R.max_bounces = d->max_bounces;
    R.cpos = make_float3(cam->position[0], cam->position[1], cam->position[2]);
    R.nv = make_float3(nv[0], nv[1], nv[2]);
    R.uv = make_float3(uv[0], uv[1], uv[2]);
    R.vv = make_float3(vv[0], vv[1], vv[2]);
    R.fd = cam->view_plane_dist > 0.f ? cam->view_plane_dist : float(1. / std::tan(double(fov)));
    R.xw2 = float(double(fd.width) / 2.0);
    R.yw2 = float(double(fd.height) / 2.0);
    R.ratio = float(fd.width) / float(fd.height);
    R.inv_spp = float(1. / double(float(d->sqrt_spp)));
    R.seed = d->seed;
    R.layers = f->layers;
    R.layer_stride = uint32_t(size_t(f->rows) * size_t(fd.width) * size_t(fd.time_bins));
    R.steady = f->d_steady;
    R.steady_comp = f->d_steady ? f->d_steady + size_t(f->rows) * size_t(fd.width) * 3 : nullptr;
    R.layer_w = f->d_layer_w;
    R.cs_bits = nullptr;  // set by the launch (wavefront buffers)
    out->scene = s;
    out->film = f;
    out->dev.S = s->view();
    out->dev.R = R;
    out->dev.path_begin = 0;
    out->paths = total;
    out->spp2 = uint32_t(spp2);
    out->max_bounces = d->max_bounces;
    return TR_OK;
}

// Everything the kernels of one launch need, shared by the per-wave enqueue.
struct Launch {
    hipStream_t stream;
    WaveBuffers* wb;
    std::vector<HostJob>* jobs;
    const LaunchCfg* cfg;
    tr_guide guide;
    trg::GuideView GV;
    int compute_units;
    hipEvent_t* ev;
    bool batch;
    int bounces;
    int group;  // bounces whose shadow rays are traced and deposited together
    bool path_launch;  // a wavefront's bounces run in one launch (path_kernel), path_per_wave paths per GPU wavefront
    uint32_t path_per_wave;
    int stack_bound;
    int trav_ext, trav_sh;  // kTrav* of the closest-hit and any-hit launches
    uint32_t pix_slots;
    size_t film_lds;
    // profiling
    std::vector<std::pair<int, int>> ev_kind;
    double kernel_ms[TR_K_COUNT] = {};
    uint32_t launches[TR_K_COUNT] = {};
    bool events_on = false;
    bool extend_only = false;  // events around the extend launches only
    bool open = false;         // begin() recorded an event that end() closes
    // events of the current extend / shadow launch, stamped by the launch itself (launch_timed)
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;

    int flush_events()
    {
        if (ev_kind.empty()) return TR_OK;
        HIP_TRY(hipEventSynchronize(ev[2 * ev_kind.back().second + 1]));
        for (auto& kv : ev_kind) {
            float ms = 0.f;
            HIP_TRY(hipEventElapsedTime(&ms, ev[2 * kv.second], ev[2 * kv.second + 1]));
            kernel_ms[kv.first] += ms;
        }
        ev_kind.clear();
        return TR_OK;
    }
    int begin(int kind)
    {
        launches[kind]++;
        open = events_on && !(extend_only && kind != TR_K_EXTEND);
        if (!open) return TR_OK;
        if (ev_kind.size() == 256) {
            int r2 = flush_events();
            if (r2) return r2;
        }
        int slot = int(ev_kind.size());
        ev_kind.push_back({kind, slot});
        if (kind == TR_K_EXTEND || kind == TR_K_SHADOW) {
            ev_start = ev[2 * slot];
            ev_stop = ev[2 * slot + 1];
        } else {
            HIP_TRY(hipEventRecord(ev[2 * slot], stream));
        }
        return TR_OK;
    }
    int end()
    {
        HIP_TRY(hipGetLastError());
        if (!open) return TR_OK;
        open = false;
        if (ev_start) {
            ev_start = ev_stop = nullptr;
            return TR_OK;
        }
        HIP_TRY(hipEventRecord(ev[2 * ev_kind.back().second + 1], stream));
        return TR_OK;
    }

    // the kernels of one wavefront: camera, then per bounce extend / shade and per group of bounces shadow /
    // film; or path, shadow, film
    int enqueue_wave()
    {
        int rc;
        const LaunchCfg& c = *cfg;
        const HostJob& j0 = (*jobs)[0];
        const SceneDev S0 = j0.dev.S;
        const RenderDev R0 = j0.dev.R;
        const JobDev* dj = batch ? wb->d_jobs : nullptr;
        const uint32_t nj = uint32_t(jobs->size());
        WaveDev Wv = wb->view();
        Wv.cpos = R0.cpos;
        const uint32_t wave = c.wave, cu = uint32_t(std::max(compute_units, 1));
        // persistent traversal grid: trace_per_cu blocks per CU, but at least kTraceRaysPerThread rays
        // per thread of a full wavefront (a smaller scene's wavefronts run faster on fewer, longer-lived
        // blocks: 8 rays per thread is 8 % faster than 4 or 16 on the 2-M-path media workload, no
        // change on 33-M-path wavefronts) as long as every CU keeps kTraceMinPerCu blocks (small
        // renders: 128 blocks for a 262,144-path wavefront left three quarters of the SIMDs idle)
        const uint32_t by_rays = std::max((wave + kTraceBlock * kTraceRaysPerThread - 1) / (kTraceBlock * kTraceRaysPerThread),
                                          cu * kTraceMinPerCu);
        const uint32_t tg = std::max(1u, std::min({(wave + kTraceBlock - 1) / kTraceBlock, cu * c.trace_per_cu, by_rays}));
        const uint32_t sblock = c.mode == kShadeGuided ? kShadeBlockGuided : kShadeBlock;
        // guided shading: 2 blocks per CU (its LDS allows no more), persistent over the wavefront, so
        // each block stages the network's 38 KB of weights once per launch instead of once per
        // 256 paths
        const uint32_t scap = cu * (c.mode == kShadeGuided ? 2u : c.shade_per_cu);
        const uint32_t sg = std::max(1u, std::min((wave + sblock - 1) / sblock, scap));
        const uint32_t cg = (wave + kBlock - 1) / kBlock;
        if (path_launch) {
            const bool onb = c.mode == kShadeOnb;
            Wv.seg_paths = path_per_wave;
            Wv.seg_cap = Wv.seg_paths * uint32_t(bounces);
            const uint32_t waves = (wave + Wv.seg_paths - 1) / Wv.seg_paths, pg = (waves * 64u + kTraceBlock - 1) / kTraceBlock;
            if ((rc = begin(TR_K_EXTEND))) return rc;
            if (trav_ext == kTravWide16 && batch)
                TR_PATH_DISPATCH_T(kTravWide16, stack_bound, true, pg, kTraceBlock, stream, S0, R0, dj, nj, Wv, onb);
            else if (trav_ext == kTravWide16)
                TR_PATH_DISPATCH_T(kTravWide16, stack_bound, false, pg, kTraceBlock, stream, S0, R0, dj, nj, Wv, onb);
            else if (batch)
                TR_PATH_DISPATCH_T(kTravWide, stack_bound, true, pg, kTraceBlock, stream, S0, R0, dj, nj, Wv, onb);
            else
                TR_PATH_DISPATCH_T(kTravWide, stack_bound, false, pg, kTraceBlock, stream, S0, R0, dj, nj, Wv, onb);
            if ((rc = end()) || (rc = enqueue_film(Wv, 0))) return rc;
            return enqueue_layer_weights();
        }
        if ((rc = begin(TR_K_CAMERA))) return rc;
        if (batch) camera_kernel<true><<<cg, kBlock, 0, stream>>>(S0, R0, dj, nj, Wv);
        else camera_kernel<false><<<cg, kBlock, 0, stream>>>(S0, R0, dj, nj, Wv);
        if ((rc = end())) return rc;
        int cur = 0;
        for (int b = 0; b < bounces; ++b) {
            if ((rc = begin(TR_K_EXTEND))) return rc;
            if (b == 0 && !batch && c.camera_packets &&
                (trav_ext == kTravWide || trav_ext == kTravWide16 || trav_ext == kTravWideKeyed)) {
                if (trav_ext == kTravWide) TR_CAMERA_DISPATCH_T(kTravWide, stack_bound, tg, kTraceBlock, stream, S0, Wv, cur);
                else if (trav_ext == kTravWide16)
                    TR_CAMERA_DISPATCH_T(kTravWide16, stack_bound, tg, kTraceBlock, stream, S0, Wv, cur);
                else TR_CAMERA_DISPATCH_T(kTravWideKeyed, stack_bound, tg, kTraceBlock, stream, S0, Wv, cur);
            } else {
                TR_TRACE_DISPATCH(trav_ext, stack_bound, batch, extend_kernel, tg, kTraceBlock, stream, S0, dj, Wv,
                                  cur | (b == 0 ? 2 : 0) | (b % group != 0 ? 4 : 0));
            }
            if ((rc = end())) return rc;
            if ((rc = begin(TR_K_SHADE))) return rc;
            if (batch) {
                if (c.mode == kShadeOnb)
                    shade_kernel<kShadeOnb, true><<<sg, kShadeBlock, 0, stream>>>(S0, R0, dj, Wv, cur | (b << 1), GV);
                else
                    shade_kernel<kShadeRef, true><<<sg, kShadeBlock, 0, stream>>>(S0, R0, dj, Wv, cur | (b << 1), GV);
            } else if (c.mode == kShadeGuided) {
                shade_kernel<kShadeGuided, false><<<sg, kShadeBlockGuided, 0, stream>>>(S0, R0, dj, Wv, cur | (b << 1), GV);
            } else if (c.mode == kShadeOnb) {
                shade_kernel<kShadeOnb, false><<<sg, kShadeBlock, 0, stream>>>(S0, R0, dj, Wv, cur | (b << 1), GV);
            } else {
                shade_kernel<kShadeRef, false><<<sg, kShadeBlock, 0, stream>>>(S0, R0, dj, Wv, cur | (b << 1), GV);
            }
            if ((rc = end())) return rc;
            if ((b + 1) % group != 0 && b + 1 < bounces) {
                cur ^= 1;
                continue;
            }
            if ((rc = begin(TR_K_SHADOW))) return rc;
            TR_TRACE_DISPATCH(trav_sh, stack_bound, batch, shadow_kernel, tg, kTraceBlock, stream, S0, dj, Wv, cur ^ 1);
            if ((rc = end()) || (rc = enqueue_film(Wv, cur ^ 1))) return rc;
            cur ^= 1;
        }
        return enqueue_layer_weights();
    }

    // the traced shadow records deposited: those of queue `sh`, or of a path launch (Wv.seg_cap)
    int enqueue_film(const WaveDev& Wv, int sh)
    {
        int rc;
        const RenderDev R0 = (*jobs)[0].dev.R;
        const uint32_t wave = cfg->wave, cu = uint32_t(std::max(compute_units, 1));
        const uint32_t fg = std::max(1u, std::min((wave + kFilmRange - 1) / kFilmRange, cu * 4u));
        const uint32_t rg = std::max(1u, std::min((wave + kBlock - 1) / kBlock, cu * 16u));
        if ((rc = begin(TR_K_FILM))) return rc;
        if (batch) film_batch_kernel<<<rg, kBlock, 0, stream>>>(wb->d_jobs, Wv, sh);
        else if (R0.layers > 0) film_mb_kernel<<<rg, kBlock, 0, stream>>>(R0, Wv, sh);
        else if (guide)
            film_kernel<kFilmGuided><<<fg, kFilmBlock, film_lds, stream>>>(R0, Wv, sh, pix_slots, GV.contrib, SamplesDev{});
        else if (Wv.seg_cap)
            film_kernel<kFilmPath><<<fg, kFilmBlock, film_lds, stream>>>(R0, Wv, sh, pix_slots, nullptr, SamplesDev{});
        else film_kernel<kFilmRender><<<fg, kFilmBlock, film_lds, stream>>>(R0, Wv, sh, pix_slots, nullptr, SamplesDev{});
        return end();
    }

    // multibounce films, after a wavefront
    int enqueue_layer_weights()
    {
        const RenderDev R0 = (*jobs)[0].dev.R;
        if (batch || R0.layers == 0) return TR_OK;
        int rc;
        if ((rc = begin(TR_K_FILM))) return rc;
        const uint32_t ncs = cfg->wave / uint32_t(R0.n_inc), cu = uint32_t(std::max(compute_units, 1));
        mb_weight_kernel<<<std::max(1u, std::min((ncs + kBlock - 1) / kBlock, cu * 16u)), kBlock, 0, stream>>>(R0, wb->view());
        return end();
    }
};

static_assert(kMaxLayersTagBits == kMbLayerTagBits, "layer tag width");

// Renders every job of `jobs` in one sequence of wavefronts on `stream`; jobs share wavefronts
// when there are several (batched kernels look up each path's job).
int run_jobs(hipStream_t stream, WaveBuffers& wb, std::vector<HostJob>& jobs, const LaunchCfg& cfg, tr_guide guide,
             int compute_units, hipEvent_t* ev, bool* ev_made, tr_render_stats* stats,
             std::chrono::steady_clock::time_point t_start)
{
    if (jobs.empty()) return fail(TR_ERR_INVALID, "render: no job");
    // every return drains the stream, so no queued copy or kernel outlives the host buffers and
    // device views it was given (the normal path synchronises as well, to read the counters)
    trb::Chunks pinned;  // (given back after that)
    struct Use {
        WaveBuffers* b;
        explicit Use(WaveBuffers* wb) : b(wb) { BufferList::get().use(b, 1); }
        ~Use() { BufferList::get().use(b, -1); }
    } use(&wb);  // (until after that)
    struct Drain {
        hipStream_t s;
        ~Drain() { (void)hipStreamSynchronize(s); }
    } drain{stream};
    if (pinned.take(1) != hipSuccess) return fail(TR_ERR_NOMEM, "render: pinned memory");
    const bool batch = jobs.size() > 1;
    if (batch && guide) return fail(TR_ERR_INVALID, "render: guided renders take one job");
    uint64_t total = 0;
    int bounces = 0, stack_bound = 0;
    uint32_t max_nodes4 = 0;
    bool wide = cfg.wide, shallow = true;
    for (auto& j : jobs) {
        wide = wide && j.scene->wide;
        shallow = shallow && j.scene->n_nodes4 <= kShallowNodes;
    }
    for (auto& j : jobs) {
        j.dev.path_begin = total;
        total += j.paths;
        bounces = std::max(bounces, j.max_bounces);
        stack_bound = std::max(stack_bound, wide ? j.scene->stack4 : j.scene->depth);
        max_nodes4 = std::max(max_nodes4, j.scene->n_nodes4);
    }
    // 16-bit stack entries hold node indices below 65,536
    const bool small = max_nodes4 <= 65536u && cfg.stack_fmt != 1;
    const int trav_ext = !wide ? kTravBinary : !small ? kTravWide : cfg.stack_fmt == 2 ? kTravWideKeyed : kTravWide16;
    const int trav_sh = !wide ? kTravBinary : !small ? kTravWide : kTravWide16;
    const bool mb = jobs[0].dev.R.layers > 0;
    for (auto& j : jobs)
        if (j.dev.R.layers > 0 && (batch || guide))
            return fail(TR_ERR_INVALID, "render: multibounce films render alone and without guiding");
    LaunchCfg c = cfg;
    c.wave = uint32_t(std::min<uint64_t>(c.wave ? c.wave : kDefaultWave, std::max<uint64_t>(total, 1)));
    if (mb) {
        // wavefronts hold whole camera samples, whose layer marks are counted per wavefront; a
        // shadow record tags its camera sample within the wavefront in 27 bits (and its layer in 5),
        // so a wavefront holds at most kMbMaxCameraSamples camera samples
        const uint32_t ni = uint32_t(jobs[0].dev.R.n_inc);
        c.wave = mb_wave(c.wave, ni);
    }
    // bounces whose shadow rays one launch takes
    uint32_t group = std::max(1u, std::min(uint32_t(std::max(bounces, 1)), kShadowRecords / c.wave));
    if (c.group) group = std::min(group, c.group);
    const uint32_t unit = guide ? c.wave : mb ? uint32_t(jobs[0].dev.R.n_inc) : 1u;
    wb.fit(c.wave, group, unit);
    bool unwarp = false;
    for (auto& j : jobs) unwarp = unwarp || j.dev.R.unwarp;
    int rc;
    for (;;) {
        const bool was = wb.cap != 0;  // (what it already has may have made the first try larger than the shape)
        rc = wb.ensure_all(c.wave, group, unwarp, mb || guide, mb ? c.wave / uint32_t(jobs[0].dev.R.n_inc) : 0u,
                           batch ? uint32_t(jobs.size()) : 0u);
        if (rc != TR_ERR_NOMEM || (!was && !WaveBuffers::smaller(c.wave, group, unit))) break;
    }
    if (rc) return rc;
    if (mb) {
        HIP_TRY(hipMemsetAsync(wb.cs_bits, 0, size_t(c.wave / uint32_t(jobs[0].dev.R.n_inc)) * sizeof(uint32_t), stream));
        jobs[0].dev.R.cs_bits = wb.cs_bits;
    }
    Launch L{};
    L.stream = stream;
    L.wb = &wb;
    L.jobs = &jobs;
    L.cfg = &c;
    L.guide = guide;
    L.compute_units = compute_units;
    L.ev = ev;
    L.batch = batch;
    L.bounces = bounces;
    L.group = int(group);
    const uint32_t path_wave = shallow ? kPathWaveShallow : trav_ext == kTravWide ? kPathWave32 : kPathWave;
    L.path_launch = c.path_launch && !guide && bounces > 0 && c.wave <= path_wave &&
                    group == uint32_t(bounces) && (trav_ext == kTravWide || trav_ext == kTravWide16);
    L.path_per_wave = 64u * std::max({1u, std::min(4u, c.wave >> 19), c.wave >> 20});
    while (L.path_per_wave > 16u && c.wave <= L.path_per_wave * 1024u) L.path_per_wave /= 2u;
    L.stack_bound = stack_bound;
    L.trav_ext = trav_ext;
    L.trav_sh = trav_sh;
    if (guide) {
        const HostJob& j = jobs[0];
        if (j.max_bounces < 1) return fail(TR_ERR_INVALID, "tr_render_transient_guided: max_bounces must be >= 1");
        if ((rc = trg::guide_begin_render(guide, c.wave, uint32_t(j.max_bounces), j.scene->bb_lo, j.scene->bb_hi,
                                          stream, &L.GV)))
            return rc;
    }
    if (batch) {
        // the previous render on this stream ended with a synchronisation, so the pinned table is
        // free to overwrite
        JobDev* dj = wb.h_jobs;
        for (size_t k = 0; k < jobs.size(); ++k) dj[k] = jobs[k].dev;
        dj[jobs.size()] = jobs.back().dev;
        dj[jobs.size()].path_begin = total;
        HIP_TRY(hipMemcpyAsync(wb.d_jobs, dj, (jobs.size() + 1) * sizeof(JobDev), hipMemcpyHostToDevice, stream));
    }
    if (c.prof && !c.graph) {
        if (!*ev_made) {
            for (int k = 0; k < 2 * 256; ++k) HIP_TRY(hipEventCreate(&ev[k]));
            *ev_made = true;
        }
        L.events_on = true;
        L.extend_only = c.prof_extend;
    }
    // LDS histogram slots of the film kernel: as many pixels x T bins x RGB FP64 partials as fit in
    // kFilmLdsBytes
    {
        const uint32_t T = uint32_t(jobs[0].dev.R.T);
        L.pix_slots = std::min<uint32_t>(kFilmMaxSlots, kFilmLdsBytes / (T * 24u));
        L.film_lds = size_t(L.pix_slots) * size_t(T) * 24u;
    }
    // pass buffers are written on this stream; order it after any pending film work
    for (auto& j : jobs) HIP_TRY(hipStreamSynchronize(j.film->stream));

    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    auto drop_graph = [&]() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    };
    uint32_t n_waves = 0;
    if (c.graph && !guide) {
        // the whole render (every wavefront's set-up, camera and bounce kernels) as one captured
        // graph, submitted with one launch; guided renders instead replay one wavefront's kernels
        // (their Adam steps between wavefronts take host-computed bias corrections)
        HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        for (uint64_t base = 0; base < total && !rc; base += c.wave) {
            const uint32_t n = uint32_t(std::min<uint64_t>(c.wave, total - base));
            ++n_waves;
            set_wave_kernel<<<1, kBlock, 0, stream>>>(wb.ctl, base, n, wb.counters);
            rc = L.enqueue_wave();
        }
        const hipError_t ce = hipStreamEndCapture(stream, &graph);
        if (rc || ce != hipSuccess) {
            drop_graph();
            return rc ? rc : fail(TR_ERR_DEVICE, std::string("hipStreamEndCapture: ") + hipGetErrorString(ce));
        }
        const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (ie != hipSuccess) {
            drop_graph();
            return fail(TR_ERR_DEVICE, std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
        }
        const hipError_t le = hipGraphLaunch(exec, stream);
        if (le != hipSuccess) {
            drop_graph();
            return fail(TR_ERR_DEVICE, std::string("hipGraphLaunch: ") + hipGetErrorString(le));
        }
    }
    for (uint64_t base = 0; base < total && !(c.graph && !guide); base += c.wave) {
        uint32_t n = uint32_t(std::min<uint64_t>(c.wave, total - base));
        ++n_waves;
        if (guide) {
            if ((rc = L.begin(TR_K_GUIDE)) || (rc = trg::guide_wave_begin(guide, stream)) || (rc = L.end())) {
                drop_graph();
                return rc;
            }
        }
        set_wave_kernel<<<1, kBlock, 0, stream>>>(wb.ctl, base, n, wb.counters);
        if (c.graph) {
            if (!exec) {
                uint32_t launches_before[TR_K_COUNT];
                std::memcpy(launches_before, L.launches, sizeof launches_before);
                HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
                rc = L.enqueue_wave();
                hipError_t ce = hipStreamEndCapture(stream, &graph);
                if (rc || ce != hipSuccess) {
                    drop_graph();
                    return rc ? rc : fail(TR_ERR_DEVICE, std::string("hipStreamEndCapture: ") + hipGetErrorString(ce));
                }
                hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
                if (ie != hipSuccess) {
                    drop_graph();
                    return fail(TR_ERR_DEVICE, std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
                }
                std::memcpy(L.launches, launches_before, sizeof launches_before);
            }
            // count the kernels each replay runs
            L.launches[TR_K_CAMERA] += 1;
            for (int k : {TR_K_EXTEND, TR_K_SHADE}) L.launches[k] += uint32_t(bounces);
            for (int k : {TR_K_SHADOW, TR_K_FILM}) L.launches[k] += (uint32_t(bounces) + group - 1) / group;
            if (mb) L.launches[TR_K_FILM] += 1;
            hipError_t le = hipGraphLaunch(exec, stream);
            if (le != hipSuccess) {
                drop_graph();
                return fail(TR_ERR_DEVICE, std::string("hipGraphLaunch: ") + hipGetErrorString(le));
            }
        } else if ((rc = L.enqueue_wave())) {
            return rc;
        }
        if (guide) {
            if ((rc = L.begin(TR_K_GUIDE)) || (rc = trg::guide_wave_end(guide, stream)) || (rc = L.end())) {
                drop_graph();
                return rc;
            }
        }
    }
    uint32_t* const counters = reinterpret_cast<uint32_t*>(pinned[0].host);
    read_counters_kernel<<<1, kBlock, 0, stream>>>(wb.counters, counters);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    drop_graph();
    if (rc) return rc;
    if (e != hipSuccess) return fail(TR_ERR_DEVICE, std::string("render: ") + hipGetErrorString(e));
    if ((rc = L.flush_events())) return rc;
    for (auto& j : jobs)
        for (double& w : j.film->weight) w += double(j.spp2);
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->paths = total;
        auto rd64 = [&](int w) { return uint64_t(counters[w]) | (uint64_t(counters[w + 1]) << 32); };
        stats->extension_rays = rd64(C_STAT_EXT);
        stats->shadow_rays = rd64(C_STAT_SHADOW);
        for (uint32_t p = 0; p < kParts; ++p) {
            stats->extension_rays += rd64(int(part_word(p, P_STAT_EXT)));
            stats->shadow_rays += rd64(int(part_word(p, P_STAT_SHADOW)));
            stats->contributions += rd64(int(part_word(p, P_STAT_CONTRIB)));
        }
        stats->waves = n_waves;
        stats->bounces_max = uint32_t(bounces);
        for (int k = 0; k < TR_K_COUNT; ++k) {
            stats->kernel_ms[k] = L.kernel_ms[k];
            stats->kernel_launches[k] = L.launches[k];
        }
        stats->render_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
    }
    return TR_OK;
}

int render_impl(tr_scene s, const tr_camera* cam, tr_film f, const tr_render_desc* d, tr_guide guide,
                tr_render_stats* stats)
{
    auto t_start = std::chrono::steady_clock::now();
    std::vector<HostJob> jobs(1);
    int rc = make_job(s, cam, f, d, &jobs[0], guide ? "tr_render_transient_guided" : "tr_render_transient");
    if (rc) return rc;
    LaunchCfg c = s->tune;
    if (d->wave_paths) c.wave = d->wave_paths;
    else if (guide && c.wave == kDefaultWave) c.wave = kSmallWave;  // (a guide trains after each wavefront)
    c.wide = (d->flags & TR_RENDER_BINARY_BVH) == 0;
    c.graph = (d->flags & TR_RENDER_GRAPH) != 0;
    c.prof = (d->flags & (TR_RENDER_PROFILE | TR_RENDER_PROFILE_EXTEND)) != 0;
    c.prof_extend = (d->flags & TR_RENDER_PROFILE) == 0 && (d->flags & TR_RENDER_PROFILE_EXTEND) != 0;
    if (d->flags & (TR_RENDER_STACK32 | TR_RENDER_STACK_KEYED | TR_RENDER_POSTPONE_LEAVES)) c.stack_fmt = stack_fmt_of(d->flags);
    c.mode = guide ? kShadeGuided : ((d->flags & TR_RENDER_ORTHONORMAL_FRAME) ? kShadeOnb : kShadeRef);
    c.camera_packets = (d->flags & TR_RENDER_NO_CAMERA_PACKETS) == 0;
    c.path_launch = (d->flags & TR_RENDER_QUEUES) == 0;
    c.group = d->flags >> 24;
    return run_jobs(s->stream, s->wave, jobs, c, guide, s->compute_units, s->ev, &s->ev_made, stats, t_start);
}

}  // namespace

extern "C" {

int tr_render_transient(tr_scene s, const tr_camera* cam, tr_film f, const tr_render_desc* d, tr_render_stats* stats)
{
    return render_impl(s, cam, f, d, nullptr, stats);
}

int tr_render_transient_guided(tr_scene s, const tr_camera* cam, tr_film f, const tr_render_desc* d, tr_guide g,
                               tr_render_stats* stats)
{
    if (!g) return fail(TR_ERR_INVALID, "tr_render_transient_guided: null guide");
    if (d && (d->flags & TR_RENDER_TIME_SAMPLING))
        return fail(TR_ERR_INVALID, "tr_render_transient_guided: guiding does not combine with TR_RENDER_TIME_SAMPLING");
    return render_impl(s, cam, f, d, g, stats);
}

}  // extern "C"

// =============================================================================================
// batched renders and the launch-shape autotuner

struct tr_batch_s {
    struct Entry {
        tr_scene s;
        tr_camera cam;
        tr_film f;
        tr_render_desc d;
    };
    std::vector<Entry> entries;
    hipStream_t stream = nullptr;
    WaveBuffers wave;
    hipEvent_t ev[2 * 256] = {};
    bool ev_made = false;
    int compute_units = 256;
    bool tuned = false;
    LaunchCfg tune;

    ~tr_batch_s()
    {
        if (stream) (void)hipStreamSynchronize(stream);
        if (ev_made)
            for (auto& e : ev) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

LaunchCfg launch_cfg(const tr_batch_s* b, const tr_launch_desc* L)
{
    LaunchCfg c = b->tuned ? b->tune : LaunchCfg{};
    if (L) {
        if (L->wave_paths) c.wave = L->wave_paths;
        if (L->trace_per_cu) c.trace_per_cu = L->trace_per_cu;
        if (L->shade_per_cu) c.shade_per_cu = L->shade_per_cu;
        c.wide = (L->flags & TR_RENDER_BINARY_BVH) == 0;
        c.graph = (L->flags & TR_RENDER_GRAPH) != 0;
        c.prof = (L->flags & (TR_RENDER_PROFILE | TR_RENDER_PROFILE_EXTEND)) != 0;
        c.prof_extend = (L->flags & TR_RENDER_PROFILE) == 0 && (L->flags & TR_RENDER_PROFILE_EXTEND) != 0;
        c.mode = (L->flags & TR_RENDER_ORTHONORMAL_FRAME) ? kShadeOnb : kShadeRef;
        c.stack_fmt = stack_fmt_of(L->flags);
        c.per_job = (L->flags & TR_RENDER_PER_JOB) != 0;
        c.path_launch = (L->flags & TR_RENDER_QUEUES) == 0;
        c.group = L->flags >> 24;
    }
    return c;
}

// Renders the jobs of a batch: one shared sequence of wavefronts, or (per_job) one job after another
// on the same stream, with their statistics summed.
int run_batch(tr_batch_s* b, std::vector<HostJob>& jobs, const LaunchCfg& c, tr_render_stats* stats,
              std::chrono::steady_clock::time_point t0);

// sqrt_spp_cap > 0 lowers every job's sqrt_spp to at most the cap (autotuner trials)
int batch_jobs(tr_batch b, std::vector<HostJob>* jobs, int sqrt_spp_cap)
{
    jobs->resize(b->entries.size());
    for (size_t k = 0; k < b->entries.size(); ++k) {
        const auto& e = b->entries[k];
        tr_render_desc d = e.d;
        if (sqrt_spp_cap > 0) d.sqrt_spp = std::min(d.sqrt_spp, sqrt_spp_cap);
        int rc = make_job(e.s, &e.cam, e.f, &d, &(*jobs)[k], "tr_batch_render");
        if (rc) return rc;
    }
    return TR_OK;
}

}  // namespace

extern "C" {

int tr_batch_create(tr_batch* out)
{
    if (!out) return fail(TR_ERR_INVALID, "tr_batch_create: null output");
    *out = nullptr;
    int rc = check_device();
    if (rc) return rc;
    tr_batch b = new (std::nothrow) tr_batch_s();
    if (!b) return fail(TR_ERR_NOMEM, "tr_batch_create: host allocation");
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
        delete b;
        return fail(TR_ERR_DEVICE, "tr_batch_create: hipStreamCreate failed");
    }
    b->compute_units = tri::compute_units();
    *out = b;
    return TR_OK;
}

int tr_batch_destroy(tr_batch b)
{
    delete b;
    return TR_OK;
}

int tr_batch_add(tr_batch b, tr_scene s, const tr_camera* cam, tr_film f, const tr_render_desc* d, uint32_t* job)
{
    if (!b || !s || !cam || !f || !d) return fail(TR_ERR_INVALID, "tr_batch_add: null argument");
    for (const auto& e : b->entries)
        if (e.f == f) return fail(TR_ERR_INVALID, "tr_batch_add: every job needs its own film");
    if (b->entries.size() >= 65535u) return fail(TR_ERR_INVALID, "tr_batch_add: too many jobs");
    HostJob probe;
    int rc = make_job(s, cam, f, d, &probe, "tr_batch_add");
    if (rc) return rc;
    b->entries.push_back({s, *cam, f, *d});
    if (job) *job = uint32_t(b->entries.size() - 1);
    return TR_OK;
}

int tr_batch_clear(tr_batch b)
{
    if (!b) return fail(TR_ERR_INVALID, "tr_batch_clear: null batch");
    b->entries.clear();
    return TR_OK;
}

int tr_batch_render(tr_batch b, const tr_launch_desc* launch, tr_render_stats* stats)
{
    auto t0 = std::chrono::steady_clock::now();
    if (!b) return fail(TR_ERR_INVALID, "tr_batch_render: null batch");
    if (b->entries.empty()) return fail(TR_ERR_INVALID, "tr_batch_render: no job");
    std::vector<HostJob> jobs;
    int rc = batch_jobs(b, &jobs, 0);
    if (rc) return rc;
    return run_batch(b, jobs, launch_cfg(b, launch), stats, t0);
}

// a trial replaces the best shape only when it is faster by more than run-to-run noise
constexpr double kTuneMargin = 0.98;

int tr_autotune(tr_batch b, tr_launch_desc* best, double* ms_best)
{
    if (!b) return fail(TR_ERR_INVALID, "tr_autotune: null batch");
    if (b->entries.empty()) return fail(TR_ERR_INVALID, "tr_autotune: no job");
    std::vector<HostJob> jobs;
    int rc = batch_jobs(b, &jobs, 0);
    if (rc) return rc;
    uint64_t total = 0;
    int max_spp = 1;
    for (auto& j : jobs) total += j.paths;
    for (auto& e : b->entries) max_spp = std::max(max_spp, e.d.sqrt_spp);
    // the trials render the jobs with sqrt_spp capped so that a trial holds about as many paths as
    // the largest candidate wavefront (or the whole batch, when it is smaller): the wavefront size
    // that wins depends on how many paths are in flight
    const uint64_t kMaxWave = 1ull << 25;
    const uint64_t target = std::min<uint64_t>(total, kMaxWave);
    uint64_t trial_total = 0;
    for (int cap = 1; cap <= max_spp; ++cap) {
        if ((rc = batch_jobs(b, &jobs, cap))) return rc;
        trial_total = 0;
        for (auto& j : jobs) trial_total += j.paths;
        if (trial_total >= target) break;
    }
    LaunchCfg base = b->tuned ? b->tune : LaunchCfg{};
    // one trial: the capped jobs, best of two runs
    auto trial = [&](const LaunchCfg& c, double* ms) -> int {
        double m = 1e300;
        for (int rep = 0; rep < 2; ++rep) {
            tr_render_stats st;
            auto t0 = std::chrono::steady_clock::now();
            int r = run_batch(b, jobs, c, &st, t0);
            if (r) return r;
            m = std::min(m, st.render_ms);
        }
        *ms = m;
        return TR_OK;
    };
    // the current shape is the incumbent; stage 1: wavefront size and graph replay; stage 2: persistent
    // grid shapes; stage 3: stack formats
    LaunchCfg bestc = base;
    bestc.prof = false;
    double best_ms;
    if ((rc = trial(bestc, &best_ms))) return rc;
    std::vector<uint32_t> waves;
    for (uint32_t w : {1u << 18, 1u << 20, 1u << 22, 1u << 24, 1u << 25})
        if (w == (1u << 18) || w / 2 < trial_total) waves.push_back(w);
    for (uint32_t w : waves)
        for (bool g : {false, true}) {
            if (w == base.wave && g == base.graph) continue;
            LaunchCfg c = base;
            c.wave = w;
            c.graph = g;
            c.prof = false;
            double ms;
            if ((rc = trial(c, &ms))) return rc;
            if (ms < best_ms * kTuneMargin) best_ms = ms, bestc = c;
        }
    for (uint32_t tpc : {8u, 16u, 24u, 32u})
        for (uint32_t spc : {1u, 2u, 4u}) {
            if (tpc == bestc.trace_per_cu && spc == bestc.shade_per_cu) continue;
            LaunchCfg c = bestc;
            c.trace_per_cu = tpc;
            c.shade_per_cu = spc;
            double ms;
            if ((rc = trial(c, &ms))) return rc;
            if (ms < best_ms * kTuneMargin) best_ms = ms, bestc = c;
        }
    // stage 3: one job after another with the best shape (jobs large enough to fill the GPU on
    // their own gain the single-job kernels and the LDS-privatised film). Per-job launch overheads
    // shrink with the job sizes, so this is decided on the full jobs, one run each.
    if (jobs.size() > 1) {
        std::vector<HostJob> full;
        if ((rc = batch_jobs(b, &full, 0))) return rc;
        double ms[2];
        for (int pj = 0; pj < 2; ++pj) {
            LaunchCfg c = bestc;
            c.per_job = pj != 0;
            tr_render_stats st;
            if ((rc = run_batch(b, full, c, &st, std::chrono::steady_clock::now()))) return rc;
            ms[pj] = st.render_ms;
        }
        if (ms[1] < ms[0] * kTuneMargin) bestc.per_job = true;
    }
    // stage 4: traversal stack formats
    for (int fmt : {1, 2}) {
        LaunchCfg c = bestc;
        if (!c.wide || c.stack_fmt == fmt) continue;
        c.stack_fmt = fmt;
        double ms;
        if ((rc = trial(c, &ms))) return rc;
        if (ms < best_ms * kTuneMargin) best_ms = ms, bestc = c;
    }
    // the trials accumulated into the films
    for (auto& e : b->entries)
        if ((rc = tr_film_clear(e.f))) return rc;
    b->tune = bestc;
    b->tuned = true;
    if (b->entries.size() == 1) b->entries[0].s->tune = bestc;
    if (best) {
        best->wave_paths = bestc.wave;
        best->flags = (bestc.wide ? 0u : TR_RENDER_BINARY_BVH) | (bestc.graph ? TR_RENDER_GRAPH : 0u) |
                      (bestc.mode == kShadeOnb ? TR_RENDER_ORTHONORMAL_FRAME : 0u) | stack_flags_of(bestc.stack_fmt) |
                      (bestc.per_job ? TR_RENDER_PER_JOB : 0u);
        best->trace_per_cu = bestc.trace_per_cu;
        best->shade_per_cu = bestc.shade_per_cu;
    }
    if (ms_best) *ms_best = best_ms;
    return TR_OK;
}

}  // extern "C"

namespace {

// Per-job mode: jobs of at least kPerJobMinPaths paths (enough to fill the GPU on their own) render
// one after another with the single-job kernels and LDS-privatised film; the smaller ones share one
// sequence of wavefronts, where launch overheads are paid once for all of them.
constexpr uint64_t kPerJobMinPaths = 1ull << 22;

int run_batch(tr_batch_s* b, std::vector<HostJob>& jobs, const LaunchCfg& c, tr_render_stats* stats,
              std::chrono::steady_clock::time_point t0)
{
    if (!c.per_job || jobs.size() == 1)
        return run_jobs(b->stream, b->wave, jobs, c, nullptr, b->compute_units, b->ev, &b->ev_made, stats, t0);
    std::vector<std::vector<HostJob>> groups;
    std::vector<HostJob> small;
    for (auto& j : jobs) {
        if (j.paths >= kPerJobMinPaths) groups.emplace_back(1, j);
        else small.push_back(j);
    }
    if (!small.empty()) groups.push_back(std::move(small));
    tr_render_stats total{};
    for (auto& g : groups) {
        tr_render_stats st{};
        int rc = run_jobs(b->stream, b->wave, g, c, nullptr, b->compute_units, b->ev, &b->ev_made, &st, t0);
        if (rc) return rc;
        total.paths += st.paths;
        total.extension_rays += st.extension_rays;
        total.shadow_rays += st.shadow_rays;
        total.contributions += st.contributions;
        total.waves += st.waves;
        total.bounces_max = std::max(total.bounces_max, st.bounces_max);
        for (int k = 0; k < TR_K_COUNT; ++k) {
            total.kernel_ms[k] += st.kernel_ms[k];
            total.kernel_launches[k] += st.kernel_launches[k];
        }
    }
    total.render_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (stats) *stats = total;
    return TR_OK;
}

}  // namespace
