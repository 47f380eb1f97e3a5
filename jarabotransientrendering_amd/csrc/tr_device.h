// Device-side building blocks for gfx950: PCG32 streams, watertight BVH traversal, light and
// BSDF sampling. Included only by HIP translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <type_traits>

#include "tr_internal.h"

namespace trd {

// ---- float3 helpers ------------------------------------------------------------------------
struct f3 {
    float x, y, z;
};
__device__ __forceinline__ f3 mk(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ f3 mk(float4 v) { return f3{v.x, v.y, v.z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ f3 mul(f3 a, f3 b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ float dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b)
{
    return mk(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ f3 normalize(f3 a)
{
    float inv = 1.0f / sqrtf(dot(a, a));
    return a * inv;
}
__device__ __forceinline__ float comp(f3 v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

// ---- PCG32 (the reference's Random::RNG, src/Utils/RandomNumbers.h:119-174, 83-98), one stream
// per (seed, sequence). The increment is (seq << 1) | 1 and is recomputed from the sequence id. --
__device__ __forceinline__ uint32_t pcg_next(uint64_t& state, uint64_t inc)
{
    uint64_t old = state;
    state = old * 6364136223846793005ULL + inc;
    uint32_t xorshifted = uint32_t(((old >> 18u) ^ old) >> 27u);
    uint32_t rot = uint32_t(old >> 59u);
    return (xorshifted >> rot) | (xorshifted << ((0u - rot) & 31u));
}
__device__ __forceinline__ float pcg_float(uint64_t& state, uint64_t inc)
{
    uint32_t bits = (pcg_next(state, inc) >> 9) | 0x3f800000u;
    return __uint_as_float(bits) - 1.0f;
}
__device__ __forceinline__ uint64_t pcg_inc(uint64_t seq) { return (seq << 1u) | 1u; }
__device__ __forceinline__ uint64_t pcg_seed(uint64_t initstate, uint64_t seq)
{
    uint64_t inc = pcg_inc(seq), s = 0u;
    pcg_next(s, inc);
    s += initstate;
    pcg_next(s, inc);
    return s;
}

// The state of the stream with increment `inc` after n draws. A step is s -> a s + inc, so n + 1 steps
// from (inc + seed) (where pcg_seed stands before its last one) give A (inc + seed) + C inc with
// A = a^(n + 1) and C = 1 + a + ... + a^n mod 2^64 (F. Brown, "Random number generation with arbitrary
// strides", 1994), read from a table: a path keeps a stream as its number of draws instead of a state.
constexpr uint32_t kPcgJumps = 768;  // three draws per vertex, at most 255 vertices
struct PcgJumps {
    uint64_t ac[kPcgJumps][2];
};
constexpr PcgJumps pcg_jumps()
{
    PcgJumps t{};
    uint64_t a = 1, c = 0;
    for (uint32_t n = 0; n < kPcgJumps; ++n) {
        c += a;
        a *= 6364136223846793005ULL;
        t.ac[n][0] = a;
        t.ac[n][1] = c;
    }
    return t;
}
__device__ __constant__ const PcgJumps kPcgJump = pcg_jumps();
__device__ __forceinline__ uint64_t pcg_at(uint64_t initstate, uint64_t inc, uint32_t n)
{
    return kPcgJump.ac[n][0] * (inc + initstate) + kPcgJump.ac[n][1] * inc;
}

// ---- wave-aggregated queue append (one atomic per wavefront) -------------------------------
__device__ __forceinline__ uint32_t wave_append(uint32_t* counter, bool pred)
{
    uint64_t mask = __ballot(pred);
    uint32_t lane = __lane_id();
    uint32_t base = 0;
    if (mask != 0) {
        int leader = __ffsll((long long)mask) - 1;
        if (int(lane) == leader) base = atomicAdd(counter, uint32_t(__popcll(mask)));
        base = __shfl(base, leader);
    }
    return base + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
}

// ---- block-aggregated append to two queues with one atomic ----------------------------------
// As block_append for two queues whose lengths are the low and high halves of one 64-bit counter
// (`pair`, 8-byte aligned): each thread passes its items for queue A (0 or 1) and queue B (0 or 1)
// and gets its positions in both; the block issues a single 64-bit atomic. Per-block counts fit
// 16 bits (blocks of at most 1024 threads), so the two scans run packed in one 32-bit value.
__device__ __forceinline__ void block_append2(uint32_t* pair, uint32_t cnt_a, uint32_t cnt_b, uint32_t* smem,
                                              uint32_t* pos_a, uint32_t* pos_b)
{
    const uint32_t lane = __lane_id(), wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    const uint32_t mine = cnt_a | (cnt_b << 16);
    uint32_t x = mine;  // inclusive scan within the wavefront, both halves at once
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) smem[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < nw; ++w) {
            uint32_t t = smem[w];
            smem[w] = total;  // exclusive prefix of wavefront totals
            total += t;
        }
        unsigned long long old = 0ull;
        if (total)
            old = atomicAdd(reinterpret_cast<unsigned long long*>(pair),
                            (unsigned long long)(total & 0xFFFFu) | ((unsigned long long)(total >> 16) << 32));
        smem[nw] = uint32_t(old);
        smem[nw + 1] = uint32_t(old >> 32);
    }
    __syncthreads();
    const uint32_t pre = smem[wid] + x - mine;
    *pos_a = smem[nw] + (pre & 0xFFFFu);
    *pos_b = smem[nw + 1] + (pre >> 16);
    __syncthreads();  // smem may be reused by the caller's next iteration
}

// ---- block-aggregated queue append ----------------------------------------------------------
// Every thread of the block calls this with its number of items (0 or more); the block issues one
// atomic on `counter` and each thread gets the first queue position of its items. `smem` holds at
// least blockDim.x / 64 + 1 words. Same-address atomics from every wavefront are the limiting
// rate at tens of millions of queue entries, hence one per block.
__device__ __forceinline__ uint32_t block_append(uint32_t* counter, uint32_t cnt, uint32_t* smem)
{
    const uint32_t lane = __lane_id(), wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    uint32_t x = cnt;  // inclusive scan within the wavefront
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) smem[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < nw; ++w) {
            uint32_t t = smem[w];
            smem[w] = total;  // exclusive prefix of wavefront totals
            total += t;
        }
        smem[nw] = total ? atomicAdd(counter, total) : 0u;
    }
    __syncthreads();
    uint32_t pos = smem[nw] + smem[wid] + x - cnt;
    __syncthreads();  // smem may be reused by the caller's next iteration
    return pos;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// ---- ray/box and watertight ray/triangle -----------------------------------------------------
struct RayPre {
    f3 o, inv;
    f3 c0, c1;            // -(o * inv) -+ k |inv|: slab offsets of entry and exit planes (4-wide BVH)
    uint32_t sx, sy, sz;  // byte selectors of the entry planes of children 0 and 1, per axis (kPermUp)
    f3 o_rot;             // origin components in (kx, ky, kz) order
    uint32_t rot4;        // 4 * kx: byte offset of the (kx, ky, kz) run in a rotated triangle vertex (TriRot)
    float Sx, Sy, Sz;
};

// reciprocal for slab tests; zero components become +-1e20 so that (lo - o) * inv never
// evaluates 0 * inf (a ray lying in a box face plane stays inside that slab)
__device__ __forceinline__ float safe_rcp(float d)
{
    return 1.0f / (fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d);
}

// Entry planes of an axis for a ray going up (down) it: the lower (upper) ones. v_perm_b32 picks
// them from the (upper, lower) plane words and spreads two of them to 16-bit halves (0x0c is a zero
// byte); with the words swapped the same selector picks the exit planes. Children 2 and 3 are two
// bytes further on.
constexpr uint32_t kPermUp = 0x0c010c00u, kPermDown = 0x0c050c04u, kPermNext = 0x00020002u;

// Offset and margin of the quantized node test. A plane at P = origin + q * step (one rounding
// on the host) is entered at (P - o) * inv; the node test evaluates it as fma(q, step * inv, b) with
// b = fma(origin, inv, c) and c = -(o * inv) -+ k |inv| (entry planes down, exit planes up), so a plane
// costs one operation and an axis three more per node. The roundings, each at most u = 2^-24 of
// its result, are: the host plane u (|origin| + 255 step) |inv|, o * inv and c together
// u (2 |o| |inv| + m) with m = k |inv|, b u (|origin| |inv| + |o| |inv| + m) and the plane distance
// u (|b| + 255 step |inv|). With C >= |origin| + 255 step for every node (plane_bound) they sum to at
// most u |inv| (4 C + 5 |o|) + 3 u m. Exit planes also make up for the 3 ulp by which box_far moves
// a hit's distance out: 6 u (C + |o|) |inv| more. k = 1e-6 (C + max |o|) (over 16 u (C + |o|))
// exceeds the sum: the entry plane is never late and the exit plane never early.
__device__ __forceinline__ RayPre ray_pre(f3 o, f3 d, float plane_bound)
{
    RayPre r;
    r.o = o;
    r.inv = mk(safe_rcp(d.x), safe_rcp(d.y), safe_rcp(d.z));
    const float k = 1e-6f * (plane_bound + fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z)));
    const f3 c = mk(-(o.x * r.inv.x), -(o.y * r.inv.y), -(o.z * r.inv.z));
    r.c0 = mk(fmaf(-k, fabsf(r.inv.x), c.x), fmaf(-k, fabsf(r.inv.y), c.y), fmaf(-k, fabsf(r.inv.z), c.z));
    r.c1 = mk(fmaf(k, fabsf(r.inv.x), c.x), fmaf(k, fabsf(r.inv.y), c.y), fmaf(k, fabsf(r.inv.z), c.z));
    r.sx = r.inv.x >= 0.0f ? kPermUp : kPermDown;
    r.sy = r.inv.y >= 0.0f ? kPermUp : kPermDown;
    r.sz = r.inv.z >= 0.0f ? kPermUp : kPermDown;
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1 == 3 ? 0 : kz + 1;
    int ky = kx + 1 == 3 ? 0 : kx + 1;
    // The paper swaps kx and ky when d[kz] < 0 to keep the winding; that only negates U, V, W, det
    // and T (each exactly), so the hit test and T / det are the same without it.
    r.rot4 = 4u * uint32_t(kx);
    r.o_rot = mk(comp(o, kx), comp(o, ky), comp(o, kz));
    // 1 / d[kz]: the slab reciprocal unless that was clamped
    const float dz = comp(d, kz);
    r.Sz = comp(r.inv, kz);
    if (fabsf(dz) < 1e-20f) r.Sz = 1.0f / dz;
    r.Sx = comp(d, kx) * r.Sz;
    r.Sy = comp(d, ky) * r.Sz;
    return r;
}

// Rotated triangle record (TriRot, 16 floats = 64 bytes, slot order): vertex v at floats
// [5v, 5v + 5) as (x, y, z, x, y), so that the components (kx, ky, kz) = (kz+1, kz+2, kz) mod 3
// of any ray are three consecutive floats starting at kx; float 15 = scene triangle index bits.
struct __attribute__((packed, aligned(4))) Packed3 {
    float x, y, z;
};

// The far bound of box tests for a hit at distance t: three ulp further (also behind the origin, where t is
// negative), so that a box whose triangle lies at exactly t is still entered.
__device__ __forceinline__ float box_far(float t) { return fmaf(fabsf(t), 0x1.8p-22f, t); }

// Tests the triangle record at byte offset `off` of `tris` (its slot is `slot`) against the current
// hit: updates hit (a slot) and tfar; equal-distance ties go to the lower scene triangle index, which
// is read only for a tie.
//
// Woop, Benthin, Wald, "Watertight Ray/Triangle Intersection", JCGT 2(1) 2013, Sec. 4 (no
// backface culling; double-precision re-evaluation when an edge function is exactly zero).
template <class Off>
__device__ __forceinline__ void tri_hit(const RayPre& r, const char* __restrict__ tris, Off off, int32_t slot,
                                        float tnear, float& tfar, int32_t& hit)
{
    // No fused multiply-adds here: an edge shared by two triangles must evaluate to exactly
    // opposite values in both, which fma(Cx, By, -Cy*Bx) vs fma(Bx, Cy, -By*Cx) does not give.
#pragma clang fp contract(off)
    const char* t = tris + (off + Off(r.rot4));
    const Packed3 a = *reinterpret_cast<const Packed3*>(t);
    const Packed3 b = *reinterpret_cast<const Packed3*>(t + 20);
    const Packed3 c = *reinterpret_cast<const Packed3*>(t + 40);
    float Akx = a.x - r.o_rot.x, Aky = a.y - r.o_rot.y, Akz = a.z - r.o_rot.z;
    float Bkx = b.x - r.o_rot.x, Bky = b.y - r.o_rot.y, Bkz = b.z - r.o_rot.z;
    float Ckx = c.x - r.o_rot.x, Cky = c.y - r.o_rot.y, Ckz = c.z - r.o_rot.z;
    float Ax = Akx - r.Sx * Akz, Ay = Aky - r.Sy * Akz;
    float Bx = Bkx - r.Sx * Bkz, By = Bky - r.Sy * Bkz;
    float Cx = Ckx - r.Sx * Ckz, Cy = Cky - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (fminf(fminf(fabsf(U), fabsf(V)), fabsf(W)) == 0.0f) {
        U = float(double(Cx) * double(By) - double(Cy) * double(Bx));
        V = float(double(Ax) * double(Cy) - double(Ay) * double(Cx));
        W = float(double(Bx) * double(Ay) - double(By) * double(Ax));
    }
    const bool neg = fminf(fminf(U, V), W) < 0.0f, pos = fmaxf(fmaxf(U, V), W) > 0.0f;
    const float det = U + V + W;
    // outside the triangle's interior and edges, or degenerate
    if ((neg & pos) | (det == 0.0f)) return;
    const float T = U * (r.Sz * Akz) + V * (r.Sz * Bkz) + W * (r.Sz * Ckz);
    // divide only when an estimate of the distance is near (tnear, tfar]
    const float te = T * __builtin_amdgcn_rcpf(det);
    if (!((te >= fmaf(fabsf(tnear), -1e-5f, tnear)) & (te <= fmaf(fabsf(tfar), 1e-5f, tfar)))) return;
    const float th = T / det;
    if (!((th > tnear) & (th <= tfar))) return;
    if (th == tfar && hit >= 0) {
        const int32_t id = *reinterpret_cast<const int32_t*>(tris + (off + Off(60)));
        const int32_t id_hit = *reinterpret_cast<const int32_t*>(tris + (Off(uint32_t(hit)) * 64 + 60));
        if (id >= id_hit) return;
    }
    hit = slot;
    tfar = th;
}

// Closest (ANY = false) or any (ANY = true) hit in (tnear, tfar]. On a closest hit `tfar` is
// updated. Equal-distance ties resolve to the lower scene triangle index. `stack` points at this
// thread's first LDS stack slot; consecutive slots are `stride` ints apart.
// Returns the triangle's slot or -1.
template <bool ANY>
__device__ __forceinline__ int32_t trace(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                         const RayPre& r, float tnear, float& tfar, int32_t* stack,
                                         int stride)
{
    int32_t hit = -1;
    int32_t node = 0;
    int sp = 0;
    for (;;) {
        const float4* n = nodes + 4 * size_t(node);
        float4 a = n[0], b = n[1], c = n[2];
        int4 dd = *reinterpret_cast<const int4*>(n + 3);
        // slab tests as (lo - o) * inv: exact at a face through the origin, three roundings per
        // bound, so the far distance is widened by 1 + 2*gamma(3) (PBRT 3.9.2)
        float lx0 = (a.x - r.o.x) * r.inv.x, lx1 = (a.y - r.o.x) * r.inv.x;
        float ly0 = (a.z - r.o.y) * r.inv.y, ly1 = (a.w - r.o.y) * r.inv.y;
        float lz0 = (c.x - r.o.z) * r.inv.z, lz1 = (c.y - r.o.z) * r.inv.z;
        float rx0 = (b.x - r.o.x) * r.inv.x, rx1 = (b.y - r.o.x) * r.inv.x;
        float ry0 = (b.z - r.o.y) * r.inv.y, ry1 = (b.w - r.o.y) * r.inv.y;
        float rz0 = (c.z - r.o.z) * r.inv.z, rz1 = (c.w - r.o.z) * r.inv.z;
        float tl0 = fmaxf(fmaxf(fminf(lx0, lx1), fminf(ly0, ly1)), fmaxf(fminf(lz0, lz1), tnear));
        float tl1 = fminf(fminf(fmaxf(lx0, lx1), fmaxf(ly0, ly1)), fminf(fmaxf(lz0, lz1), tfar));
        float tr0 = fmaxf(fmaxf(fminf(rx0, rx1), fminf(ry0, ry1)), fmaxf(fminf(rz0, rz1), tnear));
        float tr1 = fminf(fminf(fmaxf(rx0, rx1), fmaxf(ry0, ry1)), fminf(fmaxf(rz0, rz1), tfar));
        bool hl = (tl0 <= box_far(tl1)) && dd.z >= 0;
        bool hr = (tr0 <= box_far(tr1)) && dd.w >= 0;
        // leaf children: test their triangles now
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            bool h = side == 0 ? hl : hr;
            int cnt = side == 0 ? dd.z : dd.w;
            if (h && cnt > 0) {
                int first = side == 0 ? dd.x : dd.y;
                for (int i = first; i < first + cnt; ++i) {
                    tri_hit<size_t>(r, reinterpret_cast<const char*>(tris), size_t(i) * 64, i, tnear, tfar, hit);
                    if (ANY && hit >= 0) return hit;
                }
                if (side == 0) hl = false;
                else hr = false;
            }
        }
        if (hl && hr) {
            bool left_first = tl0 <= tr0;
            stack[sp * stride] = left_first ? dd.y : dd.x;
            ++sp;
            node = left_first ? dd.x : dd.y;
        } else if (hl) {
            node = dd.x;
        } else if (hr) {
            node = dd.y;
        } else {
            if (sp == 0) break;
            --sp;
            node = stack[sp * stride];
        }
    }
    return hit;
}

// Traversal stack entry formats of the 4-wide BVH, kept in LDS, one column per thread (entry e of
// thread `tid` is element e * stride + tid):
//   kStack32   : 32-bit node index;
//   kStack16   : 16-bit node index (BVHs of at most 65,536 nodes): half the LDS, so more
//                wavefronts fit on a compute unit;
//   kStackKeyed: 16-bit node index | the upper 16 bits of the child's entry distance (a lower bound
//                of it, the float truncated to 7 mantissa bits): a closest-hit query skips a popped
//                child that starts beyond the current hit without fetching the node.
enum { kStack32 = 0, kStack16 = 1, kStackKeyed = 2 };

// Per-lane state of a 4-wide BVH query between node steps.
struct Trav4 {
    uint32_t node;    // node to visit next
    uint32_t sp;      // element index of the next free stack entry
    int32_t hit;      // slot of the closest (or any) hit so far, -1 if none
    float tfar;       // current far bound (the hit distance once there is a hit)
    uint32_t leaves;  // leaf mode: triangles of the last node still to test (bit 8 k + j: slot tri0 + j)
    uint32_t tri0;    // ... and that node's first triangle slot
    uint32_t p[4];    // closest hit: the node's entered inner children, nearest first, held back in leaf mode
};

__device__ __forceinline__ void trav4_begin(Trav4& st, float tfar, uint32_t tid)
{
    st.node = 0;
    st.sp = tid;
    st.hit = -1;
    st.tfar = tfar;
    st.leaves = 0;
    st.tri0 = 0;
}

// q * a + b for the 8-bit planes q held in the halves of `p`. A byte in a 16-bit half is the
// half-precision subnormal q * 2^-24, which v_fma_mix_f32 takes as it is (exactly; a is held scaled
// by 2^24): no conversion instruction per plane.
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float plane_lo(uint32_t p, float a, float b)
{
    return fmaf(float(__builtin_bit_cast(half2v, p).x), a, b);
}
__device__ __forceinline__ float plane_hi(uint32_t p, float a, float b)
{
    return fmaf(float(__builtin_bit_cast(half2v, p).y), a, b);
}

// Entry distances t0[k] (at least tnear) of the four child boxes of a node (Bvh4DevNode) and whether
// the ray meets them in [tnear, tfar_box]. n / f: entry / exit plane pairs per axis, [2 axis] of
// children 0 and 1, [2 axis + 1] of children 2 and 3.
__device__ __forceinline__ void slabs4(const RayPre& r, const uint4& w0, const uint4& w3, const uint32_t (&n)[6],
                                       const uint32_t (&f)[6], float tnear, float tfar_box, float (&t0)[4], bool (&ent)[4])
{
    const float ox = __uint_as_float(w0.x), oy = __uint_as_float(w0.y), oz = __uint_as_float(w0.z);
    const float ax = __uint_as_float(w3.x) * r.inv.x, ay = __uint_as_float(w3.y) * r.inv.y,
                az = __uint_as_float(w3.z) * r.inv.z;
    const float bx0 = fmaf(ox, r.inv.x, r.c0.x), by0 = fmaf(oy, r.inv.y, r.c0.y), bz0 = fmaf(oz, r.inv.z, r.c0.z);
    const float bx1 = fmaf(ox, r.inv.x, r.c1.x), by1 = fmaf(oy, r.inv.y, r.c1.y), bz1 = fmaf(oz, r.inv.z, r.c1.z);
#define TR_CHILD(k, P, h)                                                                                        \
    t0[k] = fmaxf(fmaxf(P(n[h], ax, bx0), P(n[2 + h], ay, by0)), fmaxf(P(n[4 + h], az, bz0), tnear));            \
    ent[k] = t0[k] <= fminf(fminf(P(f[h], ax, bx1), P(f[2 + h], ay, by1)), fminf(P(f[4 + h], az, bz1), tfar_box));
    TR_CHILD(0, plane_lo, 0)
    TR_CHILD(1, plane_hi, 0)
    TR_CHILD(2, plane_lo, 1)
    TR_CHILD(3, plane_hi, 1)
#undef TR_CHILD
}

// the same with each lane's own entry / exit selection
__device__ __forceinline__ void node_slabs(const RayPre& r, const uint4& w0, const uint4& w1, const uint4& w2,
                                           const uint4& w3, float tnear, float tfar_box, float (&t0)[4], bool (&ent)[4])
{
    const uint32_t sx2 = r.sx + kPermNext, sy2 = r.sy + kPermNext, sz2 = r.sz + kPermNext;
    const uint32_t n[6] = {__builtin_amdgcn_perm(w1.y, w1.x, r.sx), __builtin_amdgcn_perm(w1.y, w1.x, sx2),
                           __builtin_amdgcn_perm(w1.w, w1.z, r.sy), __builtin_amdgcn_perm(w1.w, w1.z, sy2),
                           __builtin_amdgcn_perm(w2.y, w2.x, r.sz), __builtin_amdgcn_perm(w2.y, w2.x, sz2)};
    const uint32_t f[6] = {__builtin_amdgcn_perm(w1.x, w1.y, r.sx), __builtin_amdgcn_perm(w1.x, w1.y, sx2),
                           __builtin_amdgcn_perm(w1.z, w1.w, r.sy), __builtin_amdgcn_perm(w1.z, w1.w, sy2),
                           __builtin_amdgcn_perm(w2.x, w2.y, r.sz), __builtin_amdgcn_perm(w2.x, w2.y, sz2)};
    slabs4(r, w0, w3, n, f, tnear, tfar_box, t0, ent);
}

// One step of a closest (ANY = false) or any (ANY = true) hit query over the quantized 4-wide BVH
// (Bvh4DevNode: 4 x 16 bytes per node). A lane either visits a node or, while triangles of its last
// node's entered leaves are left to test, tests one of them (leaf mode), so a wavefront does not wait
// on the few lanes that loop over their leaves. The inner children the ray enters are pushed
// far-to-near and the nearest is visited next; a closest-hit query holds them back (st.p) until its
// triangles are tested and drops those behind the hit, an any-hit query pushes all of them at once,
// in slot order. Queries that take no leaf mode (32-bit stack entries, or !POS) loop over the node's
// triangles in the step. Returns true when the query is complete (st.hit, st.tfar hold the
// answer). `stack` is the block's LDS stack, `tid` this thread's column and `stride` the block size.
// POS: every tnear of the launch is positive, so that entry distances order like their bits (renders;
// not the public queries).
//
// The step is bound by VALU issue (a wavefront issues an instruction on nearly every cycle of its
// SIMD, with about half its lanes active), so what counts is instructions per step: planes taken as
// half-precision subnormals (no conversions), children as (distance, index) words sorted by integer
// min / max, triangles as one bit mask over consecutive slots, hits kept as slots (no index loads) and
// addresses in 32 bits took a node visit of a closest-hit query from about 190 to 115 VALU
// instructions and a triangle test from 90 to 70; leaf mode for closest hits saved a further tenth
// (holding the children back keeps the culling that pushing them at once loses). On the
// 81,930-triangle frame of 67 M paths: closest hits 11.8 -> 9.8 ms, any hits 9.9 -> 7.1 ms, frame
// 31.1 -> 25.5 ms. Lost: any-hit queries that loop over their triangles in the step (7.1 -> 8.7 ms),
// triangle tests only once 6 to 20 lanes wait for one (extend 9.8 -> 10.5-10.9 ms), keyed entries by
// default (12.0 ms: twice the LDS), one triangle per leaf (10.0 ms).
template <bool ANY, int SK, bool POS>
__device__ __forceinline__ bool trace4_step(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                            const RayPre& r, float tnear, Trav4& st, uint32_t* stack, uint32_t tid,
                                            uint32_t stride)
{
    static_assert(!(ANY && SK == kStackKeyed), "any-hit queries keep no entry distances");
    static_assert(!(SK == kStackKeyed && !POS), "keyed entries need positive distances");
    constexpr bool PACKED = !ANY && SK != kStack32 && POS;  // (distance, child) words of 32 bits
    // 16-bit node indices: at most 65,536 nodes with eight triangles each, so byte offsets fit 32 bits
    typedef typename std::conditional<SK == kStack32, size_t, uint32_t>::type Off;
    const char* tri_base = reinterpret_cast<const char*>(tris);
    auto push = [&](uint32_t e) {
        if constexpr (SK == kStack16) reinterpret_cast<uint16_t*>(stack)[st.sp] = uint16_t(e);
        else stack[st.sp] = e;
        st.sp += stride;
    };
    auto top = [&]() -> uint32_t {
        if constexpr (SK == kStack16) return reinterpret_cast<const uint16_t*>(stack)[st.sp];
        else return stack[st.sp];
    };
    auto test = [&](uint32_t tri0, uint32_t leaves) {
        const uint32_t slot = tri0 + (uint32_t(__builtin_ctz(leaves)) & 7u);
        tri_hit<Off>(r, tri_base, Off(slot) * 64, int32_t(slot), tnear, st.tfar, st.hit);
    };
    if ((ANY || PACKED) && st.leaves) {
        test(st.tri0, st.leaves);
        if (ANY && st.hit >= 0) return true;
        st.leaves &= st.leaves - 1u;
    } else {
        const uint4* nd = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(nodes) + Off(st.node) * 64);
        const uint4 w0 = nd[0], w1 = nd[1], w2 = nd[2], w3 = nd[3];
        const uint32_t child0 = w0.w, meta = w2.z, tri0 = w2.w, n_inner = w3.w;
        float t0[4];
        bool ent[4];
        node_slabs(r, w0, w1, w2, w3, tnear, box_far(st.tfar), t0, ent);
        // triangles of the entered leaf children: byte k of `meta` marks those of child k
        uint32_t leaves = ((ent[0] ? 0x000000FFu : 0u) | (ent[1] ? 0x0000FF00u : 0u) | (ent[2] ? 0x00FF0000u : 0u) |
                           (ent[3] ? 0xFF000000u : 0u)) & meta;
        if constexpr (ANY) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (ent[k] & (k < n_inner)) push(child0 + k);
            st.leaves = leaves;
            st.tri0 = tri0;
        } else if constexpr (PACKED) {
            // (entry distance, child) in one word, the distance truncated to its upper 16 bits: sorted
            // with integer min / max; ~0: not entered
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t e = (__float_as_uint(t0[k]) & 0xFFFF0000u) | (child0 + k);
                st.p[k] = (ent[k] & (k < n_inner)) ? e : 0xFFFFFFFFu;
            }
#define TR_CSWAP(a, b)                                                                \
    {                                                                                 \
        const uint32_t lo = min(st.p[a], st.p[b]), hi = max(st.p[a], st.p[b]);        \
        st.p[a] = lo;                                                                 \
        st.p[b] = hi;                                                                 \
    }
            TR_CSWAP(0, 1) TR_CSWAP(2, 3) TR_CSWAP(0, 2) TR_CSWAP(1, 3) TR_CSWAP(1, 2)
#undef TR_CSWAP
            st.leaves = leaves;
            st.tri0 = tri0;
        } else {
            for (; leaves; leaves &= leaves - 1u) test(tri0, leaves);
            float key[4];
            int32_t idx[4];
            const float lim = box_far(st.tfar);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool h = ent[k] & (uint32_t(k) < n_inner) & (t0[k] <= lim);
                key[k] = h ? t0[k] : __int_as_float(0x7f800000);
                idx[k] = h ? int32_t(child0 + uint32_t(k)) : -1;
            }
            // sort (key, idx) ascending: 5-comparator network; nearest child first
#define TR_CSWAP(a, b)                                                            \
    if (key[b] < key[a]) {                                                        \
        float tk = key[a]; key[a] = key[b]; key[b] = tk;                          \
        int ti = idx[a]; idx[a] = idx[b]; idx[b] = ti;                            \
    }
            TR_CSWAP(0, 1) TR_CSWAP(2, 3) TR_CSWAP(0, 2) TR_CSWAP(1, 3) TR_CSWAP(1, 2)
#undef TR_CSWAP
#pragma unroll
            for (int k = 3; k >= 1; --k)
                if (idx[k] >= 0) push(uint32_t(idx[k]));
            if (idx[0] >= 0) {
                st.node = uint32_t(idx[0]);
                return false;
            }
        }
    }
    if ((ANY || PACKED) && st.leaves) return false;
    if constexpr (PACKED) {
        // words above `lim` start behind the hit or are not entered
        const uint32_t lim = __float_as_uint(box_far(st.tfar)) | 0xFFFFu;
#pragma unroll
        for (int k = 3; k >= 1; --k)
            if (st.p[k] <= lim) push(st.p[k]);
        if (st.p[0] <= lim) {
            st.node = st.p[0] & 0xFFFFu;
            return false;
        }
        if constexpr (SK == kStackKeyed) {
            while (st.sp != tid) {
                st.sp -= stride;
                const uint32_t e = top();
                if (e <= lim) {
                    st.node = e & 0xFFFFu;
                    return false;
                }
            }
            return true;
        }
    }
    if (st.sp == tid) return true;
    st.sp -= stride;
    st.node = top();
    return false;
}

// ---- closest hit of a wavefront's rays as one packet ------------------------------------------
// The camera rays of one pixel's samples nearly share their traversal. Here the wavefront visits one
// node at a time for all its lanes: a node is visited when the ray of any active lane enters it, so
// the node index and the traversal stack are uniform, node and triangle reads are the same address
// for every lane, and every lane runs the same instruction stream (a per-lane query runs each node
// step with about half the lanes of a wavefront active). Each lane keeps its own closest hit and far
// bound, tests the triangles of a leaf its ray enters, and drops a child whose box starts beyond its
// hit. A lane's answer is the one trace4_step gives: the closest hit does not depend on the order of
// the visits or on visits of boxes the ray misses (equal distances resolve to the lower triangle
// index). Children are visited nearest first by the entry distances of the first active lane.
// When the directions of all active lanes have the same signs (nearly every pixel), entry and exit
// planes are the same for every lane and are picked and spread on the scalar unit.
// `col` is the stack column of the wavefront's first lane (all lanes write the same entries); tnear
// is positive.
template <int SK>
__device__ __forceinline__ void trace4_packet(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                              const RayPre& r, float tnear, bool active, float& tfar, int32_t& hit,
                                              uint32_t* stack, int col, int stride)
{
    typedef typename std::conditional<SK == kStack32, size_t, uint32_t>::type Off;
    const uint64_t amask = __ballot(active);
    if (amask == 0ull) return;
    const int lead = int(__builtin_ctzll(amask));
    const uint64_t upx = __ballot(active && r.sx == kPermUp), upy = __ballot(active && r.sy == kPermUp),
                   upz = __ballot(active && r.sz == kPermUp);
    const bool same = (upx == 0ull || upx == amask) && (upy == 0ull || upy == amask) && (upz == 0ull || upz == amask);
    const char* tri_base = reinterpret_cast<const char*>(tris);
    auto push = [&](int sp, uint32_t child) {
        if constexpr (SK == kStack16) reinterpret_cast<uint16_t*>(stack)[sp * stride + col] = uint16_t(child);
        else stack[sp * stride + col] = child;
    };
    auto pop = [&](int sp) -> uint32_t {
        if constexpr (SK == kStack16) return uint32_t(reinterpret_cast<const uint16_t*>(stack)[sp * stride + col]);
        else return stack[sp * stride + col];
    };
    // the node is the same for every lane: the device pass reads it through the constant address
    // space, so that the compiler uses scalar loads (one per wavefront, into scalar registers); the
    // host pass, which only parses this function, has no such address space
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(4))) const uint4 cuint4;
#else
    typedef const uint4 cuint4;
#endif
    // two plane bytes in the halves of a word, as v_perm_b32 spreads them
    auto spread01 = [](uint32_t q) { return (q & 0xFFu) | ((q & 0xFF00u) << 8); };
    auto spread23 = [](uint32_t q) { return ((q >> 16) & 0xFFu) | ((q >> 8) & 0xFF0000u); };
    uint32_t node = 0;
    int sp = 0;
    for (;;) {
        node = uint32_t(__builtin_amdgcn_readfirstlane(int(node)));
        const cuint4* nd = (const cuint4*)(reinterpret_cast<const char*>(nodes) + size_t(node) * 64);
        const uint4 w0 = nd[0], w1 = nd[1], w2 = nd[2], w3 = nd[3];
        const uint32_t child0 = w0.w, meta = w2.z, tri0 = w2.w, n_inner = w3.w;
        float t0[4];
        bool ent[4];
        if (same) {
            const uint32_t nx = upx ? w1.x : w1.y, fx = upx ? w1.y : w1.x;
            const uint32_t ny = upy ? w1.z : w1.w, fy = upy ? w1.w : w1.z;
            const uint32_t nz = upz ? w2.x : w2.y, fz = upz ? w2.y : w2.x;
            const uint32_t n[6] = {spread01(nx), spread23(nx), spread01(ny), spread23(ny), spread01(nz), spread23(nz)};
            const uint32_t f[6] = {spread01(fx), spread23(fx), spread01(fy), spread23(fy), spread01(fz), spread23(fz)};
            slabs4(r, w0, w3, n, f, tnear, box_far(tfar), t0, ent);
        } else {
            node_slabs(r, w0, w1, w2, w3, tnear, box_far(tfar), t0, ent);
        }
        // leaves first: the wavefront loops over the triangles of every leaf some lane entered;
        // each lane tests those of the leaves its ray entered
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool e = active && ent[k];
            if (k >= n_inner && __ballot(e) != 0ull) {
                for (uint32_t m = (meta >> (8 * k)) & 0xFFu; m; m &= m - 1u) {
                    const uint32_t slot = tri0 + uint32_t(__builtin_ctz(m));
                    if (e) tri_hit<Off>(r, tri_base, Off(slot) * 64, int32_t(slot), tnear, tfar, hit);
                }
            }
        }
        // inner children that some lane enters before its hit, ordered by the first active lane's
        // entry distances (children that lane does not enter last; distances are positive, so their
        // bits order like them)
        const float lim = box_far(tfar);
        uint32_t uk[4], ui[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool e = active && ent[k] && k < n_inner && t0[k] <= lim;
            const bool any = __ballot(e) != 0ull;
            const uint32_t lk = uint32_t(__builtin_amdgcn_readlane(e ? __float_as_int(t0[k]) : 0x7f800000, lead));
            uk[k] = any ? lk : 0xFFFFFFFFu;
            ui[k] = child0 + k;
        }
#define TR_PSWAP(a, b)                                                                \
    if (uk[b] < uk[a]) {                                                              \
        uint32_t tk = uk[a]; uk[a] = uk[b]; uk[b] = tk;                               \
        uint32_t ti = ui[a]; ui[a] = ui[b]; ui[b] = ti;                               \
    }
        TR_PSWAP(0, 1) TR_PSWAP(2, 3) TR_PSWAP(0, 2) TR_PSWAP(1, 3) TR_PSWAP(1, 2)
#undef TR_PSWAP
        if (uk[0] == 0xFFFFFFFFu) {
            if (sp == 0) break;
            --sp;
            node = pop(sp);
            continue;
        }
#pragma unroll
        for (int k = 3; k >= 1; --k)
            if (uk[k] != 0xFFFFFFFFu) {
                push(sp, ui[k]);
                ++sp;
            }
        node = ui[0];
    }
}

template <bool ANY, int SK, bool POS>
__device__ __forceinline__ int32_t trace4(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                          const RayPre& r, float tnear, float& tfar, uint32_t* stack, uint32_t tid,
                                          uint32_t stride)
{
    Trav4 st;
    trav4_begin(st, tfar, tid);
    while (!trace4_step<ANY, SK, POS>(nodes, tris, r, tnear, st, stack, tid, stride)) {
    }
    tfar = st.tfar;
    return st.hit;
}

}  // namespace trd
