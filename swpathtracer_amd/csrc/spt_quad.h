// spt_quad.h - persistent closest-hit traversal with four lanes per ray.
//
// One lane per ray kept 17-20 of a wave's 64 lanes active per VALU instruction
// (lanes wait for each other across node and leaf phases) and the VALU was
// the limit: about 120 wave instructions a ray. Here the four lanes of a quad
// share a ray. In a node step each lane tests one of the four children (one
// 64-B line per quad), in a block step one of the block's four triangles; the
// quad orders its hits and reduces its candidates with DPP moves inside the
// quad. A wave's 16 rays diverge far less than 64 did: a wave runs whichever
// step more of its rays are ready for (about 11 of 16).
//
// Rays enter through a pool in LDS: a wave sets up to kQuadPool rays up, one
// per lane (reciprocals, root box; rays that cannot hit anything are finished
// there), and idle quads read theirs from the pool, so the set-up's
// instructions are paid once per kQuadPool rays and the ray loads are
// coalesced (RayShares: which wave takes which rays).
//
// Once no rays are left, idle quads of a wave take stack entries of its busy
// ones, so that the longest rays (hundreds of steps at 0.7 us each) are traced
// by up to 16 quads.
//
// Measured on the 1M-triangle mesh in the box, a lane per ray before: rays off
// its surfaces, 4,096: 294 -> 32 us, 65,536: 1409 -> 94 us, 1M: 1.67 -> 0.27
// ms, 4.2M: 3.46 -> 0.70 ms, 16.8M: 7.3 -> 2.3 ms (2.3 -> 7.3 Grays/s);
// 1920x1080 primary rays 1.00 -> 0.33 ms; the extension rays of a 123M-path
// render 139 -> 84 ms. Bound by VALU issue (about 80% of the issue cycles at 42
// of 64 lanes) once a launch has millions of rays, by the longest rays' chains
// of loads below that.
//
// The closest hit is the minimum of (t, leaf-order index) over the accepted
// candidates, whatever the visiting order: a candidate is accepted as the
// reference accepts it (acceleration/sbvh.cpp:494-496: t > 0, t < best, hit
// point inside the leaf box +-1e-3).
#pragma once

#include <hip/hip_fp16.h>

#include "spt_device.h"

namespace spt {

// Rays a wave sets up at a time and stack entries of a ray kept in LDS. The set-up
// costs a wave the same for any number of rays up to 64, and seven blocks have
// to fit a CU's LDS: (32, 24), (48, 16), (64, 14): 16.8M rays 2.35, 2.30, 2.26
// ms; 4.2M 0.72, 0.67, 0.70; 2.1M 0.41, 0.415, 0.425.
constexpr int kQuadPool = 48, kQuadStack = 16;
constexpr int kQuadsPerBlock = kBlock / 4;
constexpr int kQuadWaves = 7;   // waves per SIMD the kernels are held to (72 VGPRs, a few spills in the refill
                                // code): 6 (80 VGPRs, almost none) ran extension rays 5% slower
constexpr uint32_t kDone = 0xFFFFFFFFu;

// Where a ray starts: its scene's root box and root node. Rays of several
// scenes share the node and block arrays.
struct Root {
    V3 mn, mx;
    uint32_t node;
};

__device__ inline Root scene_root(const DevScene& sc) {
    return Root{V3{sc.rmin[0], sc.rmin[1], sc.rmin[2]}, V3{sc.rmax[0], sc.rmax[1], sc.rmax[2]}, 0u};
}

// A stack entry: the child's reference (low word) and the bits of its entry
// distance (an entry farther than the best hit is dropped when popped).
// Address-space-qualified pointers keep the accesses ds_* and global_*
// instructions instead of flat ones.
typedef uint64_t QuadEntry;
typedef __attribute__((address_space(3))) QuadEntry lds_entry;
typedef __attribute__((address_space(1))) QuadEntry glb_entry;
__device__ inline QuadEntry quad_entry(uint32_t ref, float t) {
    return (QuadEntry)ref | ((QuadEntry)__float_as_uint(t) << 32);
}

// What a quad keeps of its ray outside registers.
struct QuadRay {
    uint32_t ray;    // index in the launch; kDone: none
    float slack;     // widens the boxes (ray_slack)
    uint32_t owner;  // split rays: the quad that took the ray from the pool
    int bot;         // lowest stack entry (the end mark lies below it)
    uint32_t idx, mat;  // the quad's best candidate (idx kNoHit: none of its own)
    float u, v;
    QuadEntry best;  // of the ray this quad took: the minimum (t, index) of its parts finished so far
};

struct QuadLds {
    float4 pool[kBlock / 64][3][kQuadPool];  // o + inv.x | d + inv.y | inv.z, ray, root node
    QuadRay ray[kQuadsPerBlock];
    uint8_t donor[kBlock / 64][16];  // split step: donor quads of a wave by rank
    QuadEntry stack[kQuadsPerBlock][kQuadStack + 1];  // entry 0: the end mark; odd row stride: spread over the banks
};

// Words of global spill space one block needs for a stack of `cap` entries.
__host__ __device__ inline uint32_t quad_spill_words(uint32_t cap) {
    return cap > kQuadStack ? (cap - kQuadStack) * kQuadsPerBlock * 2u : 0u;
}

// Reciprocal for the conservative box tests: a (nearly) zero component gives
// a large power of two, so products with it are exact and (lo - o) / d never
// becomes inf - inf.
__device__ inline float safe_rcp(float d) { return (fabsf(d) > 0x1p-60f) ? rcp_rn(d) : copysignf(0x1p60f, d); }

// Whether the ray meets the box [mn, mx] at t >= 0: one FMA per slab plane and
// IEEE min/max (a NaN product keeps the box).
__device__ inline bool root_test(V3 inv, V3 oi, V3 mn, V3 mx) {
    const float t0x = fmaf(mn.x, inv.x, oi.x), t1x = fmaf(mx.x, inv.x, oi.x);
    const float t0y = fmaf(mn.y, inv.y, oi.y), t1y = fmaf(mx.y, inv.y, oi.y);
    const float t0z = fmaf(mn.z, inv.z, oi.z), t1z = fmaf(mx.z, inv.z, oi.z);
    const float tmin = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fmaxf(fminf(t0z, t1z), 0.0f));
    const float tmax = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fmaxf(t0z, t1z));
    return tmin <= tmax && tmin < __builtin_inff();
}

// What a ray adds to the tree's box paddings (prim_pad in quad_tree.cpp): they
// cover rays of at most unit length whose origin is within a diagonal of the
// root box of its centre. The error they stand for grows with the distance and
// with the length; adding 1e-3 gives boxes no smaller than the reference's. The
// rounding of the box tests grows with the distance whatever the length (the
// second term: without it 25 of a million rays of length 2 from 60,000 away lost
// their hit). It opens the more boxes the farther a ray starts: 65,536 rays
// into the 1M-triangle mesh in the box, of size 2, 0.26 ms from 100 away, 0.81
// from 5,000, 11 from 60,000.
__device__ inline float ray_slack(const Root& r, V3 o, V3 d) {
    const V3 e = r.mx - r.mn, c = o - (r.mn + e * 0.5f);
    const float diag2 = dot(e, e), far2 = dot(c, c);
    float slack = dot(d, d) <= 1.002f ? 0.0f : 1e-3f;
    if (far2 > diag2) {
        const float far = sqrtf(far2);
        slack = fminf(1e-3f, slack + 1e-3f * (far / sqrtf(diag2) - 1.0f)) + 1e-6f * far;
    }
    return slack;
}

template <int CTRL>
__device__ inline uint32_t quad_swap(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
constexpr int kSwap1 = 0xB1, kSwap2 = 0x4E, kSwap3 = 0x1B;  // quad_perm: lane ^ 1, ^ 2, ^ 3

// One half (as float) of a pair of half-float denormals times a, plus b.
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ inline float fma_half(uint32_t pair, int hi, float a, float b) {
    const half2v h = __builtin_bit_cast(half2v, pair);
    return fmaf((float)(hi ? h.y : h.x), a, b);
}

// Exact acceptance test of a candidate at t (sbvh.cpp:494-496) with the box
// of its leaf, which the ray must also meet.
__device__ inline bool accept_exact(const DevScene& sc, V3 o, V3 d, float t, uint32_t box) {
    box &= ~kQuadExact;
    const float4 b0 = sc.qboxes[2 * (size_t)box], b1 = sc.qboxes[2 * (size_t)box + 1];
    const V3 mn{b0.x, b0.y, b0.z}, mx{b1.x, b1.y, b1.z};
    float tn, tf;
    return point_inside(o + d * t, mn, mx) && slab(o, V3{1.0f / d.x, 1.0f / d.y, 1.0f / d.z}, mn, mx, tn, tf);
}

// The same test answered from the primitive alone where that is certain: the
// point at (u, v) of a triangle lies inside its leaf's box where that holds the
// vertices (no kQuadExact), so a hit point within 5e-4 of it lies inside the box +-1e-3 (with
// coordinates up to 1024 the rounding of the triangle's point is below 2e-4).
// A sphere (u = v = 0, v0 = centre) reaches its radius, as its box does, and no
// further: its hit point may lie off it, and a root leaf's box, which the ray has
// to meet, has no padding. Saves the load of the box, which the whole wave would wait for.
__device__ inline bool accept_near(V3 o, V3 d, float t, float u, float v, V3 v0, V3 e1, V3 e2, float radius) {
    const V3 p = o + d * t;
    const float x = p.x - fmaf(u, e1.x, fmaf(v, e2.x, v0.x));
    const float y = p.y - fmaf(u, e1.y, fmaf(v, e2.y, v0.y));
    const float z = p.z - fmaf(u, e1.z, fmaf(v, e2.z, v0.z));
    return fmaxf(fmaxf(fabsf(x), fabsf(y)), fabsf(z)) <= (radius > 0.0f ? radius : 5e-4f);
}

// How the waves of a launch share its rays: groups of `chunk` rays dealt to
// the waves in turn without any counter (all rays of a small launch, one pool
// load per wave of a larger one); the rays from `fixed` on lie in kRayCounters
// regions with a counter each, a wave takes from its block's region and then
// from the others. Blocks go to the XCDs in turn, so a region's counter stays
// in one XCD's L2. One counter for all rays was the limit of mid-sized
// launches: about 10 ns per atomic on an address that all XCDs share, 160 us
// for 1M rays in shares of 32 to 64. A share is a quarter of what an even split
// of the region's rest would give each wave: long rays lie together in an
// image, and with half of it the last waves held 1920x1080 primary rays up
// from 0.33 to 0.41 ms (incoherent rays, 16.8M: 2.36 and 2.42 ms).
constexpr uint32_t kRayCounters = 8, kRayCounterStride = 32;  // one 128-B line each
constexpr uint32_t kRayCounterWords = kRayCounters * kRayCounterStride;
struct RayShares {
    uint32_t waves, chunk, fixed, groups, span;
    __host__ __device__ RayShares(uint32_t n, uint32_t n_waves) {
        waves = n_waves;
        const uint32_t per_wave = (n + waves - 1) / waves;  // n is at most 2^31
        if (per_wave <= 2u * kQuadPool) {  // all dealt, at least 4 to a wave
            chunk = per_wave <= 4u ? 4u : (per_wave <= (uint32_t)kQuadPool ? per_wave : (per_wave + 1u) / 2u);
            fixed = n;
        } else {
            chunk = kQuadPool;
            fixed = waves * kQuadPool;
        }
        groups = (fixed + chunk - 1) / chunk;
        span = (n - fixed + kRayCounters - 1) / kRayCounters;
    }
    // all n rays to one wave
    __device__ explicit RayShares(uint32_t n) : waves(1), chunk(kQuadPool), fixed(n), groups((n + kQuadPool - 1) / kQuadPool), span(0) {}
};

__device__ inline uint64_t ballot(bool x) { return __builtin_amdgcn_ballot_w64(x); }
__device__ inline int lanes(uint64_t mask) { return (int)__builtin_popcountll(mask); }

// Traces rays 0 .. n - 1, shared between the waves of the launch (RayShares;
// ray_counter: kRayCounterWords words, the counters 0 at the start). GetRay(i, o, d, root) loads ray i (root starts
// as the single scene's); PutHit(i, h, o, d, nodes, tris) stores a
// result: it is called by one lane per ray. `refill`: idle lanes of a wave that make it
// take new rays. spill: this block's spill space (quad_spill_words words).
template <bool FETCH, bool SMALL, typename GetRay, typename PutHit>
__device__ inline void trace_shares(const DevScene& sc, uint32_t n, RayShares sh, uint32_t first_group,
                                    uint32_t* ray_counter, QuadLds& lds, uint32_t* spill, bool& overflow,
                                    uint32_t refill, GetRay get_ray, PutHit put_hit) {
    const uint32_t lane = __lane_id(), q4 = lane & 3u, quad = threadIdx.x >> 2;
    float4(*pool)[kQuadPool] = lds.pool[threadIdx.x >> 6];
    lds_entry* stk = (lds_entry*)lds.stack[quad];
    glb_entry* deep = (glb_entry*)spill + quad;  // entry k at (k - kQuadStack) * kQuadsPerBlock
    const int cap = (int)sc.stack_cap4;
    const uint64_t lt = __lanemask_lt();
    const char* nodes_at = reinterpret_cast<const char*>(sc.qnodes);
    const char* prims_at = reinterpret_cast<const char*>(sc.qprims);
    const uint32_t child_ofs = 16 + 12 * q4, prim_ofs = 48 * q4;
    sh.waves = __builtin_amdgcn_readfirstlane(sh.waves);
    sh.chunk = __builtin_amdgcn_readfirstlane(sh.chunk);  // scalar registers
    sh.fixed = __builtin_amdgcn_readfirstlane(sh.fixed);
    sh.groups = __builtin_amdgcn_readfirstlane(sh.groups);
    sh.span = __builtin_amdgcn_readfirstlane(sh.span);
    uint32_t range = 0, range_end = 0;  // rays taken and not yet in the pool
    uint32_t pool_n = 0, pool_at = 0;   // rays in the pool, next one to hand out
    uint32_t group = __builtin_amdgcn_readfirstlane(first_group);
    uint32_t tried = 0;                 // regions found empty, the block's own first
    uint32_t left = sh.span;            // rays left in the current region at this wave's last look
    bool more = true;

    V3 o{}, d{}, inv{}, oi{};
    uint32_t sel_near = 0, sel_far = 0, sel_z = 0;
    uint32_t cur = kQuadNone;    // entry to visit; kQuadNone: idle, or finished and not yet stored
    int sp = 1;                  // next free stack entry
    float best = 0.0f;           // closest hit so far (the same in a ray's four lanes)
    uint32_t best_idx = kNoHit;
    uint32_t nodes = 0, tris = 0;
    bool split = false, wide = false;  // of the wave: some ray was split; some ray has a slack
    QuadRay& my = lds.ray[quad];
    my.ray = kDone;
    stk[0] = quad_entry(kQuadNone, -__builtin_inff());  // popped last: the ray is finished

    // What the node test needs beside o, d and inv. Byte selectors: the near
    // (far) bounds of x and y as two halves with zero high bytes, and near z
    // beside far z.
    auto set_up = [&]() {
        oi = V3{-o.x * inv.x, -o.y * inv.y, -o.z * inv.z};
        sel_near = (inv.x >= 0.0f ? 0x0C000C00u : 0x0C000C01u) | (inv.y >= 0.0f ? 0x20000u : 0x30000u);
        sel_far = sel_near ^ 0x00010001u;
        sel_z = inv.z >= 0.0f ? 0x0C010C00u : 0x0C000C01u;
    };
    // Next entry of the rays that took a step; entries beyond the best hit are
    // dropped. any_deep: some of their stacks reach beyond the part in LDS.
    auto take = [&](bool any_deep) {
        --sp;
        QuadEntry e;
        if (any_deep) {
            if (sp <= kQuadStack)
                e = stk[sp];
            else
                e = deep[(size_t)(sp - kQuadStack - 1) * kQuadsPerBlock];
        } else {
            e = stk[sp];
        }
        cur = (uint32_t)e;
        return __uint_as_float((uint32_t)(e >> 32)) > best;
    };
    auto pop = [&](bool any_deep) {
        bool again = take(any_deep);
        while (ballot(again))
            if (again) again = take(any_deep);
    };

    while (true) {
        uint64_t idle = ballot(cur == kQuadNone);
        if (idle == ~0ull || lanes(idle) >= (int)refill) {
            // ---- finished rays are stored, idle quads take new ones
            if (cur == kQuadNone && q4 == 0u && my.ray != kDone) {
                bool store = best_idx == kNoHit || my.idx == best_idx;
                if (!FETCH && split) {  // a part of a ray stores its result if it is the best of the parts so far
                    const QuadEntry k = ((QuadEntry)__float_as_uint(best) << 32) | best_idx;
                    QuadEntry& kept = lds.ray[my.owner].best;
                    if (store) atomicMin((unsigned long long*)&kept, (unsigned long long)k);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    store = store && kept == k && (best_idx != kNoHit || my.owner == quad);
                }
                if (store) {
                    Hit h;
                    h.t = best;
                    h.idx = best_idx;
                    h.mat = my.mat;
                    h.u = best_idx == kNoHit ? 0.0f : my.u;
                    h.v = best_idx == kNoHit ? 0.0f : my.v;
                    put_hit(my.ray, h, o, d, nodes, tris);
                }
                my.ray = kDone;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (!more && pool_at == pool_n) {
                if (idle == ~0ull) break;
                // ---- no rays left: each idle quad takes the lowest (largest) stack
                // entry of a busy one's ray, so that a few long rays do not keep
                // the launch alive alone
                const bool gives = !FETCH && cur != kQuadNone && sp > my.bot && my.bot <= kQuadStack;
                const uint64_t donors = ballot(gives);
                if (donors) {
                    split = true;
                    const uint32_t wave0 = (threadIdx.x >> 6) * 16u;
                    uint8_t* list = lds.donor[threadIdx.x >> 6];
                    const int pairs = min(lanes(donors), lanes(idle)) >> 2;
                    const bool is_idle = cur == kQuadNone;
                    const int rank = lanes((is_idle ? idle : donors) & lt & 0x1111111111111111ull) - (q4 ? 1 : 0);
                    if (gives && rank < pairs) list[rank] = (uint8_t)(lane >> 2);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    const bool takes = is_idle && rank < pairs;
                    const int src = takes ? (int)list[rank] * 4 : (int)(lane & 60u);
                    o = V3{__shfl(o.x, src), __shfl(o.y, src), __shfl(o.z, src)};
                    d = V3{__shfl(d.x, src), __shfl(d.y, src), __shfl(d.z, src)};
                    inv = V3{__shfl(inv.x, src), __shfl(inv.y, src), __shfl(inv.z, src)};
                    best = __shfl(best, src);
                    best_idx = __shfl(best_idx, src);
                    if (takes) {
                        const QuadRay& its = lds.ray[wave0 + (uint32_t)src / 4u];
                        const QuadEntry e = *((lds_entry*)lds.stack[wave0 + (uint32_t)src / 4u] + its.bot);
                        sp = 1;
                        if (__uint_as_float((uint32_t)(e >> 32)) <= best) {
                            set_up();
                            cur = (uint32_t)e;
                            if (q4 == 0u) {
                                my.ray = its.ray;
                                my.slack = its.slack;
                                my.owner = its.owner;
                                my.bot = 1;
                                my.idx = kNoHit;
                            }
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (gives && rank < pairs && q4 == 0u) {
                        stk[my.bot] = quad_entry(kQuadNone, -__builtin_inff());
                        ++my.bot;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    idle = ballot(cur == kQuadNone);
                }
            } else {
                if (pool_at == pool_n && more) {
                    if (range == range_end) {
                        if (group < sh.groups) {
                            range = group * sh.chunk;
                            range_end = min(range + sh.chunk, sh.fixed);
                            group += sh.waves;
                        } else {
                            range = range_end = 0;
                            while (tried < kRayCounters && sh.fixed < n) {
                                const uint32_t region = (blockIdx.x + tried) % kRayCounters;
                                const uint32_t take =
                                    max(1u, min(left * kRayCounters / (4u * sh.waves), 512u) / kQuadPool) * kQuadPool;
                                uint32_t at = 0;
                                if (lane == 0) at = atomicAdd(ray_counter + region * kRayCounterStride, take);
                                at = __builtin_amdgcn_readfirstlane(at);
                                const uint32_t r0 = sh.fixed + region * sh.span;
                                const uint32_t in_region = r0 < n ? min(sh.span, n - r0) : 0u;
                                if (at < in_region) {
                                    range = r0 + at;
                                    range_end = r0 + min(at + take, in_region);
                                    left = in_region - at;
                                    break;
                                }
                                ++tried;
                                left = 0;  // small shares from the other regions
                            }
                        }
                    }
                    const uint32_t cnt = min((uint32_t)kQuadPool, range_end - range);
                    const uint32_t base = range;
                    range += cnt;
                    more = range < range_end || group < sh.groups || (sh.fixed < n && tried < kRayCounters);
                    pool_at = 0;
                    bool keep = false;
                    V3 po{}, pd{}, pi{};
                    Root R = scene_root(sc);
                    if (lane < cnt) {
                        get_ray(base + lane, po, pd, R);
                        pi = V3{safe_rcp(pd.x), safe_rcp(pd.y), safe_rcp(pd.z)};
                        // a ray with a non-finite component cannot hit anything (every
                        // t comparison fails) but would pass every box test: a miss
                        const float sum = po.x + po.y + po.z + pd.x + pd.y + pd.z;
                        keep = (sum - sum == 0.0f) &&
                               root_test(pi, V3{-po.x * pi.x, -po.y * pi.y, -po.z * pi.z}, R.mn, R.mx);
                        if (!keep) {
                            Hit h;
                            h.t = __builtin_inff();
                            h.idx = kNoHit;
                            h.mat = 0;
                            h.u = h.v = 0.0f;
                            put_hit(base + lane, h, po, pd, 0u, 0u);
                        }
                    }
                    const uint64_t kept = ballot(keep);
                    pool_n = (uint32_t)lanes(kept);
                    if (keep) {
                        const uint32_t j = (uint32_t)lanes(kept & lt);
                        pool[0][j] = make_float4(po.x, po.y, po.z, pi.x);
                        pool[1][j] = make_float4(pd.x, pd.y, pd.z, pi.y);
                        pool[2][j] = make_float4(pi.z, __uint_as_float(base + lane), __uint_as_float(R.node),
                                                 ray_slack(R, po, pd));
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
                float slack = 0.0f;
                if (cur == kQuadNone) {
                    // rank of this quad among the idle ones
                    const uint32_t j = pool_at + (uint32_t)lanes(idle & lt & 0x1111111111111111ull) - (q4 ? 1u : 0u);
                    if (j < pool_n) {
                        const float4 a = pool[0][j], b = pool[1][j], c = pool[2][j];
                        o = V3{a.x, a.y, a.z};
                        d = V3{b.x, b.y, b.z};
                        inv = V3{a.w, b.w, c.x};
                        set_up();
                        cur = __float_as_uint(c.z);
                        sp = 1;
                        best = __builtin_inff();
                        best_idx = kNoHit;
                        if (q4 == 0u) {
                            my.ray = __float_as_uint(c.y);
                            my.slack = c.w;
                            my.owner = quad;
                            my.bot = 1;
                            my.idx = kNoHit;
                            my.best = ((QuadEntry)0x7F800000u << 32) | kNoHit;
                        }
                        slack = c.w;
                        if (FETCH) nodes = tris = 0;
                    }
                }
                pool_at = min(pool_n, pool_at + ((uint32_t)lanes(idle) >> 2));
                wide = wide || ballot(slack > 0.0f);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                continue;
            }
        }
        const bool at_node = (int)cur >= 0;
        const uint64_t node_lanes = ballot(at_node);
        if (2 * lanes(node_lanes) >= 64 - lanes(idle)) {
            // ---- node step: one child per lane
            if (at_node) {
                uint4 g;
                uint3 c;
                if (SMALL) {
                    g = *reinterpret_cast<const uint4*>(nodes_at + (cur << 6));
                    uint32_t at;  // in one instruction, and as a 32-bit offset beside a scalar base
                    asm("v_lshl_or_b32 %0, %1, 6, %2" : "=v"(at) : "v"(cur), "v"(child_ofs));
                    c = *reinterpret_cast<const uint3*>(nodes_at + at);
                } else {
                    g = *reinterpret_cast<const uint4*>(nodes_at + (uint64_t)cur * 64);
                    c = *reinterpret_cast<const uint3*>(nodes_at + (uint64_t)cur * 64 + child_ofs);
                }
                if (FETCH) nodes += 2;  // 32-B units
                const float ax = __uint_as_float(g.w) * inv.x, ay = __uint_as_float(g.w << 9) * inv.y,
                            az = __uint_as_float(g.w << 18) * inv.z;
                const float bx = fmaf(__uint_as_float(g.x), inv.x, oi.x), by = fmaf(__uint_as_float(g.y), inv.y, oi.y),
                            bz = fmaf(__uint_as_float(g.z), inv.z, oi.z);
                float fx = bx, fy = by, fz = bz, nx = bx, ny = by, nz = bz;
                if (wide) {
                    const float slack = my.slack;
                    nx = fmaf(-slack, fabsf(inv.x), bx), fx = fmaf(slack, fabsf(inv.x), bx);
                    ny = fmaf(-slack, fabsf(inv.y), by), fy = fmaf(slack, fabsf(inv.y), by);
                    nz = fmaf(-slack, fabsf(inv.z), bz), fz = fmaf(slack, fabsf(inv.z), bz);
                }
                const uint32_t nxy = __builtin_amdgcn_perm(c.x, c.x, sel_near);
                const uint32_t fxy = __builtin_amdgcn_perm(c.x, c.x, sel_far);
                const uint32_t zz = __builtin_amdgcn_perm(c.y, c.y, sel_z);
                const float tn = fmaxf(fmaxf(fma_half(nxy, 0, ax, nx), fma_half(nxy, 1, ay, ny)),
                                       fmaxf(fma_half(zz, 0, az, nz), 0.0f));
                float tf = fminf(fma_half(fxy, 0, ax, fx), fma_half(fxy, 1, ay, fy));
                // (fminf would canonicalise best, which is never a NaN, first)
                asm("v_min3_f32 %0, %1, %2, %3" : "=v"(tf) : "v"(tf), "v"(fma_half(zz, 1, az, fz)), "v"(best));
                const bool hit = (tn <= tf) && c.z != kQuadNone;
                // order among the quad's hits: entry distance, its low bits replaced by the
                // lane; before = -(hits nearer than this lane's), the differences' sign bits
                const int key = hit ? (int)((__float_as_uint(tn) & 0x7FFFFFFCu) | q4) : 0x7FFFFFFF;
                const int before = (((int)quad_swap<kSwap1>((uint32_t)key) - key) >> 31) +
                                   (((int)quad_swap<kSwap2>((uint32_t)key) - key) >> 31) +
                                   (((int)quad_swap<kSwap3>((uint32_t)key) - key) >> 31);
                // hits of the quad, from the wave's mask
                const uint64_t hit_mask = ballot(tn <= tf) & ballot(c.z != kQuadNone);
                sp += __builtin_popcount((uint32_t)(hit_mask >> (lane & 60u)) & 15u);
                const int at = sp - 1 + before;
                const bool any_deep = ballot(sp > kQuadStack + 1) != 0;
                if (any_deep) {
                    if (sp > cap + 1) {  // more entries than the tree can need: reported, the ray ends
                        overflow = true;
                        sp = 1;
                    } else if (hit) {
                        if (at <= kQuadStack)
                            stk[at] = quad_entry(c.z, tn);
                        else
                            deep[(size_t)(at - kQuadStack - 1) * kQuadsPerBlock] = quad_entry(c.z, tn);
                    }
                } else if (hit) {
                    stk[at] = quad_entry(c.z, tn);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                pop(any_deep);
            }
        } else if (!at_node && cur != kQuadNone) {
            // ---- block step: one triangle (or sphere) per lane
            float4 a, b, c;
            if (SMALL) {
                const uint32_t at = ((cur + (cur << 1)) << 6) + prim_ofs;  // 192 B a block; the leaf bit shifts out
                const float4* tp = reinterpret_cast<const float4*>(prims_at + at);
                a = tp[0];
                b = tp[1];
                c = tp[2];
            } else {
                const float4* tp =
                    reinterpret_cast<const float4*>(prims_at + (uint64_t)(cur & ~kQuadLeaf) * 192 + prim_ofs);
                a = tp[0];
                b = tp[1];
                c = tp[2];
            }
            if (FETCH) tris += 4;
            float t, u = 0.0f, v = 0.0f;
            bool pass;
            if (sc.has_spheres && (__float_as_uint(c.w) & kQuadSphere))
                pass = sphere_test(o, d, V3{a.x, a.y, a.z}, a.w, t);
            else
                pass = tri_test(o, d, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, V3{b.z, b.w, c.x}, t, u, v);
            const uint32_t idx = __float_as_uint(c.y), km = __float_as_uint(c.w);
            pass = pass & (t > 0.0f) & ((t < best) | ((t == best) & (idx < best_idx)));
            if (ballot(pass)) {
                bool ok = pass;
                const bool sure = !(__float_as_uint(c.z) & kQuadExact) &&
                                  accept_near(o, d, t, u, v, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, V3{b.z, b.w, c.x},
                                              (km & kQuadSphere) ? a.w : 0.0f);
                if (ballot(pass & !sure)) {
                    if (pass & !sure) ok = accept_exact(sc, o, d, t, __float_as_uint(c.z));
                    if (FETCH) nodes += (pass & !sure) ? 1u : 0u;
                }
                float ct = ok ? t : best;
                uint32_t ci = ok ? idx : best_idx;
                // the quad's minimum of (t, index)
                float ot = __uint_as_float(quad_swap<kSwap1>(__float_as_uint(ct)));
                uint32_t oj = quad_swap<kSwap1>(ci);
                bool less = (ot < ct) | ((ot == ct) & (oj < ci));
                ct = less ? ot : ct;
                ci = less ? oj : ci;
                ot = __uint_as_float(quad_swap<kSwap2>(__float_as_uint(ct)));
                oj = quad_swap<kSwap2>(ci);
                less = (ot < ct) | ((ot == ct) & (oj < ci));
                best = less ? ot : ct;
                best_idx = less ? oj : ci;
                if (ok && idx == best_idx) {
                    my.idx = idx;
                    my.mat = km & ~kQuadSphere;
                    my.u = u;
                    my.v = v;
                }
            }
            pop(ballot(sp > kQuadStack + 1) != 0);
        }
    }
}

// The rays of a launch, shared between all its waves.
template <bool FETCH, bool SMALL, typename GetRay, typename PutHit>
__device__ inline void trace_quads(const DevScene& sc, uint32_t n, uint32_t* ray_counter, QuadLds& lds,
                                   uint32_t* spill, bool& overflow, uint32_t refill, GetRay get_ray, PutHit put_hit) {
    trace_shares<FETCH, SMALL>(sc, n, RayShares(n, gridDim.x * (kBlock / 64)), blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6),
                        ray_counter, lds, spill, overflow, refill, get_ray, put_hit);
}

// Rays 0 .. n - 1 against a scene whose tree is one block (at most four
// primitives in a root leaf): a ray per lane, no tree, pool or stack. The same
// candidates are accepted as in the block step above, and then the ray has to
// meet the root's box, as the reference asks before it tests the leaf
// (acceleration/sbvh.cpp:423-515): that box has no padding, so a ray towards a
// vertex or edge on it may miss it by a rounding. Only hits pay for that test.
// 185x305 depth image of a sphere 3.2 us, 11.5 with the quads, whose set-up and
// rounds a wave are latency here; 1900x1050 10.3 us (9.7 without the root's box).
// Bound by VALU issue.
template <typename GetRay, typename PutHit>
__device__ inline void trace_one_block(const DevScene& sc, uint32_t n, GetRay get_ray, PutHit put_hit) {
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        V3 o, d;
        get_ray(i, o, d);
        const float sum = o.x + o.y + o.z + d.x + d.y + d.z;
        Hit miss;
        miss.t = __builtin_inff();
        miss.idx = kNoHit;
        miss.mat = 0;
        miss.u = miss.v = 0.0f;
        Hit h = miss;
        if (sum - sum == 0.0f) {
            const float4* tp = reinterpret_cast<const float4*>(sc.qprims);
            for (int k = 0; k < 4; ++k) {
                const float4 a = tp[3 * k], b = tp[3 * k + 1], c = tp[3 * k + 2];
                const uint32_t idx = __float_as_uint(c.y), km = __float_as_uint(c.w);
                if (idx == kNoHit) break;  // unused slots come last
                float t, u = 0.0f, v = 0.0f;
                bool pass;
                if (km & kQuadSphere)
                    pass = sphere_test(o, d, V3{a.x, a.y, a.z}, a.w, t);
                else
                    pass = tri_test(o, d, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, V3{b.z, b.w, c.x}, t, u, v);
                pass = pass & (t > 0.0f) & ((t < h.t) | ((t == h.t) & (idx < h.idx)));
                if (!pass) continue;
                const uint32_t box = __float_as_uint(c.z);
                const bool sure = !(box & kQuadExact) &&
                                  accept_near(o, d, t, u, v, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, V3{b.z, b.w, c.x},
                                              (km & kQuadSphere) ? a.w : 0.0f);
                if (sure || accept_exact(sc, o, d, t, box)) {
                    h.t = t;
                    h.idx = idx;
                    h.mat = km & ~kQuadSphere;
                    h.u = u;
                    h.v = v;
                }
            }
            const Root r = scene_root(sc);
            float tn, tf;
            if (h.idx != kNoHit && !slab(o, V3{1.0f / d.x, 1.0f / d.y, 1.0f / d.z}, r.mn, r.mx, tn, tf)) h = miss;
        }
        put_hit(i, h, o, d);
    }
}

}  // namespace spt
