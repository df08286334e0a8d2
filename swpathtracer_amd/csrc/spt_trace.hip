// spt_trace.hip - closest-hit ray casting kernels (batched
// AccelStructure::intersect, acceleration/accel_structure.h:29-30) and the
// three ray casters (integrators/raycaster.h:61-99).
#include <mutex>

#include "spt_quad.h"

namespace spt {

namespace {

// The reference's own node set on the binary tree (COUNT: with its counters).
template <bool COUNT>
__global__ __launch_bounds__(kBlock) void k_trace(DevScene sc, const float4* __restrict__ rays, uint64_t n,
                                                  uint2* __restrict__ hits, uint32_t* __restrict__ tests_out,
                                                  uint32_t* __restrict__ isects_out, uint32_t* __restrict__ spill,
                                                  uint32_t* __restrict__ flags) {
    __shared__ uint32_t lds[kLdsStack * kBlock];
    const uint32_t gthreads = gridDim.x * kBlock;
    const uint32_t gtid = blockIdx.x * kBlock + threadIdx.x;
    Stack st(lds + threadIdx.x, spill + gtid, gthreads, sc.stack_cap);
    bool overflow = false;
    for (uint64_t i = gtid; i < n; i += gthreads) {
        const float4 ro = rays[2 * i], rd = rays[2 * i + 1];
        Hit h;
        uint32_t tests, isects;
        trace_ray<COUNT>(sc, V3{ro.x, ro.y, ro.z}, V3{rd.x, rd.y, rd.z}, st, h, tests, isects, overflow);
        hits[i] = make_uint2(__float_as_uint(h.t), h.prim);
        if (COUNT) {
            if (tests_out) tests_out[i] = tests;
            if (isects_out) isects_out[i] = isects;
        }
    }
    if (overflow) atomicOr(flags, 1u);
}

// Scene-order id of the primitive at a leaf-order index.
__device__ inline uint32_t prim_of(const DevScene& sc, uint32_t idx) {
    return idx == kNoHit ? SPT_MISS : __float_as_uint(sc.tris[3 * (size_t)idx + 2].y);
}

// Closest-hit kernel: rays[i] -> hits[i] (FETCH: per-ray node and triangle
// record counts into nodes_out / tris_out).
template <bool FETCH, bool SMALL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kQuadWaves))) void k_trace_q(DevScene sc, const float4* __restrict__ rays, uint32_t n,
                                                    uint2* __restrict__ hits, uint32_t* __restrict__ nodes_out,
                                                    uint32_t* __restrict__ tris_out, uint32_t* __restrict__ spill,
                                                    uint32_t* __restrict__ flags, uint32_t* __restrict__ rays_taken,
                                                    uint32_t refill) {
    __shared__ QuadLds lds;
    bool overflow = false;
    trace_quads<FETCH, SMALL>(
        sc, n, rays_taken, lds, spill + (size_t)blockIdx.x * quad_spill_words(sc.stack_cap4), overflow, refill,
        [&](uint32_t i, V3& o, V3& d, Root&) {
            const float4 ro = rays[2 * (size_t)i], rd = rays[2 * (size_t)i + 1];
            o = V3{ro.x, ro.y, ro.z};
            d = V3{rd.x, rd.y, rd.z};
        },
        [&](uint32_t i, const Hit& h, V3, V3, uint32_t nn, uint32_t nt) {
            hits[i] = make_uint2(__float_as_uint(h.t), prim_of(sc, h.idx));
            if (FETCH) {
                nodes_out[i] = nn;
                tris_out[i] = nt;
            }
        });
    if (overflow) atomicOr(flags, 1u);
}

// Camera ray of pixel i: one ray per pixel centre (RegularPixelSampler(1)
// gives (0.5, 0.5), regular_pixel_sampler.cpp:3-14).
__device__ inline void pixel_ray(const DevCamera& cam, uint64_t i, V3& o, V3& d) {
    uint32_t x, y;
    if (i >> 32) {
        x = (uint32_t)(i % cam.width);
        y = (uint32_t)(i / cam.width);
    } else {  // a 32-bit division takes a fifth of the instructions
        y = (uint32_t)i / cam.width;
        x = (uint32_t)i - y * cam.width;
    }
    camera_ray(cam, x + 0.5f, y + 0.5f, o, d);
}

// Pixel value of a normal or depth ray caster.
template <int KIND>
__device__ inline void put_pixel(const DevScene& sc, float* __restrict__ out, uint64_t i, const Hit& h, V3 o, V3 d) {
    if (KIND == SPT_RAYCAST_DEPTH) {
        out[i] = (h.idx != kNoHit) ? h.t : -1.0f;
    } else {
        const V3 nrm = (h.idx != kNoHit) ? shading_normal(sc, h, o + d * h.t) : V3{0.0f, 0.0f, 0.0f};
        float* o3 = out + 3 * i;
        o3[0] = nrm.x;
        o3[1] = nrm.y;
        o3[2] = nrm.z;
    }
}

// Normal (normal_raycaster.cpp:19-31) and depth (depth_raycaster.cpp:36-48)
// ray casters over pixels [base, base + n).
template <int KIND, bool SMALL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kQuadWaves))) void k_raycast(DevScene sc, DevCamera cam, uint64_t base, uint32_t n,
                                                    float* __restrict__ out, uint32_t* __restrict__ spill,
                                                    uint32_t* __restrict__ flags, uint32_t* __restrict__ rays_taken,
                                                    uint32_t refill) {
    __shared__ QuadLds lds;
    bool overflow = false;
    trace_quads<false, SMALL>(
        sc, n, rays_taken, lds, spill + (size_t)blockIdx.x * quad_spill_words(sc.stack_cap4), overflow, refill,
        [&](uint32_t i, V3& o, V3& d, Root&) { pixel_ray(cam, base + i, o, d); },
        [&](uint32_t i, const Hit& h, V3 o, V3 d, uint32_t, uint32_t) { put_pixel<KIND>(sc, out, base + i, h, o, d); });
    if (overflow) atomicOr(flags, 1u);
}

// Closest hits and ray casters in a scene of one block.
__global__ __launch_bounds__(kBlock) void k_trace_block(DevScene sc, const float4* __restrict__ rays, uint32_t n,
                                                        uint2* __restrict__ hits) {
    trace_one_block(
        sc, n,
        [&](uint32_t i, V3& o, V3& d) {
            const float4 ro = rays[2 * (size_t)i], rd = rays[2 * (size_t)i + 1];
            o = V3{ro.x, ro.y, ro.z};
            d = V3{rd.x, rd.y, rd.z};
        },
        [&](uint32_t i, const Hit& h, V3, V3) { hits[i] = make_uint2(__float_as_uint(h.t), prim_of(sc, h.idx)); });
}
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_raycast_block(DevScene sc, DevCamera cam, uint64_t base, uint32_t n,
                                                          float* __restrict__ out) {
    trace_one_block(
        sc, n, [&](uint32_t i, V3& o, V3& d) { pixel_ray(cam, base + i, o, d); },
        [&](uint32_t i, const Hit& h, V3 o, V3 d) { put_pixel<KIND>(sc, out, base + i, h, o, d); });
}

// Intersection-test count ray caster (int_test_count_raycaster.cpp:75-85): the
// boxes and primitives the reference tests for the ray of each pixel, i.e.
// every box of the binary tree whose parent the ray's line meets (no pruning
// by t, so the order does not matter and no primitive is read).
//
// A ray per lane: bound by the longest rays' chains of node loads, and by its
// instructions in small trees.
__global__ __launch_bounds__(kBlock) void k_raycast_count_lane(DevScene sc, DevCamera cam, uint32_t* __restrict__ out,
                                                          uint32_t* __restrict__ spill, uint32_t* __restrict__ flags) {
    __shared__ uint32_t lds[kLdsStack * kBlock];
    const uint32_t gthreads = gridDim.x * kBlock;
    const uint32_t gtid = blockIdx.x * kBlock + threadIdx.x;
    Stack st(lds + threadIdx.x, spill + gtid, gthreads, sc.stack_cap);
    bool overflow = false;
    const uint64_t n = (uint64_t)cam.width * cam.height;
    for (uint64_t i = gtid; i < n; i += gthreads) {
        V3 o, d;
        pixel_ray(cam, i, o, d);
        Hit h;
        uint32_t tests, isects;
        trace_ray<true>(sc, o, d, st, h, tests, isects, overflow);
        out[i] = tests;
    }
    if (overflow) atomicOr(flags, 1u);
}

// The four lanes of a quad share a ray and its stack: each round they take its
// four top entries, a node each, and push the children that are met, those of
// deeper nodes on top. A wave's 16 rays are a tile of 4 x 4 pixels. Bound by
// the longest rays' chains of node loads, which take a quarter of the rounds
// this way. Mesh of 1M triangles, a ray per lane before: 64x48 266 -> 68 us,
// 185x305 545 -> 105, 640x480 686 -> 170, 1920x1080 852 -> 260. Tiles of 8 x 8
// pixels whose rays are set up once and taken by free quads: 72, 113, 217, 348
// (longer chains per wave).
//
// Stack entries: pops take the deepest nodes, so entries of a level are only
// added once none of it is left, at most 8, and at most 4 stay once a deeper
// level has entries: 4 per level and 8 are never exceeded (kCountSlack).
constexpr int kCountStack = 24;  // entries of a ray in LDS, deeper ones spill
constexpr uint32_t kCountSlack = 8;
__host__ __device__ inline uint32_t count_stack_cap(uint32_t stack_cap) { return 4u * stack_cap + kCountSlack; }

// Words of spill space a block needs.
inline size_t count_spill_words(uint32_t stack_cap) {
    const uint32_t cap = count_stack_cap(stack_cap);
    return cap > (uint32_t)kCountStack ? (size_t)(cap - kCountStack) * kQuadsPerBlock : 0;
}

// Whether a ray per lane counts faster: a root that is a leaf has no nodes to
// share, and with a small tree (short chains) and enough pixels to fill the chip
// the quads' extra instructions cost more than the chains. 1920x1080, lane
// against quad: 4,746 nodes 128 and 150 us, 9,568 nodes 162 and 159, 19,923
// nodes 209 and 160; 4,746 nodes, 1280x960 125 and 125, 960x720 109 and 80.
inline bool count_by_lane(const DevScene& sc, uint64_t pixels) {
    return sc.root_leaf != 0 || (sc.n_nodes < 8192u && pixels > (1u << 20));
}

__global__ __launch_bounds__(kBlock) void k_raycast_count(DevScene sc, DevCamera cam, uint32_t* __restrict__ out,
                                                          uint32_t* __restrict__ spill, uint32_t* __restrict__ flags) {
    __shared__ uint32_t lds[kQuadsPerBlock][kCountStack + 1];  // odd row stride: spread over the banks
    const uint32_t lane = __lane_id(), q4 = lane & 3u, quad = threadIdx.x >> 2, ray = lane >> 2;
    lds_u32* stk = (lds_u32*)lds[quad];
    // entry k at (k - kCountStack) * kQuadsPerBlock
    const int cap = (int)count_stack_cap(sc.stack_cap);
    glb_u32* deep = (glb_u32*)(spill + blockIdx.x * (size_t)max(cap - kCountStack, 0) * kQuadsPerBlock) + quad;
    const uint32_t after = (0xEu << q4) & 0xFu;  // lanes of the quad that hold entries further down
    const V3 rmn{sc.rmin[0], sc.rmin[1], sc.rmin[2]}, rmx{sc.rmax[0], sc.rmax[1], sc.rmax[2]};
    const uint64_t tiles_x = ((uint64_t)cam.width + 3) / 4, tiles = tiles_x * (((uint64_t)cam.height + 3) / 4);
    const uint64_t waves = (uint64_t)gridDim.x * (kBlock / 64);
    bool overflow = false;
    for (uint64_t tile = (uint64_t)blockIdx.x * (kBlock / 64) + threadIdx.x / 64; tile < tiles; tile += waves) {
        // a 32-bit division takes a fifth of the instructions
        const uint64_t ty = tile >> 32 ? tile / tiles_x : (uint32_t)tile / (uint32_t)tiles_x;
        const uint64_t x = (tile - ty * tiles_x) * 4 + (ray & 3u), y = ty * 4 + (ray >> 2);
        const bool inside = x < cam.width && y < cam.height;
        const uint64_t i = inside ? y * cam.width + x : 0;
        V3 o, d;
        pixel_ray(cam, i, o, d);
        const V3 inv{1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
        float tn, tf;
        uint32_t tests = q4 == 0u ? 1u : 0u;
        int sp = 0;
        if (inside && slab(o, inv, rmn, rmx, tn, tf)) {
            sp = 1;
            if (q4 == 0u) stk[0] = 0u;
        }
        while (ballot(sp > 0)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            bool hl = false, hr = false;
            uint4 r{};
            if ((int)q4 < sp) {
                const int at = sp - 1 - (int)q4;
                const uint32_t node = at < kCountStack ? stk[at] : deep[(size_t)(at - kCountStack) * kQuadsPerBlock];
                const float4* np = sc.nodes + 4 * (size_t)node;
                const float4 a = np[0], b = np[1], c = np[2];
                r = reinterpret_cast<const uint4*>(np)[3];
                hl = slab(o, inv, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, tn, tf);
                hr = slab(o, inv, V3{b.z, b.w, c.x}, V3{c.y, c.z, c.w}, tn, tf);
                tests += 2u + (hl ? r.y : 0u) + (hr ? r.w : 0u);  // a leaf's primitives are all tested
                hl = hl && r.y == 0u;
                hr = hr && r.w == 0u;
            }
            const uint32_t ml = (uint32_t)(ballot(hl) >> (lane & 60u)) & 0xFu;
            const uint32_t mr = (uint32_t)(ballot(hr) >> (lane & 60u)) & 0xFu;
            sp = max(sp - 4, 0);
            const int added = __popc(ml) + __popc(mr);
            if (sp + added > cap) {
                overflow = true;
                sp = 0;
                continue;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // all entries are read before their places are reused
            int at = sp + __popc(ml & after) + __popc(mr & after);
            auto put = [&](uint32_t node) {
                if (at < kCountStack)
                    stk[at] = node;
                else
                    deep[(size_t)(at - kCountStack) * kQuadsPerBlock] = node;
                ++at;
            };
            if (hr) put(r.z);
            if (hl) put(r.x);
            sp += added;
        }
        tests += (uint32_t)__shfl_xor((int)tests, 1);
        tests += (uint32_t)__shfl_xor((int)tests, 2);
        if (inside && q4 == 0u) out[i] = tests;
    }
    if (overflow) atomicOr(flags, 1u);
}

__global__ __launch_bounds__(kBlock) void k_camera_rays(DevCamera cam, float4* __restrict__ rays) {
    const uint64_t n = (uint64_t)cam.width * cam.height;
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    V3 o, d;
    pixel_ray(cam, i, o, d);
    rays[2 * i] = make_float4(o.x, o.y, o.z, 0.0f);
    rays[2 * i + 1] = make_float4(d.x, d.y, d.z, 0.0f);
}

// Scratch of the allocation-free closest-hit entry point
// (spt_trace_noalloc) in scenes with a tree: word 0 holds the overflow flag, then come the
// traversal's ray counters and the traversal stacks' spill area. Each device holds its own copy; host code reaches it
// only through the address hipGetSymbolAddress returns for that device.
static __device__ __align__(256) uint32_t scratch[SPT_NOALLOC_SCRATCH_WORDS];
constexpr uint32_t kScratchRays = 64, kScratchSpill = kScratchRays + kRayCounterWords;

__global__ void k_scratch_reset(uint32_t* __restrict__ ctl) {
    ctl[threadIdx.x] = 0u;
}

__global__ void k_scratch_fold_overflow(const uint32_t* __restrict__ ctl, uint32_t* __restrict__ ctx_flags) {
    if (threadIdx.x == 0 && ctl[0] != 0u) atomicOr(ctx_flags, 1u);
}

uint32_t grid_for(const spt_ctx* ctx, uint64_t n) {
    uint64_t want = (n + kBlock - 1) / kBlock;
    uint64_t cap = (uint64_t)ctx->num_cus * 16;  // resident-size grid, stride loop beyond
    if (want > cap) want = cap;
    if (want == 0) want = 1;
    return (uint32_t)want;
}

}  // namespace

namespace {

// Idle lanes of a wave that make it take new rays (spt_tuning.refill_lanes).
uint32_t refill_of(const spt_ctx* ctx) {
    const uint32_t want = ctx->tuning.refill_lanes ? ctx->tuning.refill_lanes : kRefillLanes;
    return std::min<uint32_t>(kMaxRefillLanes, std::max<uint32_t>(1, want));
}

// Grid of a quad kernel over n rays: what the chip holds at once, or a block
// per 16 rays when that is fewer (a wave takes at least 4).
uint32_t quad_grid(spt_ctx* ctx, const void* kernel, uint64_t n) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess || per_cu <= 0)
        per_cu = 4;
    return (uint32_t)std::min<uint64_t>((uint64_t)per_cu * ctx->num_cus, (n + 15) / 16);
}

constexpr uint64_t kMaxLaunchRays = 1ull << 31;  // rays of one launch (32-bit ray counter)

// Launches `launch(base, n, grid)` over [0, total) with the ray counters
// reset before each launch that uses them.
template <typename Launch>
spt_status quad_launches(spt_ctx* ctx, const void* kernel, uint64_t total, Launch launch, const char* what) {
    for (uint64_t base = 0; base < total; base += kMaxLaunchRays) {
        const uint32_t n = (uint32_t)std::min(kMaxLaunchRays, total - base);
        const uint32_t grid = quad_grid(ctx, kernel, n);
        spt_status s = ensure_spill(ctx, std::max<size_t>(1, (size_t)grid * quad_spill_words(ctx->stack_cap4)));
        if (s != SPT_OK) return s;
        if (RayShares(n, grid * (kBlock / 64)).fixed < n) {  // only larger launches use the counters
            s = check_hip(ctx, hipMemsetAsync(ctx->d_rays, 0, kRayCounterWords * 4, ctx->stream), "ray counters");
            if (s != SPT_OK) return s;
        }
        launch(base, n, grid);
        s = check_hip(ctx, hipGetLastError(), what);
        if (s != SPT_OK) return s;
    }
    return SPT_OK;
}

// The same for the kernels of a scene of one block, a ray per lane.
template <typename Launch>
spt_status block_launches(spt_ctx* ctx, uint64_t total, Launch launch, const char* what) {
    for (uint64_t base = 0; base < total; base += kMaxLaunchRays) {
        const uint32_t n = (uint32_t)std::min(kMaxLaunchRays, total - base);
        launch(base, n, grid_for(ctx, n));
        const spt_status s = check_hip(ctx, hipGetLastError(), what);
        if (s != SPT_OK) return s;
    }
    return SPT_OK;
}

}  // namespace

spt_status launch_trace(spt_ctx* ctx, const spt_ray32* d_rays, uint64_t n, spt_hit* d_hits, uint32_t mode,
                        uint32_t* d_tests, uint32_t* d_isects) {
    if (n == 0) return SPT_OK;
    DevScene sc = ctx->scene();
    const float4* rays = reinterpret_cast<const float4*>(d_rays);
    uint2* hits = reinterpret_cast<uint2*>(d_hits);
    if (mode == SPT_TRACE_CLOSEST && ctx->one_block)
        return block_launches(
            ctx, n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL(k_trace_block, dim3(grid), dim3(kBlock), 0, ctx->stream, sc, rays + 2 * base, cnt,
                                   hits + base);
            },
            "trace launch");
    if (mode == SPT_TRACE_CLOSEST)
        return quad_launches(
            ctx, reinterpret_cast<const void*>(&k_trace_q<false, true>), n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL((sc.small_tree ? k_trace_q<false, true> : k_trace_q<false, false>), dim3(grid),
                                   dim3(kBlock), 0, ctx->stream, sc, rays + 2 * base, cnt,
                                   hits + base, nullptr, nullptr, ctx->d_spill, ctx->d_flags, ctx->d_rays, refill_of(ctx));
            },
            "trace launch");
    if (mode == SPT_TRACE_FETCH)
        return quad_launches(
            ctx, reinterpret_cast<const void*>(&k_trace_q<true, false>), n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL((k_trace_q<true, false>), dim3(grid), dim3(kBlock), 0, ctx->stream, sc, rays + 2 * base, cnt,
                                   hits + base, d_tests + base, d_isects + base, ctx->d_spill, ctx->d_flags,
                                   ctx->d_rays, refill_of(ctx));
            },
            "trace launch");
    const uint32_t grid = grid_for(ctx, n);
    spt_status s = ensure_spill(ctx, (size_t)grid * kBlock * (ctx->stack_cap > kLdsStack ? ctx->stack_cap - kLdsStack : 1));
    if (s != SPT_OK) return s;
    if (mode == SPT_TRACE_COUNT)
        hipLaunchKernelGGL((k_trace<true>), dim3(grid), dim3(kBlock), 0, ctx->stream, sc, rays, n, hits, d_tests,
                           d_isects, ctx->d_spill, ctx->d_flags);
    else
        hipLaunchKernelGGL((k_trace<false>), dim3(grid), dim3(kBlock), 0, ctx->stream, sc, rays, n, hits, nullptr,
                           nullptr, ctx->d_spill, ctx->d_flags);
    return check_hip(ctx, hipGetLastError(), "trace launch");
}

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};
bool g_scratch_done[kMaxScratchDevices] = {};
}  // namespace

spt_status init_static_scratch(spt_ctx* ctx) {
    if (ctx->device < 0 || ctx->device >= kMaxScratchDevices) {
        ctx->scratch = nullptr;
        return SPT_OK;  // the allocation-free entry point reports it when called
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_done[ctx->device]) {
        // the calling thread has ctx->device current (spt_create set it)
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) {
            (void)hipGetLastError();
            ctx->scratch = nullptr;
            return check_hip(ctx, e, "static scratch address");
        }
        g_scratch_ptr[ctx->device] = ptr;
        g_scratch_done[ctx->device] = true;
    }
    ctx->scratch = static_cast<uint32_t*>(g_scratch_ptr[ctx->device]);
    return SPT_OK;
}

spt_status launch_trace_noalloc(spt_ctx* ctx, const spt_ray32* d_rays, uint64_t n, spt_hit* d_hits) {
    if (n > SPT_NOALLOC_MAX_RAYS)
        return set_error(ctx, SPT_ERR_INVALID, "spt_trace_noalloc: more than SPT_NOALLOC_MAX_RAYS rays");
    if (!ctx->scratch) return set_error(ctx, SPT_ERR_STATE, "spt_trace_noalloc: no static scratch on this device");
    if (n == 0) return SPT_OK;
    if (ctx->one_block) {  // no stack, no counters: the kernel of spt_trace, and its results
        const DevScene sc = ctx->scene();
        return block_launches(
            ctx, n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL(k_trace_block, dim3(grid), dim3(kBlock), 0, ctx->stream, sc,
                                   reinterpret_cast<const float4*>(d_rays) + 2 * base, cnt,
                                   reinterpret_cast<uint2*>(d_hits) + base);
            },
            "trace (no allocation) launch");
    }
    const void* kern = reinterpret_cast<const void*>(&k_trace_q<false, true>);
    // blocks whose stack entries beyond the LDS part fit the scratch
    const uint64_t per_block = quad_spill_words(ctx->stack_cap4);
    const uint64_t room = (uint64_t)SPT_NOALLOC_SCRATCH_WORDS - kScratchSpill;
    const uint64_t max_blocks = per_block ? room / per_block : ~0ull;
    if (max_blocks == 0)
        return set_error(ctx, SPT_ERR_UNSUPPORTED, "spt_trace_noalloc: the tree is too deep for the static scratch");
    uint32_t* ctl = ctx->scratch;
    uint32_t* spill = ctx->scratch + kScratchSpill;
    const float4* rays = reinterpret_cast<const float4*>(d_rays);
    uint2* hits = reinterpret_cast<uint2*>(d_hits);
    for (uint64_t base = 0; base < n; base += kMaxLaunchRays) {
        const uint32_t cnt = (uint32_t)std::min(kMaxLaunchRays, n - base);
        const uint32_t grid = (uint32_t)std::min<uint64_t>(quad_grid(ctx, kern, cnt), max_blocks);
        // a fill kernel, not a memset node: callers may capture this in a graph
        hipLaunchKernelGGL(k_scratch_reset, dim3(1), dim3(kScratchSpill), 0, ctx->stream, ctl);
        hipLaunchKernelGGL((ctx->small_tree ? k_trace_q<false, true> : k_trace_q<false, false>), dim3(grid), dim3(kBlock),
                           0, ctx->stream, ctx->scene(), rays + 2 * base,
                           cnt, hits + base, nullptr, nullptr, spill, ctl, ctl + kScratchRays, refill_of(ctx));
        // a stack overflow is reported by spt_sync, as for spt_trace
        hipLaunchKernelGGL(k_scratch_fold_overflow, dim3(1), dim3(64), 0, ctx->stream, ctl, ctx->d_flags);
    }
    return check_hip(ctx, hipGetLastError(), "trace (no allocation) launch");
}

spt_status launch_camera_rays(spt_ctx* ctx, const spt_camera* cam, spt_ray32* d_rays) {
    const uint64_t n = (uint64_t)cam->width * cam->height;
    const uint32_t grid = (uint32_t)((n + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(k_camera_rays, dim3(grid), dim3(kBlock), 0, ctx->stream, make_camera(*cam),
                       reinterpret_cast<float4*>(d_rays));
    return check_hip(ctx, hipGetLastError(), "camera rays launch");
}

spt_status launch_raycast(spt_ctx* ctx, const spt_camera* cam, uint32_t kind, void* d_out) {
    const uint64_t n = (uint64_t)cam->width * cam->height;
    if (n == 0) return SPT_OK;
    DevScene sc = ctx->scene();
    DevCamera dc = make_camera(*cam);
    float* out = reinterpret_cast<float*>(d_out);
    if (ctx->one_block && kind != SPT_RAYCAST_COUNT)
        return block_launches(
            ctx, n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL(
                    (kind == SPT_RAYCAST_NORMAL ? k_raycast_block<SPT_RAYCAST_NORMAL> : k_raycast_block<SPT_RAYCAST_DEPTH>),
                    dim3(grid), dim3(kBlock), 0, ctx->stream, sc, dc, base, cnt, out);
            },
            "raycast launch");
    if (kind == SPT_RAYCAST_NORMAL)
        return quad_launches(
            ctx, reinterpret_cast<const void*>(&k_raycast<SPT_RAYCAST_NORMAL, true>), n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL((sc.small_tree ? k_raycast<SPT_RAYCAST_NORMAL, true> : k_raycast<SPT_RAYCAST_NORMAL, false>),
                                   dim3(grid), dim3(kBlock), 0, ctx->stream, sc, dc,
                                   base, cnt, out, ctx->d_spill, ctx->d_flags, ctx->d_rays, refill_of(ctx));
            },
            "raycast launch");
    if (kind == SPT_RAYCAST_DEPTH)
        return quad_launches(
            ctx, reinterpret_cast<const void*>(&k_raycast<SPT_RAYCAST_DEPTH, true>), n,
            [&](uint64_t base, uint32_t cnt, uint32_t grid) {
                hipLaunchKernelGGL((sc.small_tree ? k_raycast<SPT_RAYCAST_DEPTH, true> : k_raycast<SPT_RAYCAST_DEPTH, false>),
                                   dim3(grid), dim3(kBlock), 0, ctx->stream, sc, dc,
                                   base, cnt, out, ctx->d_spill, ctx->d_flags, ctx->d_rays, refill_of(ctx));
            },
            "raycast launch");
    uint32_t* counts = reinterpret_cast<uint32_t*>(d_out);
    if (count_by_lane(sc, n)) {
        const uint32_t grid = grid_for(ctx, n);
        spt_status s = ensure_spill(ctx, (size_t)grid * kBlock * (ctx->stack_cap > kLdsStack ? ctx->stack_cap - kLdsStack : 1));
        if (s != SPT_OK) return s;
        hipLaunchKernelGGL(k_raycast_count_lane, dim3(grid), dim3(kBlock), 0, ctx->stream, sc, dc, counts, ctx->d_spill,
                           ctx->d_flags);
    } else {
        const uint64_t tiles = (((uint64_t)dc.width + 3) / 4) * (((uint64_t)dc.height + 3) / 4);
        const uint32_t grid = (uint32_t)std::min<uint64_t>((tiles + kBlock / 64 - 1) / (kBlock / 64), (uint64_t)ctx->num_cus * 16);
        spt_status s = ensure_spill(ctx, std::max<size_t>(1, grid * count_spill_words(sc.stack_cap)));
        if (s != SPT_OK) return s;
        hipLaunchKernelGGL(k_raycast_count, dim3(grid), dim3(kBlock), 0, ctx->stream, sc, dc, counts, ctx->d_spill,
                           ctx->d_flags);
    }
    return check_hip(ctx, hipGetLastError(), "raycast launch");
}

}  // namespace spt
