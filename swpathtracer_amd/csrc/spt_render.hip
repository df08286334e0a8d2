// spt_render.hip - wavefront path tracer (replaces PathTracer::render and the
// recursive estimator of integrators/pathtracer.cpp:12-147).
//
// Pipeline per bounce, each a separate kernel over a queue of live paths:
//   generate (camera sample + primary ray) -> extend (closest hit) ->
//   [walk: the random walks through layered materials] -> shade (emission,
//   BSDF sample, Russian roulette, next ray; finished paths write the film) ->
//   the survivors form the next queue.
// The last paths of a call run to their end in one kernel (k_finish).
// The recursion L = Le + f * L' * cos / pdf is evaluated forwards with a
// throughput: L = sum_d (prod_{j<d} f_j cos_j / pdf_j) * Le_d.
#include <algorithm>
#include <chrono>
#include <mutex>
#include <thread>

#include "spt_bsdf.h"
#include "spt_guide.h"
#include "spt_quad.h"

namespace spt {

namespace {

constexpr uint32_t kLdsMats = 48;         // shading stages up to this many materials in LDS
constexpr int kWalkRefill = 32;           // lanes of a wave without a walk that make it take new ones

// Path state of one buffer (structure of arrays, one slot per live path).
// Two buffers alternate: shade reads buffer A and appends survivors to B.
struct PathBuf {
    float4* o;       // ray origin; .w: pixel index (bits)
    float4* d;       // ray direction; .w: scene of the path in a multi-scene call (bits)
    float4* thr;     // throughput; .w: draws consumed (bits)
    float4* rad;     // radiance so far; .w: depth (bits)
    uint64_t* key;   // RNG key (counter mode) or replay-stream row
    uint64_t* local; // path index within this render call (per-path output)
    uint4* grec;     // guide training records of this path: 3 slots + count
};
constexpr size_t kBufBytes = 16 * 5 + 8 * 2;
constexpr uint32_t kNoRec = 0xFFFFFFFFu;

// Per-bounce scratch shared by both buffers.
struct Work {
    float4* hit;       // t, leaf-order triangle index (bits), u, v   (indexed like buffer A)
    uint32_t* skey;    // material of the hit, n_mats for a miss
    float2* walk;      // layered walks: cosine and density of the sampled direction
    uint32_t* cnt;     // [0], [1]: live counts of the two buffers; [2]: replay overflows;
                       // u64 at [10]: rays, u64 at [12]: bounces
    uint32_t* rays;    // ray counters of the extend kernel (kRayCounterWords)
};
constexpr size_t kWorkBytes = 16 + 4 + 8;

struct RenderArgs {
    DevScene sc;
    Job job;                    // single-scene call
    const Job* jobs;            // multi-scene call: per-job parameters (path d.w = job)
    const BatchTile* tiles;     // multi-scene call: generation order
    const uint64_t* tile_start; // first path of each tile (n_tiles + 1 entries)
    uint32_t n_tiles;
    uint32_t n_jobs;
    uint32_t* job_done;         // paths finished per job
    uint64_t* job_clock;        // [0] start, [1 + j] finish of job j (device wall clock)
    uint32_t flags;
    uint32_t per_path;  // some job writes per-path radiance: paths carry their output index
    uint32_t refill;  // idle lanes that trigger a ray refill in the traversal
    uint32_t walk;  // k_walk runs the walks of materials of several layers
    uint64_t gen_base;  // number of this wavefront's first path in the call's numbering
    // learned guide
    uint32_t guided, train;
    uint32_t gflags;          // SPT_GUIDE_*
    const uint8_t* guidable;  // per material: kGuideSingle / kGuideCoated / 0
    float bsdf_frac;
    unsigned short* gout;     // per path slot: 40 raw network outputs (IEEE half)
    float* records;           // training records (guide::kRecord floats each)
    uint32_t* rec_count;  // [0]: records written, [1]: candidate vertices (one 8-B aligned u64)
    uint32_t* rec_shared; // concurrent wavefronts: one rec_count for all (else nullptr: the work words)
    const float* theta;          // guide parameters (FP32 master copy)
    const unsigned short* wbf;   // guide weights in bf16
    GuideBox gbox;               // encoding box of the guide
    uint32_t rec_cap;
    uint32_t rec_stride;  // record 1 in rec_stride candidates (hash of key and depth)
    uint32_t rec_ring;    // in-call training: record slots wrap around rec_cap
};

__device__ inline float lum(V3 c) { return 0.2126f * c.x + 0.7152f * c.y + 0.0722f * c.z; }

// Tag of record k of the path with RNG key `key`, kept in the record: with a
// ring of record slots a slot can be reused while its first path is alive,
// and that path must then leave the new record alone.
__device__ inline uint32_t rec_tag(uint64_t key, uint32_t k) {
    return (uint32_t)mix64(key * 3u + k + 1u);
}

// Training targets of a finished path: the radiance that arrived along each
// recorded wi is (L - radiance before it) / throughput after it.
__device__ inline void finish_records(const RenderArgs& a, uint4 gr, float4 L, uint64_t key) {
    const uint32_t sl[3] = {gr.x, gr.y, gr.z};
    for (uint32_t k = 0; k < gr.w && k < 3; ++k) {
        float* r = a.records + (size_t)sl[k] * guide::kRecord;
        if (__float_as_uint(r[20]) != rec_tag(key, k)) continue;  // slot reused
        const float lt = lum(V3{r[17], r[18], r[19]});
        const float li = lum(V3{L.x - r[14], L.y - r[15], L.z - r[16]});
        r[12] = (lt > 0.0f && li > 0.0f) ? r[13] * li / lt : 0.0f;
    }
}

// Guide mode of a material in this call: coated layers only with SPT_GUIDE_COATED.
__device__ inline uint32_t guide_mode(const RenderArgs& a, uint32_t mid) {
    const uint32_t g = a.guidable[mid];
    return (g == kGuideCoated && !(a.gflags & SPT_GUIDE_COATED)) ? 0u : g;
}

template <bool MULTI>
__device__ inline const Job& job_of(const RenderArgs& a, uint32_t j) {
    if (MULTI) return a.jobs[j];
    return a.job;
}

// Adds finished paths to a job's count and stamps the job's finish time when
// its last path is counted.
__device__ inline void count_done(const RenderArgs& a, uint32_t jid, uint32_t n) {
    const uint32_t k = atomicAdd(&a.job_done[jid], n);
    if ((uint64_t)k + n == a.jobs[jid].n_paths) a.job_clock[1 + jid] = wall_clock64();
}

// Film and per-path output of a finished path. A multi-scene call also counts
// the job's finished paths: in the block's LDS counters (`done`, added to the
// job's at the block's end: one global atomic per block and job instead of one
// per wave, whose addresses all XCDs share) when the jobs fit them.
constexpr uint32_t kDoneJobs = 512;
template <bool MULTI>
__device__ __forceinline__ void finish_path(const RenderArgs& a, const Job& jb, uint32_t jid, uint32_t pix, uint64_t local,
                                   float4 L, uint32_t* done) {
    if (MULTI) {
        if (a.n_jobs <= kDoneJobs)
            atomicAdd(&done[jid], 1u);
        else
            count_done(a, jid, 1u);
    }
    if (jb.film32) {
        float* f = jb.film32 + 3 * (size_t)pix;
        // adding 0 changes nothing, and most paths end without light: 28M paths
        // shaded in 1.37 ms instead of 1.65 (blocks of 256)
        if (L.x != 0.0f) unsafeAtomicAdd(f + 0, L.x);
        if (L.y != 0.0f) unsafeAtomicAdd(f + 1, L.y);
        if (L.z != 0.0f) unsafeAtomicAdd(f + 2, L.z);
    }
    if (jb.film64) {
        double* f = jb.film64 + 3 * (size_t)pix;
        if (L.x != 0.0f) unsafeAtomicAdd(f + 0, (double)L.x);
        if (L.y != 0.0f) unsafeAtomicAdd(f + 1, (double)L.y);
        if (L.z != 0.0f) unsafeAtomicAdd(f + 2, (double)L.z);
    }
    if (jb.path_rgb) {
        float* o = jb.path_rgb + 3 * (size_t)local;
        o[0] = L.x;
        o[1] = L.y;
        o[2] = L.z;
    }
}

__device__ inline Draws make_draws(const Job& jb, uint64_t key, uint32_t k) {
    Draws r;
    r.k = k;
    r.overflow = false;
    r.stride = jb.stride;
    if (jb.stream) {
        r.key = 0;
        r.stream = jb.stream + key * (uint64_t)jb.stride;
    } else {
        r.key = key + (uint64_t)(k + 1) * kGolden;
        r.stream = nullptr;
    }
    return r;
}

// Camera sample of path g into slot s of buffer A:
// integrators/pathtracer.cpp:104-113. A single-scene call numbers its paths
// sample by sample over the viewport's pixels; a multi-scene call walks its
// tile list. The per-path output index is pixel * spp_count + sample either way.
// With max depth 0 (single-scene calls only) the path finishes here.
template <bool MULTI>
__device__ inline void gen_path(const RenderArgs& a, PathBuf& A, const Work& w, uint32_t s, uint64_t g) {
    g += a.gen_base;  // a wavefront numbers its own paths from 0
    uint32_t jid = 0;
    uint64_t pl, local;
    uint32_t smp;
    if (MULTI) {
        uint32_t lo = 0, hi = a.n_tiles - 1;  // last tile starting at or before g
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (a.tile_start[mid] <= g)
                lo = mid;
            else
                hi = mid - 1;
        }
        const BatchTile tl = a.tiles[lo];
        const uint64_t q = g - a.tile_start[lo];
        jid = tl.job;
        pl = tl.p0 + q % tl.np;
        smp = tl.s0 + (uint32_t)(q / tl.np);
        local = pl * a.jobs[jid].spp_count + (smp - a.jobs[jid].spp_begin);
    } else {
        // pixel-minor: consecutive paths are neighbouring pixels (coherent
        // primary rays, and no pile-up of one pixel's film atomics in a wave)
        const uint64_t npl = (uint64_t)a.job.vw * a.job.vh;
        pl = g % npl;
        smp = a.job.spp_begin + (uint32_t)(g / npl);
        local = pl * a.job.spp_count + (smp - a.job.spp_begin);
    }
    const Job& jb = job_of<MULTI>(a, jid);
    const uint32_t x = jb.vl + (uint32_t)(pl % jb.vw), y = jb.vt + (uint32_t)(pl / jb.vw);
    const uint64_t path = ((uint64_t)y * jb.cam.width + x) * jb.spp + smp;
    const uint32_t pix = y * jb.cam.width + x;
    const uint64_t key = jb.stream ? local : rng_key(jb.seed, path);
    Draws r = make_draws(jb, key, 0);
    float sx, sy;
    pixel_offset(jb.sampler, jb.n_sub, jb.w_sub, smp, r, sx, sy);
    const float xs = x + sx, ys = y + sy;
    V3 o, d;
    camera_ray(jb.cam, xs, ys, o, d);
    if (r.overflow) atomicAdd(&w.cnt[2], 1u);
    if (jb.max_depth == 0) {  // depth >= path_length before the first trace
        finish_path<MULTI>(a, jb, jid, pix, local, make_float4(0.0f, 0.0f, 0.0f, 0.0f), nullptr);
        return;
    }
    A.o[s] = make_float4(o.x, o.y, o.z, __uint_as_float(pix));
    A.d[s] = make_float4(d.x, d.y, d.z, __uint_as_float(jid));
    A.thr[s] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(r.k));
    A.rad[s] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(0u));
    A.key[s] = key;
    if (a.per_path) A.local[s] = local;
    if (a.train) A.grec[s] = make_uint4(kNoRec, kNoRec, kNoRec, 0u);
}

// Paths [base, base + n) (of this wavefront) into slots [0, n) of buffer A;
// a call with max depth 0 finishes them all here.
template <bool MULTI>
__global__ __launch_bounds__(kBlock) void k_generate(RenderArgs a, PathBuf A, Work w, uint64_t base, uint32_t n) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s < n) gen_path<MULTI>(a, A, w, s, base + s);
}

// Work-word layout (w.cnt, 64 words): [0], [1] live counts of the two
// buffers; [2] replay overflows; u64 [10] rays, u64 [12] bounces; [16] guide records, [17] candidates;
// u64 [20] next path to generate; [24] first slot and [25] number of the
// planned new paths, u64 [26] their first path index; [28] plans made.
// A ray counter's line (w.rays) also holds, for the blocks that share it: u64
// [2] rays k_finish traced, [4] the segments of its longest path, u64 [6]
// hits evaluated by the guide network.
// Live paths from which k_finish takes over once none is left to generate: two
// for each lane of the waves that fit the chip. 2^17, 2^18, 2^19, 2^20: 800x600
// mesh image, 4 samples 4.28, 4.06, 3.94, 3.83 ms; 256x256 box image, 16
// samples 1.35, 1.35, 1.35, 1.46 ms; batch of 8 scenes 7.11, 7.06, 7.03, 7.02.
constexpr uint32_t kFinishPaths = 1u << 19;
// Live paths below which the host follows each bounce closely.
constexpr uint32_t kNearEnd = 1u << 21;
constexpr int kFinishRays = 2, kFinishBounces = 4, kGuideQueries = 6;
constexpr int kGen = 20, kPlanSlot = 24, kPlanN = 25, kPlanPath = 26, kPlanSeq = 28;

// Between bounces (one wave): the consumed buffer's count and the extend
// kernel's ray counters go back to zero (a kernel, not a memset, so the bounce
// can be graph-captured), and new camera paths are planned into the free
// tail of the survivors' buffer B: n = min(capacity - survivors, paths not
// yet generated). Progress goes to mapped host memory: status[1] = live
// paths after the refill, status[2] = all paths generated, then status[0] =
// the plan's sequence number, so the host can stop issuing bounces without
// waiting on the stream.
__global__ void k_plan(uint32_t* cntA, uint32_t* cntB, uint32_t* cnt, uint32_t* rays, uint32_t cap, uint64_t total,
                       uint32_t* status, uint64_t* job_clock) {
    if (threadIdx.x < kRayCounters) rays[threadIdx.x * kRayCounterStride] = 0;
    if (threadIdx.x != 0) return;
    if (cntA) *cntA = 0;
    const uint32_t have = *cntB;
    uint64_t* gen = reinterpret_cast<uint64_t*>(cnt + kGen);
    const uint64_t g0 = *gen;
    if (g0 == 0 && job_clock) job_clock[0] = wall_clock64();
    const uint32_t n = (uint32_t)min((uint64_t)(cap - have), total - g0);
    cnt[kPlanSlot] = have;
    cnt[kPlanN] = n;
    *reinterpret_cast<uint64_t*>(cnt + kPlanPath) = g0;
    *cntB = have + n;
    *gen = g0 + n;
    const uint32_t seq = cnt[kPlanSeq] + 1;
    cnt[kPlanSeq] = seq;
    if (status) {
        volatile uint32_t* hs = status;
        hs[1] = have + n;
        hs[2] = (g0 + n == total) ? 1u : 0u;
        hs[3] = cnt[16];  // guide records written so far
        __threadfence_system();
        hs[0] = seq;
    }
}

// The paths k_plan planned, generated into buffer B (grid-stride).
template <bool MULTI>
__global__ __launch_bounds__(kBlock) void k_refill(RenderArgs a, PathBuf B, Work w) {
    const uint32_t slot0 = w.cnt[kPlanSlot], n = w.cnt[kPlanN];
    const uint64_t g0 = *reinterpret_cast<const uint64_t*>(w.cnt + kPlanPath);
    for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < n; s += gridDim.x * kBlock)
        gen_path<MULTI>(a, B, w, slot0 + s, g0 + s);
}

// Closest hit of every live path of buffer A (count *cntA). Persistent
// traversal; hit record and material written at the path's slot. FETCH adds
// node / triangle record fetch counts to the two 64-bit counters at flags + 4.
template <bool FETCH, bool MULTI, bool SMALL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kQuadWaves))) void k_extend(RenderArgs a, PathBuf A, Work w, const uint32_t* __restrict__ cntA,
                                                   uint32_t* __restrict__ spill, uint32_t* __restrict__ flags) {
    __shared__ QuadLds lds;
    __shared__ unsigned long long fetched[2];
    const uint32_t n = *cntA;
    if (n == 0) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(reinterpret_cast<unsigned long long*>(w.cnt + 10), (unsigned long long)n);
        atomicAdd(reinterpret_cast<unsigned long long*>(w.cnt + 12), 1ull);
    }
    bool overflow = false;
    unsigned long long my_nodes = 0, my_tris = 0;
    if (FETCH) {
        if (threadIdx.x < 2) fetched[threadIdx.x] = 0;
        __syncthreads();
    }
    trace_quads<FETCH, SMALL>(
        a.sc, n, w.rays, lds, spill + (size_t)blockIdx.x * quad_spill_words(a.sc.stack_cap4), overflow, a.refill,
        [&](uint32_t i, V3& o, V3& d, Root& root) {
            const float4 o4 = A.o[i], d4 = A.d[i];
            o = V3{o4.x, o4.y, o4.z};
            d = V3{d4.x, d4.y, d4.z};
            if (MULTI) {
                const Job& jb = a.jobs[__float_as_uint(d4.w)];
                root = Root{V3{jb.rmin[0], jb.rmin[1], jb.rmin[2]}, V3{jb.rmax[0], jb.rmax[1], jb.rmax[2]}, jb.node0};
            }
        },
        [&](uint32_t i, const Hit& h, V3, V3, uint32_t nn, uint32_t nt) {
            w.hit[i] = make_float4(h.t, __uint_as_float(h.idx), h.u, h.v);
            w.skey[i] = (h.idx == kNoHit) ? a.sc.n_mats : h.mat;
            if (FETCH) {
                my_nodes += nn;
                my_tris += nt;
            }
        });
    if (overflow) atomicOr(flags, 1u);
    if (FETCH) {
        atomicAdd(&fetched[0], my_nodes);
        atomicAdd(&fetched[1], my_tris);
        __syncthreads();
        if (threadIdx.x < 2)
            atomicAdd(reinterpret_cast<unsigned long long*>(flags + 4) + threadIdx.x, fetched[threadIdx.x]);
    }
}

// Guide inference for the live hits of buffer A whose material is guidable:
// each wave encodes 64 hits (one per lane) and runs the
// register-resident MLP; raw outputs go to gout[slot] as half floats.
__global__ __launch_bounds__(kBlock) void k_guide_paths(RenderArgs a, PathBuf A, Work w,
                                                        const uint32_t* __restrict__ cntA,
                                                        const float* __restrict__ theta,
                                                        const unsigned short* __restrict__ wbf, GuideBox box) {
    using namespace guide;
    extern __shared__ float dyn[];
    FwdWeights& sw = *reinterpret_cast<FwdWeights*>(dyn);
    WaveStage* stages = reinterpret_cast<WaveStage*>(reinterpret_cast<char*>(dyn) + sizeof(FwdWeights));
    const uint32_t n = *cntA;
    if (n == 0) return;
    load_weights(sw, wbf, theta);
    __syncthreads();
    const int wave = threadIdx.x >> 6, l = __lane_id(), r = l & 15;
    WaveStage& st = stages[wave];
    uint32_t queries = 0;
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        const uint32_t slot = base + threadIdx.x;
        bool mine = false;
        float f[kEnc];
        if (slot < n) {
            const float4 hv = w.hit[slot];
            const uint32_t idx = __float_as_uint(hv.y);
            mine = (idx != kNoHit) && guide_mode(a, w.skey[slot]) != 0u;
            if (mine) {
                const float4 o4 = A.o[slot], d4 = A.d[slot];
                const V3 d{d4.x, d4.y, d4.z};
                Hit h;
                h.t = hv.x;
                h.idx = idx;
                h.u = hv.z;
                h.v = hv.w;
                const V3 pos = V3{o4.x, o4.y, o4.z} + d * h.t;
                encode(pos, shading_normal(a.sc, h, pos), -d, box.bmin, box.bext, f);
            }
        }
        if (!mine)
            for (int i = 0; i < kEnc; ++i) f[i] = 0.0f;
        const uint64_t any = __ballot(mine);
        queries += (uint32_t)__popcll(any);
        stage_row(st, f);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a stage belongs to one wave
        if (any)
            mlp_stage_fwd(sw, st, [&](int g16, const f32x4 y[3]) {
                const int src = 16 * g16 + r;
                const uint32_t s = __shfl(slot, src);
                if ((any >> src) & 1ull) store_outputs_h(a.gout + (size_t)s * kOut, y);
            });
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (l == 0 && queries)
        atomicAdd(reinterpret_cast<unsigned long long*>(w.rays + (blockIdx.x % kRayCounters) * kRayCounterStride + kGuideQueries),
                  (unsigned long long)queries);
}

// Density of a single BSDF layer's own sampler (guidable layers only).
__device__ inline float layer_density(const spt_layer& l, V3 wo, V3 wi) {
    if (l.type == SPT_BSDF_LAMBERTIAN) {
        if (wi.y <= 0.0f) return 0.0f;
        return (l.sampler == SPT_SAMPLER_UNIFORM) ? 1.0f / (2.0f * kPi) : wi.y / kPi;
    }
    return ggx_pdf(l, wo, wi);
}

// Guide density of a direction w2 inside a smooth dielectric coat of IOR eta
// (local frame, pointing up): the guide proposes the exit direction above the
// coat, and w2 is the direction that refracts to it (tangential part scaled
// by 1/eta). p(w2) = p(exit) |d exit / d w2| = p(exit) eta^2 cos(w2) /
// cos(exit). Directions past the critical angle are never proposed.
__device__ __forceinline__ float coat_guide_density(const guide::Lobe* lobes, const Frame& fr, V3 w2, float eta) {
    const float t2 = eta * eta * (w2.x * w2.x + w2.z * w2.z);
    if (w2.y <= 0.0f || t2 >= 1.0f) return 0.0f;
    const float cy = sqrtf(1.0f - t2);
    const V3 out{eta * w2.x, cy, eta * w2.z};
    return guide::mixture_pdf(lobes, to_world(fr, out)) * (eta * eta * w2.y / cy);
}

// vMF stand-in (local frame) for the lobe of a guided layer, multiplied with
// the learned incident radiance to propose directions: Lambertian, the
// normal with kappa 3 (mean cosine 2/3, that of the cosine lobe); GGX, the
// mirror direction with kappa 1 / (4 alpha^2) (reflected spread about twice
// the microfacet spread alpha), widened by 'widen' (the IOR of a smooth coat
// above the layer, which scales exit angles).
__device__ inline void bsdf_lobe(const spt_layer& l, V3 wo, float widen, V3& mb, float& kb) {
    if (l.type == SPT_BSDF_LAMBERTIAN) {
        mb = V3{0.0f, 1.0f, 0.0f};
        kb = 3.0f;
        return;
    }
    mb = V3{-wo.x, wo.y, -wo.z};
    const float s = l.roughness * widen;
    kb = fminf(fmaxf(0.25f / fmaxf(s * s, 1e-8f), guide::kKappaMin), 1e3f);
}

// The layered random walk of layered_eval (materials/layered_bsdf.cpp:10-74)
// for a smooth dielectric coat over one opaque layer with an evaluable
// density, where the first visit of the opaque layer draws its direction from
// a one-sample mixture: the layer's own sampler with probability c, else the
// guide's exit direction mapped under the coat. The step density is the
// mixture's, so the walk weight estimates the same BSDF without bias. Later
// visits (after total internal reflection under the coat, where the guide
// has no density) use the layer's own sampler: mixing there would double the
// weight of every such revisit. 'via' is set when the walk reached the
// opaque layer.
__device__ __forceinline__ void layered_eval_guided(const spt_material& m, V3 wo, const Frame& frm, const guide::Lobe* lobes,
                                           float c, V3& bsdf, V3& refl, float& pdf, V3& wi, Draws& r, bool& via) {
    const spt_layer& coat = m.layers[0];
    const spt_layer& base = m.layers[1];
    const float eta = coat.ior, ieta = 1.0f / coat.ior;
    V3 fb{1.0f, 1.0f, 1.0f}, fr{1.0f, 1.0f, 1.0f};
    float fp = 1.0f;
    V3 nwo = wo;
    bool reached_inf = false;
    int bounce = 0;
    int id = (nwo.y > 0.0f) ? 0 : 1;
    const float inf = __builtin_inff();
    via = false;
    while ((id > -1) && (id < 2) && (fp > 0.0f) && (!reached_inf) && (bounce < 500)) {
        if (id == 0) {  // coat: the layer's own sampler, as in layered_eval
            const BSample s = layer_sample(coat, nwo, r);
            wi = s.wi;
            fp *= s.pdf;
            if (!(fp < inf)) reached_inf = true;
            if (wi.y > 0.0f) {
                fb = fb * layer_f(coat, nwo, wi);
                fr = fr * layer_reflectance(coat, nwo, wi);
                --id;
            } else if (wi.y < 0.0f) {
                fb = fb * (layer_f(coat, nwo, wi) * wi.y);
                fr = fr * layer_reflectance(coat, nwo, wi);
                ++id;
            } else {
                fp = 0.0f;
            }
        } else if (via) {  // opaque base, revisited: its own sampler, as in layered_eval
            const BSample s = layer_sample(base, nwo, r);
            wi = s.wi;
            fp *= s.pdf;
            if (!(fp < inf)) reached_inf = true;
            if (wi.y > 0.0f) {
                fb = fb * (layer_f(base, nwo, wi) * wi.y);
                fr = fr * layer_reflectance(base, nwo, wi);
                --id;
            } else {
                fp = 0.0f;
            }
        } else {  // opaque base, first visit: one-sample mixture with the guide
            via = true;
            if (r.next() < c) {
                wi = layer_sample(base, nwo, r).wi;
            } else {
                const float u0 = r.next(), u1 = r.next(), u2 = r.next();
                const V3 g = to_local(frm, guide::mixture_sample(lobes, u0, u1, u2));
                if (g.y > 0.0f) {
                    const float tx = g.x * ieta, tz = g.z * ieta;
                    wi = V3{tx, sqrtf(gmax(0.0f, 1.0f - tx * tx - tz * tz)), tz};
                } else {
                    wi = V3{0.0f, -1.0f, 0.0f};  // exit below the surface: no contribution
                }
            }
            const float p = c * layer_density(base, nwo, wi) + (1.0f - c) * coat_guide_density(lobes, frm, wi, eta);
            if ((wi.y > 0.0f) && (p > 0.0f)) {
                fp *= p;
                if (!(fp < inf)) reached_inf = true;
                fb = fb * (layer_f(base, nwo, wi) * wi.y);
                fr = fr * layer_reflectance(base, nwo, wi);
                --id;
            } else {
                fp = 0.0f;
            }
        }
        if (!((fb.x < inf) && (fb.y < inf) && (fb.z < inf))) reached_inf = true;
        nwo = -wi;
        ++bounce;
    }
    if ((bounce < 500) && !reached_inf && (fp > 0.0f)) {
        pdf = fp;
        bsdf = fb;
        refl = fr;
    } else {
        pdf = 1.0f;
        bsdf = V3{0.0f, 0.0f, 0.0f};
        refl = V3{0.0f, 0.0f, 0.0f};
    }
}

// What a path that goes on carries into the next bounce.
struct Survivor {
    float4 o, d, thr, rad;
    uint64_t key, local;
    uint4 gr;
};

template <bool GUIDED>
__device__ __forceinline__ void store_survivor(const RenderArgs& a, const PathBuf& B, const Survivor& sv, uint32_t slot) {
    B.o[slot] = sv.o;
    B.d[slot] = sv.d;
    B.thr[slot] = sv.thr;
    B.rad[slot] = sv.rad;
    B.key[slot] = sv.key;
    if (a.per_path) B.local[slot] = sv.local;
    if (GUIDED && a.train) B.grec[slot] = sv.gr;
}

// A path's vertex at its hit: position, shading normal, local frame and
// outgoing direction in it.
__device__ __forceinline__ void path_vertex(const RenderArgs& a, V3 o, V3 d, float4 hv, V3& pos, V3& nrm, Frame& fr, V3& wo) {
    Hit h;
    h.t = hv.x;
    h.idx = __float_as_uint(hv.y);
    h.u = hv.z;
    h.v = hv.w;
    pos = o + d * h.t;  // triangle.cpp:69
    nrm = shading_normal(a.sc, h, pos);
    fr = frame_from_up(nrm);          // pathtracer.cpp:28
    wo = normalize(to_local(fr, -d));    // pathtracer.cpp:30
}

// Shading of one vertex (integrators/pathtracer.cpp:21-54) of path j in
// shading order; go_on(survivor) is called for a path that does not end here.
template <bool MULTI, bool GUIDED, bool WALKS, typename GoOn>
__device__ __forceinline__ void shade_path(const RenderArgs& a, const PathBuf& A, const Work& w, const spt_material* smats,
                                  bool lds_mats, uint32_t i, uint32_t* done, GoOn go_on) {
    const float4 hv = w.hit[i];
    float4 rad = A.rad[i];
    const float4 thr = A.thr[i];
    const float4 o4 = A.o[i], d4 = A.d[i];
    const uint32_t pix = __float_as_uint(o4.w), jid = __float_as_uint(d4.w);
    const Job& jb = job_of<MULTI>(a, jid);
    const uint32_t depth = __float_as_uint(rad.w);
    const uint32_t idx = __float_as_uint(hv.y);
    const uint32_t mid = w.skey[i];
    // the path's walk is done: hit, o and d hold its results
    const bool walked = !WALKS && mid < a.sc.n_mats && (lds_mats ? smats[mid] : a.sc.mats[mid]).n_layers > 1;
    if (!walked && idx == kNoHit) {  // miss: background at depth 0, else 0 (pathtracer.cpp:21-26)
        if (depth == 0) {
            rad.x += thr.x * jb.bg[0];
            rad.y += thr.y * jb.bg[1];
            rad.z += thr.z * jb.bg[2];
        }
        if (GUIDED && a.train) finish_records(a, A.grec[i], rad, A.key[i]);
        finish_path<MULTI>(a, jb, jid, pix, a.per_path ? A.local[i] : 0ull, rad, done);
        return;
    }
    const spt_material& m = lds_mats ? smats[mid] : a.sc.mats[mid];
    const V3 o{o4.x, o4.y, o4.z}, d{d4.x, d4.y, d4.z};
    V3 pos{}, nrm{}, wo{};
    Frame fr{};
    if (!walked) path_vertex(a, o, d, hv, pos, nrm, fr, wo);
    const uint64_t key = A.key[i];
    Draws r = make_draws(jb, key, __float_as_uint(thr.w));
    V3 bsdf, refl, wi;
    float pdf;
    const uint32_t gmode = GUIDED ? guide_mode(a, mid) : 0u;
    const bool prod = GUIDED && (a.gflags & SPT_GUIDE_PRODUCT);
    const bool guided = gmode != 0u;
    bool via = true;  // the sampled direction came from a guided step
    float pmarg = 0.0f;  // PRODUCT: density of wi, the training weight's 1/p
    if (gmode == kGuideCoated) {
        // with PRODUCT: the learned incident radiance times the coated
        // lobe in exit space
        using namespace guide;
        Lobe lobes[kLobes];
        mixture_params(HalfRow{a.gout + (size_t)i * kOut}, lobes);
        V3 mb;
        float kb;
        bsdf_lobe(m.layers[1], wo, m.layers[0].ior, mb, kb);
        const V3 mbw = to_world(fr, mb);
        if (prod) mixture_product(lobes, mbw, kb);
        layered_eval_guided(m, wo, fr, lobes, a.bsdf_frac, bsdf, refl, pdf, wi, r, via);
        if (prod && a.train && via && wi.y > 0.0f) {  // exit density, the lobe standing in for the walk
            const V3 e = to_world(fr, wi);
            Lobe bl;
            bl.mu = mbw;
            bl.kappa = kb;
            pmarg = a.bsdf_frac * expf(log_vmf(bl, e)) + (1.0f - a.bsdf_frac) * mixture_pdf(lobes, e);
        }
    } else if (guided) {
        // one-sample mixture of the layer's sampler and the learned
        // incident radiance times a vMF stand-in of the layer's lobe
        using namespace guide;
        const spt_layer& l = m.layers[0];
        Lobe lobes[kLobes];
        mixture_params(HalfRow{a.gout + (size_t)i * kOut}, lobes);
        if (prod) {
            V3 mb;
            float kb;
            bsdf_lobe(l, wo, 1.0f, mb, kb);
            mixture_product(lobes, to_world(fr, mb), kb);
        }
        if (r.next() < a.bsdf_frac) {
            wi = layer_sample(l, wo, r).wi;
        } else {
            const float u0 = r.next(), u1 = r.next(), u2 = r.next();
            wi = to_local(fr, mixture_sample(lobes, u0, u1, u2));
        }
        pdf = a.bsdf_frac * layer_density(l, wo, wi) +
              (1.0f - a.bsdf_frac) * mixture_pdf(lobes, to_world(fr, wi));
        pmarg = pdf;
        if (wi.y > 0.0f && pdf > 0.0f) {
            bsdf = layer_f(l, wo, wi);
            refl = layer_reflectance(l, wo, wi);
        } else {
            bsdf = V3{0.0f, 0.0f, 0.0f};
            refl = V3{0.0f, 0.0f, 0.0f};
            pdf = 1.0f;
        }
    } else if (WALKS) {
        layered_eval(m, wo, bsdf, refl, pdf, wi, r);  // pathtracer.cpp:36
    } else if (!walked) {  // one layer: the walk is one step
        Walk k;
        k.start(m, wo);
        k.step(m, r);
        wi = k.wi;
        k.result(bsdf, refl, pdf);
    }
    V3 wwi, no;
    float kk;
    if (walked) {
        const float2 cp = w.walk[i];
        wi.y = cp.x;
        pdf = cp.y;
        bsdf = V3{hv.x, hv.y, hv.z};
        kk = hv.w;
        wwi = d;
        no = o;
    } else {
        wwi = to_world(fr, wi);              // pathtracer.cpp:37
        no = pos + wwi * 1e-3f;              // pathtracer.cpp:38
        kk = gmax(gmax(refl.x, refl.y), refl.z);  // pathtracer.cpp:41
    }
    rad.x += thr.x * m.emission[0];
    rad.y += thr.y * m.emission[1];
    rad.z += thr.z * m.emission[2];
    // training weight before roulette: L_i / p (PRODUCT, radiance target)
    // or f cos / p L_i (the product target)
    const float rec_w = prod ? ((pmarg > 0.0f) ? 1.0f / pmarg : 0.0f) : lum(bsdf) * wi.y / pdf;
    bool alive = true;
    if ((jb.rr_depth >= 0) && ((int32_t)depth >= jb.rr_depth)) {  // pathtracer.cpp:43-49
        if ((r.next() < kk) && (depth < 1000u))
            bsdf = bsdf / kk;
        else
            alive = false;
    }
    if (r.overflow) atomicAdd(&w.cnt[2], 1u);
    const uint32_t nd = depth + 1;
    if (alive && (jb.max_depth >= 0) && ((int32_t)nd >= jb.max_depth)) alive = false;  // pathtracer.cpp:18
    if (!alive) {
        if (GUIDED && a.train) finish_records(a, A.grec[i], rad, A.key[i]);
        finish_path<MULTI>(a, jb, jid, pix, a.per_path ? A.local[i] : 0ull, rad, done);
        return;
    }
    // pathtracer.cpp:52-54, forwards: throughput *= f * cos / pdf
    const V3 wgt = (bsdf * wi.y) / pdf;
    uint4 gr = (GUIDED && a.train) ? A.grec[i] : make_uint4(0u, 0u, 0u, 0u);
    const bool cand = GUIDED && a.train && guided && via && gr.w < 3u && wi.y > 0.0f && bsdf.x + bsdf.y + bsdf.z > 0.0f;
    const bool take = cand && (a.rec_stride <= 1u ||
                               mix64(key + (uint64_t)(depth + 1) * 0x9E3779B97F4A7C15ull) % a.rec_stride == 0u);
    uint32_t rs = 0;
    if (GUIDED && a.train) {
        // one 64-bit atomic per wave adds the wave's candidates (high
        // word) and records (low word); the record slots of the wave are
        // consecutive from the old low word
        const uint64_t cb = __ballot(cand), tb = __ballot(take);
        const int leader = __ffsll((unsigned long long)cb) - 1;
        const unsigned long long inc = ((unsigned long long)__popcll(cb) << 32) | (unsigned long long)__popcll(tb);
        unsigned long long* rc = reinterpret_cast<unsigned long long*>(a.rec_count);
        if (tb) {
            unsigned long long old = 0;
            if (__lane_id() == (unsigned)leader) old = atomicAdd(rc, inc);
            rs = __shfl((uint32_t)old, leader) + (uint32_t)__popcll(tb & __lanemask_lt());
        } else if (cb && __lane_id() == (unsigned)leader) {
            atomicAdd(rc, inc);
        }
    }
    if (take) {
        if (a.rec_ring) rs %= a.rec_cap;
        if (rs < a.rec_cap) {
            float* rec = a.records + (size_t)rs * guide::kRecord;
            rec[20] = __uint_as_float(rec_tag(key, gr.w));
            const V3 wdir = to_world(fr, wi);
            const float vals[20] = {pos.x, pos.y, pos.z, nrm.x, nrm.y, nrm.z, -d.x, -d.y, -d.z, wdir.x, wdir.y,
                                    wdir.z, 0.0f, rec_w, rad.x, rad.y, rad.z,
                                    thr.x * wgt.x, thr.y * wgt.y, thr.z * wgt.z};
            for (int k = 0; k < 20; ++k) rec[k] = vals[k];
            if (gr.w == 0) gr.x = rs;
            else if (gr.w == 1) gr.y = rs;
            else gr.z = rs;
            ++gr.w;
        }
    }
    Survivor sv;
    sv.o = make_float4(no.x, no.y, no.z, __uint_as_float(pix));
    sv.d = make_float4(wwi.x, wwi.y, wwi.z, __uint_as_float(jid));
    sv.thr = make_float4(thr.x * wgt.x, thr.y * wgt.y, thr.z * wgt.z, __uint_as_float(r.k));
    sv.rad = make_float4(rad.x, rad.y, rad.z, __uint_as_float(nd));
    sv.key = key;
    if (a.per_path) sv.local = A.local[i];
    if (GUIDED && a.train) sv.gr = gr;
    go_on(sv);
}

// The walks through materials of several layers (pathtracer.cpp:28-38) of
// the live paths of A, before k_shade, which only weighs and appends these
// paths: new origin and direction, BSDF value, largest reflectance component,
// cosine and density replace ray and hit in the path's slot.
//
// Walks of coated metal take 4 steps on average, the longest of 64 lanes 23;
// walked inside k_shade they left 16 lanes active, unless the paths were
// sorted by material first, which then cost the sort and the gathers of every
// array in that order (3 TB/s of partly used lines). Here a wave looks its
// share of the queue through for such paths (one word each) and takes new
// ones once half of its lanes have finished; each round it steps the lanes at
// a dielectric or the others, whichever are more, so that lanes line up.
// 123M-path mesh image (28M live paths a launch): sort, walks and shading 2.5
// -> 0.88 (walks) + 1.01 ms (k_shade), the rays of the unsorted queue 5% faster
// as well. Bound by VALU issue at 20 lanes.
template <bool MULTI>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_walk(RenderArgs a, PathBuf A, Work w,
                                                                                           const uint32_t* __restrict__ cntA) {
    __shared__ spt_material smats[kLdsMats];
    __shared__ uint32_t lists[kBlock / 64][128];  // slots found and not yet taken
    __shared__ float park[6][kBlock];  // position and normal of a lane's vertex
    if (*cntA == 0) return;
    const bool lds_mats = a.sc.n_mats <= kLdsMats;
    if (lds_mats) {
        const uint32_t words = a.sc.n_mats * (uint32_t)(sizeof(spt_material) / 4);
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.sc.mats);
        uint32_t* dst = reinterpret_cast<uint32_t*>(smats);
        for (uint32_t k = threadIdx.x; k < words; k += kBlock) dst[k] = src[k];
    }
    __syncthreads();
    const uint64_t lt = __lanemask_lt();
    const uint32_t n = *cntA, waves = gridDim.x * (kBlock / 64);
    uint32_t* list = lists[threadIdx.x / 64];
    // 64 slots at a time, dealt to the waves in turn: layered paths lie together
    uint32_t next = (blockIdx.x * (kBlock / 64) + threadIdx.x / 64) * 64, found = 0;
    uint32_t slot = kDone, mid = 0;
    bool walking = false;
    Walk wk{};
    Draws r{};
    while (true) {
        const uint64_t idle = __ballot(!walking);
        if (idle == ~0ull || ((next < n || found) && __popcll(idle) >= kWalkRefill)) {
            if (!walking && slot != kDone) {
                V3 bsdf, refl;
                float pdf;
                wk.result(bsdf, refl, pdf);
                const V3 pos{park[0][threadIdx.x], park[1][threadIdx.x], park[2][threadIdx.x]};
                const Frame fr = frame_from_up(V3{park[3][threadIdx.x], park[4][threadIdx.x], park[5][threadIdx.x]});
                const V3 wwi = to_world(fr, wk.wi);  // pathtracer.cpp:37
                const V3 no = pos + wwi * 1e-3f;     // pathtracer.cpp:38
                float* p = reinterpret_cast<float*>(A.o + slot);
                p[0] = no.x;
                p[1] = no.y;
                p[2] = no.z;
                p = reinterpret_cast<float*>(A.d + slot);
                p[0] = wwi.x;
                p[1] = wwi.y;
                p[2] = wwi.z;
                A.thr[slot].w = __uint_as_float(r.k);
                w.hit[slot] = make_float4(bsdf.x, bsdf.y, bsdf.z, gmax(gmax(refl.x, refl.y), refl.z));
                w.walk[slot] = make_float2(wk.wi.y, pdf);
                if (r.overflow) atomicAdd(&w.cnt[2], 1u);
                slot = kDone;
            }
            while (found < (uint32_t)__popcll(idle) && next < n) {
                const uint32_t e = next + __lane_id();
                const uint32_t k = e < n ? w.skey[e] : a.sc.n_mats;
                const bool layered = k < a.sc.n_mats && (lds_mats ? smats[k] : a.sc.mats[k]).n_layers > 1;
                const uint64_t lm = __ballot(layered);
                if (layered) list[found + (uint32_t)__popcll(lm & lt)] = e;
                found += (uint32_t)__popcll(lm);
                next += 64 * waves;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (!walking) {
                const uint32_t q = (uint32_t)__popcll(idle & lt);
                if (q < found) {
                    slot = list[found - 1 - q];
                    mid = w.skey[slot];
                    const float4 hv = w.hit[slot], o4 = A.o[slot], d4 = A.d[slot];
                    const uint32_t k = __float_as_uint(A.thr[slot].w);
                    r = make_draws(job_of<MULTI>(a, __float_as_uint(d4.w)), A.key[slot], k);
                    V3 pos, nrm, wo;
                    Frame fr;
                    path_vertex(a, V3{o4.x, o4.y, o4.z}, V3{d4.x, d4.y, d4.z}, hv, pos, nrm, fr, wo);
                    park[0][threadIdx.x] = pos.x;
                    park[1][threadIdx.x] = pos.y;
                    park[2][threadIdx.x] = pos.z;
                    park[3][threadIdx.x] = nrm.x;
                    park[4][threadIdx.x] = nrm.y;
                    park[5][threadIdx.x] = nrm.z;
                    const spt_material& mm = lds_mats ? smats[mid] : a.sc.mats[mid];
                    wk.start(mm, wo);
                    walking = wk.running(mm);
                }
            }
            found -= min(found, (uint32_t)__popcll(idle));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (!__ballot(slot != kDone)) break;
        }
        const spt_material& m = lds_mats ? smats[mid] : a.sc.mats[mid];
        const bool coat = walking && m.layers[wk.id].type == SPT_BSDF_SMOOTH_DIELECTRIC;
        const bool coats = 2 * __popcll(__ballot(coat)) >= __popcll(__ballot(walking));
        if (walking && coat == coats) {
            wk.step(m, r);
            walking = wk.running(m);
        }
    }
}

// Shading of one bounce (integrators/pathtracer.cpp:21-54) for every live
// path of A, in the queue's order; survivors are appended to B, with one atomic
// on B's count per block and turn: one per wave (the compiler's aggregation)
// made that address the limit, about 10 ns per atomic that all XCDs share (61M
// paths: 950k atomics in a 10.2-ms launch).
// GUIDED instantiates the guide's sampling and record capture and walks in
// place (a bounce's launches are shorter there, and a launch more costs the
// length of its longest walk, 60 us); the plain instantiation carries none of
// their registers and leaves layered materials to k_walk. Bound by the queue's
// traffic, about 200 B a path (28M paths 1.01 ms); five or six waves per SIMD
// instead of four do not help.
// Threads of a shading block, which takes its survivors' slots with one
// atomic: 28M paths shaded in 1.45 ms with 256, 1.01 with 512, 1.09 with 1024.
// Guided shading is bound by its own instructions and its waves wait for each
// other less in smaller blocks (400x300, 36-sample pass 10.6 ms with 256, 11.0
// with 512).
template <bool GUIDED>
constexpr uint32_t kShadeBlock = GUIDED ? 256 : 512;

// Guided shading keeps the survivors of a block in LDS across the barriers:
// held in registers they spill 72 of them.
template <bool GUIDED>
struct Park {
    float4 o[kShadeBlock<true>], d[kShadeBlock<true>], thr[kShadeBlock<true>], rad[kShadeBlock<true>];
    uint4 gr[kShadeBlock<true>];
    uint64_t key[kShadeBlock<true>], local[kShadeBlock<true>];
    __device__ __forceinline__ void put(const RenderArgs& a, const Survivor& sv) {
        const uint32_t i = threadIdx.x;
        o[i] = sv.o;
        d[i] = sv.d;
        thr[i] = sv.thr;
        rad[i] = sv.rad;
        key[i] = sv.key;
        if (a.per_path) local[i] = sv.local;
        if (a.train) gr[i] = sv.gr;
    }
    __device__ __forceinline__ void get(const RenderArgs& a, Survivor& sv) {
        const uint32_t i = threadIdx.x;
        sv.o = o[i];
        sv.d = d[i];
        sv.thr = thr[i];
        sv.rad = rad[i];
        sv.key = key[i];
        if (a.per_path) sv.local = local[i];
        if (a.train) sv.gr = gr[i];
    }
};
template <>
struct Park<false> {
    __device__ void put(const RenderArgs&, const Survivor&) {}
    __device__ void get(const RenderArgs&, Survivor&) {}
};

template <bool MULTI, bool GUIDED>
__global__ __launch_bounds__(kShadeBlock<GUIDED>) __attribute__((amdgpu_waves_per_eu(4))) void k_shade(RenderArgs a, PathBuf A, PathBuf B, Work w,
                                                  const uint32_t* __restrict__ cntA, uint32_t* __restrict__ cntB) {
    constexpr uint32_t kThreads = kShadeBlock<GUIDED>;
    // the material table in LDS when it is small (each lane reads its
    // layered material field by field)
    __shared__ spt_material smats[kLdsMats];
    const bool lds_mats = a.sc.n_mats <= kLdsMats;
    if (lds_mats) {
        const uint32_t words = a.sc.n_mats * (uint32_t)(sizeof(spt_material) / 4);
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.sc.mats);
        uint32_t* dst = reinterpret_cast<uint32_t*>(smats);
        for (uint32_t k = threadIdx.x; k < words; k += kThreads) dst[k] = src[k];
    }
    __shared__ uint32_t done[MULTI ? kDoneJobs : 1];  // finished paths of the block per job
    if (MULTI)
        for (uint32_t k = threadIdx.x; k < kDoneJobs; k += kThreads) done[k] = 0;
    __syncthreads();
    __shared__ Park<GUIDED> park;
    // survivors of the block's waves (two sets, used in turn) and their first slot
    __shared__ uint32_t survivors[2][kThreads / 64 + 1];
    const uint32_t n = *cntA;
    const uint32_t gthreads = gridDim.x * kThreads;
    const uint32_t wave = threadIdx.x / 64;
    uint32_t turn = 0;
    for (uint32_t j0 = blockIdx.x * kThreads; j0 < n; j0 += gthreads, turn ^= 1u) {
        const uint32_t j = j0 + threadIdx.x;
        Survivor sv;
        bool alive = false;
        if (j < n)
            shade_path<MULTI, GUIDED, GUIDED>(a, A, w, smats, lds_mats, j, done, [&](const Survivor& next) {
                if (GUIDED)
                    park.put(a, next);
                else
                    sv = next;
                alive = true;
            });
        const uint64_t am = __ballot(alive);
        if (__lane_id() == 0) survivors[turn][wave] = (uint32_t)__popcll(am);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t sum = 0;
            for (uint32_t v = 0; v < kThreads / 64; ++v) sum += survivors[turn][v];
            survivors[turn][kThreads / 64] = sum ? atomicAdd(cntB, sum) : 0u;
        }
        __syncthreads();
        if (!alive) continue;
        uint32_t slot = survivors[turn][kThreads / 64] + (uint32_t)__popcll(am & __lanemask_lt());
        for (uint32_t v = 0; v < wave; ++v) slot += survivors[turn][v];
        if (GUIDED) park.get(a, sv);
        store_survivor<GUIDED>(a, B, sv, slot);
    }
    if (MULTI && a.n_jobs <= kDoneJobs) {
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < a.n_jobs; k += kThreads)
            if (done[k]) count_done(a, k, done[k]);
    }
}

// Every path of buffer A (count *cntA) run to its end in one launch: a wave
// owns a share of the paths, up to 64 at a time in its lanes, and
// alternates between tracing their rays with its 16 quads and shading them in
// place, at its own pace. For the last paths of a call, and all paths of a
// small one, whose bounces would each take seven launches and wait for the
// longest ray (up to 100 us) and the longest layered walk (500 steps, 110 us)
// of any path: here a path waits for those of its own wave. Bound by the
// latency of those chains; the path state and hits stay in the queue's arrays,
// read back from the caches. 128 VGPRs and 36 KB of LDS: four blocks a CU.
// 97x61 box image, 1 sample: 590 -> 150 us; 800x600 mesh image, 4 samples,
// where it takes the bounces from the seventh on: 6.1 -> 4.4 ms.
template <bool MULTI, bool SMALL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_finish(
    RenderArgs a, PathBuf A, Work w, const uint32_t* __restrict__ cntA, uint32_t* __restrict__ spill,
    uint32_t* __restrict__ flags) {
    __shared__ QuadLds lds;
    __shared__ spt_material smats[kLdsMats];
    __shared__ uint32_t slots[kBlock / 64][64];
    __shared__ uint32_t done[MULTI ? kDoneJobs : 1];
    const bool lds_mats = a.sc.n_mats <= kLdsMats;
    if (lds_mats) {
        const uint32_t words = a.sc.n_mats * (uint32_t)(sizeof(spt_material) / 4);
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.sc.mats);
        uint32_t* dst = reinterpret_cast<uint32_t*>(smats);
        for (uint32_t k = threadIdx.x; k < words; k += kBlock) dst[k] = src[k];
    }
    if (MULTI)
        for (uint32_t k = threadIdx.x; k < kDoneJobs; k += kBlock) done[k] = 0;
    __syncthreads();
    const uint32_t n = *cntA;
    const uint32_t waves = gridDim.x * (kBlock / 64);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
    // this wave's paths, in chunks dealt to the waves in turn: long ones lie together
    const uint32_t chunk = min(16u, (n + waves - 1) / waves);
    const uint32_t end = n ? (n + waves * chunk - 1) / (waves * chunk) * chunk : 0u;
    uint32_t next = 0;
    uint32_t* mine = slots[threadIdx.x >> 6];
    const uint64_t lt = __lanemask_lt();
    bool overflow = false;
    uint32_t slot = kDone, segments = 0, longest = 0;
    uint32_t rays = 0;
    while (true) {
        const uint64_t need = ballot(slot == kDone);
        if (slot == kDone) {
            const uint32_t k = next + (uint32_t)lanes(need & lt);
            const uint32_t at = k < end ? ((k / chunk) * waves + wave) * chunk + k % chunk : n;
            if (at < n) {
                slot = at;
                segments = 0;
            }
        }
        next = min(end, next + (uint32_t)lanes(need));
        const uint64_t live = ballot(slot != kDone);
        if (!live) {
            if (next < end) continue;
            break;
        }
        const uint32_t m = (uint32_t)lanes(live);
        rays += m;
        if (slot != kDone) mine[lanes(live & lt)] = slot;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        trace_shares<false, SMALL>(
            a.sc, m, RayShares(m), 0u, w.rays, lds, spill + (size_t)blockIdx.x * quad_spill_words(a.sc.stack_cap4), overflow,
            a.refill,
            [&](uint32_t i, V3& o, V3& d, Root& root) {
                const uint32_t s = mine[i];
                const float4 o4 = A.o[s], d4 = A.d[s];
                o = V3{o4.x, o4.y, o4.z};
                d = V3{d4.x, d4.y, d4.z};
                if (MULTI) {
                    const Job& jb = a.jobs[__float_as_uint(d4.w)];
                    root = Root{V3{jb.rmin[0], jb.rmin[1], jb.rmin[2]}, V3{jb.rmax[0], jb.rmax[1], jb.rmax[2]}, jb.node0};
                }
            },
            [&](uint32_t i, const Hit& h, V3, V3, uint32_t, uint32_t) {
                const uint32_t s = mine[i];
                w.hit[s] = make_float4(h.t, __uint_as_float(h.idx), h.u, h.v);
                w.skey[s] = h.mat;
            });
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        if (slot != kDone) {
            bool alive = false;
            longest = max(longest, ++segments);
            shade_path<MULTI, false, true>(a, A, w, smats, lds_mats, slot, done, [&](const Survivor& sv) {
                store_survivor<false>(a, A, sv, slot);
                alive = true;
            });
            if (!alive) slot = kDone;
        }
    }
    if (overflow) atomicOr(flags, 1u);
    for (int k = 32; k > 0; k >>= 1) longest = max(longest, (uint32_t)__shfl_xor(longest, k));
    if (__lane_id() == 0 && rays) {
        uint32_t* c = w.rays + (blockIdx.x % kRayCounters) * kRayCounterStride;
        atomicAdd(reinterpret_cast<unsigned long long*>(c + kFinishRays), (unsigned long long)rays);
        atomicMax(c + kFinishBounces, longest);
    }
    if (MULTI && a.n_jobs <= kDoneJobs) {
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < a.n_jobs; k += kBlock)
            if (done[k]) count_done(a, k, done[k]);
    }
}

uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

size_t guide_paths_lds_bytes() {
    return sizeof(guide::FwdWeights) + sizeof(guide::WaveStage) * (kBlock / 64);
}

}  // namespace

// Validates one render's parameters and fills its job (everything but the
// tree root). total = paths of the call.
spt_status make_job(spt_ctx* ctx, const spt_camera* cam, const spt_render_params* prm, float* d_rgb32, double* d_rgb64,
                    float* d_path_rgb, Job& jb, uint64_t& total) {
    jb = Job{};
    jb.cam = make_camera(*cam);
    jb.sampler = prm->pixel_sampler;
    if (jb.sampler > SPT_PIXEL_UNIFORM) return set_error(ctx, SPT_ERR_INVALID, "unknown pixel sampler");
    if (prm->spp == 0) return set_error(ctx, SPT_ERR_INVALID, "spp must be > 0");
    if (jb.sampler == SPT_PIXEL_UNIFORM) {
        jb.n_sub = 1;
        jb.spp = prm->spp;
        jb.w_sub = 1.0f;
    } else {  // n = ceil(sqrt(spp)), spp := n^2 (jittered_pixel_sampler.cpp:6-8)
        jb.n_sub = (uint32_t)std::ceil(std::sqrt((double)prm->spp));
        jb.spp = jb.n_sub * jb.n_sub;
        jb.w_sub = 1.0f / jb.n_sub;
    }
    jb.spp_begin = prm->spp_begin;
    jb.spp_count = prm->spp_count ? prm->spp_count : jb.spp - std::min(prm->spp_begin, jb.spp);
    if ((uint64_t)jb.spp_begin + jb.spp_count > jb.spp || jb.spp_count == 0)
        return set_error(ctx, SPT_ERR_INVALID, "sample range outside [0, spp)");
    jb.vt = prm->viewport[0];
    jb.vl = prm->viewport[1];
    jb.vw = prm->viewport[2];
    jb.vh = prm->viewport[3];
    if (jb.vw == 0) {
        jb.vt = jb.vl = 0;
        jb.vw = cam->width;
        jb.vh = cam->height;
    }
    if ((uint64_t)jb.vl + jb.vw > cam->width || (uint64_t)jb.vt + jb.vh > cam->height || jb.vh == 0)
        return set_error(ctx, SPT_ERR_INVALID, "viewport outside the image");
    jb.max_depth = prm->max_depth;
    jb.rr_depth = prm->rr_depth;
    if (jb.max_depth < 0 && jb.rr_depth < 0)
        return set_error(ctx, SPT_ERR_INVALID, "need max_depth >= 0 or rr_depth >= 0 (paths must terminate)");
    jb.seed = prm->seed;
    for (int i = 0; i < 3; ++i) jb.bg[i] = prm->background[i];
    jb.film32 = (prm->flags & SPT_RENDER_FILM32) ? d_rgb32 : nullptr;
    jb.film64 = (prm->flags & SPT_RENDER_FILM64) ? d_rgb64 : nullptr;
    jb.path_rgb = (prm->flags & SPT_RENDER_PER_PATH) ? d_path_rgb : nullptr;
    if ((prm->flags & SPT_RENDER_FILM32) && !d_rgb32) return set_error(ctx, SPT_ERR_INVALID, "FILM32 without buffer");
    if ((prm->flags & SPT_RENDER_FILM64) && !d_rgb64) return set_error(ctx, SPT_ERR_INVALID, "FILM64 without buffer");
    if ((prm->flags & SPT_RENDER_PER_PATH) && !d_path_rgb)
        return set_error(ctx, SPT_ERR_INVALID, "PER_PATH without buffer");
    if (prm->rng == SPT_RNG_STREAM) {
        if (!prm->d_stream || prm->stream_stride == 0)
            return set_error(ctx, SPT_ERR_INVALID, "replay stream missing");
        jb.stream = prm->d_stream;
        jb.stride = prm->stream_stride;
    } else if (prm->rng != SPT_RNG_COUNTER) {
        return set_error(ctx, SPT_ERR_INVALID, "unknown rng mode");
    }
    total = (uint64_t)jb.vw * jb.vh * jb.spp_count;
    jb.n_paths = total;
    return SPT_OK;
}

namespace {

// The dynamic LDS size of the guide inference kernel, set once per process
// (thread-safe: concurrent wavefronts start their calls together).
spt_status allow_guide_paths_lds(spt_ctx* ctx) {
    static std::once_flag once;
    static hipError_t e = hipSuccess;
    std::call_once(once, []() {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_guide_paths),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)guide_paths_lds_bytes());
    });
    return check_hip(ctx, e, "guide LDS size");
}

// Runs `total` paths through the wavefront: the queue is filled to its
// capacity, then every bounce refills it from the paths not yet generated,
// until every path is generated and none is live.
template <bool MULTI>
spt_status run_paths(spt_ctx* ctx, RenderArgs& a, uint64_t total, const spt_tuning& tn, spt_render_stats& stats) {
    uint64_t cap = std::min<uint64_t>(total, tn.path_capacity);
    auto state_bytes = [](uint64_t c) {
        return (size_t)c * (2 * kBufBytes + kWorkBytes + 4 * 8) + 8192;
    };
    if (state_bytes(cap) > ctx->paths_bytes) {
        (void)hipStreamSynchronize(ctx->stream);
        if (ctx->d_paths) (void)hipFree(ctx->d_paths);
        ctx->d_paths = nullptr;
        ctx->paths_bytes = 0;
        // a device without room for the queue gets a smaller one (slower,
        // same results), down to 2^20 paths
        while (true) {
            const hipError_t e = hipMalloc(&ctx->d_paths, state_bytes(cap));
            if (e == hipSuccess) break;
            (void)hipGetLastError();  // the failed allocation is not the next launch's error
            ctx->d_paths = nullptr;
            if (e != hipErrorOutOfMemory || cap <= (1u << 20)) return check_hip(ctx, e, "path state");
            cap = std::max<uint64_t>(cap / 2, 1u << 20);
        }
        ctx->paths_bytes = state_bytes(cap);
    }
    char* base = reinterpret_cast<char*>(ctx->d_paths);
    auto take = [&](size_t sz) {
        char* r = base;
        base += (sz + 255) & ~size_t(255);
        return r;
    };
    PathBuf buf[2];
    for (PathBuf& b : buf) {
        b.o = (float4*)take(cap * 16);
        b.d = (float4*)take(cap * 16);
        b.thr = (float4*)take(cap * 16);
        b.rad = (float4*)take(cap * 16);
        b.key = (uint64_t*)take(cap * 8);
        b.local = (uint64_t*)take(cap * 8);
        b.grec = (uint4*)take(cap * 16);
    }
    Work w;
    w.hit = (float4*)take(cap * 16);
    w.skey = (uint32_t*)take(cap * 4);
    w.walk = (float2*)take(cap * 8);
    w.cnt = (uint32_t*)take((64 + kRayCounterWords) * 4);
    w.rays = w.cnt + 64;
    if ((size_t)(base - reinterpret_cast<char*>(ctx->d_paths)) > ctx->paths_bytes)
        return set_error(ctx, SPT_ERR_NOMEM, "path state layout exceeds its allocation");
    a.rec_count = a.rec_shared ? a.rec_shared : w.cnt + 16;
    a.refill = std::min<uint32_t>(kMaxRefillLanes, std::max<uint32_t>(1, tn.refill_lanes));
    if (a.guided) {
        const size_t need = (size_t)cap * guide::kOut * sizeof(unsigned short);
        if (need > ctx->guide.gout_cap) {
            (void)hipStreamSynchronize(ctx->stream);
            if (ctx->guide.d_gout) (void)hipFree(ctx->guide.d_gout);
            ctx->guide.d_gout = nullptr;
            ctx->guide.gout_cap = 0;
            spt_status s = check_hip(ctx, hipMalloc(&ctx->guide.d_gout, need), "guide outputs");
            if (s != SPT_OK) return s;
            ctx->guide.gout_cap = need;
        }
        a.gout = ctx->guide.d_gout;
    }

    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(&k_extend<true, MULTI, false>),
                                                     kBlock, 0) != hipSuccess ||
        per_cu <= 0)
        per_cu = 4;
    if (tn.extend_blocks_per_cu)
        per_cu = std::min<int>(per_cu, (int)tn.extend_blocks_per_cu);
    else if (tn.wavefronts > 1)  // concurrent wavefronts share the CUs: three with 3, 4, 5, 7 blocks each ran
                                 // the 1024-spp mesh image at 911, 948, 897, 914 Mpaths/s
        per_cu = std::min<int>(per_cu, tn.wavefronts == 2 ? 5 : 4);
    const uint32_t ext_grid = std::min<uint32_t>(blocks_for(cap), (uint32_t)(per_cu * ctx->num_cus));
    // tn.shade_blocks_per_cu counts blocks of kBlock threads
    const uint32_t shade_block = a.guided ? kShadeBlock<true> : kShadeBlock<false>;
    const uint32_t shade_grid = std::max<uint32_t>(
        1, std::min<uint32_t>(blocks_for(cap), (uint32_t)ctx->num_cus * tn.shade_blocks_per_cu) / (shade_block / kBlock));
    const uint32_t walk_grid = std::min<uint32_t>(blocks_for(cap), (uint32_t)ctx->num_cus * 4);
    const uint32_t refill_grid = std::min<uint32_t>(blocks_for(cap), (uint32_t)ctx->num_cus * 8);
    hipStream_t st = ctx->stream;
    const bool timed = (a.flags & SPT_RENDER_TIME_KERNELS) != 0;
    const bool fetch_stats = (a.flags & SPT_RENDER_FETCH_STATS) != 0;
    const uint64_t finish_at = (a.guided || timed || fetch_stats) ? 0 : kFinishPaths;
    const uint32_t finish_grid = std::min<uint32_t>(blocks_for(std::min<uint64_t>(cap, finish_at) * 64), (uint32_t)ctx->num_cus * 4);
    spt_status s = ensure_spill(
        ctx, std::max<size_t>(1, (size_t)std::max(ext_grid, finish_grid) * quad_spill_words(a.sc.stack_cap4)));
    if (s != SPT_OK) return s;
    s = check_hip(ctx, hipMemsetAsync(w.cnt, 0, (64 + kRayCounterWords) * 4, st), "counters");
    if (s != SPT_OK) return s;
    if (a.train && !a.rec_shared) {  // records continue after those collected since the last training step
        s = check_hip(ctx,
                      hipMemsetD32Async((hipDeviceptr_t)(w.cnt + 16), a.rec_ring ? 0 : (int)ctx->guide.collected, 1, st),
                      "record counter");
        if (s != SPT_OK) return s;
    }
    if (a.guided) {
        s = allow_guide_paths_lds(ctx);
        if (s != SPT_OK) return s;
    }
    if (fetch_stats) {
        s = check_hip(ctx, hipMemsetAsync(ctx->d_flags + 4, 0, 16, st), "fetch counters");
        if (s != SPT_OK) return s;
    }
    std::vector<hipEvent_t> gev;  // guide inference launches (TIME_KERNELS)
    bool generated = total <= cap;  // no bounce plans new paths any more, as far as the host has seen
    // One bounce over buffer (b & 1) into the other buffer.
    auto bounce = [&](uint32_t b) -> spt_status {
        PathBuf& A = buf[b & 1];
        PathBuf& B = buf[(b + 1) & 1];
        uint32_t* cntA = w.cnt + (b & 1);
        uint32_t* cntB = w.cnt + ((b + 1) & 1);
        if (timed) {
            while (ctx->tev.size() < 2 * (stats.extend_launches + 1)) {
                hipEvent_t e;
                spt_status es = check_hip(ctx, hipEventCreate(&e), "event");
                if (es != SPT_OK) return es;
                ctx->tev.push_back(e);
            }
            (void)hipEventRecord(ctx->tev[2 * stats.extend_launches], st);
        }
        hipLaunchKernelGGL((fetch_stats       ? k_extend<true, MULTI, false>
                            : a.sc.small_tree ? k_extend<false, MULTI, true>
                                              : k_extend<false, MULTI, false>),
                           dim3(ext_grid), dim3(kBlock), 0, st, a, A, w, cntA, ctx->d_spill, ctx->d_flags);
        if (timed) {
            (void)hipEventRecord(ctx->tev[2 * stats.extend_launches + 1], st);
            ++stats.extend_launches;
        }
        if (a.guided) {
            if (timed) {
                hipEvent_t e0, e1;
                if (hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
                    gev.push_back(e0);
                    gev.push_back(e1);
                    (void)hipEventRecord(e0, st);
                }
            }
            hipLaunchKernelGGL(k_guide_paths, dim3((uint32_t)ctx->num_cus * 3), dim3(kBlock), guide_paths_lds_bytes(),
                               st, a, A, w, cntA, a.theta, a.wbf, a.gbox);
            if (timed && !gev.empty()) (void)hipEventRecord(gev.back(), st);
        }
        if (a.walk) hipLaunchKernelGGL((k_walk<MULTI>), dim3(walk_grid), dim3(kBlock), 0, st, a, A, w, cntA);
        hipLaunchKernelGGL((a.guided ? k_shade<MULTI, true> : k_shade<MULTI, false>), dim3(shade_grid), dim3(shade_block), 0, st, a, A, B, w, cntA, cntB);
        // regeneration: the survivors' buffer is topped up with new camera paths
        hipLaunchKernelGGL(k_plan, dim3(1), dim3(64), 0, st, cntA, cntB, w.cnt, w.rays, (uint32_t)cap, total, ctx->d_status,
                           a.job_clock);
        if (!generated) hipLaunchKernelGGL((k_refill<MULTI>), dim3(refill_grid), dim3(kBlock), 0, st, a, B, w);
        return check_hip(ctx, hipGetLastError(), "bounce launch");
    };
    // Graph mode: two bounces (one per buffer parity) captured once and
    // replayed; every kernel reads its live count from device memory, so the
    // same graph serves every bounce. No memset nodes are recorded.
    const bool graph_on = tn.use_graph == 1 && !timed && !fetch_stats;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    auto drop_graph = [&]() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    };
    if (graph_on) {
        s = check_hip(ctx, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "graph capture");
        if (s != SPT_OK) return s;
        spt_status s0 = bounce(0);
        spt_status s1 = bounce(1);
        hipError_t e = hipStreamEndCapture(st, &graph);
        if (s0 != SPT_OK || s1 != SPT_OK) {
            drop_graph();
            return s0 != SPT_OK ? s0 : s1;
        }
        s = check_hip(ctx, e, "graph capture end");
        if (s == SPT_OK) s = check_hip(ctx, hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0), "graph instantiate");
        if (s != SPT_OK) {
            drop_graph();
            return s;
        }
    }
    // The host stays at most `lag` bounces ahead of the device and stops once
    // a plan reports every path generated and none live; the bounces issued
    // after that one find empty queues (a few empty launches each: 30 us).
    // Once few paths are left it stays one bounce ahead, so that it sees the
    // end, or the point for k_finish, sooner.
    const uint32_t lag = std::max<uint32_t>(2, graph_on ? (tn.check_every + 1) & ~1u : tn.check_every);
    if (!MULTI && a.job.max_depth == 0) {  // every path finishes at generation
        for (uint64_t done = 0; done < total && s == SPT_OK; done += cap) {
            const uint32_t n = (uint32_t)std::min<uint64_t>(cap, total - done);
            hipLaunchKernelGGL((k_generate<MULTI>), dim3(blocks_for(n)), dim3(kBlock), 0, st, a, buf[0], w, done, n);
            s = check_hip(ctx, hipGetLastError(), "generate launch");
        }
    } else {
        ctx->h_status[0] = 0;
        hipLaunchKernelGGL(k_plan, dim3(1), dim3(64), 0, st, nullptr, w.cnt, w.cnt, w.rays, (uint32_t)cap, total, ctx->d_status,
                           a.job_clock);
        hipLaunchKernelGGL((k_refill<MULTI>), dim3(refill_grid), dim3(kBlock), 0, st, a, buf[0], w);
        s = check_hip(ctx, hipGetLastError(), "generate launch");
        uint32_t b = 0;
        // in-call training (ring of records): train aligned batches of the
        // records counted one round earlier; skip what is about to be reused
        uint32_t next_train = ctx->guide.train_every, prev_count = 0, trained = 0;
        auto finish = [&]() {  // reads its count on the device: may be queued behind a bounce still running
            hipLaunchKernelGGL((a.sc.small_tree ? k_finish<MULTI, true> : k_finish<MULTI, false>), dim3(finish_grid), dim3(kBlock), 0, st, a, buf[b & 1], w, w.cnt + (b & 1),
                               ctx->d_spill, ctx->d_flags);
            return check_hip(ctx, hipGetLastError(), "finish launch");
        };
        auto few = [&](uint64_t live) { return live <= kNearEnd && !a.rec_ring; };
        bool near_end = generated && few(total);
        const bool at_once = generated && total <= finish_at;
        if (s == SPT_OK && at_once) s = finish();
        while (s == SPT_OK && !at_once) {
            if (graph_on) {
                s = check_hip(ctx, hipGraphLaunch(exec, st), "graph launch");
                b += 2;
            } else {
                s = bounce(b);
                ++b;
            }
            const uint32_t behind = near_end ? (graph_on ? 2u : 1u) : lag;
            if (s != SPT_OK || b <= behind) continue;
            // plan number 1 is the initial one; bounce j's plan is number j + 2
            const uint32_t want = b - behind + 1;
            bool idle = false;
            while (ctx->h_status[0] < want && !idle) {
                const hipError_t q = hipStreamQuery(st);
                if (q == hipSuccess) idle = true;  // drained: the status below is final
                else if (q != hipErrorNotReady) s = check_hip(ctx, q, "bounce");
                if (s != SPT_OK) break;
                __builtin_ia32_pause();
            }
            if (s == SPT_OK && ctx->h_status[2]) {
                generated = true;
                const uint32_t live = ctx->h_status[1];
                if (live == 0) break;
                if (live <= finish_at) {
                    s = finish();
                    break;
                }
                near_end = few(live);
            }
            if (idle && ctx->h_status[0] < want) {
                s = set_error(ctx, SPT_ERR_DEVICE, "bounce status did not advance");
                break;
            }
            if (a.rec_ring && s == SPT_OK && b >= next_train) {
                const uint32_t now = ctx->h_status[3], upto = prev_count, bt = ctx->guide.batch;
                prev_count = now;
                next_train = b + ctx->guide.train_every;
                if (now > a.rec_cap / 2) trained = std::max(trained, (now - a.rec_cap / 2 + bt - 1) / bt * bt);
                while (s == SPT_OK && trained + bt <= upto) {
                    s = guide_train_launch(ctx, ctx->guide.d_records + (size_t)(trained % a.rec_cap) * guide::kRecord, bt,
                                           nullptr, 1u);
                    trained += bt;
                }
            }
        }
    }
    if (s != SPT_OK) {
        (void)stream_wait(ctx, "render abort");
        drop_graph();
        return s;
    }
    uint32_t cnt[64 + kRayCounterWords];  // the work words and the ray counters' lines
    uint32_t flags = 0;
    s = read_small(ctx, cnt, w.cnt, sizeof(cnt), "render", &flags, ctx->d_flags, sizeof(flags));
    drop_graph();
    if (s != SPT_OK) return s;
    stats.stream_overflows = cnt[2];
    if (a.train && !a.rec_shared) {
        GuideState& gs = ctx->guide;
        // a ring of records was trained inside the call; otherwise the
        // records wait for spt_guide_train_collected
        gs.collected = a.rec_ring ? 0 : std::min<uint64_t>(cnt[16], a.rec_cap);
        gs.candidates = cnt[17];
        // next pass: record about one batch worth of candidates
        gs.cand_per_path = total ? (double)cnt[17] / (double)total : 0.0;
    }
    for (size_t i = 0; i + 1 < gev.size(); i += 2) {
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, gev[i], gev[i + 1]) == hipSuccess) stats.guide_ms += ms;
    }
    for (hipEvent_t e : gev) (void)hipEventDestroy(e);
    stats.rays = (uint64_t)cnt[10] | ((uint64_t)cnt[11] << 32);
    if (a.train && !a.rec_shared && total) ctx->guide.rays_per_path = std::max(1.0, (double)stats.rays / (double)total);
    stats.bounces = (uint64_t)cnt[12] | ((uint64_t)cnt[13] << 32);
    uint32_t longest = 0;
    for (uint32_t k = 0; k < kRayCounters; ++k) {
        const uint32_t* c = cnt + 64 + k * kRayCounterStride;
        stats.rays += (uint64_t)c[kFinishRays] | ((uint64_t)c[kFinishRays + 1] << 32);
        longest = std::max(longest, c[kFinishBounces]);
        stats.guide_queries += (uint64_t)c[kGuideQueries] | ((uint64_t)c[kGuideQueries + 1] << 32);
    }
    stats.bounces += longest;
    if (timed) {
        for (uint64_t i = 0; i < stats.extend_launches; ++i) {
            float ms = 0.0f;
            if (hipEventElapsedTime(&ms, ctx->tev[2 * i], ctx->tev[2 * i + 1]) == hipSuccess) stats.extend_ms += ms;
        }
    }
    if (fetch_stats) {
        unsigned long long f[2] = {0, 0};
        s = read_small(ctx, f, ctx->d_flags + 4, 16, "fetch counters");
        if (s != SPT_OK) return s;
        stats.node_fetches = f[0];
        stats.tri_fetches = f[1];
    }
    if (flags & 1u) {
        (void)hipMemset(ctx->d_flags, 0, 4);
        return set_error(ctx, SPT_ERR_OVERFLOW, "traversal stack overflow");
    }
    if (stats.stream_overflows) return set_error(ctx, SPT_ERR_OVERFLOW, "replay stream exhausted");
    return SPT_OK;
}

// Runs `total` paths as tn.wavefronts independent wavefronts at once: each
// on its own stream, with its own queue (the capacity split between them),
// status word, flags and stack spill buffer, taking a contiguous share of
// the call's path numbering. One wavefront's traversal (bound by VALU issue)
// then overlaps another's gathers. Per-path results do not depend on the
// wavefront a path runs in. Calls of fewer than 2^21 paths per wavefront use
// fewer.
template <bool MULTI>
spt_status run_fronts(spt_ctx* ctx, RenderArgs& a, uint64_t total, const spt_tuning& tn, spt_render_stats& stats) {
    spt_tuning t1 = tn;
    uint32_t k = std::max<uint32_t>(1, std::min<uint32_t>(4, tn.wavefronts));
    if (a.rec_ring) k = 1;  // in-call training trains from one wavefront's ring
    while (k > 1 && total / k < (1ull << 21)) --k;
    if (k == 1) {
        t1.wavefronts = 1;
        resolve_front_defaults(ctx->tuning, t1, 1);
        return run_paths<MULTI>(ctx, a, total, t1, stats);
    }
    resolve_front_defaults(ctx->tuning, t1, k);
    while (ctx->fronts.size() < k - 1) {
        spt_ctx* f = nullptr;
        const spt_status cs = spt_create(ctx->device, &f);
        if (cs != SPT_OK) return set_error(ctx, cs, "context of a concurrent wavefront");
        ctx->fronts.push_back(f);
    }
    t1.wavefronts = k;
    t1.path_capacity = std::max<uint32_t>(1u << 20, tn.path_capacity / k);
    std::vector<RenderArgs> args(k, a);
    std::vector<spt_render_stats> st(k, stats);
    std::vector<spt_status> res(k, SPT_OK);
    std::vector<uint64_t> n(k);
    for (uint32_t i = 0; i < k; ++i) {
        const uint64_t lo = total * i / k, hi = total * (i + 1) / k;
        args[i].gen_base = lo;
        n[i] = hi - lo;
    }
    // training records of all wavefronts go to one buffer through one
    // counter pair (records written, candidate vertices) in the calling
    // context's flag words 12-13, starting after the records collected so far
    if (a.train) {
        const uint32_t init[2] = {(uint32_t)ctx->guide.collected, 0u};
        spt_status cs = check_hip(ctx, hipMemcpyAsync(ctx->d_flags + 12, init, sizeof(init), hipMemcpyHostToDevice,
                                                      ctx->stream), "record counter");
        if (cs != SPT_OK) return cs;
        for (RenderArgs& x : args) x.rec_shared = ctx->d_flags + 12;
    }
    if (a.guided) {
        spt_status ls = allow_guide_paths_lds(ctx);
        if (ls != SPT_OK) return ls;
    }
    // the stream of the calling context orders this call after earlier work
    // on it; the other wavefronts start once that work is done
    spt_status s = stream_wait(ctx, "render start");
    if (s != SPT_OK) return s;
    auto run = [&](uint32_t i) {
        if (hipSetDevice(ctx->device) != hipSuccess) {
            res[i] = SPT_ERR_DEVICE;
            return;
        }
        res[i] = run_paths<MULTI>(i ? ctx->fronts[i - 1] : ctx, args[i], n[i], t1, st[i]);
    };
    std::vector<std::thread> th;
    std::vector<uint32_t> inline_fronts;
    for (uint32_t i = 1; i < k; ++i) {
        try {
            th.emplace_back(run, i);
        } catch (...) {  // no thread: that wavefront runs after the others
            inline_fronts.push_back(i);
        }
    }
    run(0);
    for (std::thread& x : th) x.join();
    for (uint32_t i : inline_fronts) run(i);
    for (uint32_t i = 0; i < k; ++i) {
        if (res[i] != SPT_OK) {
            if (i > 0) ctx->err = ctx->fronts[i - 1]->err;
            return res[i];
        }
    }
    stats = st[0];
    for (uint32_t i = 1; i < k; ++i) {
        stats.rays += st[i].rays;
        stats.bounces = std::max(stats.bounces, st[i].bounces);
        stats.stream_overflows += st[i].stream_overflows;
        stats.extend_ms += st[i].extend_ms;
        stats.extend_launches += st[i].extend_launches;
        stats.node_fetches += st[i].node_fetches;
        stats.tri_fetches += st[i].tri_fetches;
        stats.guide_ms += st[i].guide_ms;
        stats.guide_queries += st[i].guide_queries;
    }
    if (a.train) {
        uint32_t rc[2];
        s = read_small(ctx, rc, ctx->d_flags + 12, sizeof(rc), "record counter");
        if (s != SPT_OK) return s;
        GuideState& gs = ctx->guide;
        gs.collected = std::min<uint64_t>(rc[0], a.rec_cap);
        gs.candidates = rc[1];
        gs.cand_per_path = total ? (double)rc[1] / (double)total : 0.0;
        if (total) gs.rays_per_path = std::max(1.0, (double)stats.rays / (double)total);
    }
    return SPT_OK;
}

}  // namespace

spt_status launch_render(spt_ctx* ctx, const spt_camera* cam, const spt_render_params* prm, float* d_rgb32,
                         double* d_rgb64, float* d_path_rgb) {
    auto t0 = std::chrono::steady_clock::now();
    RenderArgs a{};
    a.sc = ctx->scene();
    uint64_t total = 0;
    spt_status s = make_job(ctx, cam, prm, d_rgb32, d_rgb64, d_path_rgb, a.job, total);
    if (s != SPT_OK) return s;
    for (int i = 0; i < 3; ++i) {
        a.job.rmin[i] = ctx->root_box[i];
        a.job.rmax[i] = ctx->root_box[3 + i];
    }
    a.flags = prm->flags;
    a.per_path = a.job.path_rgb ? 1u : 0u;
    a.guided = (prm->flags & SPT_RENDER_GUIDED) ? 1u : 0u;
    a.train = (a.guided && (prm->flags & SPT_RENDER_GUIDE_TRAIN)) ? 1u : 0u;
    if ((prm->flags & SPT_RENDER_GUIDE_TRAIN) && !a.guided)
        return set_error(ctx, SPT_ERR_INVALID, "GUIDE_TRAIN needs GUIDED");
    if (a.guided && !ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "guided rendering needs spt_guide_init");
    a.guidable = ctx->d_guidable;
    a.theta = ctx->guide.d_theta;
    a.wbf = ctx->guide.d_wbf;
    a.gbox = guide_box(ctx);
    a.bsdf_frac = ctx->guide.bsdf_fraction;
    a.gflags = ctx->guide.flags;
    a.records = ctx->guide.d_records;
    a.rec_cap = ctx->guide.records_cap;
    // record about records_cap of this render's candidate vertices, estimated
    // from the candidates per path of the previous training render. With
    // in-call training the ring must not wrap between the count a training
    // round reads and the moment its steps run: the host runs up to
    // check_every bounces ahead of the device, so one round spans
    // train_every + check_every + 1 bounces, and that span writes at most a
    // quarter of the ring (a bounce of a full queue meets about capacity /
    // rays-per-path paths); the host skips batches older than half a ring
    a.rec_ring = (a.train && ctx->guide.train_every) ? 1u : 0u;
    if (ctx->guide.cand_per_path > 0.0 && ctx->guide.records_cap > 0) {
        double want = ctx->guide.cand_per_path * (double)total;
        if (a.rec_ring) {
            const spt_tuning tn = running_tuning(ctx->tuning);
            const double per_bounce = ctx->guide.cand_per_path / ctx->guide.rays_per_path *
                                      (double)std::min<uint64_t>(total, tn.path_capacity);
            want = per_bounce * (double)(ctx->guide.train_every + tn.check_every + 1) * 4.0;
        }
        ctx->guide.rec_stride =
            (uint32_t)std::min<double>(1 << 30, std::max(1.0, std::ceil(want / ctx->guide.records_cap)));
    }
    a.rec_stride = ctx->guide.rec_stride;
    a.walk = ctx->layered && !a.guided;
    spt_render_stats stats{};
    stats.paths = total;
    s = run_fronts<false>(ctx, a, total, running_tuning(ctx->tuning), stats);
    stats.ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    ctx->stats = stats;
    return s;
}

spt_status launch_batch(spt_ctx* ctx, BatchData& b, uint32_t sample_div) {
    auto t0 = std::chrono::steady_clock::now();
    const spt_tuning tn = running_tuning(ctx->tuning);
    const uint32_t nj = (uint32_t)b.jobs.size();
    std::vector<Job> jobs = b.jobs;
    for (Job& jb : jobs) {
        if (sample_div > 1) {  // tuning trial: a share of the samples, outputs untouched
            jb.spp_count = std::max<uint32_t>(1, jb.spp_count / sample_div);
            jb.film32 = nullptr;
            jb.film64 = nullptr;
            jb.path_rgb = nullptr;
        }
        jb.n_paths = (uint64_t)jb.vw * jb.vh * jb.spp_count;
    }
    // generation tiles, taken round-robin from the jobs; within a job samples
    // advance slowest, so every pixel gets its first samples early
    std::vector<std::vector<BatchTile>> per(nj);
    for (uint32_t j = 0; j < nj; ++j) {
        const Job& jb = jobs[j];
        const uint32_t npix = jb.vw * jb.vh;
        for (uint32_t s0 = 0; s0 < jb.spp_count; s0 += tn.tile_samples)
            for (uint32_t p0 = 0; p0 < npix; p0 += tn.tile_pixels) {
                BatchTile t{};
                t.job = j;
                t.p0 = p0;
                t.np = std::min(tn.tile_pixels, npix - p0);
                t.s0 = jb.spp_begin + s0;
                t.ns = std::min(tn.tile_samples, jb.spp_count - s0);
                per[j].push_back(t);
            }
    }
    std::vector<BatchTile> tiles;
    std::vector<uint64_t> start;
    uint64_t total = 0;
    for (size_t r = 0;; ++r) {
        bool any = false;
        for (uint32_t j = 0; j < nj; ++j) {
            if (r >= per[j].size()) continue;
            any = true;
            tiles.push_back(per[j][r]);
            start.push_back(total);
            total += (uint64_t)per[j][r].np * per[j][r].ns;
        }
        if (!any) break;
    }
    start.push_back(total);
    if (tiles.empty() || tiles.size() >= (1u << 31)) return set_error(ctx, SPT_ERR_INVALID, "empty or oversized batch");
    if (tiles.size() > b.tiles_cap) {
        if (b.d_tiles) (void)hipFree(b.d_tiles);
        if (b.d_tile_start) (void)hipFree(b.d_tile_start);
        b.d_tiles = nullptr;
        b.d_tile_start = nullptr;
        b.tiles_cap = 0;
        spt_status s = check_hip(ctx, hipMalloc(&b.d_tiles, tiles.size() * sizeof(BatchTile)), "batch tiles");
        if (s == SPT_OK)
            s = check_hip(ctx, hipMalloc(&b.d_tile_start, (tiles.size() + 1) * sizeof(uint64_t)), "batch tiles");
        if (s != SPT_OK) return s;
        b.tiles_cap = tiles.size();
    }
    hipStream_t st = ctx->stream;
    spt_status s = check_hip(ctx, hipMemcpyAsync(b.d_tiles, tiles.data(), tiles.size() * sizeof(BatchTile),
                                                 hipMemcpyHostToDevice, st), "tiles upload");
    if (s == SPT_OK)
        s = check_hip(ctx, hipMemcpyAsync(b.d_tile_start, start.data(), start.size() * sizeof(uint64_t),
                                          hipMemcpyHostToDevice, st), "tiles upload");
    if (s == SPT_OK)
        s = check_hip(ctx, hipMemcpyAsync(b.d_jobs, jobs.data(), nj * sizeof(Job), hipMemcpyHostToDevice, st),
                      "jobs upload");
    if (s == SPT_OK) s = check_hip(ctx, hipMemsetAsync(b.d_done, 0, nj * sizeof(uint32_t), st), "job counters");
    if (s == SPT_OK) s = check_hip(ctx, hipMemsetAsync(b.d_clock, 0, (nj + 1) * sizeof(uint64_t), st), "job clocks");
    if (s == SPT_OK) s = check_hip(ctx, hipStreamSynchronize(st), "batch upload");  // host vectors go out of scope
    if (s != SPT_OK) return s;

    RenderArgs a{};  // no binary tree: only casters and counting traversals read it
    a.sc.qnodes = reinterpret_cast<const uint32_t*>(b.d_qnodes);
    a.sc.qprims = reinterpret_cast<const float4*>(b.d_qprims);
    a.sc.qboxes = reinterpret_cast<const float4*>(b.d_qboxes);
    a.sc.small_tree = b.small_tree ? 1u : 0u;
    a.sc.stack_cap4 = b.stack_cap4;
    a.sc.shading = b.d_shading;
    a.sc.mats = b.d_mats;
    a.sc.n_tris = b.n_tris;
    a.sc.n_mats = b.n_mats;
    a.sc.has_spheres = b.has_spheres ? 1u : 0u;
    a.jobs = b.d_jobs;
    a.tiles = b.d_tiles;
    a.tile_start = b.d_tile_start;
    a.n_tiles = (uint32_t)tiles.size();
    a.n_jobs = nj;
    a.job_done = b.d_done;
    a.job_clock = b.d_clock;
    a.flags = 0;
    for (const Job& jb : jobs) a.per_path |= jb.path_rgb ? 1u : 0u;
    a.walk = b.layered;
    spt_render_stats stats{};
    stats.paths = total;
    s = run_fronts<true>(ctx, a, total, tn, stats);
    if (s != SPT_OK) return s;
    std::vector<uint64_t> clk(nj + 1, 0);
    std::vector<uint32_t> done(nj, 0);
    s = check_hip(ctx, hipMemcpy(clk.data(), b.d_clock, clk.size() * sizeof(uint64_t), hipMemcpyDeviceToHost),
                  "job clocks");
    if (s == SPT_OK)
        s = check_hip(ctx, hipMemcpy(done.data(), b.d_done, done.size() * sizeof(uint32_t), hipMemcpyDeviceToHost),
                      "job counters");
    if (s != SPT_OK) return s;
    b.scene_ms.assign(nj, 0.0);
    for (uint32_t j = 0; j < nj; ++j) {
        if (done[j] != jobs[j].n_paths) return set_error(ctx, SPT_ERR_DEVICE, "a scene did not finish all its paths");
        b.scene_ms[j] = (double)(clk[1 + j] - clk[0]) / (double)ctx->wall_clock_khz;
    }
    b.stats = spt_batch_stats{};
    b.stats.scenes = nj;
    b.stats.paths = total;
    b.stats.rays = stats.rays;
    b.stats.bounces = stats.bounces;
    b.stats.tiles = tiles.size();
    b.stats.triangles = b.n_tris;
    b.stats.device_bytes = b.device_bytes;
    b.stats.ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    ctx->stats = stats;
    ctx->stats.ms = b.stats.ms;
    return SPT_OK;
}

}  // namespace spt
