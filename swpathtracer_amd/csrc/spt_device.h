// spt_device.h - device-side scene layout, context and closest-hit traversal.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "spt.h"
#include "quad_tree.h"
#include "spt_tuning.h"
#include "spt_internal.h"
#include "spt_math.h"

namespace spt {

constexpr int kBlock = 256;       // threads per block of the ray kernels (4 wave64)
// normal kind of a shading record (word 10): flat n0, smooth n0 n1 n2, sphere centre n0
constexpr uint32_t kShadeFlat = 0, kShadeSmooth = 1, kShadeSphere = 2;
constexpr int kLdsStack = 16;     // traversal stack entries per lane kept in LDS
constexpr uint32_t kNoHit = SPT_MISS;

// Materials the learned guide samples: one Lambertian / importance-sampled
// GGX layer (kGuideSingle), or such a layer under one smooth dielectric coat
// of IOR >= 1 (kGuideCoated: the guide drives the base layer's directions).
constexpr uint8_t kGuideSingle = 1, kGuideCoated = 2;

// Scene as the kernels see it.
struct DevScene {
    const uint32_t* qnodes; // QuadNode x 16 words, quad traversal
    const float4* qprims;   // QuadPrim x 3 float4, blocks of four
    const float4* qboxes;   // QuadBox x 2 float4
    const float4* nodes;    // n_nodes x 4 float4 (spt_node64)
    const float4* tris;     // n_tris x 3 float4 (spt_tri48; .pad[0] = material id)
    const float4* shading;  // n_tris x 3 float4: n0 n1 n2, material, smooth flag, pad
    const spt_material* mats;
    float rmin[3], rmax[3];
    uint32_t root_leaf;  // > 0: the root is a leaf holding this many triangles
    uint32_t n_tris;
    uint32_t n_nodes;
    uint32_t n_mats;
    uint32_t stack_cap;  // traversal stack entries a lane may need (inner-node depth + 1)
    uint32_t stack_cap4; // same for the quad traversal's tree (3 per level + 1)
    uint32_t small_tree;   // the quad nodes and blocks are under 4 GiB each (32-bit offsets)
    uint32_t has_spheres;  // some primitive record is a sphere (uniform branch in the leaf loops)
};

// Closest-hit test of one primitive record (a, b, c = its three float4):
// Moller-Trumbore for a triangle, Hultquist for a sphere (centre a.xyz,
// radius a.w, kind in c.w). u, v are the triangle's barycentrics (0 for a
// sphere). `spheres` is the scene's uniform flag: without spheres the kind is
// never read.
__device__ inline bool prim_test(bool spheres, V3 o, V3 d, float4 a, float4 b, float4 c, float& t, float& u,
                                 float& v) {
    if (spheres && __float_as_uint(c.w) == SPT_PRIM_SPHERE) {
        u = v = 0.0f;
        return sphere_test(o, d, V3{a.x, a.y, a.z}, a.w, t);
    }
    return tri_test(o, d, V3{a.x, a.y, a.z}, V3{a.w, b.x, b.y}, V3{b.z, b.w, c.x}, t, u, v);
}

// Closest-hit result of one ray.
struct Hit {
    float t;
    uint32_t idx;   // triangle index in leaf order (kNoHit: miss)
    uint32_t prim;  // primitive id in scene order
    uint32_t mat;
    float u, v;
};

// Traversal stack: the first kLdsStack entries of a lane live in LDS
// (layout [entry][lane], conflict-free), deeper entries spill to a global
// buffer laid out [entry - kLdsStack][thread] so a wave's accesses coalesce.
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(1))) uint32_t glb_u32;

struct Stack {
    lds_u32* lds;       // &lds[threadIdx.x], stride kBlock
    glb_u32* spill;     // &spill[global thread], stride spill_stride
    uint32_t spill_stride;
    uint32_t cap;       // total entries available
    // Address-space-qualified pointers keep LDS and global accesses as ds_* and
    // global_* instructions instead of one merged flat access.
    __device__ Stack(uint32_t* lds_lane, uint32_t* spill_lane, uint32_t stride, uint32_t capacity)
        : lds((lds_u32*)lds_lane), spill((glb_u32*)spill_lane), spill_stride(stride), cap(capacity) {}
    __device__ void put(int i, uint32_t v) {
        if (i < kLdsStack)
            lds[i * kBlock] = v;
        else
            spill[(size_t)(i - kLdsStack) * spill_stride] = v;
    }
    __device__ uint32_t get(int i) const {
        if (i < kLdsStack) return lds[i * kBlock];
        return spill[(size_t)(i - kLdsStack) * spill_stride];
    }
};

// Leaf: tests triangles [first, first+cnt) against the ray. A candidate is
// accepted exactly when the reference accepts it (sbvh.cpp:494-496: t > 0,
// t < best, hit point inside the leaf box +-1e-3); among equal t the smaller
// leaf-order index wins, which is the reference's depth-first left-first
// first-come rule (strict '<').
template <bool COUNT>
__device__ inline void leaf_test(const DevScene& sc, V3 o, V3 d, uint32_t first, uint32_t cnt, V3 bmn, V3 bmx,
                                 Hit& h, uint32_t& tests, uint32_t& isects) {
    for (uint32_t k = first; k < first + cnt; ++k) {
        const float4* tp = sc.tris + 3 * (size_t)k;
        const float4 a = tp[0], b = tp[1], c = tp[2];
        if (COUNT) ++tests;
        float t, u, v;
        if (prim_test(sc.has_spheres != 0u, o, d, a, b, c, t, u, v)) {
            if (COUNT) ++isects;
            if ((t > 0.0f) && ((t < h.t) || ((t == h.t) && (k < h.idx)))) {
                V3 p = o + d * t;
                if (point_inside(p, bmn, bmx)) {
                    h.t = t;
                    h.idx = k;
                    h.prim = __float_as_uint(c.y);
                    h.mat = __float_as_uint(c.z);
                    h.u = u;
                    h.v = v;
                }
            }
        }
    }
}

// Closest hit of one ray on the binary tree, visiting exactly the nodes the
// reference visits (acceleration/sbvh.cpp:423-515: every box the ray's line
// meets); with COUNT it reproduces num_intersection_tests /
// num_intersections.
template <bool COUNT>
__device__ inline void trace_ray(const DevScene& sc, V3 o, V3 d, Stack& st, Hit& h, uint32_t& tests,
                                 uint32_t& isects, bool& overflow) {
    h.t = __builtin_inff();
    h.idx = kNoHit;
    h.prim = kNoHit;
    h.mat = 0;
    h.u = h.v = 0.0f;
    tests = 0;
    isects = 0;
    const V3 inv{1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
    float tn, tf;
    const V3 rmn{sc.rmin[0], sc.rmin[1], sc.rmin[2]}, rmx{sc.rmax[0], sc.rmax[1], sc.rmax[2]};
    if (COUNT) tests = 1;
    if (!slab(o, inv, rmn, rmx, tn, tf)) return;
    if (COUNT) isects = 1;
    if (sc.root_leaf) {
        leaf_test<COUNT>(sc, o, d, 0, sc.root_leaf, rmn, rmx, h, tests, isects);
        return;
    }
    uint32_t node = 0;
    int sp = 0;
    while (true) {
        const float4* np = sc.nodes + 4 * (size_t)node;
        const float4 a = np[0], b = np[1], c = np[2];
        const uint4 r = reinterpret_cast<const uint4*>(np)[3];
        const V3 lmn{a.x, a.y, a.z}, lmx{a.w, b.x, b.y}, rmn2{b.z, b.w, c.x}, rmx2{c.y, c.z, c.w};
        float tnl = 0.0f, tfl = 0.0f, tnr = 0.0f, tfr = 0.0f;
        bool hl = slab(o, inv, lmn, lmx, tnl, tfl);
        bool hr = slab(o, inv, rmn2, rmx2, tnr, tfr);
        if (COUNT) {
            tests += 2;
            isects += (uint32_t)hl + (uint32_t)hr;
        }
        if (hl && r.y) {
            leaf_test<COUNT>(sc, o, d, r.x, r.y, lmn, lmx, h, tests, isects);
            hl = false;
        }
        if (hr && r.w) {
            leaf_test<COUNT>(sc, o, d, r.z, r.w, rmn2, rmx2, h, tests, isects);
            hr = false;
        }
        if (hl && hr) {
            if (sp >= (int)st.cap) {
                overflow = true;
                return;
            }
            st.put(sp++, r.z);
            node = r.x;
        } else if (hl) {
            node = r.x;
        } else if (hr) {
            node = r.z;
        } else {
            if (sp == 0) break;
            node = st.get(--sp);
        }
    }
}

// Camera ray through image point (x, y): PinholeCamera::getRay
// (cameras/pinhole_camera.cpp:14-18), OrthographicCamera::getRay
// (cameras/orthographic_camera.cpp:21-25).
__device__ inline void camera_ray(const DevCamera& c, float x, float y, V3& o, V3& d) {
    if (c.type == SPT_CAMERA_PINHOLE) {
        V3 ld = normalize(c.ulc + V3{x, -y, 0.0f});
        o = c.position;
        d = to_world(c.frame, ld);
    } else {
        V3 lo = c.ulc + V3{x * c.pdx, y * -c.pdy, 0.0f};
        o = to_world(c.frame, lo) + c.position;
        d = c.ortho_dir;
    }
}

// Shading normal of a hit at pos: SmoothTriangle::getNormal
// (primitives/smooth_triangle.h:11-13), the stored flat normal
// (primitives/triangle.cpp:5-6) or a sphere's normalize(pos - centre)
// (primitives/sphere.cpp:35).
__device__ inline V3 shading_normal(const DevScene& sc, const Hit& h, V3 pos) {
    const float4* sp = sc.shading + 3 * (size_t)h.idx;
    const float4 a = sp[0], b = sp[1], c = sp[2];
    const V3 n0{a.x, a.y, a.z};
    const uint32_t kind = __float_as_uint(c.z);
    if (kind == kShadeFlat) return n0;
    if (kind == kShadeSphere) return normalize(pos - n0);
    const V3 n1{a.w, b.x, b.y}, n2{b.z, b.w, c.x};
    return normalize(n0 * (1.0f - h.u - h.v) + n1 * h.u + n2 * h.v);
}

// One scene's share of a render call: camera, sampling, termination,
// outputs and where its tree starts in the (shared) node/triangle arrays.
struct Job {
    DevCamera cam;
    uint32_t sampler, n_sub, spp, spp_begin, spp_count;
    float w_sub;
    int32_t max_depth, rr_depth;
    uint64_t seed;
    uint32_t vt, vl, vw, vh;
    float bg[3];
    const float* stream;
    uint32_t stride;
    float* film32;
    double* film64;
    float* path_rgb;
    float rmin[3], rmax[3];
    uint32_t node0;     // root in the quad tree
    uint64_t n_paths;  // paths of this job in the call
};

// A run of consecutive paths of one job: pixels [p0, p0 + np) of its
// viewport (row-major), samples [s0, s0 + ns) of each; the paths run over the
// pixels for one sample, then the next sample.
struct BatchTile {
    uint32_t job, p0, np, s0, ns, pad[3];
};

// Device arrays and per-scene jobs of a batch (spt_batch_*).
struct BatchData {
    QuadNode* d_qnodes = nullptr;
    QuadPrim* d_qprims = nullptr;
    QuadBox* d_qboxes = nullptr;
    float4* d_shading = nullptr;
    spt_material* d_mats = nullptr;
    bool layered = false;  // some material has several layers
    uint32_t n_tris = 0, n_mats = 0, stack_cap4 = 0;
    bool has_spheres = false, small_tree = false;
    std::vector<Job> jobs;  // host copy: sampling, outputs, roots
    Job* d_jobs = nullptr;
    BatchTile* d_tiles = nullptr;
    uint64_t* d_tile_start = nullptr;
    size_t tiles_cap = 0;
    uint32_t* d_done = nullptr;   // finished paths per job
    uint64_t* d_clock = nullptr;  // start, then finish time per job
    uint64_t device_bytes = 0;
    spt_batch_stats stats{};
    std::vector<double> scene_ms;
};

// Scene box used by the guide's input encoding.
struct GuideBox {
    float bmin[3], bext[3];
};

// Device-resident training state of the guide (64-float area after the
// gradient): the host never waits for a step; it reads this block when it
// asks for statistics or a loss.
struct GuideCtl {
    float wsum;       // sum of the current step's record weights
    float loss;       // loss of the current step
    uint32_t bad;     // a gradient entry was not finite
    float scale;      // loss scale (halved on overflow)
    uint32_t steps;   // successful steps (Adam step number - 1)
    uint32_t skipped; // skipped steps
    float last_loss;  // loss of the last successful step
    uint32_t pad;
    unsigned long long trained;  // records consumed by successful steps
};

// Learned guide state of a context (spt_guide.hip).
struct GuideState {
    bool ready = false;
    float* d_theta = nullptr;  // fp32 master parameters, then m, v, grad, control block (64 floats)
    float* d_m = nullptr;
    float* d_v = nullptr;
    float* d_grad = nullptr;
    float* d_acc = nullptr;
    unsigned short* d_wbf = nullptr;  // bf16 copy of the parameters, in the order of guide::FwdWeights
    float* d_records = nullptr;
    uint32_t records_cap = 0;    // batch x steps_per_pass
    uint32_t records_alloc = 0;  // allocated record slots
    uint64_t collected = 0;
    float lr = 5e-3f, loss_scale = 65536.0f, bsdf_fraction = 0.5f;  // loss_scale: the configured start
    uint32_t flags = 0;  // SPT_GUIDE_*
    uint32_t train_every = 0;      // in-call training rounds every this many bounces (0: none)
    double rays_per_path = 4.0;    // extension rays per path of the last training render
    uint32_t batch = 262144;
    double train_ms = 0.0;
    unsigned short* d_gout = nullptr;  // per-path raw outputs (half floats) during a guided render
    size_t gout_cap = 0;
    uint32_t rec_stride = 1;      // 1 in rec_stride candidate vertices is recorded
    double cand_per_path = 0.0;   // candidate vertices per path of the last training render
    uint64_t candidates = 0;      // candidate vertices of the last training render
    double kernel_ms = 0.0;       // device time of the training kernels (settled steps)
    // training scratch: the partial gradients of the training kernel's blocks, f32 [blocks][params]
    char* d_scratch = nullptr;
    size_t scratch_bytes = 0;
    std::vector<hipEvent_t> ev_free, ev_pending;  // event pairs around training kernels

    GuideCtl* ctl() const { return reinterpret_cast<GuideCtl*>(d_acc); }
    // an event pair for one training kernel (false: none available)
    bool event_pair(hipEvent_t& a, hipEvent_t& b) {
        for (int k = 0; k < 2; ++k) {
            if (ev_free.empty()) {
                hipEvent_t e;
                if (hipEventCreate(&e) != hipSuccess) return false;
                ev_free.push_back(e);
            }
            (k == 0 ? a : b) = ev_free.back();
            ev_free.pop_back();
            ev_pending.push_back(k == 0 ? a : b);
        }
        return true;
    }
    // adds the device time of completed pairs (call after the stream is idle)
    void settle_events() {
        for (size_t i = 0; i + 1 < ev_pending.size(); i += 2) {
            float ms = 0.0f;
            if (hipEventElapsedTime(&ms, ev_pending[i], ev_pending[i + 1]) == hipSuccess) kernel_ms += ms;
        }
        ev_free.insert(ev_free.end(), ev_pending.begin(), ev_pending.end());
        ev_pending.clear();
    }
    void destroy_events() {
        for (hipEvent_t e : ev_free) (void)hipEventDestroy(e);
        for (hipEvent_t e : ev_pending) (void)hipEventDestroy(e);
        ev_free.clear();
        ev_pending.clear();
    }
};

}  // namespace spt

// The context: one device, one stream, the uploaded scene and scratch buffers.
struct spt_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    int num_cus = 256;
    // scene
    float4* d_nodes = nullptr;
    spt::QuadNode* d_qnodes = nullptr;
    spt::QuadPrim* d_qprims = nullptr;
    spt::QuadBox* d_qboxes = nullptr;
    uint32_t stack_cap4 = 0;
    float4* d_tris = nullptr;
    float4* d_shading = nullptr;
    spt_material* d_mats = nullptr;
    bool layered = false;  // some material has several layers
    uint32_t n_nodes = 0, n_tris = 0, n_mats = 0;
    float root_box[6] = {0, 0, 0, 0, 0, 0};
    uint32_t root_leaf = 0;
    uint32_t stack_cap = 0;
    uint32_t max_mat = 0;  // largest material id referenced by a triangle
    bool has_spheres = false, small_tree = false;
    bool one_block = false;  // at most four primitives: closest hits without a tree
    bool has_scene = false;
    std::vector<spt_material> h_mats;
    uint8_t* d_guidable = nullptr;  // per material: kGuideSingle / kGuideCoated, 0 = not guide-sampled
    // traversal stack spill buffer
    uint32_t* d_spill = nullptr;
    size_t spill_words = 0;
    // status word written by kernels (1 = stack overflow), then two 64-bit
    // fetch counters (nodes, triangles) at byte offset 16
    uint32_t* d_flags = nullptr;
    uint32_t* d_rays = nullptr;   // ray counters of the traversal launches (spt_quad.h)
    uint32_t* scratch = nullptr;  // this device's static scratch (spt_trace_noalloc), never freed
    // HIP events: [0..1] bracket extend launches, [2..9] user slots (spt_event_*)
    hipEvent_t ev[10] = {};
    // event pairs bracketing the extend launches of one render call
    std::vector<hipEvent_t> tev;
    // path-tracing state (grown on demand)
    void* d_paths = nullptr;
    size_t paths_bytes = 0;
    spt_render_stats stats{};
    spt::GuideState guide;
    spt_tuning tuning{};  // zero fields: defaults
    bool told_default = false;  // the last three wavefronts spt_get_tuning reported were the default's
    int wall_clock_khz = 100000;
    void* h_pin = nullptr;  // kPinBytes of pinned host memory for small read-backs
    // mapped host memory the bounce loop reports its progress to (see k_plan)
    volatile uint32_t* h_status = nullptr;
    uint32_t* d_status = nullptr;
    // contexts of the extra concurrent wavefronts of a render (their own
    // stream, queue, status, flags and spill buffer), created on first use
    std::vector<spt_ctx*> fronts;

    spt::DevScene scene() const {
        spt::DevScene s;
        s.nodes = d_nodes;
        s.qnodes = reinterpret_cast<const uint32_t*>(d_qnodes);
        s.qprims = reinterpret_cast<const float4*>(d_qprims);
        s.qboxes = reinterpret_cast<const float4*>(d_qboxes);
        s.small_tree = small_tree ? 1u : 0u;
        s.stack_cap4 = stack_cap4;
        s.tris = d_tris;
        s.shading = d_shading;
        s.mats = d_mats;
        for (int i = 0; i < 3; ++i) {
            s.rmin[i] = root_box[i];
            s.rmax[i] = root_box[3 + i];
        }
        s.root_leaf = root_leaf;
        s.n_tris = n_tris;
        s.n_nodes = n_nodes;
        s.n_mats = n_mats;
        s.stack_cap = stack_cap;
        s.has_spheres = has_spheres ? 1u : 0u;
        return s;
    }
};

namespace spt {
spt_status set_error(spt_ctx* ctx, spt_status code, const std::string& msg);
spt_status check_hip(spt_ctx* ctx, hipError_t e, const char* what);
// A material as the kernels read it: constants of its layers in the fields
// that their type leaves unused or only reads through them, with the bits the
// kernels would compute. Lambertian: r0 = kd / pi; smooth dielectric: r0 =
// Schlick reflectance of 1 and ior (the same from both sides: its root only
// changes sign), 1 / ior, 1 / ior^2; GGX conductor: eta, k = eta^2 - k^2,
// 4 eta^2 k^2.
spt_material prepare_material(const spt_material& m);
// Waits for the context stream by polling it (no blocking wait on an
// interrupt: those have been seen to wake up hundreds of ms late).
spt_status stream_wait(spt_ctx* ctx, const char* what);
// Copies up to 64 KiB, from one or two places, from the device through pinned
// memory and waits once.
constexpr size_t kPinBytes = 64 * 1024;
spt_status read_small(spt_ctx* ctx, void* dst, const void* d_src, size_t bytes, const char* what, void* dst2 = nullptr,
                      const void* d_src2 = nullptr, size_t bytes2 = 0);
// grows ctx->d_spill to hold `words` entries; returns false on failure
spt_status ensure_spill(spt_ctx* ctx, size_t words);
// launch helpers implemented by the kernel translation units
spt_status launch_trace(spt_ctx* ctx, const spt_ray32* d_rays, uint64_t n, spt_hit* d_hits, uint32_t mode,
                        uint32_t* d_tests, uint32_t* d_isects);
spt_status launch_raycast(spt_ctx* ctx, const spt_camera* cam, uint32_t kind, void* d_out);
// The allocation-free closest-hit path (spt_trace_noalloc) and the lookup of
// its static scratch on the context's device (from spt_create).
constexpr int kMaxScratchDevices = 64;
spt_status init_static_scratch(spt_ctx* ctx);
spt_status launch_trace_noalloc(spt_ctx* ctx, const spt_ray32* d_rays, uint64_t n, spt_hit* d_hits);
spt_status launch_camera_rays(spt_ctx* ctx, const spt_camera* cam, spt_ray32* d_rays);
GuideBox guide_box(const spt_ctx* ctx);
spt_status guide_eval_launch(spt_ctx* ctx, const float* d_q, uint32_t stride, uint32_t n, float* d_out);
// One Adam step on n records, record i at d_rec + i * rs records (queued on
// the context stream; loss_out, when given, waits for the step).
spt_status guide_train_launch(spt_ctx* ctx, const float* d_rec, uint32_t n, float* loss_out, uint32_t rs);
spt_status launch_render(spt_ctx* ctx, const spt_camera* cam, const spt_render_params* p, float* d_rgb32,
                         double* d_rgb64, float* d_path_rgb);
void scene_arrays(const spt_bvh* bvh, const float* verts, const float* normals, const uint32_t* mat_ids,
                  std::vector<spt_tri48>& tris, std::vector<float>& sh);
spt_status make_job(spt_ctx* ctx, const spt_camera* cam, const spt_render_params* prm, float* d_rgb32, double* d_rgb64,
                    float* d_path_rgb, Job& jb, uint64_t& total);
// A multi-scene render (spt_batch_*): every job of the batch, or with
// sample_div > 1 the first 1/sample_div of each job's samples.
spt_status launch_batch(spt_ctx* ctx, BatchData& b, uint32_t sample_div);
}  // namespace spt
