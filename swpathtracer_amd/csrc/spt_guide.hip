// spt_guide.hip - the learned guide's kernels (batched inference, fused
// training step, Adam) and their C ABI (include/spt.h, spt_guide_*).
#include <chrono>
#include <cmath>
#include <cstring>

#include "spt_guide.h"

namespace spt {

using namespace guide;

namespace {

// Raw outputs for queries (p, n, wo) as 9 floats with a stride: each wave
// encodes 64 queries (one per lane) into its stage, then runs the
// register-resident MLP on 4 groups of 16. Three blocks a CU, as many as their
// LDS lets in at once (a million queries 51.7 us, with four 56.7, six 52.0,
// sixteen 55.5), and no block-wide waits. Bound by the 196 B a query moves: a
// million queries 50 us (before: 62), 41 at the rate of a large copy.
__global__ __launch_bounds__(kBlock) void k_guide_eval(const float* __restrict__ theta,
                                                       const unsigned short* __restrict__ wbf,
                                                       const float* __restrict__ q, uint32_t stride, uint32_t n,
                                                       float* __restrict__ out, GuideBox box) {
    extern __shared__ float dyn[];
    FwdWeights& sw = *reinterpret_cast<FwdWeights*>(dyn);
    WaveStage* stages = reinterpret_cast<WaveStage*>(reinterpret_cast<char*>(dyn) + sizeof(FwdWeights));
    load_weights(sw, wbf, theta);
    __syncthreads();
    const int wave = threadIdx.x >> 6, r = __lane_id() & 15;
    WaveStage& st = stages[wave];
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        const uint32_t row = base + threadIdx.x;
        float f[kEnc];
        if (row < n) {
            const float* p = q + (size_t)row * stride;
            encode(V3{p[0], p[1], p[2]}, V3{p[3], p[4], p[5]}, V3{p[6], p[7], p[8]}, box.bmin, box.bext, f);
        } else {
            for (int i = 0; i < kEnc; ++i) f[i] = 0.0f;
        }
        stage_row(st, f);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a stage belongs to one wave
        const uint32_t wbase = base + (uint32_t)wave * 64;
        if (wbase < n)
            mlp_stage_fwd(sw, st, [&](int g16, const f32x4 y[3]) {
                const uint32_t smp = wbase + 16 * g16 + r;
                if (smp < n) store_outputs(out + (size_t)smp * kOut, y);
            });
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// Sum of the record weights (for the batch-mean normalisation), one atomic
// per block.
__global__ __launch_bounds__(kBlock) void k_guide_wsum(const float* __restrict__ rec, uint32_t n, uint32_t rs,
                                                       float* __restrict__ acc) {
    __shared__ float part[kBlock / 64];
    float s = 0.0f;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        s += rec[(size_t)i * rs * kRecord + 12];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (__lane_id() == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(acc, (part[0] + part[1]) + (part[2] + part[3]));
}

// ---------------------------------------------------------------------------
// The gradient of a training batch in one kernel: a block takes tiles of 128
// records through encoding, forward pass, loss gradient and backward pass and
// adds the weight gradients up in its accumulators, which it writes once.
// Nothing but the records is read and nothing but a partial gradient written:
// activations and their gradients as bf16 lie in LDS, feature-major, so that
// a weight gradient dW[o][k] = sum_s dz[o][s] in[k][s] reads both of its MFMA
// operands as 16-B rows of samples. LDS (150 KB of 160) allows one block of
// eight waves a CU: a wave owns 16 samples of a tile in the passes (column
// form, as in inference) and one or two 16 x 16 tiles of each layer's gradient.
// The loss gradient of a record takes four lanes, two lobes each.
//
// 262,144 records: 75 us; as three kernels with all of that in global memory
// (0.5 GB written and read again) 342 us. Bound by the chain of a tile's
// stages at two waves a SIMD.
// ---------------------------------------------------------------------------
constexpr int kTrainTile = 128, kTrainBlock = 512, kTrainRow = kTrainTile + 8;  // 272 B: 16 rows on distinct banks

struct TrainLds {
    FwdWeights fw;
    // W2^T, W3^T, W4^T as MFMA operands of the backward pass (as in FwdWeights,
    // rows = inputs; W4 with 16 more outputs of weight 0). A third k-tile of 16
    // as a v_mfma 16x16x16 is not safe here: the compiler puts no wait between it
    // and a 16x16x32 whose result it adds to, and as a pair on one accumulator,
    // two instructions apart, they give wrong sums (nearly every element off; exact
    // with three other products in between, or with a second 16x16x32).
    uint4 w2t[4 * 2 * 64], w3t[4 * 2 * 64], w4t[4 * 2 * 64];
    unsigned short x[2][kEnc][kTrainRow];  // two tiles in turn
    unsigned short h1[kHid][kTrainRow], h2[kHid][kTrainRow], h3[kHid][kTrainRow];
    unsigned short dy[kOutP][kTrainRow];   // rows 40..47 stay zero
    union {
        float y[kTrainTile][kOut + 1];
        unsigned short dz[kHid][kTrainRow];
    };
};

__device__ inline bf16x8 bf8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// D += A B, 32 samples from s0 on as the reduction axis: rows o0 + r of T and
// rows k0 + r of U.
__device__ inline f32x4 mfma_rows(const unsigned short (*T)[kTrainRow], int o0, const unsigned short (*U)[kTrainRow],
                                  int k0, int s0, f32x4 c) {
    const int r = __lane_id() & 15, g = __lane_id() >> 4;
    const uint4 a = *reinterpret_cast<const uint4*>(&T[o0 + r][s0 + 8 * g]);
    const uint4 b = *reinterpret_cast<const uint4*>(&U[k0 + r][s0 + 8 * g]);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf8(a), bf8(b), c, 0, 0, 0);
}
// The same with B = 1: every column of D gets the sums of the rows of T.
__device__ inline f32x4 mfma_row_sums(const unsigned short (*T)[kTrainRow], int o0, int s0, f32x4 c) {
    const int r = __lane_id() & 15, g = __lane_id() >> 4;
    const uint4 a = *reinterpret_cast<const uint4*>(&T[o0 + r][s0 + 8 * g]);
    const uint32_t ones = 0x3F803F80u;
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf8(a), bf8(make_uint4(ones, ones, ones, ones)), c, 0, 0, 0);
}

// Features f0 + 0..3 of sample s.
__device__ inline bf16x4 ld_col4(const unsigned short (*T)[kTrainRow], int f0, int s) {
    return bf16x4{(short)T[f0][s], (short)T[f0 + 1][s], (short)T[f0 + 2][s], (short)T[f0 + 3][s]};
}
__device__ inline void st_col4(unsigned short (*T)[kTrainRow], int f0, int s, bf16x4 v) {
    T[f0][s] = (unsigned short)v[0];
    T[f0 + 1][s] = (unsigned short)v[1];
    T[f0 + 2][s] = (unsigned short)v[2];
    T[f0 + 3][s] = (unsigned short)v[3];
}
// Gradients through the ReLU whose outputs are h, as bf16.
__device__ inline bf16x4 relu_grad(f32x4 v, bf16x4 h) {
    for (int i = 0; i < 4; ++i)
        if (h[i] <= 0) v[i] = 0.0f;  // the sign of a bf16 is that of its bits
    return __builtin_bit_cast(bf16x4, (u32x2){pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])});
}

// W^T of a layer of 64 inputs as MFMA operands: block (t, p) holds
// for lane r + 16 g W[32 p + 4 g + 0..3][16 t + r] and W[32 p + 16 + 4 g + 0..3][16 t + r].
// Rows from `rows` on count as 0.
__device__ inline void transpose_layer(uint4* dst, const unsigned short* w, int rows) {
    for (int i = threadIdx.x; i < 4 * 2 * 64; i += blockDim.x) {
        const int l = i & 63, p = (i >> 6) & 1, t = i >> 7;
        uint32_t v[4];
        for (int k = 0; k < 4; ++k) {
            const int row = 32 * p + 4 * (l >> 4) + (k >> 1) * 16 + (k & 1) * 2;
            const int col = 16 * t + (l & 15);
            v[k] = row < rows ? (uint32_t)w[bf_at(kHid, row, col)] | ((uint32_t)w[bf_at(kHid, row + 1, col)] << 16) : 0u;
        }
        dst[i] = make_uint4(v[0], v[1], v[2], v[3]);
    }
}

// Sum and maximum over the four lanes of a quad.
template <int CTRL>
__device__ inline float quad_swap_f(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xF, 0xF, true));
}
__device__ inline float quad_sum(float v) {
    v += quad_swap_f<0xB1>(v);
    return v + quad_swap_f<0x4E>(v);
}
__device__ inline float quad_max(float v) {
    v = fmaxf(v, quad_swap_f<0xB1>(v));
    return fmaxf(v, quad_swap_f<0x4E>(v));
}

// Gradient of -W log q(d) w.r.t. the 40 raw outputs, by the four lanes of a
// quad: y and dy are the lane's two lobes (10 outputs); every lane returns the
// loss.
__device__ inline float loss_grad_quad(const float y[10], V3 d, float W, float dy[10]) {
    const float amax = quad_max(fmaxf(y[4], y[9]));
    const float lse = amax + logf(quad_sum(expf(y[4] - amax) + expf(y[9] - amax)));
    Lobe L[2];
    float lv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const V3 raw{y[5 * i], y[5 * i + 1], y[5 * i + 2]};
        const float nr = sqrtf(dot(raw, raw) + 1e-12f);
        L[i].mu = raw * (1.0f / nr);
        L[i].norm = nr;
        const float s = y[5 * i + 3];
        const float sc = fminf(fmaxf(s, logf(kKappaMin)), logf(kKappaMax));
        L[i].inside = (s == sc);
        L[i].kappa = expf(sc);
        L[i].logw = y[5 * i + 4] - lse;
        lv[i] = L[i].logw + log_vmf(L[i], d);
    }
    const float m = quad_max(fmaxf(lv[0], lv[1]));
    const float logq = m + logf(quad_sum(expf(lv[0] - m) + expf(lv[1] - m)));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float r = expf(lv[i] - logq);
        const float w = expf(L[i].logw);
        const float c = dot(L[i].mu, d);
        dy[5 * i + 4] = -W * (r - w);
        const float kap = L[i].kappa;
        const float dlv = 1.0f - 2.0f * kap / expm1f(2.0f * kap) + kap * (c - 1.0f);
        dy[5 * i + 3] = L[i].inside ? -W * r * dlv : 0.0f;
        const V3 gmu = d * (-W * r * kap);
        const V3 proj = (gmu - L[i].mu * dot(gmu, L[i].mu)) * (1.0f / L[i].norm);
        dy[5 * i + 0] = proj.x;
        dy[5 * i + 1] = proj.y;
        dy[5 * i + 2] = proj.z;
    }
    return -W * logq;
}

// Gradients of the records' loss, scaled by loss_scale / n, as one partial
// gradient per block; the loss goes to ctl->loss. Tiles past n count zero.
__global__ __launch_bounds__(kTrainBlock) void k_train_grad(const float* __restrict__ theta,
                                                            const unsigned short* __restrict__ wbf,
                                                            const float* __restrict__ rec, uint32_t n, uint32_t rs,
                                                            GuideCtl* __restrict__ ctl, GuideBox box,
                                                            float* __restrict__ partial) {
    extern __shared__ float dyn[];
    TrainLds& t = *reinterpret_cast<TrainLds*>(dyn);
    load_weights(t.fw, wbf, theta);
    transpose_layer(t.w2t, wbf + kW2, kHid);
    transpose_layer(t.w3t, wbf + kW3, kHid);
    transpose_layer(t.w4t, wbf + kW4, kOutP);
    for (int i = threadIdx.x; i < (kOutP - kOut) * kTrainRow; i += kTrainBlock) t.dy[kOut + i / kTrainRow][i % kTrainRow] = 0;
    const int wave = threadIdx.x >> 6, l = __lane_id(), r = l & 15, g = l >> 4;
    const int col = 16 * wave + r;              // this lane's sample of the tile in the passes
    const int lrec = 16 * wave + (l >> 2), part = l & 3;  // its record and lobe pair in the loss
    const int ot = wave & 3, half = wave >> 2;  // its tiles of the weight gradients
    const float wmean = fmaxf(ctl->wsum / (float)n, 1e-30f);
    const float scale = ctl->scale / (float)n;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 g4[2] = {zero, zero}, g3[2] = {zero, zero}, g2[2] = {zero, zero}, g1 = zero, b3 = zero, b2 = zero, b1 = zero;
    float b4[10] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    float loss = 0.0f;
    uint32_t turn = 0;
    for (uint32_t base = blockIdx.x * kTrainTile; base < n; base += gridDim.x * kTrainTile, turn ^= 1u) {
        unsigned short(*x)[kTrainRow] = t.x[turn];
        if (threadIdx.x < kTrainTile) {
            const uint32_t s = base + threadIdx.x;
            float f[kEnc];
            if (s < n) {
                const float* p = rec + (size_t)s * rs * kRecord;
                encode(V3{p[0], p[1], p[2]}, V3{p[3], p[4], p[5]}, V3{p[6], p[7], p[8]}, box.bmin, box.bext, f);
            } else {
                for (int i = 0; i < kEnc; ++i) f[i] = 0.0f;
            }
#pragma unroll
            for (int i = 0; i < kEnc; i += 2) {
                const uint32_t v = pack_bf2(f[i], f[i + 1]);
                x[i][threadIdx.x] = (unsigned short)v;
                x[i + 1][threadIdx.x] = (unsigned short)(v >> 16);
            }
        }
        __syncthreads();  // encoded; the tile before has been read
        bf16x4 h1[4], h2[4], h3[4];
        {
            const bf16x4 x0 = ld_col4(x, 4 * g, col), x1 = ld_col4(x, 16 + 4 * g, col);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                h1[k] = pack_relu(mfma_w(t.fw.w1 + 64 * k, x0, x1, bias4(t.fw.b1 + 16 * k + 4 * g)));
                st_col4(t.h1, 16 * k + 4 * g, col, h1[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f32x4 acc = bias4(t.fw.b2 + 16 * k + 4 * g);
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = mfma_w(t.fw.w2 + 64 * (2 * k + p), h1[2 * p], h1[2 * p + 1], acc);
                h2[k] = pack_relu(acc);
                st_col4(t.h2, 16 * k + 4 * g, col, h2[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f32x4 acc = bias4(t.fw.b3 + 16 * k + 4 * g);
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = mfma_w(t.fw.w3 + 64 * (2 * k + p), h2[2 * p], h2[2 * p + 1], acc);
                h3[k] = pack_relu(acc);
                st_col4(t.h3, 16 * k + 4 * g, col, h3[k]);
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                f32x4 acc = bias4(t.fw.b4 + 16 * k + 4 * g);
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = mfma_w(t.fw.w4 + 64 * (2 * k + p), h3[2 * p], h3[2 * p + 1], acc);
                if (16 * k + 4 * g < kOut)
                    for (int i = 0; i < 4; ++i) t.y[col][16 * k + 4 * g + i] = acc[i];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // a wave reads its own samples' outputs
        {
            float y[10], dy[10];
#pragma unroll
            for (int i = 0; i < 10; ++i) y[i] = t.y[lrec][10 * part + i];
            const uint32_t s = base + (uint32_t)lrec;
            if (s < n) {
                const float* p = rec + (size_t)s * rs * kRecord;
                const float v = loss_grad_quad(y, V3{p[9], p[10], p[11]}, p[12] / wmean, dy);
                loss += part == 0 ? v : 0.0f;
#pragma unroll
                for (int i = 0; i < 10; ++i) dy[i] *= scale;
            } else {
#pragma unroll
                for (int i = 0; i < 10; ++i) dy[i] = 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 10; i += 2) {
                b4[i] += dy[i];
                b4[i + 1] += dy[i + 1];
                const uint32_t v = pack_bf2(dy[i], dy[i + 1]);
                t.dy[10 * part + i][lrec] = (unsigned short)v;
                t.dy[10 * part + i + 1][lrec] = (unsigned short)(v >> 16);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        bf16x4 z3[4], z2[4], z1[4];  // gradients of the hidden pre-activations
        {
            const bf16x4 d0 = ld_col4(t.dy, 4 * g, col), d1 = ld_col4(t.dy, 16 + 4 * g, col),
                         d2 = ld_col4(t.dy, 32 + 4 * g, col);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f32x4 acc = mfma_w(t.w4t + 64 * (2 * k), d0, d1, zero);
                acc = mfma_w(t.w4t + 64 * (2 * k + 1), d2, bf16x4{0, 0, 0, 0}, acc);
                z3[k] = relu_grad(acc, h3[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f32x4 acc = zero;
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = mfma_w(t.w3t + 64 * (2 * k + p), z3[2 * p], z3[2 * p + 1], acc);
                z2[k] = relu_grad(acc, h2[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f32x4 acc = zero;
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = mfma_w(t.w2t + 64 * (2 * k + p), z2[2 * p], z2[2 * p + 1], acc);
                z1[k] = relu_grad(acc, h1[k]);
            }
        }
        __syncthreads();  // activations and dy of the whole tile lie in LDS; y has been read
#pragma unroll
        for (int k = 0; k < 4; ++k) st_col4(t.dz, 16 * k + 4 * g, col, z3[k]);
        if (ot < 3)
            for (int s0 = 0; s0 < kTrainTile; s0 += 32)
                for (int k = 0; k < 2; ++k) g4[k] = mfma_rows(t.dy, 16 * ot, t.h3, 16 * (2 * half + k), s0, g4[k]);
        __syncthreads();  // dz3 is there, h3 has been read
#pragma unroll
        for (int k = 0; k < 4; ++k) st_col4(t.h3, 16 * k + 4 * g, col, z2[k]);
        for (int s0 = 0; s0 < kTrainTile; s0 += 32) {
            for (int k = 0; k < 2; ++k) g3[k] = mfma_rows(t.dz, 16 * ot, t.h2, 16 * (2 * half + k), s0, g3[k]);
            if (half == 0) b3 = mfma_row_sums(t.dz, 16 * ot, s0, b3);
        }
        __syncthreads();  // dz2 is there (in h3), h2 has been read
#pragma unroll
        for (int k = 0; k < 4; ++k) st_col4(t.h2, 16 * k + 4 * g, col, z1[k]);
        for (int s0 = 0; s0 < kTrainTile; s0 += 32) {
            for (int k = 0; k < 2; ++k) g2[k] = mfma_rows(t.h3, 16 * ot, t.h1, 16 * (2 * half + k), s0, g2[k]);
            if (half == 0) b2 = mfma_row_sums(t.h3, 16 * ot, s0, b2);
        }
        __syncthreads();  // dz1 is there (in h2)
        for (int s0 = 0; s0 < kTrainTile; s0 += 32) {
            g1 = mfma_rows(t.h2, 16 * ot, x, 16 * half, s0, g1);
            if (half == 0) b1 = mfma_row_sums(t.h2, 16 * ot, s0, b1);
        }
    }
    // the block's partial gradient
    float* out = partial + (size_t)blockIdx.x * kParams;
    auto put = [&](int wofs, int K, int kt, f32x4 v) {
        for (int i = 0; i < 4; ++i) out[wofs + (16 * ot + 4 * g + i) * K + 16 * kt + r] = v[i];
    };
    for (int k = 0; k < 2; ++k) {
        if (ot < 3) put(kW4, kHid, 2 * half + k, g4[k]);
        put(kW3, kHid, 2 * half + k, g3[k]);
        put(kW2, kHid, 2 * half + k, g2[k]);
    }
    put(kW1, kEnc, half, g1);
    if (half == 0 && r == 0)
        for (int i = 0; i < 4; ++i) {
            out[kB3 + 16 * ot + 4 * g + i] = b3[i];
            out[kB2 + 16 * ot + 4 * g + i] = b2[i];
            out[kB1 + 16 * ot + 4 * g + i] = b1[i];
        }
    // output biases and loss: sums over the lanes of one lobe pair, then the waves
    for (int o = 4; o < 64; o <<= 1) {
        for (int i = 0; i < 10; ++i) b4[i] += __shfl_xor(b4[i], o);
        loss += __shfl_xor(loss, o);
    }
    __syncthreads();  // y lies where dz was read
    if (l < 4) {
        for (int i = 0; i < 10; ++i) t.y[wave][10 * part + i] = b4[i];
        if (l == 0) t.y[wave][kOut] = loss;
    }
    __syncthreads();
    if (threadIdx.x <= kOut) {
        float v = 0.0f;
        for (int w = 0; w < kTrainBlock / 64; ++w) v += t.y[w][threadIdx.x];
        if (threadIdx.x < kOut)
            out[kB4 + threadIdx.x] = v;
        else
            atomicAdd(&ctl->loss, v / (float)n);
    } else if (threadIdx.x < kOutP + 1) {
        out[kB4 + threadIdx.x - 1] = 0.0f;  // the padding outputs'
    }
}

// grad = sum of the blocks' partial gradients (grad holds the scaled
// gradient): 64 parameters a block, four threads each, so that 256 partials
// are 64 loads deep instead of 256 (5 instead of 64 us).
__global__ __launch_bounds__(kBlock) void k_train_reduce(const float* __restrict__ partial, uint32_t splits,
                                                         float* __restrict__ grad) {
    __shared__ float part[kBlock / 64][64];
    const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
    float acc = 0.0f;
    if (i < (uint32_t)kParams) {
#pragma unroll 8
        for (uint32_t sp = w; sp < splits; sp += kBlock / 64) acc += partial[(size_t)sp * kParams + i];
    }
    part[w][threadIdx.x & 63] = acc;
    __syncthreads();
    if (w == 0 && i < (uint32_t)kParams)
        grad[i] = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
}

// Start of a step: clears the per-step fields of the control block.
__global__ void k_guide_begin(GuideCtl* ctl) {
    if (threadIdx.x == 0) {
        ctl->wsum = 0.0f;
        ctl->loss = 0.0f;
        ctl->bad = 0u;
    }
}

// ctl->bad = 1 when any gradient entry is not finite (loss-scale overflow)
__global__ __launch_bounds__(kBlock) void k_guide_check(const float* __restrict__ grad, GuideCtl* ctl) {
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < (uint32_t)kParams; i += gridDim.x * kBlock)
        if (!isfinite(grad[i])) atomicOr(&ctl->bad, 1u);
}

// FP32 Adam on the unscaled gradient, skipped when the gradient overflowed or
// the batch carried no weight; refreshes the bf16 copy and clears grad. The
// step number (for the bias corrections) is the count of successful steps + 1.
__global__ __launch_bounds__(kBlock) void k_guide_adam(float* __restrict__ theta, float* __restrict__ m,
                                                       float* __restrict__ v, float* __restrict__ grad,
                                                       unsigned short* __restrict__ wbf, const GuideCtl* ctl,
                                                       float lr) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= (uint32_t)kParams) return;
    if (ctl->bad == 0u && ctl->wsum > 0.0f) {
        const float t = (float)(ctl->steps + 1u);
        const float bc1 = 1.0f - powf(0.9f, t), bc2 = 1.0f - powf(0.99f, t);
        const float g = grad[i] * (1.0f / ctl->scale);
        const float mi = 0.9f * m[i] + 0.1f * g;
        const float vi = 0.99f * v[i] + 0.01f * g * g;
        m[i] = mi;
        v[i] = vi;
        theta[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + 1e-8f);
    }
    wbf[bf_at((int)i)] = f2bf(theta[i]);
    grad[i] = 0.0f;
}

// End of a step: counters, last loss, and the loss scale halved on overflow.
__global__ void k_guide_post(GuideCtl* ctl, uint32_t n) {
    if (threadIdx.x != 0) return;
    if (ctl->bad == 0u && ctl->wsum > 0.0f) {
        ctl->steps += 1u;
        ctl->trained += n;
        ctl->last_loss = ctl->loss;
    } else {
        ctl->skipped += 1u;
        if (ctl->bad) ctl->scale *= 0.5f;
    }
}

__global__ void k_guide_tobf16(const float* __restrict__ theta, unsigned short* __restrict__ wbf) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (uint32_t)kParams) wbf[bf_at((int)i)] = f2bf(theta[i]);
}

size_t eval_lds_bytes() { return sizeof(FwdWeights) + sizeof(WaveStage) * (kBlock / 64); }

// The inference and training kernels use more than the default 64 KiB of
// dynamic LDS (gfx950 has 160 KiB per CU).
spt_status allow_lds(spt_ctx* ctx) {
    static bool done = false;
    if (done) return SPT_OK;
    spt_status s = check_hip(ctx,
                             hipFuncSetAttribute(reinterpret_cast<const void*>(&k_train_grad),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(TrainLds)),
                             "training LDS size");
    if (s == SPT_OK)
        s = check_hip(ctx,
                      hipFuncSetAttribute(reinterpret_cast<const void*>(&k_guide_eval),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)eval_lds_bytes()),
                      "eval LDS size");
    done = (s == SPT_OK);
    return s;
}

// Queues the gradient of one step (ctl->wsum and ctl->loss, grad = scaled
// gradient) on the context stream.
spt_status queue_gradient(spt_ctx* ctx, const float* d_rec, uint32_t n, uint32_t rs, hipEvent_t e0, hipEvent_t e1) {
    GuideState& gs = ctx->guide;
    hipStream_t st = ctx->stream;
    GuideCtl* ctl = gs.ctl();
    const uint32_t blocks = std::min<uint32_t>((n + kTrainTile - 1) / kTrainTile, (uint32_t)ctx->num_cus);
    const size_t need = (size_t)blocks * kParams * sizeof(float);  // the blocks' partial gradients
    if (need > gs.scratch_bytes) {
        spt_status s = stream_wait(ctx, "guide scratch");
        if (s != SPT_OK) return s;
        if (gs.d_scratch) (void)hipFree(gs.d_scratch);
        gs.d_scratch = nullptr;
        gs.scratch_bytes = 0;
        s = check_hip(ctx, hipMalloc(&gs.d_scratch, need), "guide scratch");
        if (s != SPT_OK) return s;
        gs.scratch_bytes = need;
    }
    float* partial = reinterpret_cast<float*>(gs.d_scratch);
    hipLaunchKernelGGL(k_guide_wsum, dim3(std::min<uint32_t>((n + kBlock - 1) / kBlock, 256)), dim3(kBlock), 0, st, d_rec, n,
                       rs, &ctl->wsum);
    if (e0) (void)hipEventRecord(e0, st);
    hipLaunchKernelGGL(k_train_grad, dim3(blocks), dim3(kTrainBlock), sizeof(TrainLds), st, gs.d_theta, gs.d_wbf, d_rec,
                       n, rs, ctl, guide_box(ctx), partial);
    hipLaunchKernelGGL(k_train_reduce, dim3((kParams + 63) / 64), dim3(kBlock), 0, st, partial, blocks, gs.d_grad);
    if (e1) (void)hipEventRecord(e1, st);
    return check_hip(ctx, hipGetLastError(), "guide gradient launch");
}

}  // namespace

GuideBox guide_box(const spt_ctx* ctx) {
    GuideBox b;
    for (int i = 0; i < 3; ++i) {
        b.bmin[i] = ctx->root_box[i];
        b.bext[i] = fmaxf(ctx->root_box[3 + i] - ctx->root_box[i], 1e-6f);
    }
    return b;
}

spt_status guide_eval_launch(spt_ctx* ctx, const float* d_q, uint32_t stride, uint32_t n, float* d_out) {
    GuideState& gs = ctx->guide;
    spt_status ls = allow_lds(ctx);
    if (ls != SPT_OK) return ls;
    const uint32_t grid = std::min<uint32_t>((n + kBlock - 1) / kBlock, (uint32_t)ctx->num_cus * 3);
    hipLaunchKernelGGL(k_guide_eval, dim3(grid), dim3(kBlock), eval_lds_bytes(), ctx->stream, gs.d_theta, gs.d_wbf,
                       d_q, stride, n, d_out, guide_box(ctx));
    return check_hip(ctx, hipGetLastError(), "guide eval launch");
}

spt_status guide_train_launch(spt_ctx* ctx, const float* d_rec, uint32_t n, float* loss_out, uint32_t rs) {
    GuideState& gs = ctx->guide;
    spt_status ls = allow_lds(ctx);
    if (ls != SPT_OK) return ls;
    auto t0 = std::chrono::steady_clock::now();
    hipStream_t st = ctx->stream;
    GuideCtl* ctl = gs.ctl();
    hipLaunchKernelGGL(k_guide_begin, dim3(1), dim3(64), 0, st, ctl);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (!gs.event_pair(e0, e1)) e0 = e1 = nullptr;
    spt_status qs = queue_gradient(ctx, d_rec, n, rs, e0, e1);
    if (qs != SPT_OK) return qs;
    hipLaunchKernelGGL(k_guide_check, dim3(64), dim3(kBlock), 0, st, gs.d_grad, ctl);
    hipLaunchKernelGGL(k_guide_adam, dim3((kParams + kBlock - 1) / kBlock), dim3(kBlock), 0, st, gs.d_theta, gs.d_m,
                       gs.d_v, gs.d_grad, gs.d_wbf, ctl, gs.lr);
    hipLaunchKernelGGL(k_guide_post, dim3(1), dim3(64), 0, st, ctl, n);
    spt_status s = check_hip(ctx, hipGetLastError(), "guide train launch");
    if (s == SPT_OK && loss_out) {  // only a caller that wants the loss waits for it
        GuideCtl h;
        s = read_small(ctx, &h, ctl, sizeof(h), "guide step");
        if (s == SPT_OK) *loss_out = h.loss;
    }
    gs.train_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return s;
}

spt_status guide_grad_launch(spt_ctx* ctx, const float* d_rec, uint32_t n, float* grad_out, float* loss_out) {
    GuideState& gs = ctx->guide;
    spt_status ls = allow_lds(ctx);
    if (ls != SPT_OK) return ls;
    hipStream_t st = ctx->stream;
    GuideCtl* ctl = gs.ctl();
    hipLaunchKernelGGL(k_guide_begin, dim3(1), dim3(64), 0, st, ctl);
    spt_status s = queue_gradient(ctx, d_rec, n, 1u, nullptr, nullptr);
    if (s != SPT_OK) return s;
    GuideCtl h;
    s = read_small(ctx, grad_out, gs.d_grad, kParams * sizeof(float), "guide grad", &h, ctl, sizeof(h));
    if (s != SPT_OK) return s;
    for (int i = 0; i < kParams; ++i) grad_out[i] /= h.scale;
    if (loss_out) *loss_out = h.loss;
    return check_hip(ctx, hipMemsetAsync(gs.d_grad, 0, kParams * sizeof(float), st), "guide grad clear");
}

}  // namespace spt

using namespace spt;

namespace {

uint64_t sm64(uint64_t& s) {
    s += 0x9E3779B97F4A7C15ull;
    uint64_t z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

spt_status upload_theta(spt_ctx* ctx, const float* theta) {
    GuideState& gs = ctx->guide;
    spt_status s = check_hip(ctx, hipMemcpy(gs.d_theta, theta, kParams * sizeof(float), hipMemcpyHostToDevice), "theta");
    if (s != SPT_OK) return s;
    (void)hipMemset(gs.d_m, 0, kParams * sizeof(float));
    (void)hipMemset(gs.d_v, 0, kParams * sizeof(float));
    (void)hipMemset(gs.d_grad, 0, kParams * sizeof(float));
    hipLaunchKernelGGL(k_guide_tobf16, dim3((kParams + 255) / 256), dim3(256), 0, ctx->stream, gs.d_theta, gs.d_wbf);
    // fresh moments: step count and statistics restart; the loss scale is the configured one
    GuideCtl c{};
    c.scale = gs.loss_scale;
    s = check_hip(ctx, hipMemcpyAsync(gs.ctl(), &c, sizeof(c), hipMemcpyHostToDevice, ctx->stream), "guide control");
    if (s == SPT_OK) s = stream_wait(ctx, "guide upload");
    return s;
}

}  // namespace

extern "C" {

spt_status spt_guide_init(spt_ctx* ctx, const spt_guide_config* cfg) {
    if (!ctx) return SPT_ERR_INVALID;
    spt_guide_config c{};
    c.seed = 1;
    c.learning_rate = 5e-3f;
    c.loss_scale = 65536.0f;
    c.bsdf_fraction = 0.5f;
    c.batch = 262144;
    c.steps_per_pass = 1;
    if (cfg) c = *cfg;
    if (c.steps_per_pass == 0) c.steps_per_pass = 1;
    if (!(c.bsdf_fraction > 0.0f && c.bsdf_fraction < 1.0f) || c.batch == 0 || !(c.learning_rate > 0.0f) ||
        !(c.loss_scale > 0.0f) || c.steps_per_pass > 64 || (uint64_t)c.batch * c.steps_per_pass >= (1ull << 31) ||
        (c.flags & ~(SPT_GUIDE_COATED | SPT_GUIDE_PRODUCT)))
        return set_error(ctx, SPT_ERR_INVALID, "guide config out of range");
    const uint32_t cap = c.batch * c.steps_per_pass;
    GuideState& gs = ctx->guide;
    if (!gs.d_theta) {
        void* p = nullptr;
        const size_t bytes = (size_t)kParams * (4 * 4 + 2) + 256;
        spt_status s = check_hip(ctx, hipMalloc(&p, bytes), "guide state");
        if (s != SPT_OK) return s;
        char* b = reinterpret_cast<char*>(p);
        gs.d_theta = reinterpret_cast<float*>(b);
        gs.d_m = gs.d_theta + kParams;
        gs.d_v = gs.d_m + kParams;
        gs.d_grad = gs.d_v + kParams;
        gs.d_acc = gs.d_grad + kParams;
        gs.d_wbf = reinterpret_cast<unsigned short*>(gs.d_acc + 64);
    }
    if (gs.records_alloc < cap) {
        if (gs.d_records) (void)hipFree(gs.d_records);
        gs.d_records = nullptr;
        gs.records_alloc = 0;
        spt_status s = check_hip(ctx, hipMalloc(&gs.d_records, (size_t)cap * kRecord * sizeof(float) + 256),
                                 "guide records");
        if (s != SPT_OK) return s;
        gs.records_alloc = cap;
    }
    gs.records_cap = cap;
    gs.lr = c.learning_rate;
    gs.loss_scale = c.loss_scale;
    gs.bsdf_fraction = c.bsdf_fraction;
    gs.flags = c.flags;
    gs.train_every = c.train_every;
    gs.batch = c.batch;
    gs.train_ms = 0.0;
    gs.kernel_ms = 0.0;
    gs.candidates = 0;
    gs.rec_stride = 1;
    gs.cand_per_path = 0.0;
    gs.collected = 0;
    gs.settle_events();
    // Uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) weights, zero biases; output
    // layer scaled by 0.1 so the first mixtures are broad.
    std::vector<float> th(kParams, 0.0f);
    uint64_t s = c.seed;
    auto unif = [&](float lim) { return (float)(((sm64(s) >> 11) * (1.0 / 9007199254740992.0)) * 2.0 - 1.0) * lim; };
    for (int i = 0; i < kHid * kEnc; ++i) th[kW1 + i] = unif(1.0f / std::sqrt((float)kEnc));
    for (int i = 0; i < kHid * kHid; ++i) th[kW2 + i] = unif(1.0f / 8.0f);
    for (int i = 0; i < kHid * kHid; ++i) th[kW3 + i] = unif(1.0f / 8.0f);
    for (int i = 0; i < kOut * kHid; ++i) th[kW4 + i] = 0.1f * unif(1.0f / 8.0f);
    gs.ready = true;
    return upload_theta(ctx, th.data());
}

spt_status spt_guide_set_params(spt_ctx* ctx, const float* theta) {
    if (!ctx || !theta) return SPT_ERR_INVALID;
    if (!ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    std::vector<float> th(theta, theta + kParams);
    for (int i = kOut * kHid; i < kOutP * kHid; ++i) th[kW4 + i] = 0.0f;  // padding rows stay zero
    for (int i = kOut; i < kOutP; ++i) th[kB4 + i] = 0.0f;
    return upload_theta(ctx, th.data());
}

spt_status spt_guide_get_params(spt_ctx* ctx, float* theta) {
    if (!ctx || !theta) return SPT_ERR_INVALID;
    if (!ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    return check_hip(ctx, hipMemcpy(theta, ctx->guide.d_theta, kParams * sizeof(float), hipMemcpyDeviceToHost),
                     "theta read");
}

spt_status spt_guide_eval(spt_ctx* ctx, const float* d_queries, uint64_t n, float* d_out) {
    if (!ctx || (n && (!d_queries || !d_out)) || n >= (1ull << 32)) return SPT_ERR_INVALID;
    if (!ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    if (!ctx->has_scene) return set_error(ctx, SPT_ERR_STATE, "the encoding needs the scene box: upload a scene");
    if (n == 0) return SPT_OK;
    return guide_eval_launch(ctx, d_queries, 9, (uint32_t)n, d_out);
}

spt_status spt_guide_train(spt_ctx* ctx, const float* d_records, uint32_t n, float* loss) {
    if (!ctx || !d_records || n == 0) return SPT_ERR_INVALID;
    if (!ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    if (!ctx->has_scene) return set_error(ctx, SPT_ERR_STATE, "the encoding needs the scene box: upload a scene");
    return guide_train_launch(ctx, d_records, n, loss, 1u);
}

spt_status spt_guide_gradient(spt_ctx* ctx, const float* d_records, uint32_t n, float* grad, float* loss) {
    if (!ctx || !d_records || n == 0 || !grad) return SPT_ERR_INVALID;
    if (!ctx->guide.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    if (!ctx->has_scene) return set_error(ctx, SPT_ERR_STATE, "the encoding needs the scene box: upload a scene");
    return guide_grad_launch(ctx, d_records, n, grad, loss);
}

spt_status spt_guide_train_collected(spt_ctx* ctx, float* loss) {
    if (!ctx) return SPT_ERR_INVALID;
    GuideState& gs = ctx->guide;
    if (!gs.ready) return set_error(ctx, SPT_ERR_STATE, "spt_guide_init first");
    if (gs.collected == 0) {
        if (loss) *loss = 0.0f;
        return SPT_OK;
    }
    const uint32_t n = (uint32_t)std::min<uint64_t>(gs.collected, gs.records_cap);
    spt_status s = SPT_OK;
    // one step per batch (a remainder shorter than half a batch is spread over
    // the others); step k takes records k, k + steps, k + 2 steps, ...: the
    // records were appended in shading order, grouped by material and region,
    // and interleaved batches sample the whole pass
    const uint32_t steps = std::max<uint32_t>(1, n / gs.batch + ((n % gs.batch) >= gs.batch / 2 ? 1u : 0u));
    for (uint32_t k = 0; k < steps && s == SPT_OK; ++k) {
        const uint32_t len = (n - k + steps - 1) / steps;
        s = guide_train_launch(ctx, gs.d_records + (size_t)k * kRecord, len, k + 1 == steps ? loss : nullptr, steps);
    }
    gs.collected = 0;
    return s;
}

spt_status spt_guide_get_stats(spt_ctx* ctx, spt_guide_stats* out) {
    if (!ctx || !out) return SPT_ERR_INVALID;
    GuideState& gs = ctx->guide;
    GuideCtl h{};
    if (gs.ready) {
        spt_status s = read_small(ctx, &h, gs.ctl(), sizeof(h), "guide stats");
        if (s != SPT_OK) return s;
        gs.settle_events();
    } else {
        h.scale = gs.loss_scale;
    }
    out->steps = h.steps;
    out->skipped_steps = h.skipped;
    out->records = gs.collected;
    out->last_loss = h.last_loss;
    out->loss_scale = h.scale;
    out->train_ms = gs.train_ms;
    out->train_kernel_ms = gs.kernel_ms;
    out->trained_records = h.trained;
    out->candidates = gs.candidates;
    out->record_stride = gs.rec_stride;
    out->pad = 0;
    return SPT_OK;
}

spt_status spt_guide_records(spt_ctx* ctx, float** d_records, uint32_t* n) {
    if (!ctx || !d_records || !n) return SPT_ERR_INVALID;
    *d_records = ctx->guide.d_records;
    *n = (uint32_t)std::min<uint64_t>(ctx->guide.collected, ctx->guide.records_cap);
    return SPT_OK;
}

}  // extern "C"
