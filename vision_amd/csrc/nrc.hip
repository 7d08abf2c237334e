// Radiance-cache kernels for gfx950: rendering with early termination into
// the cache, training paths, the MLP forward (inference) and backward on
// BF16 MFMA tiles, Adam.
#include <hip/hip_runtime.h>

#include "dev_nrc.h"
#include "dev_pt.h"
#include "nrc.h"

#include <algorithm>
#include <cstddef>

namespace vs {

using namespace dev;

namespace {

constexpr int kBlock = 256;// 4 waves
constexpr uint32_t kTrainStream = 1u << 30;

// The rows of a launch: the min(*count, cap) (or cap) present from `offset` on,
// the offset taken modulo that number, at most `batch`
__device__ __forceinline__ uint32_t nrc_rows(const uint32_t *count, uint32_t cap, uint32_t &offset, uint32_t batch) {
    const uint32_t total = count ? min(*count, cap) : cap;
    if (total) offset %= total;
    return min(total - (total ? offset : 0u), batch);
}

// Between a wave's stores to LDS and its other lanes' loads of them, and back.
// The hardware carries out a wave's LDS accesses in order; the fences (no
// instruction at this scope) keep the compiler to it, for which the barrier
// alone is no memory access.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// per-wave LDS of the forward-only kernels: one 16-row tile at a time
// (features, two hidden buffers used in turn, outputs), so that twelve
// waves per CU fit beside the block's weights
struct NrcFwdLds {
    uint16_t x[16 * kXs];
    uint16_t h[2][16 * kHs];
    float y[16 * 4];
};

// forward of one row tile, the hidden buffers reused: H3 overwrites H1 once
// layer 2 has read it
__device__ __forceinline__ void fwd_tile(const NrcWeightsLds &w, NrcFwdLds &s, int lane) {
    nrc_fwd_tile<kNrcIn, kNrcHidden>(s.x, kXs, w.w1t, kXs, s.h[0], lane);
    wave_lds_sync();
    nrc_fwd_tile<kNrcHidden, kNrcHidden>(s.h[0], kHs, w.w2t, kHs, s.h[1], lane);
    wave_lds_sync();
    nrc_fwd_tile<kNrcHidden, kNrcHidden>(s.h[1], kHs, w.w3t, kHs, s.h[0], lane);
    wave_lds_sync();
    nrc_out_tile(s.h[0], w.w4, s.y, lane);
    wave_lds_sync();
}

// Features of the rows [first, first + span) of a list of positions, `stride`
// floats apart, `count` (on the device, when given; at most cap) or cap of them
// in all: feat[level][row - first], two bf16 a word.
// A wave takes Q x 64 rows and goes through the levels in the outer loop, so
// that the whole GPU gathers from about one level's table (2 MB of 32) at a
// time: it stays in every XCD's L2, and the coarse ones in L1.  With a row's
// levels one after the other the gathers missed L2 half the time and ran at
// the Infinity Cache's bandwidth (7.5 TB/s): a full-HD frame's queries took
// 1.92 ms, now 1.15 ms with the network.
template <int Q>
__global__ void __launch_bounds__(kBlock) nrc_encode_kernel(NrcView v, const float *__restrict__ pos, uint32_t stride,
                                                            const uint32_t *__restrict__ count, uint32_t cap,
                                                            uint32_t offset, uint32_t batch, uint32_t first,
                                                            uint32_t span, uint32_t *__restrict__ feat) {
    const uint32_t n = nrc_rows(count, cap, offset, batch);
    const uint32_t end = min(n, first + span);
    const uint32_t base = first + (blockIdx.x * kBlock + (threadIdx.x & ~63u)) * Q + (threadIdx.x & 63u);
    if (first + blockIdx.x * kBlock * Q >= end) return;
    float u[Q][3];
#pragma unroll
    for (int j = 0; j < Q; ++j) {
        float p[3] = {0.f, 0.f, 0.f};
        const uint32_t row = base + 64u * j;
        if (row < end) {
            const float *src = pos + size_t(offset + row) * stride;
            p[0] = src[0];
            p[1] = src[1];
            p[2] = src[2];
        }
        nrc_unit(v, p, u[j]);
    }
    const uint32_t *table = reinterpret_cast<const uint32_t *>(v.grid_f16);
#pragma unroll 1
    for (int l = 0; l < kNrcLevels; ++l, table += kNrcTable) {
        const bool dense = (v.dense_mask >> l) & 1u;
#pragma unroll
        for (int j = 0; j < Q; ++j) {
            const uint32_t row = base + 64u * j;
            if (row >= end) continue;
            float a0, a1;
            if (dense) nrc_level<true>(table, v.res[l], u[j], a0, a1);
            else nrc_level<false>(table, v.res[l], u[j], a0, a1);
            feat[size_t(l) * span + (row - first)] = uint32_t(f2bf(a0)) | uint32_t(f2bf(a1)) << 16;
        }
    }
}

// The network over encoded rows.  INFER: rows are queries (count on the
// device), their radiance goes into L; otherwise outputs go to out[row][3]
template <bool INFER>
__global__ void __launch_bounds__(kBlock) nrc_forward_kernel(NrcView v, const uint32_t *__restrict__ feat,
                                                             const NrcQuery *__restrict__ q,
                                                             const uint32_t *__restrict__ count, uint32_t cap,
                                                             uint32_t first, uint32_t span, float *__restrict__ out,
                                                             float4 *__restrict__ L) {
    __shared__ NrcWeightsLds w;
    __shared__ NrcFwdLds ws[kBlock / 64];
    const uint32_t n = INFER ? min(*count, cap) : cap;
    const uint32_t end = min(n, first + span);
    if (first + blockIdx.x * kBlock >= end) return;
    nrc_load_weights<kBlock>(v, w, nullptr, threadIdx.x);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    NrcFwdLds &s = ws[wave];
    for (uint32_t base = first + (blockIdx.x * (kBlock / 64) + wave) * 64u; base < end; base += gridDim.x * kBlock) {
        const uint32_t row = base + lane;
        const bool valid = row < end;
        uint32_t x[kNrcLevels];
#pragma unroll
        for (int l = 0; l < kNrcLevels; ++l) x[l] = valid ? feat[size_t(l) * span + (row - first)] : 0u;
        for (int rt = 0; rt < 4; ++rt) {
            if ((lane >> 4) == rt) {
#pragma unroll
                for (int l = 0; l < kNrcLevels; l += 2)
                    *reinterpret_cast<uint2 *>(s.x + (lane & 15) * kXs + 2 * l) = make_uint2(x[l], x[l + 1]);
            }
            wave_lds_sync();
            fwd_tile(w, s, lane);
            if ((lane >> 4) == rt && valid) {
                const int i = lane & 15;
                float y0 = s.y[i * 4], y1 = s.y[i * 4 + 1], y2 = s.y[i * 4 + 2];
                if (INFER) {
                    const NrcQuery &qq = q[row];
                    float4 l = L[qq.slot];
                    l.x += qq.beta[0] * fmaxf(y0, 0.f);
                    l.y += qq.beta[1] * fmaxf(y1, 0.f);
                    l.z += qq.beta[2] * fmaxf(y2, 0.f);
                    L[qq.slot] = l;
                } else {
                    out[3 * size_t(row)] = y0;
                    out[3 * size_t(row) + 1] = y1;
                    out[3 * size_t(row) + 2] = y2;
                }
            }
            wave_lds_sync();
        }
    }
}

// The network forward and backward over encoded training samples, rows
// [first, first + span) of the step's; the features' gradients go to
// dx[row - first][32].  A wave takes 16 rows at a time.  The weight gradients
// stay in MFMA accumulators over all rows of a wave and meet in LDS once (added
// to LDS tile by tile they were 2300 LDS atomics a wave), and a layer's
// gradient overwrites its activations, so that eight waves fit beside the
// weights.  Blocks hand their sums to nrc_reduce_kernel: 256 blocks' atomics on
// the same 10432 parameters took 100 of 135 us.
// A step's gradients for 65536 samples took 1030 us in one kernel of four waves
// a CU that also gathered and scattered a row a lane; now 430 us: encoding
// 29, this and the reduction 135, scatter 220 to 265.
constexpr int kBackWaves = 8;
constexpr int kBackBlock = 64 * kBackWaves;
struct NrcBackWaveLds {
    uint16_t x[16 * kXs];   // features of the tile
    uint16_t h[3][16 * kHs];// H1..H3 (post-ReLU), then the gradients there
    float y[16 * 4];        // outputs, then dL/dy
};
struct NrcGradLds {
    float w1[kNrcIn * kNrcHidden];
    float w2[kNrcHidden * kNrcHidden];
    float w3[kNrcHidden * kNrcHidden];
    float w4[kNrcHidden * kNrcOut];
    float loss;
};
static_assert(offsetof(NrcGradLds, loss) == sizeof(float) * kNrcMlpParams && kNrcW1 == 0, "layers in parameter order");

__global__ void __launch_bounds__(kBackBlock) nrc_backward_kernel(NrcView v, const NrcSample *__restrict__ samples,
                                                                  const uint32_t *__restrict__ feat,
                                                                  const uint32_t *__restrict__ count, uint32_t cap,
                                                                  uint32_t offset, uint32_t batch, uint32_t first,
                                                                  uint32_t span, float *__restrict__ dx,
                                                                  float *__restrict__ partial) {
    __shared__ NrcWeightsLds w;
    __shared__ NrcBackWeightsLds wb;
    __shared__ union {
        NrcBackWaveLds wave[kBackWaves];
        NrcGradLds grad;// once the waves are through
    } sh;
    const uint32_t n = nrc_rows(count, cap, offset, batch);
    const uint32_t end = min(n, first + span);
    partial += size_t(blockIdx.x) * kNrcPartial;
    if (first + blockIdx.x * uint32_t(kBackWaves * 16) >= end) {
        for (int i = threadIdx.x; i < kNrcPartial; i += kBackBlock) partial[i] = 0.f;
        return;
    }
    samples += offset;
    nrc_load_weights<kBackBlock>(v, w, &wb, threadIdx.x);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    NrcBackWaveLds &s = sh.wave[wave];
    const float inv = 1.f / (3.f * float(n));
    float loss_acc = 0.f;
    f32x4 g1[kNrcIn / 16][4] = {}, g2[4][4] = {}, g3[4][4] = {};
    float g4[3] = {0.f, 0.f, 0.f};
    const float w4r[3] = {w.w4[lane * 3], w.w4[lane * 3 + 1], w.w4[lane * 3 + 2]};
    const uint32_t step = gridDim.x * uint32_t(kBackWaves * 16);
    for (uint32_t base = first + (blockIdx.x * kBackWaves + wave) * 16u; base < end; base += step) {
        // lane: row of 16 x a quarter of the levels
        const int i = lane & 15;
        const bool valid = base + i < end;
        const uint32_t present = uint32_t(__ballot(valid)) & 0xFFFFu;
#pragma unroll
        for (int k = 0; k < kNrcLevels / 4; ++k) {
            const int l = (lane >> 4) * (kNrcLevels / 4) + k;
            const uint32_t f = valid ? feat[size_t(l) * span + (base + i - first)] : 0u;
            // a vector type, which may alias: nrc_weight_grad reads the tile as uint16_t
            *reinterpret_cast<bf16x2 *>(s.x + i * kXs + 2 * l) = __builtin_bit_cast(bf16x2, f);
        }
        wave_lds_sync();
        nrc_fwd_tile<kNrcIn, kNrcHidden>(s.x, kXs, w.w1t, kXs, s.h[0], lane);
        wave_lds_sync();
        nrc_fwd_tile<kNrcHidden, kNrcHidden>(s.h[0], kHs, w.w2t, kHs, s.h[1], lane);
        wave_lds_sync();
        nrc_fwd_tile<kNrcHidden, kNrcHidden>(s.h[1], kHs, w.w3t, kHs, s.h[2], lane);
        wave_lds_sync();
        nrc_out_tile(s.h[2], w.w4, s.y, lane);
        wave_lds_sync();
        if (lane < 16) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float t = valid ? samples[base + i].t[c] : 0.f;
                const float y = s.y[i * 4 + c];
                const float d = y - t;
                const float den = y * y + 0.01f;
                loss_acc += valid ? d * d / den * inv : 0.f;
                s.y[i * 4 + c] = valid ? 2.f * d / den * inv : 0.f;
            }
        }
        wave_lds_sync();
        // output layer: dW4[k][c] = sum_rows h3[row][k] dy[row][c]; G3 = dy W4^T x relu'(h3)
#pragma unroll 4
        for (int row = 0; row < 16; ++row) {
            const float hv = bf2f(s.h[2][row * kHs + lane]);
            const float y0 = s.y[row * 4], y1 = s.y[row * 4 + 1], y2 = s.y[row * 4 + 2];
            g4[0] += hv * y0;
            g4[1] += hv * y1;
            g4[2] += hv * y2;
            const float gs = y0 * w4r[0] + y1 * w4r[1] + y2 * w4r[2];
            s.h[2][row * kHs + lane] = f2bf(hv > 0.f ? gs : 0.f);
        }
        wave_lds_sync();
        nrc_weight_grad<kNrcHidden>(s.h[1], kHs, s.h[2], g3, lane);             // dW3 = H2^T G3
        wave_lds_sync();
        nrc_input_grad<kNrcHidden>(s.h[2], wb.w3, s.h[1], nullptr, 0u, lane);   // G2
        wave_lds_sync();
        nrc_weight_grad<kNrcHidden>(s.h[0], kHs, s.h[1], g2, lane);             // dW2 = H1^T G2
        wave_lds_sync();
        nrc_input_grad<kNrcHidden>(s.h[1], wb.w2, s.h[0], nullptr, 0u, lane);   // G1
        wave_lds_sync();
        nrc_weight_grad<kNrcIn>(s.x, kXs, s.h[0], g1, lane);                    // dW1 = X^T G1
        nrc_input_grad<kNrcIn>(s.h[0], wb.w1, nullptr, dx + size_t(base - first) * kNrcIn, present, lane);// dX
        wave_lds_sync();
    }
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off);
    __syncthreads();
    NrcGradLds &gl = sh.grad;
    float *flat = gl.w1;
    for (int i = threadIdx.x; i < kNrcPartial; i += kBackBlock) flat[i] = 0.f;
    __syncthreads();
    if (lane == 0) atomicAdd(&sh.grad.loss, loss_acc);
    nrc_add_weight_grad<kNrcIn>(g1, gl.w1, lane);
    nrc_add_weight_grad<kNrcHidden>(g2, gl.w2, lane);
    nrc_add_weight_grad<kNrcHidden>(g3, gl.w3, lane);
    for (int c = 0; c < 3; ++c) atomicAdd(gl.w4 + lane * 3 + c, g4[c]);
    __syncthreads();
    for (int i = threadIdx.x; i < kNrcPartial; i += kBackBlock) partial[i] = flat[i];
}

// the blocks' weight gradients and losses added to v.mlp_g and *loss: 32
// parameters a block, eight lanes' sums each
__global__ void __launch_bounds__(kBlock) nrc_reduce_kernel(NrcView v, const float *__restrict__ partial,
                                                            uint32_t blocks, float *__restrict__ loss) {
    __shared__ float sum[8][32];
    const uint32_t c = threadIdx.x & 31u, part = threadIdx.x >> 5, i = blockIdx.x * 32u + c;
    float acc = 0.f;
    if (i < uint32_t(kNrcPartial)) {
#pragma unroll 8
        for (uint32_t b = part; b < blocks; b += 8u) acc += partial[size_t(b) * kNrcPartial + i];
    }
    sum[part][c] = acc;
    __syncthreads();
    if (part == 0 && i < uint32_t(kNrcPartial)) {
        for (int k = 1; k < 8; ++k) acc += sum[k][c];
        if (i < uint32_t(kNrcMlpParams)) v.mlp_g[i] += acc;
        else *loss += acc;
    }
}

// The features' gradients dx[row - first][32] into the grid's.  Lane = row 4 x
// corner 8 x feature 2: a corner's two features, and mostly the corners along
// x, are neighbours in memory, so the 64 atomics of an instruction touch some
// 20 lines, and the atomics, which are carried out at the memory side, bound
// this.  Each wave starts at a level of its own, which spreads the atomics on
// the few entries of the coarse levels over time.
__global__ void __launch_bounds__(kBlock) nrc_scatter_kernel(NrcView v, const NrcSample *__restrict__ samples,
                                                             const uint32_t *__restrict__ count, uint32_t cap,
                                                             uint32_t offset, uint32_t batch, uint32_t first,
                                                             uint32_t span, const float *__restrict__ dx) {
    __shared__ uint32_t res[kNrcLevels];
    if (threadIdx.x < kNrcLevels) res[threadIdx.x] = v.res[threadIdx.x];
    __syncthreads();
    const uint32_t n = nrc_rows(count, cap, offset, batch);
    const uint32_t end = min(n, first + span);
    const int lane = threadIdx.x & 63;
    const uint32_t wave = blockIdx.x * (kBlock / 64) + threadIdx.x / 64;
    const uint32_t row = first + wave * 4u + uint32_t(lane >> 4);
    if (row >= end) return;
    const int ft = lane & 1, k = (lane >> 1) & 7;
    float u[3];
    nrc_unit(v, samples[offset + row].p, u);
    const float *d = dx + size_t(row - first) * kNrcIn;
#pragma unroll 4
    for (int i = 0; i < kNrcLevels; ++i) {
        const int l = (i + int(wave)) & (kNrcLevels - 1);
        const float d0 = d[2 * l], d1 = d[2 * l + 1];
        if (d0 == 0.f && d1 == 0.f) continue;
        uint32_t c[3];
        float f[3];
        nrc_cell(res[l], u, c, f);
        float *gg = v.grid_g + size_t(l) * kNrcTable * kNrcFeatures;
        const uint32_t idx = nrc_index((v.dense_mask >> l) & 1u, res[l], c[0] + (k & 1), c[1] + ((k >> 1) & 1),
                                       c[2] + ((k >> 2) & 1));
        atomicAdd(gg + 2 * idx + ft, nrc_corner_weight(k, f) * (ft ? d1 : d0));
    }
}

__device__ __forceinline__ float adam_update(float &p, float &m, float &vv, float &g, float lr, float c1, float c2) {
    const float b1 = 0.9f, b2 = 0.99f, eps = 1e-15f;
    float gr = g;
    m = b1 * m + (1.f - b1) * gr;
    vv = b2 * vv + (1.f - b2) * gr * gr;
    p -= lr * (m * c1) / (sqrtf(vv * c2) + eps);
    g = 0.f;
    return p;
}

// blockIdx.y: a level of the grid, or the network's weights.  Bound by HBM (34 B
// a parameter); the tail of a directly indexed level's table, which no position
// reaches, has no gradient and no moments and is left out (27 % of the table at
// the default resolutions: 112 -> 80 us a step)
__global__ void __launch_bounds__(256) nrc_adam_kernel(NrcView v, float lr, float c1, float c2) {
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    const uint32_t l = blockIdx.y;
    if (l < uint32_t(kNrcLevels)) {
        const size_t n1 = v.res[l] + 1u;
        const size_t used = ((v.dense_mask >> l) & 1u ? n1 * n1 * n1 : size_t(kNrcTable)) * kNrcFeatures;
        const size_t base = size_t(l) * kNrcTable * kNrcFeatures;
        for (size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x; k < used; k += stride) {
            const size_t i = base + k;
            float p = adam_update(v.grid[i], v.grid_m[i], v.grid_v[i], v.grid_g[i], lr, c1, c2);
            v.grid_f16[i] = f2h(p);
        }
    } else {
        for (size_t j = size_t(blockIdx.x) * blockDim.x + threadIdx.x; j < kNrcMlpParams; j += stride) {
            float p = adam_update(v.mlp[j], v.mlp_m[j], v.mlp_v[j], v.mlp_g[j], lr, c1, c2);
            v.mlp_bf16[j] = f2bf(p);
        }
    }
}

__global__ void __launch_bounds__(256) nrc_sync_kernel(NrcView v) {
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < kNrcGridParams + kNrcMlpParams; i += stride) {
        if (i < kNrcGridParams) {
            v.grid_f16[i] = f2h(v.grid[i]);
        } else {
            size_t j = i - kNrcGridParams;
            v.mlp_bf16[j] = f2bf(v.mlp[j]);
        }
    }
}

// lanes with `active` get consecutive slots of *counter (one atomic per wave)
__device__ __forceinline__ uint32_t wave_append(uint32_t *counter, bool active) {
    const uint64_t mask = __ballot(active);
    const uint32_t lane = __lane_id();
    uint32_t base = 0;
    if (mask) {
        const uint32_t leader = uint32_t(__ffsll((unsigned long long)mask) - 1);
        if (lane == leader) base = atomicAdd(counter, uint32_t(__popcll(mask)));
        base = __shfl(base, int(leader));
    }
    return base + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
}

// the cache learns radiance divided by the surface's diffuse albedo (sharp
// colour edges then need no resolution in the grid): the constant albedo of
// diffuse and Oren-Nayar materials, 1 for the others, for textured colours
// and for black surfaces
__device__ __forceinline__ f3 nrc_albedo(const SceneView &sc, uint32_t mat) {
    const MaterialRecord &m = sc.mat[mat];
    if ((m.type == MAT_DIFFUSE || m.type == MAT_OREN_NAYAR) && !(m.flags & MATF_TEXTURE_SLOT0)) {
        f3 a = mk3(m.p[0], m.p[1], m.p[2]);
        if (a.x > 1e-4f && a.y > 1e-4f && a.z > 1e-4f) return a;
    }
    return mk3(1.f, 1.f, 1.f);
}

// the emitter term of a hit, as path_shade adds it (integrator.cpp:188-196)
template <int MS>
__device__ __forceinline__ void emission_at(const SceneView &sc, const RenderView &rv, PathState<3> &ps,
                                            const TraceHit &h, const Surface &it, const InstanceRecord &inst) {
    if (inst.light == kInvalid) return;
    Spec<3> Le;
    float lpdf;
    eval_hit_light<3, true>(sc, it, inst.light, h.tri, ps.o, ps.swl, Le, lpdf);
    float w = mis_weight(ps.scatter_pdf, lpdf);
    if (rv.mis_mode == 2) w = 1.f;
    else if (rv.mis_mode == 1) w = ps.bounce == 0 ? w : 0.f;
    ps.L += to_linear_srgb<3, true>(sc, Le * ps.thr * w, ps.swl);
}

template <int MS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) nrc_render_kernel(SceneView sc, CameraView cam, RenderView rv, uint32_t frame0,
                                                        uint32_t spp, uint32_t term, float4 *__restrict__ L,
                                                        NrcQuery *__restrict__ q, uint32_t *__restrict__ qcount,
                                                        uint32_t qcap) {
    extern __shared__ uint2 lds_stack[];
    const uint32_t px = blockIdx.x * 8u + (threadIdx.x & 7u);
    const uint32_t py = blockIdx.y * 8u + (threadIdx.x >> 3);
    const bool inside = px < cam.width && py < cam.height;
    const uint32_t pix = inside ? py * cam.width + px : 0u;
    uint32_t nf = 0, tf = 0;
    for (uint32_t s = 0; s < spp; ++s) {
        PathState<3> ps;
        path_begin<3, true>(cam, rv, inside ? px : 0u, inside ? py : 0u, frame0 + s, ps);
        if (!inside) ps.alive = 0u;
        bool has_q = false;
        f3 qp = mk3(0.f, 0.f, 0.f), qa = mk3(1.f, 1.f, 1.f);
        while (ps.alive) {
            TraceHit h = traverse<false>(sc, ps.o, ps.d, 0.f, 3.402823466e38f, lds_stack + threadIdx.x, 64u, nf, tf);
            if (term && ps.bounce == term && !ps.tail && h.tri != kInvalid) {
                Surface it = surface_at(sc, h.tri, h.b1, h.b2, false);
                const InstanceRecord inst = sc.inst[it.inst];
                if (inst.mat != kInvalid) {
                    emission_at<MS>(sc, rv, ps, h, it, inst);
                    has_q = true;
                    qp = it.pos;
                    qa = nrc_albedo(sc, inst.mat);
                    ps.alive = 0u;
                    break;
                }
            }
            ShadowRay sr;
            path_shade<3, true, MS>(sc, rv, ps, h, sr);
            if (sr.valid) {
                TraceHit sh = traverse<true>(sc, sr.o, sr.d, 0.f, 1.f - kShadowEpsilon, lds_stack + threadIdx.x, 64u,
                                             nf, tf);
                if (sh.tri == kInvalid) ps.L += sr.c;
            }
        }
        const uint32_t slot = pix * spp + s;
        if (inside) {
            f3 l = ps.L * ps.fw;
            L[slot] = make_float4(l.x, l.y, l.z, 0.f);
        }
        const uint32_t k = wave_append(qcount, has_q);
        if (has_q && k < qcap) {
            NrcQuery &o = q[k];
            o.p[0] = qp.x;
            o.p[1] = qp.y;
            o.p[2] = qp.z;
            o.slot = slot;
            o.beta[0] = ps.thr.v[0] * qa.x * ps.fw;
            o.beta[1] = ps.thr.v[1] * qa.y * ps.fw;
            o.beta[2] = ps.thr.v[2] * qa.z * ps.fw;
            o.pad = 0u;
        }
    }
}

template <int MS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) nrc_train_paths_kernel(SceneView sc, CameraView cam, RenderView rv,
                                                             uint32_t frame, uint32_t stride, uint32_t offset,
                                                             uint32_t n_paths, float *__restrict__ staging,
                                                             NrcSample *__restrict__ out, uint32_t *__restrict__ count,
                                                             uint32_t cap) {
    extern __shared__ uint2 lds_stack[];
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    if (i >= n_paths) return;
    const uint32_t pixel = i * stride + offset;
    const uint32_t px = pixel % cam.width, py = pixel / cam.width;
    if (py >= cam.height) return;
    const uint32_t maxv = rv.max_depth;
    float *st = staging + size_t(i) * maxv * 9u;
    PathState<3> ps;
    path_begin<3, true>(cam, rv, px, py, kTrainStream + frame, ps);
    uint32_t nv = 0, nf = 0, tf = 0;
    while (ps.alive) {
        TraceHit h = traverse<false>(sc, ps.o, ps.d, 0.f, 3.402823466e38f, lds_stack + threadIdx.x, 64u, nf, tf);
        bool record = false;
        f3 pos = mk3(0.f, 0.f, 0.f);
        f3 beta = mk3(ps.thr.v[0], ps.thr.v[1], ps.thr.v[2]);
        if (h.tri != kInvalid && !ps.tail) {
            Surface it = surface_at(sc, h.tri, h.b1, h.b2, false);
            const uint32_t mat = sc.inst[it.inst].mat;
            if (mat != kInvalid) {
                record = true;
                pos = it.pos;
                f3 a = nrc_albedo(sc, mat);
                beta = mk3(beta.x * a.x, beta.y * a.y, beta.z * a.z);
            }
        }
        ShadowRay sr;
        path_shade<3, true, MS>(sc, rv, ps, h, sr);
        if (record && nv < maxv) {
            // the radiance gathered so far includes this vertex's emission
            float *r = st + nv * 9u;
            r[0] = pos.x;
            r[1] = pos.y;
            r[2] = pos.z;
            r[3] = beta.x;
            r[4] = beta.y;
            r[5] = beta.z;
            r[6] = ps.L.x;
            r[7] = ps.L.y;
            r[8] = ps.L.z;
            ++nv;
        }
        if (sr.valid) {
            TraceHit sh = traverse<true>(sc, sr.o, sr.d, 0.f, 1.f - kShadowEpsilon, lds_stack + threadIdx.x, 64u,
                                         nf, tf);
            if (sh.tri == kInvalid) ps.L += sr.c;
        }
    }
    uint32_t good = 0;
    for (uint32_t j = 0; j < nv; ++j) {
        const float *r = st + j * 9u;
        good += (r[3] > 0.f && r[4] > 0.f && r[5] > 0.f) ? 1u : 0u;
    }
    if (!good) return;
    uint32_t k = atomicAdd(count, good);
    for (uint32_t j = 0; j < nv; ++j) {
        const float *r = st + j * 9u;
        if (!(r[3] > 0.f && r[4] > 0.f && r[5] > 0.f)) continue;
        if (k < cap) {
            NrcSample &o = out[k];
            o.p[0] = r[0];
            o.p[1] = r[1];
            o.p[2] = r[2];
            o.t[0] = (ps.L.x - r[6]) / r[3];
            o.t[1] = (ps.L.y - r[7]) / r[4];
            o.t[2] = (ps.L.z - r[8]) / r[5];
        }
        ++k;
    }
}

__global__ void __launch_bounds__(256) nrc_accumulate_kernel(RenderView rv, const float4 *__restrict__ L,
                                                             uint32_t pixels, uint32_t spp, uint32_t frame0,
                                                             float4 *__restrict__ rt, float4 *__restrict__ out) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= pixels) return;
    float4 acc = rt[p];
    for (uint32_t s = 0; s < spp; ++s) {
        float4 l = L[size_t(p) * spp + s];
        acc = film_add(rv, acc, mk3(l.x, l.y, l.z), frame0 + s);
    }
    rt[p] = acc;
    out[p] = film_output(rv, acc);
}

__global__ void nrc_zero_kernel(uint32_t *p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

uint32_t grid_blocks() {
    int dev = 0, cus = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return uint32_t(cus > 0 ? cus : 64);
}

}// namespace

namespace {

// features of rows [first, first + span), sixteen rows a lane from half a
// million on: 1 M rows took 437 us at one row a lane, 381 at four, 344 at eight
// and 270 at sixteen (a wave a SIMD), 65536 rows 29 us at one.  Whole lookups from
// host arrays, at one / eight / sixteen rows: 65536 136 / 277 / 449 us, 200 k 422 /
// 447 / 584, 262144 491 / 503 / 624, 350 k 684 / 656 / 737, 460 k 853 / 765 / 851,
// 524288 937 / 849 / 921, 600 k 1055 / 1142 / 991, 800 k 1434 / 1400 / 1294: one
// and sixteen cross below half a million, and eight rows, not built, would be up
// to a tenth of the call faster from 350 to 530 k.
hipError_t encode(const NrcView &v, const float *pos, uint32_t stride, const uint32_t *count, uint32_t cap,
                  uint32_t offset, uint32_t batch, uint32_t first, uint32_t span, uint32_t *feat, hipStream_t s) {
    if (span >= (1u << 19))
        hipLaunchKernelGGL(nrc_encode_kernel<16>, dim3((span + kBlock * 16 - 1) / (kBlock * 16)), dim3(kBlock), 0, s, v,
                           pos, stride, count, cap, offset, batch, first, span, feat);
    else
        hipLaunchKernelGGL(nrc_encode_kernel<1>, dim3((span + kBlock - 1) / kBlock), dim3(kBlock), 0, s, v, pos,
                           stride, count, cap, offset, batch, first, span, feat);
    return hipGetLastError();
}

uint32_t forward_blocks(uint32_t span) { return std::min<uint32_t>((span + kBlock - 1) / kBlock, 8u * grid_blocks()); }

}// namespace

hipError_t nrc_forward(const NrcView &v, const float *pos, uint32_t n, float *out, const NrcScratch &sc,
                       hipStream_t s) {
    for (uint32_t first = 0, span; first < n; first += span) {
        span = std::min(sc.rows, n - first);
        hipError_t e = encode(v, pos, 3, nullptr, n, 0, n, first, span, sc.feat, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(nrc_forward_kernel<false>, dim3(forward_blocks(span)), dim3(kBlock), 0, s, v, sc.feat,
                           nullptr, nullptr, n, first, span, out, nullptr);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t nrc_infer(const NrcView &v, const NrcQuery *q, const uint32_t *count, uint32_t capacity, float4 *L,
                     const NrcScratch &sc, hipStream_t s) {
    static_assert(sizeof(NrcQuery) == 32 && offsetof(NrcQuery, p) == 0, "query layout");
    for (uint32_t first = 0, span; first < capacity; first += span) {
        span = std::min(sc.rows, capacity - first);
        hipError_t e = encode(v, q->p, 8, count, capacity, 0, capacity, first, span, sc.feat, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(nrc_forward_kernel<true>, dim3(forward_blocks(span)), dim3(kBlock), 0, s, v, sc.feat, q,
                           count, capacity, first, span, nullptr, L);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

uint32_t nrc_backward_blocks() { return grid_blocks(); }

hipError_t nrc_backward(const NrcView &v, const NrcSample *samples, const uint32_t *count, uint32_t capacity,
                        uint32_t offset, uint32_t batch, float *loss, const NrcScratch &sc, hipStream_t s) {
    static_assert(sizeof(NrcSample) == 24 && offsetof(NrcSample, p) == 0, "sample layout");
    const uint32_t rows = std::min(batch, capacity);
    for (uint32_t first = 0, span; first < rows; first += span) {
        span = std::min(sc.rows, rows - first);
        hipError_t e = encode(v, samples->p, 6, count, capacity, offset, batch, first, span, sc.feat, s);
        if (e != hipSuccess) return e;
        const uint32_t blocks = std::min((span + kBackWaves * 16 - 1) / (kBackWaves * 16), grid_blocks());
        hipLaunchKernelGGL(nrc_backward_kernel, dim3(blocks), dim3(kBackBlock), 0, s, v, samples, sc.feat, count,
                           capacity, offset, batch, first, span, sc.dx, sc.partial);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(nrc_reduce_kernel, dim3((kNrcPartial + 31) / 32), dim3(kBlock), 0, s, v, sc.partial, blocks,
                           loss);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        const uint32_t per = 4u * (kBlock / 64);
        hipLaunchKernelGGL(nrc_scatter_kernel, dim3((span + per - 1) / per), dim3(kBlock), 0, s, v, samples, count,
                           capacity, offset, batch, first, span, sc.dx);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t nrc_adam(const NrcView &v, float lr, float c1, float c2, hipStream_t s) {
    hipLaunchKernelGGL(nrc_adam_kernel, dim3(grid_blocks(), kNrcLevels + 1), dim3(256), 0, s, v, lr, c1, c2);
    return hipGetLastError();
}

hipError_t nrc_sync_copies(const NrcView &v, hipStream_t s) {
    hipLaunchKernelGGL(nrc_sync_kernel, dim3(8u * grid_blocks()), dim3(256), 0, s, v);
    return hipGetLastError();
}

hipError_t nrc_render(const SceneView &sc, const CameraView &cam, const RenderView &rv, uint32_t frame0,
                      uint32_t spp, uint32_t term, float4 *L, NrcQuery *q, uint32_t *qcount, uint32_t qcap,
                      bool diffuse_only, hipStream_t s) {
    if (!sc.spectrum_rgb) return hipErrorInvalidValue;
    dim3 grid((cam.width + 7) / 8, (cam.height + 7) / 8);
    size_t lds = size_t(sc.stack_size) * 64 * sizeof(uint2);
    if (diffuse_only)
        hipLaunchKernelGGL(nrc_render_kernel<MS_DIFFUSE>, grid, dim3(64), lds, s, sc, cam, rv, frame0, spp, term, L,
                           q, qcount, qcap);
    else
        hipLaunchKernelGGL(nrc_render_kernel<MS_ALL>, grid, dim3(64), lds, s, sc, cam, rv, frame0, spp, term, L, q,
                           qcount, qcap);
    return hipGetLastError();
}

hipError_t nrc_train_paths(const SceneView &sc, const CameraView &cam, const RenderView &rv, uint32_t frame,
                           uint32_t stride, float *staging, NrcSample *out, uint32_t *count, uint32_t cap,
                           bool diffuse_only, hipStream_t s) {
    if (!sc.spectrum_rgb || !stride || !rv.max_depth) return hipErrorInvalidValue;
    const uint32_t pixels = cam.width * cam.height;
    const uint32_t offset = (frame * 2654435761u >> 8) % stride;
    const uint32_t n_paths = pixels > offset ? (pixels - offset + stride - 1) / stride : 0u;
    if (!n_paths) return hipSuccess;
    size_t lds = size_t(sc.stack_size) * 64 * sizeof(uint2);
    dim3 grid((n_paths + 63) / 64);
    if (diffuse_only)
        hipLaunchKernelGGL(nrc_train_paths_kernel<MS_DIFFUSE>, grid, dim3(64), lds, s, sc, cam, rv, frame, stride,
                           offset, n_paths, staging, out, count, cap);
    else
        hipLaunchKernelGGL(nrc_train_paths_kernel<MS_ALL>, grid, dim3(64), lds, s, sc, cam, rv, frame, stride, offset,
                           n_paths, staging, out, count, cap);
    return hipGetLastError();
}

hipError_t nrc_accumulate(const RenderView &rv, const float4 *L, uint32_t pixels, uint32_t spp, uint32_t frame0,
                          float4 *rt, float4 *out, hipStream_t s) {
    if (!pixels) return hipSuccess;
    hipLaunchKernelGGL(nrc_accumulate_kernel, dim3((pixels + 255) / 256), dim3(256), 0, s, rv, L, pixels, spp, frame0,
                       rt, out);
    return hipGetLastError();
}

hipError_t nrc_zero(uint32_t *p, uint32_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(nrc_zero_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

}// namespace vs
