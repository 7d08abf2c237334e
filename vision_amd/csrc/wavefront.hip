// Wavefront path tracer for gfx950: the bounce loop of the megakernel split at
// its traversals.  Per bounce: closest-hit over the live-path queue (lean
// kernel, high occupancy), shading (path_shade: emission, NEE set-up, BSDF
// sample, RR; appends live paths and shadow rays, an atomic per wave and
// buffer), any-hit over the shadow rays.  Paths run the same path_shade
// arithmetic as the megakernel, so both forms give the same film.
#include <hip/hip_runtime.h>

#include "dev_pt.h"
#include "wavefront.h"

namespace vs {

using namespace dev;

namespace {

// The state a bounce reads.  The radiance gathered so far stays in memory: a
// bounce adds to it at most once (store_state), most not at all.
template <int NS, bool RGB>
__device__ __forceinline__ void load_state(const WavefrontView &w, uint32_t i, PathState<NS> &ps) {
    float4 a = w.o[i], b = w.d[i], t = w.thr[i];
    uint4 m = w.meta[i];
    ps.o = mk3(a.x, a.y, a.z);
    ps.scatter_pdf = a.w;
    ps.d = mk3(b.x, b.y, b.z);
    ps.eta_scale = b.w;
    const float tv[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int k = 0; k < NS; ++k) ps.thr.v[k] = tv[k];
    ps.L = mk3(0.f, 0.f, 0.f);
    ps.fw = 0.f;
    ps.sampler.state = m.x;
    ps.bounce = m.y & 0xFFFFu;
    ps.skips = m.y >> 16;
    ps.alive = m.z;
    ps.tail = m.w;
    if (RGB) {
        ps.swl = sample_wavelengths<NS, true>(0u, 0u, 0u);
    } else {
        float4 lm = w.lam[i], lp = w.lpdf[i];
        const float lv[4] = {lm.x, lm.y, lm.z, lm.w}, pv[4] = {lp.x, lp.y, lp.z, lp.w};
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            ps.swl.lambda[k] = lv[k];
            ps.swl.pdf[k] = pv[k];
        }
    }
}

template <int NS>
__device__ __forceinline__ void store_pdfs(const WavefrontView &w, uint32_t i, const PathState<NS> &ps) {
    float pv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NS; ++k) pv[k] = ps.swl.pdf[k];
    w.lpdf[i] = make_float4(pv[0], pv[1], pv[2], pv[3]);
}

// ray, throughput and sampler for the next bounce
template <int NS>
__device__ __forceinline__ void store_next(const WavefrontView &w, uint32_t i, const PathState<NS> &ps) {
    w.o[i] = make_float4(ps.o.x, ps.o.y, ps.o.z, ps.scatter_pdf);
    w.d[i] = make_float4(ps.d.x, ps.d.y, ps.d.z, ps.eta_scale);
    float tv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NS; ++k) tv[k] = ps.thr.v[k];
    w.thr[i] = make_float4(tv[0], tv[1], tv[2], tv[3]);
    w.meta[i] = make_uint4(ps.sampler.state, ps.bounce | (ps.skips << 16), ps.alive, ps.tail);
}

template <int NS, bool RGB>
__device__ __forceinline__ void store_begin(const WavefrontView &w, uint32_t i, const PathState<NS> &ps) {
    store_next(w, i, ps);
    w.L[i] = make_float4(ps.L.x, ps.L.y, ps.L.z, ps.fw);
    if (!RGB) {
        float lv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NS; ++k) lv[k] = ps.swl.lambda[k];
        w.lam[i] = make_float4(lv[0], lv[1], lv[2], lv[3]);
        store_pdfs(w, i, ps);
    }
}

// where item k of a queue is
__device__ __forceinline__ uint32_t queue_slot(const uint32_t *__restrict__ first, uint32_t segment, uint32_t k) {
    uint32_t s = 0;
#pragma unroll
    for (uint32_t j = 1; j < kWfSegments; ++j) s += k >= first[j] ? 1u : 0u;
    return s * segment + (k - first[s]);
}
__device__ __forceinline__ uint32_t queue_item(const WavefrontQueue &q, uint32_t k) {
    return q.items ? q.items[queue_slot(q.first, q.segment, k)] : k;
}

template <int NS, bool RGB>
__global__ void __launch_bounds__(256) begin_kernel(CameraView cam, RenderView rv, WavefrontView w, uint32_t frame0,
                                                    uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t p = i % w.pixels, s = i / w.pixels;
    PathState<NS> ps;
    path_begin<NS, RGB>(cam, rv, p % w.width, p / w.width, frame0 + s, ps);
    store_begin<NS, RGB>(w, i, ps);
}

// The traversal kernels at seven waves per SIMD (72 VGPRs): the 1080p 64-spp
// hero-4 job of 320k triangles traces in 61.7 / 38.0 ms (closest / any hit), with
// byte-to-float conversions and selects in the slab tests in 70.3 / 40.8.  The
// budgets were compared on a node with tighter boxes (6 % fewer visits): 59.3 /
// 36.5 at seven waves, 59.4 / 36.9 at six, 60.1 / 39.6 at eight, which spill; and
// waves that own 512 rays of the queue and refill their finished lanes were no
// faster there (62.1 / 38.2): a node's triangles, not the rays' lengths, leave
// lanes idle.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7)))
trace_queue_kernel(SceneView sc, WavefrontView w, WavefrontQueue queue, uint32_t count,
                   unsigned long long *__restrict__ counters) {
    extern __shared__ uint2 lds_stack[];
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    uint32_t i = queue_item(queue, k);
    float4 a = w.o[i], b = w.d[i];
    uint32_t nf = 0, tf = 0;
    TraceHit h = traverse<false>(sc, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), 0.f, 3.402823466e38f,
                                 lds_stack + threadIdx.x, blockDim.x, nf, tf);
    w.hit[i] = make_float4(h.t, __uint_as_float(h.tri), h.b1, h.b2);
    if (counters) {
        atomicAdd(counters + 0, 1ull);
        atomicAdd(counters + 1, (unsigned long long)nf);
        atomicAdd(counters + 2, (unsigned long long)tf);
    }
}

// Three resident waves per SIMD (168 VGPRs, 250-420 B of scratch per lane):
// left free the compiler takes 256 VGPRs and one wave (figures at shade_waves).
// Before shading, a block sorts its paths by what they hit (the miss branch,
// a material-less surface, or the material's kind) in LDS, so that a wave
// mostly runs one branch of path_shade; the block's paths stay the same 256
// queue entries, so their state loads stay within the same cache lines.  A wave
// appends its survivors and shadow rays to its block's segments by itself, and
// ends without waiting for the block's slowest.  Latency bounds this kernel
// (2.8 waves a SIMD, a third of the vector rate): shading the procedural job
// of 64 frames at 1920x1080 took 95.2 ms with one append a block behind a
// barrier and all state written back, and takes 77.9 (blocks of 128: 78.3,
// 512: 80.3).
constexpr uint32_t kShadeKeys = 16;// the last key: no path (past the queue's end)

__device__ __forceinline__ uint32_t shade_key(const SceneView &sc, uint32_t tri) {
    if (tri == kInvalid) return 0u;
    const uint32_t m = sc.inst[sc.tri_inst[tri]].mat;
    if (m == kInvalid) return 1u;
    return 2u + min(sc.mat[m].type, kShadeKeys - 3u);
}

// register budget of the shading kernel, in waves per SIMD: three for every
// material (measured on the procedural job: 2 -> 89.5, 3 -> 77.9, 4 -> 85.2
// ms of shading per 64-frame job), more for the diffuse family, whose
// smaller code needs fewer registers
constexpr int shade_waves(int ms) { return ms == MS_ALL ? 3 : 4; }

template <int NS, bool RGB, int MS>
__global__ void __launch_bounds__(kShadeBlock) __attribute__((amdgpu_waves_per_eu(shade_waves(MS))))
shade_kernel(SceneView sc, RenderView rv, WavefrontView w, WavefrontQueue qin, uint32_t count,
             uint32_t *__restrict__ qout, uint32_t *__restrict__ counts) {
    __shared__ uint32_t s_key[kShadeKeys];
    __shared__ uint32_t s_path[kShadeBlock];
    __shared__ float4 s_hit[kShadeBlock];
    if (threadIdx.x < kShadeKeys) s_key[threadIdx.x] = 0u;
    __syncthreads();
    {
        const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
        uint32_t i0 = 0u, key = kShadeKeys - 1u;
        float4 hv0 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k < count) {
            i0 = queue_item(qin, k);
            hv0 = w.hit[i0];
            key = shade_key(sc, __float_as_uint(hv0.y));
        }
        const uint32_t rank = atomicAdd(&s_key[key], 1u);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t sum = 0u;
            for (uint32_t j = 0; j < kShadeKeys; ++j) {
                const uint32_t c = s_key[j];
                s_key[j] = sum;
                sum += c;
            }
        }
        __syncthreads();
        const uint32_t pos = s_key[key] + rank;
        s_path[pos] = key == kShadeKeys - 1u ? kInvalid : i0;
        s_hit[pos] = hv0;
        __syncthreads();
    }
    const uint32_t i = s_path[threadIdx.x];
    bool live = false;
    ShadowRay sr;
    sr.valid = 0u;
    if (i != kInvalid) {
        PathState<NS> ps;
        load_state<NS, RGB>(w, i, ps);
        const float pdf1 = NS > 1 ? ps.swl.pdf[NS - 1] : 0.f;
        float4 hv = s_hit[threadIdx.x];
        TraceHit h;
        h.t = hv.x;
        h.tri = __float_as_uint(hv.y);
        h.b1 = hv.z;
        h.b2 = hv.w;
        path_shade<NS, RGB, MS>(sc, rv, ps, h, sr);
        live = ps.alive != 0u;
        if (ps.L.x != 0.f || ps.L.y != 0.f || ps.L.z != 0.f) {
            const float4 l = w.L[i];
            w.L[i] = make_float4(l.x + ps.L.x, l.y + ps.L.y, l.z + ps.L.z, l.w);
        }
        if (live) {
            store_next(w, i, ps);
            // dispersion drops the secondary wavelengths
            if (!RGB && ps.swl.pdf[NS - 1] != pdf1) store_pdfs(w, i, ps);
        }
    }
    const bool shadow = sr.valid != 0u;
    const unsigned long long below = (1ull << __lane_id()) - 1ull;
    const unsigned long long ml = __ballot(live), ms = __ballot(shadow);
    const uint32_t seg = blockIdx.x % kWfSegments;
    const uint32_t start = seg * wf_segment(count);
    uint32_t nl = 0u, ns = 0u;
    if (__lane_id() == 0u) {
        if (ml) nl = atomicAdd(counts + seg * kWfCounterStride, uint32_t(__popcll(ml)));
        if (ms) ns = atomicAdd(counts + kWfShadow + seg * kWfCounterStride, uint32_t(__popcll(ms)));
    }
    nl = start + __shfl(nl, 0);
    ns = start + __shfl(ns, 0);
    if (shadow) {
        const uint32_t slot = ns + uint32_t(__popcll(ms & below));
        w.sh_o[slot] = make_float4(sr.o.x, sr.o.y, sr.o.z, __uint_as_float(i));
        w.sh_d[slot] = make_float4(sr.d.x, sr.d.y, sr.d.z, 0.f);
        w.sh_c[slot] = make_float4(sr.c.x, sr.c.y, sr.c.z, 0.f);
    }
    if (live) qout[nl + uint32_t(__popcll(ml & below))] = i;
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7)))
shadow_kernel(SceneView sc, WavefrontView w, const uint32_t *__restrict__ counts, uint32_t max_count, uint32_t segment,
              unsigned long long *__restrict__ counters) {
    extern __shared__ uint2 lds_stack[];
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t *first = counts + kWfShadowFirst;
    if (k >= max_count || k >= first[kWfSegments]) return;
    k = queue_slot(first, segment, k);
    float4 a = w.sh_o[k], b = w.sh_d[k];
    uint32_t nf = 0, tf = 0;
    TraceHit h = traverse<true>(sc, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), 0.f, 1.f - kShadowEpsilon,
                                lds_stack + threadIdx.x, blockDim.x, nf, tf);
    if (h.tri == kInvalid) {
        uint32_t i = __float_as_uint(a.w);
        float4 c = w.sh_c[k], l = w.L[i];
        f3 L = mk3(l.x, l.y, l.z);
        L += mk3(c.x, c.y, c.z);
        w.L[i] = make_float4(L.x, L.y, L.z, l.w);
    }
    if (counters) {
        atomicAdd(counters + 0, 1ull);
        atomicAdd(counters + 1, (unsigned long long)nf);
        atomicAdd(counters + 2, (unsigned long long)tf);
    }
}

// one wave: lanes 0..15 the live segments, 16..31 the shadow rays'
__global__ void __launch_bounds__(64) fold_kernel(uint32_t *counts) {
    const uint32_t t = threadIdx.x, s = t % kWfSegments;
    uint32_t c = 0u;
    if (t < 2u * kWfSegments) {
        c = counts[t * kWfCounterStride];
        counts[t * kWfCounterStride] = 0u;
    }
    uint32_t sum = c;
#pragma unroll
    for (uint32_t d = 1; d < kWfSegments; d *= 2) {
        const uint32_t up = __shfl_up(sum, d);
        if (s >= d) sum += up;
    }
    if (t < 2u * kWfSegments) {
        uint32_t *first = counts + (t < kWfSegments ? kWfLiveFirst : kWfShadowFirst);
        first[s] = sum - c;
        if (s == kWfSegments - 1u) first[kWfSegments] = sum;
    }
}
static_assert(2 * kWfSegments <= 64, "segments of both queues fit one wave");

__global__ void __launch_bounds__(256) zero_kernel(uint32_t *counts) {
    for (uint32_t k = threadIdx.x; k < kWfWords; k += 256u) counts[k] = 0u;
}

// fold the chunk's samples into the film in frame order, as the megakernel's
// per-pixel loop does
__global__ void __launch_bounds__(256) accumulate_kernel(RenderView rv, WavefrontView w, uint32_t frame0,
                                                         uint32_t frames, float4 *__restrict__ rt,
                                                         float4 *__restrict__ out) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= w.pixels) return;
    float4 acc = rt[p];
    for (uint32_t s = 0; s < frames; ++s) {
        float4 l = w.L[size_t(s) * w.pixels + p];
        acc = film_add(rv, acc, mk3(l.x, l.y, l.z) * l.w, frame0 + s);
    }
    rt[p] = acc;
    if (rv.write_output) out[p] = film_output(rv, acc);
}

uint32_t blocks(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

}// namespace

hipError_t wf_begin(const CameraView &cam, const RenderView &rv, const WavefrontView &w, uint32_t spectrum_dim,
                    bool rgb, uint32_t frame0, uint32_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    dim3 g(blocks(n, 256)), b(256);
    if (rgb) hipLaunchKernelGGL((begin_kernel<3, true>), g, b, 0, stream, cam, rv, w, frame0, n);
    else if (spectrum_dim == 4) hipLaunchKernelGGL((begin_kernel<4, false>), g, b, 0, stream, cam, rv, w, frame0, n);
    else if (spectrum_dim == 3) hipLaunchKernelGGL((begin_kernel<3, false>), g, b, 0, stream, cam, rv, w, frame0, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t wf_trace(const SceneView &sc, const WavefrontView &w, const WavefrontQueue &queue, uint32_t count,
                    unsigned long long *counters, uint32_t block, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    if (block != 64 && block != 128 && block != 256) return hipErrorInvalidValue;
    size_t lds = size_t(sc.stack_size) * block * sizeof(uint2);
    hipLaunchKernelGGL(trace_queue_kernel, dim3(blocks(count, block)), dim3(block), lds, stream, sc, w, queue, count,
                       counters);
    return hipGetLastError();
}

namespace {
template <int MS>
hipError_t shade_ms(const SceneView &sc, const RenderView &rv, const WavefrontView &w, uint32_t spectrum_dim,
                    bool rgb, const WavefrontQueue &qin, uint32_t count, uint32_t *qout, uint32_t *counts,
                    hipStream_t stream) {
    dim3 g(blocks(count, kShadeBlock)), b(kShadeBlock);
    if (rgb) hipLaunchKernelGGL((shade_kernel<3, true, MS>), g, b, 0, stream, sc, rv, w, qin, count, qout, counts);
    else if (spectrum_dim == 4)
        hipLaunchKernelGGL((shade_kernel<4, false, MS>), g, b, 0, stream, sc, rv, w, qin, count, qout, counts);
    else if (spectrum_dim == 3)
        hipLaunchKernelGGL((shade_kernel<3, false, MS>), g, b, 0, stream, sc, rv, w, qin, count, qout, counts);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
}// namespace

hipError_t wf_shade(const SceneView &sc, const RenderView &rv, const WavefrontView &w, uint32_t spectrum_dim,
                    bool rgb, int material_set, const WavefrontQueue &qin, uint32_t count, uint32_t *qout,
                    uint32_t *counts, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    if (material_set == MS_DIFFUSE)
        return shade_ms<MS_DIFFUSE>(sc, rv, w, spectrum_dim, rgb, qin, count, qout, counts, stream);
    if (material_set != MS_ALL) return hipErrorInvalidValue;
    return shade_ms<MS_ALL>(sc, rv, w, spectrum_dim, rgb, qin, count, qout, counts, stream);
}

hipError_t wf_shadow(const SceneView &sc, const WavefrontView &w, const uint32_t *counts, uint32_t max_count,
                     uint32_t segment, unsigned long long *counters, uint32_t block, hipStream_t stream) {
    if (max_count == 0) return hipSuccess;
    if (block != 64 && block != 128 && block != 256) return hipErrorInvalidValue;
    size_t lds = size_t(sc.stack_size) * block * sizeof(uint2);
    hipLaunchKernelGGL(shadow_kernel, dim3(blocks(max_count, block)), dim3(block), lds, stream, sc, w, counts,
                       max_count, segment, counters);
    return hipGetLastError();
}

hipError_t wf_zero(uint32_t *counts, hipStream_t stream) {
    hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(256), 0, stream, counts);
    return hipGetLastError();
}

hipError_t wf_fold(uint32_t *counts, hipStream_t stream) {
    hipLaunchKernelGGL(fold_kernel, dim3(1), dim3(64), 0, stream, counts);
    return hipGetLastError();
}

hipError_t wf_accumulate(const RenderView &rv, const WavefrontView &w, uint32_t frame0, uint32_t frames, float4 *rt,
                         float4 *out, hipStream_t stream) {
    hipLaunchKernelGGL(accumulate_kernel, dim3(blocks(w.pixels, 256)), dim3(256), 0, stream, rv, w, frame0, frames,
                       rt, out);
    return hipGetLastError();
}

}// namespace vs
