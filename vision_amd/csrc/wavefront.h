// Wavefront form of the path tracer: per-path state in HBM (one array per
// field, so a wave's loads coalesce), queues of live paths between the
// kernels of a bounce.  Shared by the host driver (capi.cpp) and the kernels
// (wavefront.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dev_scene.h"

namespace vs {

struct WavefrontView {
    float4 *o;    // ray origin xyz, scatter pdf
    float4 *d;    // ray direction xyz, eta scale
    float4 *thr;  // throughput (up to 4 wavelengths)
    float4 *L;    // radiance gathered xyz, film weight
    uint4 *meta;  // sampler state, bounce | skips << 16, alive, tail bounce
    float4 *lam;  // hero wavelengths
    float4 *lpdf; // their pdfs
    float4 *hit;  // t, triangle id bits, b1, b2
    float4 *sh_o; // shadow ray origin xyz, path index bits
    float4 *sh_d; // shadow ray direction xyz
    float4 *sh_c; // shadow ray contribution xyz
    uint32_t pixels;
    uint32_t width;
};

// Queues are written in kWfSegments segments, each with an append counter in a
// memory line of its own: waves append by themselves, and some 100 M atomics a
// second on one address would hold them up.  Counter words: the segments' live
// paths, then their shadow rays, kWfCounterStride words apart; then what
// wf_fold makes of them, the segments' first indices in the whole queue and its
// length, for both.
constexpr uint32_t kWfSegments = 16;
constexpr uint32_t kWfCounterStride = 64;
constexpr uint32_t kWfShadow = kWfSegments * kWfCounterStride;
constexpr uint32_t kWfLiveFirst = 2 * kWfShadow;
constexpr uint32_t kWfShadowFirst = kWfLiveFirst + kWfSegments + 1;
constexpr uint32_t kWfWords = kWfShadowFirst + kWfSegments + 1;
// paths of a block of the shading kernel, and what a queue of `paths` paths
// that blocks of it append to needs
constexpr uint32_t kShadeBlock = 256;
constexpr uint32_t wf_segment(uint32_t paths) {
    return ((paths + kShadeBlock - 1u) / kShadeBlock + kWfSegments - 1u) / kWfSegments * kShadeBlock;
}
constexpr size_t wf_queue_capacity(size_t paths) { return paths + size_t(2) * kWfSegments * kShadeBlock; }

// a queue as the kernels read it: item k of the whole queue is in the segment
// whose first index is the last not above k.  No items: path k itself.
struct WavefrontQueue {
    const uint32_t *items;
    const uint32_t *first;// kWfSegments + 1 words
    uint32_t segment;     // capacity of a segment
};

hipError_t wf_begin(const CameraView &cam, const RenderView &rv, const WavefrontView &w, uint32_t spectrum_dim,
                    bool rgb, uint32_t frame0, uint32_t n, hipStream_t stream);
hipError_t wf_trace(const SceneView &sc, const WavefrontView &w, const WavefrontQueue &queue, uint32_t count,
                    unsigned long long *counters, uint32_t block, hipStream_t stream);
// material_set: 0 every material, 1 the diffuse family only (a smaller
// kernel for scenes of diffuse / Oren-Nayar / black materials).  Survivors go
// to qout, shadow rays to w.sh_*, in segments of wf_segment(count).
hipError_t wf_shade(const SceneView &sc, const RenderView &rv, const WavefrontView &w, uint32_t spectrum_dim,
                    bool rgb, int material_set, const WavefrontQueue &qin, uint32_t count, uint32_t *qout,
                    uint32_t *counts, hipStream_t stream);
// the segments' counters into first indices and lengths; clears the counters
hipError_t wf_fold(uint32_t *counts, hipStream_t stream);
hipError_t wf_shadow(const SceneView &sc, const WavefrontView &w, const uint32_t *counts, uint32_t max_count,
                     uint32_t segment, unsigned long long *counters, uint32_t block, hipStream_t stream);
hipError_t wf_zero(uint32_t *counts, hipStream_t stream);
hipError_t wf_accumulate(const RenderView &rv, const WavefrontView &w, uint32_t frame0, uint32_t frames,
                         float4 *rt, float4 *out, hipStream_t stream);

}// namespace vs
