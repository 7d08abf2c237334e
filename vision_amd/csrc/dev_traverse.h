// BVH8 closest-hit / any-hit traversal for gfx950 (replaces the reference's
// OptiX Accel::trace_closest / trace_occlusion, src/base/mgr/geometry.cpp:167-184).
//
// Per lane: one stack of node groups in LDS (entry = child_base, remaining
// hit bits by slot, internal-child mask), at most one entry per tree level; the
// nearest slot is picked by the ray's octant when a child is fetched
// (first_slot).  Leaf triangles of a node are tested before the next
// node is fetched, so closest-hit culling uses the tightest t.
//
// The ray/triangle test is the watertight test of Woop, Benthin and Wald
// (JCGT 2013) with FP contraction disabled, so the oracle's scalar restatement
// produces bit-identical (t, barycentrics, triangle) for identical rays.
// Valid hits satisfy tmin < t < tmax; equal t resolves to the lower triangle id.
#pragma once

#include "dev_common.h"
#include "dev_scene.h"

namespace vs {
namespace dev {

struct RayPre {
    f3 o;
    float tmin;
    f3 idir;
    // visiting order: the halves, quarters and eighths of the slots that the
    // ray meets first
    uint32_t first4, first2, first1;
    // byte selectors of the planes the ray enters by: slots 0 and 1 of a low
    // and a high plane word, into the low bytes of the two halves
    uint32_t near_x, near_y, near_z;
    int kx, ky, kz;
    float Sx, Sy, Sz;
};

__device__ __forceinline__ float sel3(f3 a, int k) { return k == 0 ? a.x : (k == 1 ? a.y : a.z); }

__device__ __forceinline__ float safe_rcp(float d) {
    const float eps = 1e-12f;
    return 1.f / (fabsf(d) > eps ? d : copysignf(eps, d));
}

__device__ __forceinline__ RayPre make_ray_pre(f3 o, f3 d, float tmin) {
    RayPre r;
    r.o = o;
    r.tmin = tmin;
    r.idir = mk3(safe_rcp(d.x), safe_rcp(d.y), safe_rcp(d.z));
    r.first1 = d.x < 0.f ? 0xAAu : 0x55u;
    r.first2 = d.y < 0.f ? 0xCCu : 0x33u;
    r.first4 = d.z < 0.f ? 0xF0u : 0x0Fu;
    r.near_x = r.idir.x >= 0.f ? 0x0C010C00u : 0x0C050C04u;
    r.near_y = r.idir.y >= 0.f ? 0x0C010C00u : 0x0C050C04u;
    r.near_z = r.idir.z >= 0.f ? 0x0C010C00u : 0x0C050C04u;
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = ax > ay ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1 == 3 ? 0 : kz + 1;
    int ky = kx + 1 == 3 ? 0 : kx + 1;
    if (sel3(d, kz) < 0.f) {
        int t = kx;
        kx = ky;
        ky = t;
    }
    r.kx = kx;
    r.ky = ky;
    r.kz = kz;
    float dz = sel3(d, kz);
    r.Sx = sel3(d, kx) / dz;
    r.Sy = sel3(d, ky) / dz;
    r.Sz = 1.f / dz;
    return r;
}

// watertight ray/triangle test; returns false on a miss.  The barycentrics
// of a hit are V / det and W / det: only the closest hit's are divided.
__device__ __forceinline__ bool intersect_triangle(const RayPre &r, f3 v0, f3 v1, f3 v2, float &t, float &V, float &W,
                                                   float &det) {
#pragma clang fp contract(off)
    f3 A = v0 - r.o, B = v1 - r.o, C = v2 - r.o;
    float Akz = sel3(A, r.kz), Bkz = sel3(B, r.kz), Ckz = sel3(C, r.kz);
    float Ax = sel3(A, r.kx) - r.Sx * Akz;
    float Ay = sel3(A, r.ky) - r.Sy * Akz;
    float Bx = sel3(B, r.kx) - r.Sx * Bkz;
    float By = sel3(B, r.ky) - r.Sy * Bkz;
    float Cx = sel3(C, r.kx) - r.Sx * Ckz;
    float Cy = sel3(C, r.ky) - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    V = Ax * Cy - Ay * Cx;
    W = Bx * Ay - By * Ax;
    if (fminf(fminf(fabsf(U), fabsf(V)), fabsf(W)) == 0.f) {
        double CxBy = double(Cx) * double(By), CyBx = double(Cy) * double(Bx);
        U = float(CxBy - CyBx);
        double AxCy = double(Ax) * double(Cy), AyCx = double(Ay) * double(Cx);
        V = float(AxCy - AyCx);
        double BxAy = double(Bx) * double(Ay), ByAx = double(By) * double(Ax);
        W = float(BxAy - ByAx);
    }
    det = U + V + W;
    // both signs among the three: outside
    const bool out = (fminf(fminf(U, V), W) < 0.f) & (fmaxf(fmaxf(U, V), W) > 0.f);
    if (out | (det == 0.f)) return false;
    float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    float T = U * Az + V * Bz + W * Cz;
    t = T / det;
    return true;
}

struct TraceHit {
    float t;
    uint32_t tri;// global triangle id, kInvalid on a miss
    float b1, b2;
};

// byte i of the result: byte sel[i] of lo (0..3) or hi (4..7), or zero (0x0C)
__device__ __forceinline__ uint32_t pick_bytes(uint32_t hi, uint32_t lo, uint32_t sel) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_perm(hi, lo, sel);
#else
    uint32_t r = 0;
    for (int i = 0; i < 4; ++i) {
        const uint32_t b = (sel >> (8 * i)) & 0xFFu;
        if (b < 8u) r |= (((b < 4u ? lo : hi) >> (8u * (b & 3u))) & 0xFFu) << (8 * i);
    }
    return r;
#endif
}

// the low (0) or high (1) half of a word whose halves hold bytes, read as a
// half-precision value: byte * 2^-24
__device__ __forceinline__ float byte_half(uint32_t w, int hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    return float(__builtin_bit_cast(_Float16, uint16_t(hi ? w >> 16 : w)));
#else
    return float(hi ? w >> 16 : w & 0xFFFFu) * 0x1p-24f;
#endif
}

// Intersect the 8 child boxes of node `idx` (layout in bvh.h).  Out: the
// internal children hit, by slot, with child_base and imask; the triangles of
// the leaves hit as bits of the node's leaf mask, with that mask and the
// node's first triangle.
// Bound by VALU issue and, close behind, by the texture addresser, which
// takes a 16-byte load's 64 lanes some 20 cycles whether active or not.  So
// the node stays at five loads, and a child costs 3 byte picks (two planes
// each; they choose near and far on the way), 6 mixed-precision FMAs on the
// picked bytes as half denormals, 4 min / max, and a subtract whose sign bit
// is shifted into the miss mask: 15 instructions for 21 with a conversion a
// plane, selects and a compare.
__device__ __forceinline__ void process_node(const uint4 *__restrict__ nodes, uint32_t idx, const RayPre &r, float tmax,
                                             uint32_t &cbase, uint32_t &chits, uint32_t &cimask, uint32_t &tbase,
                                             uint32_t &tleaf, uint32_t &tmask, uint32_t &nfetch) {
    const uint4 *np = nodes + size_t(idx) * 5;
    const uint4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3], n4 = np[4];
    ++nfetch;
    const float sx = __uint_as_float(n0.w << 16) * r.idir.x;
    const float sy = __uint_as_float(n0.w & 0xFFFF0000u) * r.idir.y;
    const float sz = __uint_as_float(n1.w & 0xFFFF0000u) * r.idir.z;
    const float ax = (__uint_as_float(n0.x) - r.o.x) * r.idir.x;
    const float ay = (__uint_as_float(n0.y) - r.o.y) * r.idir.y;
    const float az = (__uint_as_float(n0.z) - r.o.z) * r.idir.z;
    uint32_t miss = 0;
#pragma unroll
    for (int k = 3; k >= 0; --k) {
        // slots 2 k and 2 k + 1
        const uint32_t up = (k & 1) ? 0x00020002u : 0u;
        const uint32_t lx = k < 2 ? n2.x : n2.y, ly = k < 2 ? n2.z : n2.w, lz = k < 2 ? n3.x : n3.y;
        const uint32_t hx = k < 2 ? n3.z : n3.w, hy = k < 2 ? n4.x : n4.y, hz = k < 2 ? n4.z : n4.w;
        const uint32_t nx = pick_bytes(hx, lx, r.near_x + up), fx = pick_bytes(lx, hx, r.near_x + up);
        const uint32_t ny = pick_bytes(hy, ly, r.near_y + up), fy = pick_bytes(ly, hy, r.near_y + up);
        const uint32_t nz = pick_bytes(hz, lz, r.near_z + up), fz = pick_bytes(lz, hz, r.near_z + up);
#pragma unroll
        for (int b = 1; b >= 0; --b) {
            const float tn = fmaxf(fmaxf(fmaf(byte_half(nx, b), sx, ax), fmaf(byte_half(ny, b), sy, ay)),
                                   fmaxf(fmaf(byte_half(nz, b), sz, az), r.tmin));
            const float tf = fminf(fminf(fmaf(byte_half(fx, b), sx, ax), fmaf(byte_half(fy, b), sy, ay)),
                                   fminf(fmaf(byte_half(fz, b), sz, az), tmax));
            miss = (miss << 1) | (__float_as_uint(tf - tn) >> 31);
        }
    }
    const uint32_t hits = ~miss & 0xFFu;
    cimask = n1.z >> 24;
    chits = hits & cimask;
    // slot s to bits 3 s .. 3 s + 2; slots that are no leaves are not in the leaf mask
    uint32_t m = hits;
    m = (m | (m << 8)) & 0x00F00Fu;
    m = (m | (m << 4)) & 0x0C30C3u;
    m = (m | (m << 2)) & 0x249249u;
    tleaf = n1.z;// its high byte lies above every triangle's bit
    tmask = (m | (m << 1) | (m << 2)) & n1.z;
    tbase = n1.y;
    cbase = n1.x;
}

// the slot of `hits` that the ray meets first: its mask bit
__device__ __forceinline__ uint32_t first_slot(uint32_t hits, const RayPre &r) {
    uint32_t m = hits & r.first4;
    m = m ? m : hits;
    uint32_t n = m & r.first2;
    n = n ? n : m;
    m = n & r.first1;
    return m ? m : n;
}

template <bool ANY>
__device__ __forceinline__ TraceHit traverse(const SceneView &sc, f3 o, f3 d, float tmin, float tmax,
                                             uint2 *stack, uint32_t stride, uint32_t &nfetch, uint32_t &tfetch) {
    const uint4 *__restrict__ nodes = reinterpret_cast<const uint4 *>(sc.nodes);
    const float4 *__restrict__ ltri = reinterpret_cast<const float4 *>(sc.leaf_tris);
    RayPre r = make_ray_pre(o, d, tmin);
    TraceHit h;
    h.t = tmax;
    h.tri = kInvalid;
    float hV = 0.f, hW = 0.f, hdet = 1.f;
    uint32_t sp = 0;
    uint32_t gbase, ghits, gimask, tbase, tleaf, tmask;
    process_node(nodes, 0, r, tmax, gbase, ghits, gimask, tbase, tleaf, tmask, nfetch);
    while (true) {
        while (tmask) {
            const uint32_t bit = tmask & (0u - tmask);
            tmask ^= bit;
            const float4 *tp = ltri + size_t(tbase + uint32_t(__popc(tleaf & (bit - 1u)))) * 3;
            float4 a = tp[0], b = tp[1], c = tp[2];
            ++tfetch;
            float t, V, W, det;
            if (intersect_triangle(r, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), mk3(c.x, c.y, c.z), t, V, W, det)) {
                const uint32_t id = __float_as_uint(a.w);
                if ((t > tmin) & (t < tmax) & ((t < h.t) | ((t == h.t) & (id < h.tri)))) {
                    h.t = t;
                    h.tri = id;
                    hV = V;
                    hW = W;
                    hdet = det;
                    if (ANY) {
                        h.b1 = V / det;
                        h.b2 = W / det;
                        return h;
                    }
                }
            }
        }
        if (ghits == 0) {
            if (sp == 0) break;
            --sp;
            uint2 e = stack[sp * stride];
            gbase = e.x;
            ghits = e.y & 0xFFu;
            gimask = e.y >> 8;
        }
        const uint32_t bit = first_slot(ghits, r);
        ghits ^= bit;
        const uint32_t child = gbase + uint32_t(__popc(gimask & (bit - 1u)));
        uint32_t nb, nh, ni;
        process_node(nodes, child, r, ANY ? tmax : h.t, nb, nh, ni, tbase, tleaf, tmask, nfetch);
        if (nh) {
            if (ghits) {
                if (sp < sc.stack_size) stack[sp * stride] = make_uint2(gbase, ghits | (gimask << 8));
                ++sp;
                if (sp > sc.stack_size) sp = sc.stack_size;// unreachable: stack sized to tree depth
            }
            gbase = nb;
            ghits = nh;
            gimask = ni;
        }
    }
    // zero on a miss (0 / 1)
    h.b1 = hV / hdet;
    h.b2 = hW / hdet;
    return h;
}

}// namespace dev
}// namespace vs
