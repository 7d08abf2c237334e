// Device code of the radiance cache: hash-grid encoding, the MLP on BF16
// MFMA tiles (16x16x16, FP32 accumulation) and its backward pass.
//
// The encoding is a kernel of its own.  A wave of the network's kernels takes 64
// encoded rows (queries) or 16 (training samples) at a time and sends them
// through the network in tiles of 16.  Tile operands live in LDS:
// activations row-major (bf16), weights transposed (wt[n][k] = W[k][n]) and,
// for the backward pass, also as they are, so that a lane's four consecutive k
// of an MFMA operand are one 8-byte load.  MFMA lane layout (16x16x16 bf16):
// the A operand of lane l holds row l % 16, k = 4 (l / 16) + e; the B operand
// holds column l % 16, k = 4 (l / 16) + e; the accumulator holds rows
// 4 (l / 16) + e of column l % 16, e = 0..3.  A layer is computed transposed
// (weights as A, activations as B), so that a lane's accumulator is four
// neighbouring neurons of one row: an 8-byte store.
#pragma once

#include "dev_common.h"
#include "nrc.h"

namespace vs {
namespace dev {

typedef short bf16x2 __attribute__((ext_vector_type(2)));
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ float h2f(uint16_t h) { return float(__builtin_bit_cast(_Float16, h)); }
__device__ __forceinline__ uint16_t f2h(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }

__device__ __forceinline__ f32x4 mma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x4 ld4(const uint16_t *p) { return *reinterpret_cast<const bf16x4 *>(p); }
__device__ __forceinline__ bf16x4 gather4(const uint16_t *p, int stride) {
    bf16x4 r;
    r.x = short(p[0]);
    r.y = short(p[stride]);
    r.z = short(p[2 * stride]);
    r.w = short(p[3 * stride]);
    return r;
}

// ---- encoding ----------------------------------------------------------------

__device__ __forceinline__ uint32_t nrc_index(bool dense, uint32_t res, uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t n = res + 1u;
    return dense ? x + n * (y + n * z) : (x ^ (y * 2654435761u) ^ (z * 805459861u)) & (kNrcTable - 1u);
}

// the cell of a position in a level of `res` cells an axis: integer corner and fractions
__device__ __forceinline__ void nrc_cell(uint32_t res, const float u[3], uint32_t c[3], float f[3]) {
    float s = float(res);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float q = u[a] * s;
        float fl = floorf(q);
        uint32_t ci = uint32_t(fl);
        if (ci >= res) ci = res - 1u;
        c[a] = ci;
        f[a] = q - float(ci);
    }
}

__device__ __forceinline__ void nrc_unit(const NrcView &v, const float p[3], float u[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) u[a] = fminf(fmaxf((p[a] - v.lo[a]) * v.inv_ext[a], 0.f), 1.f);
}

// trilinear weight of corner k (bit 0: x, bit 1: y, bit 2: z)
__device__ __forceinline__ float nrc_corner_weight(int k, const float f[3]) {
    float wx = (k & 1) ? f[0] : 1.f - f[0];
    float wy = (k & 2) ? f[1] : 1.f - f[1];
    float wz = (k & 4) ? f[2] : 1.f - f[2];
    return (wx * wy) * wz;
}

typedef uint32_t u32pair __attribute__((ext_vector_type(2), aligned(4)));

// The features of one level (its table at g) at u, before rounding.  The two
// corners along x are one 8-byte load where they are neighbours in the table:
// always in a directly indexed level, in a hashed one where x is even (the
// hash of x is x itself, so x + 1 flips the lowest bit); else the second is a
// load of its own: 86 gathers a position instead of 128.  Corners are summed
// in the order of nrc_corner_weight's bits.
template <bool dense>
__device__ __forceinline__ void nrc_level(const uint32_t *__restrict__ g, uint32_t res, const float u[3], float &a0,
                                          float &a1) {
    uint32_t c[3];
    float f[3];
    nrc_cell(res, u, c, f);
    const uint32_t n = res + 1u;
    const uint32_t hy = c[1] * 2654435761u, hz = c[2] * 805459861u;
    uint32_t row[4];// of the corners (y, z), (y + 1, z), (y, z + 1), (y + 1, z + 1)
    row[0] = dense ? n * (c[1] + n * c[2]) : hy ^ hz;
    row[1] = dense ? row[0] + n : (hy + 2654435761u) ^ hz;
    row[2] = dense ? row[0] + n * n : hy ^ (hz + 805459861u);
    row[3] = dense ? row[2] + n : (hy + 2654435761u) ^ (hz + 805459861u);
    uint32_t at[4], e0[4], e1[4];
    u32pair p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        at[k] = dense ? row[k] + c[0] : (row[k] ^ c[0]) & (kNrcTable - 1u);
        p[k] = *reinterpret_cast<const u32pair *>(g + (dense ? at[k] : at[k] & ~1u));
    }
    const bool apart = !dense && (c[0] & 1u);
    uint32_t other[4] = {0, 0, 0, 0};
    if (apart) {
#pragma unroll
        for (int k = 0; k < 4; ++k) other[k] = g[(row[k] ^ (c[0] + 1u)) & (kNrcTable - 1u)];
    }
    a0 = a1 = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const bool swap = !dense && (at[k] & 1u);
        e0[k] = swap ? p[k].y : p[k].x;
        e1[k] = apart ? other[k] : (swap ? p[k].x : p[k].y);
        const float w0 = nrc_corner_weight(2 * k, f), w1 = nrc_corner_weight(2 * k + 1, f);
        a0 += w0 * h2f(uint16_t(e0[k] & 0xFFFFu));
        a1 += w0 * h2f(uint16_t(e0[k] >> 16));
        a0 += w1 * h2f(uint16_t(e1[k] & 0xFFFFu));
        a1 += w1 * h2f(uint16_t(e1[k] >> 16));
    }
}

// ---- network tiles -------------------------------------------------------------

constexpr int kXs = 40;// row stride of the feature tile (32 + pad)
constexpr int kHs = 72;// row stride of hidden tiles (64 + pad)

// weights of one block in LDS
struct NrcWeightsLds {
    uint16_t w1t[kNrcHidden * kXs];// [n][k], k < 32
    uint16_t w2t[kNrcHidden * kHs];
    uint16_t w3t[kNrcHidden * kHs];
    float w4[kNrcHidden * kNrcOut];// [k][c]
};
// and, for the backward pass, W[k][n]
struct alignas(16) NrcBackWeightsLds {
    uint16_t w1[kNrcIn * kHs];
    uint16_t w2[kNrcHidden * kHs];
    uint16_t w3[kNrcHidden * kHs];
};

// Weights to LDS by a block of `threads` (256 or 512): eight bf16 a load, all
// of a thread's loads in flight before the first store.  wb: the copies of the
// backward pass, or null.
template <int threads>
__device__ __forceinline__ void nrc_load_weights(const NrcView &v, NrcWeightsLds &w, NrcBackWeightsLds *wb, int tid) {
    constexpr int kVecs = kNrcW4 / 8;// W1, W2 and W3 are neighbours in the parameter array
    constexpr int kEach = (kVecs + threads - 1) / threads;
    const uint4 *src = reinterpret_cast<const uint4 *>(v.mlp_bf16);
    uint4 q[kEach];
#pragma unroll
    for (int e = 0; e < kEach; ++e)
        if (e * threads + tid < kVecs) q[e] = src[e * threads + tid];
    if (tid < kNrcHidden * kNrcOut) w.w4[tid] = v.mlp[kNrcW4 + tid];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
        const int at = (e * threads + tid) * 8;
        if (at >= kNrcW4) break;
        const bool first = at < kNrcW2, second = at < kNrcW3;
        const int i = at - (first ? kNrcW1 : (second ? kNrcW2 : kNrcW3));
        const int k = i / kNrcHidden, n = i % kNrcHidden;
        uint16_t *t = first ? w.w1t : (second ? w.w2t : w.w3t);
        const int ts = first ? kXs : kHs;
        const uint32_t word[4] = {q[e].x, q[e].y, q[e].z, q[e].w};
#pragma unroll
        for (int c = 0; c < 8; ++c) t[(n + c) * ts + k] = uint16_t(word[c >> 1] >> (16 * (c & 1)));
        if (wb) *reinterpret_cast<uint4 *>((first ? wb->w1 : (second ? wb->w2 : wb->w3)) + k * kHs + n) = q[e];
    }
}

// out[16][N] = relu(in[16][K] W), in rows at `in` (stride is), wt = W^T (stride ws)
template <int K, int N>
__device__ __forceinline__ void nrc_fwd_tile(const uint16_t *in, int is, const uint16_t *wt, int ws, uint16_t *out,
                                             int lane) {
    const int r = lane & 15, q = lane >> 4;
    bf16x4 b[K / 16];
#pragma unroll
    for (int kt = 0; kt < K / 16; ++kt) b[kt] = ld4(in + r * is + kt * 16 + 4 * q);
#pragma unroll
    for (int nt = 0; nt < N / 16; ++nt) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < K / 16; ++kt) acc = mma16(ld4(wt + (nt * 16 + r) * ws + kt * 16 + 4 * q), b[kt], acc);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = short(f2bf(fmaxf(acc[e], 0.f)));
        *reinterpret_cast<bf16x4 *>(out + r * kHs + nt * 16 + 4 * q) = o;
    }
}

// y[16][3] = h[16][64] W4, in single precision, k in order
__device__ __forceinline__ void nrc_out_tile(const uint16_t *h, const float *w4, float *y, int lane) {
    if (lane < 48) {
        const int row = lane / 3, c = lane % 3;
        float acc = 0.f;
#pragma unroll
        for (int k = 0; k < kNrcHidden; k += 4) {
            const bf16x4 hv = ld4(h + row * kHs + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc += bf2f(uint16_t(hv[e])) * w4[(k + e) * kNrcOut + c];
        }
        y[row * 4 + c] = acc;
    }
}

// acc[i][j] += sum over the tile's 16 rows of A[row][i] G[row][j]; A rows at
// `a` (stride as, I columns), G at `g` (stride kHs, 64 columns)
template <int I>
__device__ __forceinline__ void nrc_weight_grad(const uint16_t *a, int as, const uint16_t *g,
                                                f32x4 (&acc)[I / 16][kNrcHidden / 16], int lane) {
    const int r = lane & 15, q = lane >> 4;
    bf16x4 gv[kNrcHidden / 16];
#pragma unroll
    for (int jt = 0; jt < kNrcHidden / 16; ++jt) gv[jt] = gather4(g + (4 * q) * kHs + jt * 16 + r, kHs);
#pragma unroll
    for (int it = 0; it < I / 16; ++it) {
        const bf16x4 av = gather4(a + (4 * q) * as + it * 16 + r, as);
#pragma unroll
        for (int jt = 0; jt < kNrcHidden / 16; ++jt) acc[it][jt] = mma16(av, gv[jt], acc[it][jt]);
    }
}

// the accumulators of nrc_weight_grad added to dw[I][64] in LDS
template <int I>
__device__ __forceinline__ void nrc_add_weight_grad(const f32x4 (&acc)[I / 16][kNrcHidden / 16], float *dw, int lane) {
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int it = 0; it < I / 16; ++it)
#pragma unroll
        for (int jt = 0; jt < kNrcHidden / 16; ++jt)
#pragma unroll
            for (int e = 0; e < 4; ++e) atomicAdd(dw + (it * 16 + 4 * q + e) * kNrcHidden + jt * 16 + r, acc[it][jt][e]);
}

// G[16][64] W^T for W[J][64] (stride kHs): times relu'(h) into h itself, or
// (h null) into out[16][J], the rows whose bit in `rows` is set
template <int J>
__device__ __forceinline__ void nrc_input_grad(const uint16_t *g, const uint16_t *w, uint16_t *h, float *out,
                                               uint32_t rows, int lane) {
    const int r = lane & 15, q = lane >> 4;
    bf16x4 b[kNrcHidden / 16];
#pragma unroll
    for (int kt = 0; kt < kNrcHidden / 16; ++kt) b[kt] = ld4(g + r * kHs + kt * 16 + 4 * q);
#pragma unroll
    for (int jt = 0; jt < J / 16; ++jt) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < kNrcHidden / 16; ++kt)
            acc = mma16(ld4(w + (jt * 16 + r) * kHs + kt * 16 + 4 * q), b[kt], acc);
        if (h) {
            uint16_t *at = h + r * kHs + jt * 16 + 4 * q;
            const bf16x4 hv = ld4(at);
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = short(f2bf(bf2f(uint16_t(hv[e])) > 0.f ? acc[e] : 0.f));
            *reinterpret_cast<bf16x4 *>(at) = o;
        } else if ((rows >> r) & 1u) {
            *reinterpret_cast<f32x4 *>(out + r * J + jt * 16 + 4 * q) = acc;
        }
    }
}

}// namespace dev
}// namespace vs
