// What a GEMV workgroup does before it touches its weights' values: produce the
// activation vector in LDS.  Three sources, selected at run time:
//
//   kPlain      x as given                                   (Matvec, MatvecQkv, MatvecGateUpGelu)
//   kRms        (x * rsqrt(mean(x^2)+eps)) * w_norm          (RmsNormMatvec*, kernel.rs:303-339)
//   kAddThenRms x_new = res + (y*inv)*w_post, written back by workgroup 0 as the
//               residual stream, then (x_new*inv2)*w_norm     (RmsNormAddThenRmsNorm, lower.rs:3926-4077,
//               folded into the consumer GEMV)
//   kMergeParts the merge of a split-KV attention's partitions (SdpaMwgReduce,
//               lower.rs:5897-6087): x = sum_p w_p o_p / sum_p w_p l_p with
//               w_p = exp(m_p - max m); one float4 per thread, no reduction
//
// and two LDS formats, selected at compile time:
//
//   F32   floats with 4 of padding per 64 (lane stride 68 dwords: conflict-free b128 reads)
//   I8x3  per 32-element sub-block a scale s = amax/(2^20-1) and X = rint(x/s) as three
//         balanced base-128 int8 digits (X = 16384 h + 128 m + l), laid out per 64
//         elements as H[64] M[64] L[64] + 16 bytes of padding (lane stride 52 dwords),
//         followed by s[] and the exact f32 sub-block sums Sx[].  |x - s X| <= s/2, i.e.
//         2^-21 of the sub-block's largest magnitude: below f32 summation noise of a
//         2048-term dot, so the integer dot products (exact) keep f32-class accuracy.
//   I8x2  the same with s = amax/32767 and two digits, X = 256 m + l with m a signed and l an unsigned byte (the
//         nibbles are non-negative, so l meets them in the unsigned dot instruction), M[64] L[64] + 16 bytes of
//         padding per 64 elements (lane stride 36 dwords): |x - s X| <= 2^-16 of the sub-block's largest magnitude
//         -- finer than the half-precision activations of the reference -- for a third fewer integer dot
//         instructions per weight.
#pragma once

#include "ksh_device.hpp"

namespace ksh {

enum { kPlain = 0, kRms = 1, kAddThenRms = 2, kMergeParts = 3 };
constexpr int kMergeMaxParts = 8;
enum { kXF32 = 0, kXI2 = 2, kXI8 = 3, kXQ6 = 6 };

struct Prologue {
    const float *x;        // kPlain/kRms: the vector; kAddThenRms: y; kMergeParts: o[heads][nwg][hd]
    const float *w_norm;   // kRms / kAddThenRms; kMergeParts: (m, l)[heads][nwg]
    const float *w_post;   // kAddThenRms
    const float *res;      // kAddThenRms
    float *x_out;          // kAddThenRms: residual stream out
    float eps;
    int kind;
    int nwg, hd_log2;      // kMergeParts.  kAddThenRms: nwg carries the bits of the stream scale s, x_out = s * (res + rms(y) * w_post)
};

__host__ __device__ constexpr int xs_f32_floats(int cols) { return cols + (cols >> 6) * 4; }
__host__ __device__ constexpr int xs_i8_bytes(int cols) { return (cols >> 6) * 208 + (cols >> 5) * 8; }
__host__ __device__ constexpr int xs_i2_bytes(int cols) { return (cols >> 6) * 144 + (cols >> 5) * 8; }
__device__ __forceinline__ int xs_f32_index(int e) { return e + ((e >> 6) << 2); }

// Q6 planes: per 128 elements H[128] M[128] L[128], then for each run of 8
// elements minus the sum of its X (int32 x 16), then the scale (one per 128).
constexpr int kQ6HalfBytes = 464;
__host__ __device__ constexpr int xs_q6_bytes(int cols) { return (cols >> 7) * kQ6HalfBytes; }

template <int XF>
__host__ __device__ constexpr size_t xs_image_bytes(int cols)
{
    return XF == kXI8 ? (size_t)xs_i8_bytes(cols) : XF == kXI2 ? (size_t)xs_i2_bytes(cols) : XF == kXQ6 ? (size_t)xs_q6_bytes(cols) : (size_t)xs_f32_floats(cols) * 4;
}
template <int XF>
__host__ __device__ constexpr size_t xs_bytes(int cols)
{
    return xs_image_bytes<XF>(cols) + 128;   // + reduction scratch (4 sums x up to 8 waves)
}

// max / sum over 8 consecutive lanes (one 32-element sub-block at 4 elements per lane)
__device__ __forceinline__ float oct_max(float v)
{
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    return fmaxf(v, dpp_f32<0x141>(v));
}
__device__ __forceinline__ float oct_sum(float v)
{
    v += dpp_f32<0xB1>(v);
    v += dpp_f32<0x4E>(v);
    return v + dpp_f32<0x141>(v);
}

template <int NT>
__device__ __forceinline__ float block_sum(float v, float *red)
{
    const float w = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = w;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) s += red[i];
    return s;
}

__device__ __forceinline__ uint32_t pack4_i8(int a, int b, int c, int d)
{
    return ((uint32_t)a & 0xFFu) | (((uint32_t)b & 0xFFu) << 8) | (((uint32_t)c & 0xFFu) << 16) | ((uint32_t)d << 24);
}

// one float4 (elements 4i..4i+3) into the LDS image
template <int XF>
__device__ __forceinline__ void store_x4(uint8_t *lds, int cols, int i, float4 v)
{
    if (XF == kXF32) {
        *reinterpret_cast<float4 *>(reinterpret_cast<float *>(lds) + xs_f32_index(i * 4)) = v;
        return;
    }
    if (XF == kXQ6) {
        // 32 consecutive lanes hold one run of 128 elements: one scale for the run
        float amax = oct_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        amax = fmaxf(amax, dpp_f32<0x140>(amax));                 // row_mirror: the other 8 of the 16-lane row
        amax = fmaxf(amax, __shfl_xor(amax, 16, 64));             // the other row of the 32
        const float inv = amax > 0.f ? 1048575.0f / amax : 0.f;
        const float xs4[4] = {v.x, v.y, v.z, v.w};
        int h[4], m[4], l[4], sx = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int X = (int)rintf(xs4[k] * inv);
            sx += X;
            l[k] = (X << 25) >> 25;
            const int X1 = (X - l[k]) >> 7;
            m[k] = (X1 << 25) >> 25;
            h[k] = (X1 - m[k]) >> 7;
        }
        sx += __builtin_amdgcn_update_dpp(0, sx, 0xB1, 0xF, 0xF, true);   // the neighbour's four: a run of 8
        uint8_t *half = lds + (i >> 5) * kQ6HalfBytes;
        const int o = (i & 31) * 4;
        *reinterpret_cast<uint32_t *>(half + o) = pack4_i8(h[0], h[1], h[2], h[3]);
        *reinterpret_cast<uint32_t *>(half + 128 + o) = pack4_i8(m[0], m[1], m[2], m[3]);
        *reinterpret_cast<uint32_t *>(half + 256 + o) = pack4_i8(l[0], l[1], l[2], l[3]);
        if ((i & 1) == 0) reinterpret_cast<int *>(half + 384)[(i & 31) >> 1] = -sx;
        if ((i & 31) == 0) *reinterpret_cast<float *>(half + 448) = amax * (1.0f / 1048575.0f);
        return;
    }
    const float amax = oct_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    const float sum = oct_sum((v.x + v.y) + (v.z + v.w));
    if (XF == kXI2) {
        const float inv = amax > 0.f ? 32767.0f / amax : 0.f;
        const float xs4[4] = {v.x, v.y, v.z, v.w};
        int m[4], l[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int X = (int)rintf(xs4[k] * inv);
            l[k] = X & 255;
            m[k] = X >> 8;
        }
        uint8_t *chunk = lds + (i >> 4) * 144 + (i & 15) * 4;
        *reinterpret_cast<uint32_t *>(chunk) = pack4_i8(m[0], m[1], m[2], m[3]);
        *reinterpret_cast<uint32_t *>(chunk + 64) = pack4_i8(l[0], l[1], l[2], l[3]);
        if ((threadIdx.x & 7) == 0) {
            float *sc = reinterpret_cast<float *>(lds + (cols >> 6) * 144);
            sc[2 * (i >> 3)] = amax * (1.0f / 32767.0f);
            sc[2 * (i >> 3) + 1] = sum;
        }
        return;
    }
    const float inv = amax > 0.f ? 1048575.0f / amax : 0.f;
    const float s = amax * (1.0f / 1048575.0f);
    const float xs4[4] = {v.x, v.y, v.z, v.w};
    int h[4], m[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int X = (int)rintf(xs4[k] * inv);
        l[k] = (X << 25) >> 25;
        const int X1 = (X - l[k]) >> 7;
        m[k] = (X1 << 25) >> 25;
        h[k] = (X1 - m[k]) >> 7;
    }
    uint8_t *chunk = lds + (i >> 4) * 208 + (i & 15) * 4;
    *reinterpret_cast<uint32_t *>(chunk) = pack4_i8(h[0], h[1], h[2], h[3]);
    *reinterpret_cast<uint32_t *>(chunk + 64) = pack4_i8(m[0], m[1], m[2], m[3]);
    *reinterpret_cast<uint32_t *>(chunk + 128) = pack4_i8(l[0], l[1], l[2], l[3]);
    if ((threadIdx.x & 7) == 0) {
        float *sc = reinterpret_cast<float *>(lds + (cols >> 6) * 208);
        sc[2 * (i >> 3)] = s;
        sc[2 * (i >> 3) + 1] = sum;
    }
}

// Staging is split in two so that a GEMV can put its weight loads between the
// halves: vector memory loads return in issue order within a wave, so whatever
// is fetched after the (HBM-cold) weights also waits for them.  stage_fetch
// issues every load the prologue needs (the vector and the norm weights are
// L2-resident after the first workgroup), the caller then issues its weight
// loads, and stage_finish does the arithmetic and the LDS writes while the
// weights are still in flight.
constexpr int kStageX = 8;   // float4 per thread of x kept in registers (plain: longer vectors stream later)
constexpr int kStageP = 4;   // float4 per thread of w_norm / w_post / res (normalising prologues; host-checked)

struct StageRegs {
    float4 x[kStageX];
    float4 wn[kStageP], wp[kStageP], rs[kStageP];
};

// kMerge: whether the kernel is built with the kMergeParts source at all (the Q4_K kernels' prologue instances are)
// KMAX: a compile-time bound on the float4 per thread (kernels built for a fixed row length): what lies past it
// takes no registers, which is what decides the occupancy of the long-running LM head.
// KIND: the prologue kind when the kernel is built for one (-1: read from the descriptor at run time).  With it and a
// row length known at compile time the front of the kernel is a straight run of loads with constant offsets; with
// neither it is a chain of compare-and-branch pairs, one per possible float4, in front of the first weight load.
// H: the vectors (x, norm weights, residual, x_out) are half buffers; the partitions of kMergeParts stay f32.
template <int NT, bool kMerge = false, int KMAX = kStageX, int KIND = -1, bool H = false>
__device__ __forceinline__ void stage_fetch(const Prologue &pr_in, int cols, StageRegs &s)
{
    Prologue pr = pr_in;
    if (KIND >= 0) pr.kind = KIND;
    constexpr int KX = KMAX < kStageX ? KMAX : kStageX, KP = KMAX < kStageP ? KMAX : kStageP;
    // n4 is a multiple of 64, so "this float4 exists" is a per-wave fact: keep it
    // in scalar registers and the loads stay unpredicated
    const int wbase = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63), tid = wbase + (threadIdx.x & 63), n4 = cols / 4;
    if (kMerge && pr.kind == kMergeParts) {
        // one float4 of the output per thread (host-checked: n4 <= NT, nwg <= 8): its
        // eight partitions' values and (m, l) pairs; partitions past nwg re-read the
        // last one, so that the number of loads is fixed
        if (wbase < n4) {
            // byte offsets in 32 bits against the two base pointers (the buffers are a few hundred KB): one add per load
            // where 64-bit addresses cost a shift and an add-with-carry pair each, in front of the first weight load
            const uint32_t e = (uint32_t)tid * 4, h = e >> pr.hd_log2, d = e - (h << pr.hd_log2);
            const uint32_t o0 = (((h * (uint32_t)pr.nwg) << pr.hd_log2) + d) * 4, ml0 = h * (uint32_t)pr.nwg * 8;
            const KSH_GLOBAL char *ob = (const KSH_GLOBAL char *)pr.x, *mb = (const KSH_GLOBAL char *)pr.w_norm;
            typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int q = 0; q < kMergeMaxParts; q++) {
                const f32x4_t v = *(const KSH_GLOBAL f32x4_t *)(ob + (o0 + (((uint32_t)min(q, pr.nwg - 1) << pr.hd_log2) * 4)));
                s.x[q] = make_float4(v.x, v.y, v.z, v.w);
            }
#pragma unroll
            for (int q = 0; q < kMergeMaxParts / 2; q++) {
                const f32x2_t a = *(const KSH_GLOBAL f32x2_t *)(mb + (ml0 + (uint32_t)min(2 * q, pr.nwg - 1) * 8));
                const f32x2_t b = *(const KSH_GLOBAL f32x2_t *)(mb + (ml0 + (uint32_t)min(2 * q + 1, pr.nwg - 1) * 8));
                s.wn[q] = make_float4(a.x, a.y, b.x, b.y);
            }
        }
        return;
    }
    if (KMAX >= kStageX && n4 > NT * kStageX) return;
#pragma unroll
    for (int k = 0; k < KX; k++) {
        const int i = tid + k * NT;
        if (wbase + k * NT < n4) s.x[k] = act_ld4<H>(pr.x, i);
    }
    if (pr.kind == kPlain) return;
#pragma unroll
    for (int k = 0; k < KP; k++) {
        const int i = tid + k * NT;
        if (wbase + k * NT < n4) s.wn[k] = act_ld4<H>(pr.w_norm, i);
    }
    if (pr.kind != kAddThenRms) return;
#pragma unroll
    for (int k = 0; k < KP; k++) {
        const int i = tid + k * NT;
        if (wbase + k * NT < n4) { s.wp[k] = act_ld4<H>(pr.w_post, i); s.rs[k] = act_ld4<H>(pr.res, i); }
    }
}

// Waits for what stage_fetch has asked for.  Requests straight into LDS that follow it (to_lds16) are not known to the compiler, whose
// wait in stage_finish would be for all of them; behind this there is nothing left to wait for.
template <int KMAX>
__device__ __forceinline__ void stage_arrived(StageRegs &s)
{
    constexpr int KX = KMAX < kStageX ? KMAX : kStageX, KP = KMAX < kStageP ? KMAX : kStageP;
    auto one = [](float4 &v) __attribute__((always_inline)) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); };
#pragma unroll
    for (int k = 0; k < KX; k++) one(s.x[k]);
#pragma unroll
    for (int k = 0; k < KP; k++) { one(s.wn[k]); one(s.wp[k]); one(s.rs[k]); }
}

// Every thread must call this (it contains barriers); the LDS image is complete
// after the caller's next __syncthreads().
template <int XF, int NT, bool kMerge = false, int KMAX = kStageX, int KIND = -1, bool H = false>
__device__ __forceinline__ void stage_finish(const Prologue &pr_in, uint8_t *lds, int cols, StageRegs &s)
{
    Prologue pr = pr_in;
    if (KIND >= 0) pr.kind = KIND;
    constexpr int KX = KMAX < kStageX ? KMAX : kStageX, KP = KMAX < kStageP ? KMAX : kStageP;
    const int wbase = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63), tid = wbase + (threadIdx.x & 63), n4 = cols / 4;
    float *red = reinterpret_cast<float *>(lds + xs_image_bytes<XF>(cols));
    if (kMerge && pr.kind == kMergeParts) {
        if (wbase < n4) {
            float m[kMergeMaxParts], l[kMergeMaxParts];
#pragma unroll
            for (int q = 0; q < kMergeMaxParts / 2; q++) {
                m[2 * q] = s.wn[q].x; l[2 * q] = s.wn[q].y;
                m[2 * q + 1] = s.wn[q].z; l[2 * q + 1] = s.wn[q].w;
            }
            float M = m[0];
#pragma unroll
            for (int q = 1; q < kMergeMaxParts; q++) M = fmaxf(M, m[q]);
            float L = 0.f;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int q = 0; q < kMergeMaxParts; q++) {
                const float w = q < pr.nwg ? __expf(m[q] - M) : 0.f;
                L = fmaf(w, l[q], L);
                a.x = fmaf(w, s.x[q].x, a.x);
                a.y = fmaf(w, s.x[q].y, a.y);
                a.z = fmaf(w, s.x[q].z, a.z);
                a.w = fmaf(w, s.x[q].w, a.w);
            }
            const float rl = 1.0f / L;   // (the merging attention launch divides; the two differ by an ulp)
            store_x4<XF>(lds, cols, tid, make_float4(a.x * rl, a.y * rl, a.z * rl, a.w * rl));
        }
        return;
    }
    if (pr.kind == kPlain) {
        if (KMAX >= kStageX && n4 > NT * kStageX) {
            for (int i = tid; i < n4; i += NT) store_x4<XF>(lds, cols, i, act_ld4<H>(pr.x, i));
            return;
        }
#pragma unroll
        for (int k = 0; k < KX; k++) {
            const int i = tid + k * NT;
            if (wbase + k * NT < n4) store_x4<XF>(lds, cols, i, s.x[k]);
        }
        return;
    }
    // One pass, one reduction: with a = rsqrt(mean(y^2) + eps) the second norm's sum of squares is
    //   sum (res + a*y*wp)^2 = sum res^2 + 2a sum res*(y*wp) + a^2 sum (y*wp)^2,
    // so all four sums are taken together and cross the workgroup behind a single barrier.
    float4 *v = s.x;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const bool add = pr.kind == kAddThenRms;
#pragma unroll
    for (int k = 0; k < KP; k++) {
        if (wbase + k * NT < n4) {
            const float y4[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
            const float r4[4] = {s.rs[k].x, s.rs[k].y, s.rs[k].z, s.rs[k].w};
            const float w4[4] = {s.wp[k].x, s.wp[k].y, s.wp[k].z, s.wp[k].w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc[0] = fmaf(y4[e], y4[e], acc[0]);
                if (add) {
                    const float yw = y4[e] * w4[e];
                    acc[1] = fmaf(r4[e], r4[e], acc[1]);
                    acc[2] = fmaf(r4[e], yw, acc[2]);
                    acc[3] = fmaf(yw, yw, acc[3]);
                }
            }
        }
    }
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        // (of 16 waves some have no share of a short vector: zeros to add, nothing to do behind the barrier, and a SIMD's
        // other waves waiting for what they would issue)
        const bool share = NT < 1024 || wbase < n4;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j == 0 || add) {
                const float wsum = share ? wave_sum(acc[j]) : 0.f;
                if (lane == 0) red[wave * 4 + j] = wsum;
            }
        }
        __syncthreads();   // `red` has no earlier use in the kernel, so one barrier is enough
        if (!share) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] = 0.f;
            if (j == 0 || add) {
#pragma unroll
                for (int w = 0; w < NT / 64; w++) acc[j] += red[w * 4 + j];
            }
        }
    }
    float inv = 1.0f / sqrtf(acc[0] / (float)cols + pr.eps);
    if (add) {
        const float sc = __int_as_float(pr.nwg);   // 1 except where per-layer embeddings scale the stream
#pragma unroll
        for (int k = 0; k < KP; k++) {
            const int i = tid + k * NT;
            if (wbase + k * NT < n4) {
                const float4 r = s.rs[k], w = s.wp[k];
                v[k].x = (r.x + v[k].x * inv * w.x) * sc;
                v[k].y = (r.y + v[k].y * inv * w.y) * sc;
                v[k].z = (r.z + v[k].z * inv * w.z) * sc;
                v[k].w = (r.w + v[k].w * inv * w.w) * sc;
                if (blockIdx.x == 0) act_st4<H>(pr.x_out, i, v[k]);
            }
        }
        const float ss2 = (sc * sc) * fmaf(inv * inv, acc[3], fmaf(2.0f * inv, acc[2], acc[1]));
        inv = 1.0f / sqrtf(ss2 / (float)cols + pr.eps);
    }
#pragma unroll
    for (int k = 0; k < KP; k++) {
        const int i = tid + k * NT;
        if (wbase + k * NT < n4) {
            const float4 w = s.wn[k];
            store_x4<XF>(lds, cols, i, make_float4(v[k].x * inv * w.x, v[k].y * inv * w.y, v[k].z * inv * w.z, v[k].w * inv * w.w));
        }
    }
}

}  // namespace ksh
