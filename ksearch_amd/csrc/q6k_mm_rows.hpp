// The GEMM over Q6_K weights and a few bf16 rows, Y[t, r] = sum_c deq(W[r, c]) * X[t, c]: every wave converts its own 32 weight
// rows and multiplies them with fragments of 32 or 64 rows of X that the workgroup converts and shares in LDS.  Products, their
// order and so the results' bits are q6k_mul_mm_kernel's, whose 128 tokens a workgroup are mostly padding then.
//
// What bounds it: the vector instructions (640 a superblock and wave for 64 tokens, 5.1 of some 7 thousand cycles with two waves a
// SIMD; the matrix instructions 2).  What bounded the first form was the rate of L1: a row a lane, at the odd addresses of
// blocks of 210 bytes, cost 186 cycles a load.  So a wave loads 16-byte pieces at 16-byte addresses, lane after lane along the
// rows, and passes them through LDS.  (The 128-token tile as it was -> this kernel now) 2 tokens, 12288 x 6144 41.0 -> 23.6 us, 32
// tokens 45.3 -> 28.0, 64 tokens 47.1 -> 35.9; 20 tokens, 4096 x 2048 11.2 -> 8.7; 77 tokens, 1000 x 3072 13.0 -> 10.4; 300
// tokens, 12288 x 1536 49.0 -> 34.3.  Beyond (512 tokens, 8192 x 2048 30.8 in that tile or 40.9 here) converting for 64 tokens is
// the dearer way, and for 128 here one wave a SIMD is left.
#pragma once
#include "ksh_device.hpp"
#include "ksh_internal.hpp"

namespace ksh {
namespace {

// A workgroup has TM = 32 MT tokens x 128 weight rows: four waves of 32 rows each.
template <int MT_>
struct Mm6Rows {
    static constexpr int MT = MT_, TM = 32 * MT, TN = 128, kThreads = 256;
    static constexpr int kHalf = 512 + 16, kFrag = 2 * kHalf;   // bytes of a fragment's half (eight writes of a row in eight places)
    static constexpr int kStage = MT * 4 * kFrag;           // 64 columns: [token tile][k slice][lane][16]
    static constexpr int kLds = 2 * kStage + 4 * Q6Way::kBytes;
};

template <int MT_>
__global__ __launch_bounds__(256, 2) void q6k_mm_rows_kernel(MmParams p)
{
    using S = Mm6Rows<MT_>;
    constexpr int MT = MT_;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds6[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 31, h = lane >> 5;
    int by = blockIdx.y, ycol = 0;
    const int rows_all = p.rows + p.rows1 + p.rows2;
    if (p.rows1) {
        const int ty0 = (p.rows + S::TN - 1) / S::TN, ty1 = (p.rows1 + S::TN - 1) / S::TN;
        if (by >= ty0 + ty1) { by -= ty0 + ty1; ycol = p.rows + p.rows1; p.W = p.W2; p.Y = p.Y2; p.rows = p.rows2; }
        else if (by >= ty0) { by -= ty0; ycol = p.rows; p.W = p.W1; p.Y = p.Y1; p.rows = p.rows1; }
    }
    const int t0 = blockIdx.x * S::TM, r0 = by * S::TN + wave * 32;
    const int nsb_row = p.cols / 256;
    int nsb = nsb_row, sb0 = 0;
    size_t ystride = (size_t)p.rows;
    if (p.ksplit) {
        const int slice = blockIdx.z;
        sb0 = nsb_row * slice / p.ksplit;
        nsb = nsb_row * (slice + 1) / p.ksplit - sb0;
        p.Y = p.Y_parts + (size_t)slice * p.batch * rows_all + ycol;   // partial sums: all matrices' columns side by side
        ystride = (size_t)rows_all;
    }
    const int nsteps = 4 * nsb;

    // ---- rows of X: a thread has eight columns of MT rows of a step of 64
    const int xq = tid & 7, xt = tid >> 3;
    const uint8_t *xsrc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++)
        xsrc[i] = reinterpret_cast<const uint8_t *>(p.Xf) + ((size_t)min(t0 + xt + 32 * i, p.batch - 1) * p.cols + (size_t)sb0 * 256 + 8 * xq) * 2;
    struct XRegs { u32x4_t v[MT]; };
    auto fetch_x = [&](int step, XRegs &x) __attribute__((always_inline)) {
        const size_t off = (size_t)min(step, nsteps - 1) * 128;
#pragma unroll
        for (int i = 0; i < MT; i++) x.v[i] = *reinterpret_cast<const u32x4_t *>(xsrc[i] + off);
    };
    auto put_x = [&](int stage, const XRegs &x) __attribute__((always_inline)) {
        uint8_t *f = lds6 + stage * S::kStage + (xq >> 1) * S::kFrag + (xq & 1) * S::kHalf + xt * 16;
#pragma unroll
        for (int i = 0; i < MT; i++) *reinterpret_cast<h8 *>(f + 4 * i * S::kFrag) = from_bf16(__builtin_bit_cast(h8, x.v[i]));
    };

    // ---- weights
    const Q6Way rows(p.W, r0, p.rows, nsb_row, sb0, nsb, lds6 + 2 * S::kStage + wave * Q6Way::kBytes, lane);
    // lane (lm, h): bytes 8h .. 8h+7 of every 16 of its row's codes, the scales, d
    struct WRegs { uint32_t ql[8][2], qh[4][2], sc[4], d; };
    auto take_w = [&](int sb, WRegs &w) __attribute__((always_inline)) {
        uint32_t bits;
        const uint32_t *q = rows.row(sb, lm, bits);
#pragma unroll
        for (int i = 0; i < 8; i++) q6_words<2>(q, bits, 4 * i + 2 * h, w.ql[i]);
#pragma unroll
        for (int i = 0; i < 4; i++) q6_words<2>(q, bits, 32 + 4 * i + 2 * h, w.qh[i]);
        q6_words<4>(q, bits, 48, w.sc);
        w.d = (q[52] >> bits) & 0xFFFFu;
    };

    f16v F[MT], C[MT];
    const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < MT; mt++) F[mt] = C[mt] = kZero16;
    const uint8_t *fr = lds6 + h * S::kHalf + lm * 16;

    XRegs x[4];
    Q6Way::Pieces wp;
    WRegs w;
    fetch_x(0, x[0]);
    rows.fetch(0, wp);
    fetch_x(1, x[1]);
    fetch_x(2, x[2]);
    fetch_x(3, x[3]);
    put_x(0, x[0]);
    rows.put(wp);
    take_w(0, w);
    __syncthreads();
    auto step_body = [&](int sb, auto gtag) __attribute__((always_inline)) {
        constexpr int g = decltype(gtag)::value, H = g >> 1, P = g & 1;
        const int step = 4 * sb + g;
        fetch_x(step + 4, x[g]);
        if (g == 0) rows.fetch(sb + 1, wp);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t sc4 = w.sc[g];
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            h8 a[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) a[mt] = *reinterpret_cast<const h8 *>(fr + (g & 1) * S::kStage + (mt * 4 + ks) * S::kFrag);
            const h2 s2 = q6_scale((int8_t)(sc4 >> (8 * ks))), off2 = s2 * kQ6Offset;
            u32x4_t o;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t L = w.ql[4 * H + ks][i], Q = w.qh[2 * H + (ks & 1)][i];
                const int sh = 4 * P + 2 * (ks >> 1);
                const uint32_t hi = sh < 4 ? Q << (4 - sh) : Q >> (sh - 4);
                const uint32_t c = (hi & 0x30303030u) | ((P ? L >> 4 : L) & 0x0F0F0F0Fu);
                o[2 * i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, c, 0x0C020C00u)), s2, off2));
                o[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, c, 0x0C030C01u)), s2, off2));
            }
            const h8 b = __builtin_bit_cast(h8, o);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                C[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt], b, (g == 0 && ks == 0) ? kZero16 : C[mt], 0, 0, 0);
            if (ks == 1) put_x((g + 1) & 1, x[(g + 1) & 3]);
        }
        if (g == 3) {
            const float d = half_bits_to_f32(w.d) * kQ6Unit;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 16; i++) F[mt][i] = fmaf(d, C[mt][i], F[mt][i]);
            rows.put(wp);
            take_w(sb + 1, w);
        }
        __syncthreads();
    };
    for (int sb = 0; sb < nsb; sb++) {
        step_body(sb, std::integral_constant<int, 0>{});
        step_body(sb, std::integral_constant<int, 1>{});
        step_body(sb, std::integral_constant<int, 2>{});
        step_body(sb, std::integral_constant<int, 3>{});
    }
    const int r = r0 + lm;
    if (r >= p.rows) return;
    auto store = [&](auto keep) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int tb = t0 + mt * 32 + 4 * h, left = p.batch - tb;
            float *y = p.Y + (size_t)tb * ystride + r;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = 8 * (i / 4) + (i & 3);
                if (t < left) mm_store<decltype(keep)::value>(&y[(size_t)t * ystride], (float)F[mt][i]);
            }
        }
    };
    if (p.keep) store(std::true_type{});
    else store(std::false_type{});
}

}  // namespace
}  // namespace ksh
