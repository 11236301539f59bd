// Attention of a prompt chunk's tokens (KSH_SDPA_BATCH, heads of 256 and 512, one partition): sdpa_mfma_kernel's workgroup of one
// token, or of two, T -- the same products, scores and states in the same order, the same bits.
//
// What bounds it: the vector ALU (1208 instructions a tile of a 512-wide head and wave in that kernel, 55 % of the cycles; heads
// of 256 1336, 72 %) and a wave's waits for its tile (45 and 32 % of its time).  Here K and V come straight into LDS, K of a
// wave's next tile under this one's softmax and products and V under the next one's scores, so that one set of buffers covers
// both ways, and a block's operands are read from there while the last block is worked on.
// T = 2: tokens t and t + 32 of one prompt attend the same tiles of 32 rows -- rows from the cache's start on, or windows that
// begin 32 rows apart -- and what a tile costs beside its products is paid once for the two: its way into LDS, the tables of
// block scales, the K codes as matrix operands, the V codes gathered bytewise.  q's operands stay in LDS, since the registers
// hold two tokens' accumulators.
// us, (one token in sdpa_mfma_kernel, T = 1, T = 2): heads of 512, 2048 tokens from an empty cache 452, 359, 311; 952 behind 2048
// rows 485, 379, 309; 512 49, 40.5, 40.7; 63 behind 700 41.5, 33.7, 52.7; heads of 256, window of 512, 2048 tokens 87, 75, 71; 952
// behind 2048 47, 42, 38; 699 from an empty cache 34, 30, 34.5.  The vector ALU is busy for 77 % of the cycles now (heads of 512, 2048
// tokens; 83 with heads of 256, 67 with one token to a workgroup), the matrix pipe 10.
#pragma once
// (included by sdpa_q40_lanes.hip, behind sdpa_mfma_kernel)
namespace ksh {
namespace {

template <int HD, int T>      // T tokens to a workgroup
struct SdpaPrompt {
    static constexpr int VH = HD / 256, NW = 4, WAVES = NW * VH, NB = HD / 32, NBV = 8, TRK = 32 / VH;   // (512: two waves a tile, see sdpa_mfma_kernel)
    static constexpr int ROWB = NB * 18, ROWBV = NBV * 18, KPITCH = mfma_k_pitch<HD>();
    static constexpr int kTile = 5 * 1024;                                                  // a wave's K rows, or its share of V rows, in whole kilobytes
    static constexpr int kStrip = 2 * kTile + TRK * NB * 4 + 32 * NBV * 4;                  // K | V | K scales | V scales
    static constexpr int kQ = NB * 64 * (16 + 4);                                           // q's operands and 24 * its sums, of a token
    static constexpr int kTrade = VH == 2 ? 2 * NW * 2 * 32 * 16 : 0;                       // the scores two waves trade, two buffers, of a token
    static constexpr int kState = VH * NW * 8 * 256 * 4 + NW * 8 * 2 * 4;                   // the waves' states, of a token
    static constexpr int kFront = WAVES * kStrip + T * kQ + T * kTrade;
    static constexpr int kLds = kFront > T * kState ? kFront : T * kState;
    static_assert(TRK * KPITCH <= kTile && 32 * ROWBV <= kTile && KPITCH % 16 == 0, "");
};

// LDS by address: what follows a base is in the instruction (of pointers into one array the compiler keeps dozens)
template <class T>
__device__ __forceinline__ T lds_at(uint32_t addr)
{
    return *(const __attribute__((address_space(3))) T *)(uintptr_t)addr;
}
template <class T>
__device__ __forceinline__ void lds_put(uint32_t addr, T v)
{
    *(__attribute__((address_space(3))) T *)(uintptr_t)addr = v;
}
__device__ __forceinline__ uint32_t lds_base(uint32_t addr)
{
    asm volatile("" : "+v"(addr));
    return addr;
}

template <int I, int N, class F>
__device__ __forceinline__ void each(F &f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        each<I + 1, N>(f);
    }
}

template <int HD, int T>
__global__ __launch_bounds__((SdpaPrompt<HD, T>::WAVES * 64), 2) void sdpa_prompt_kernel(LaneParams p, int n_tok)
{
    using S = SdpaPrompt<HD, T>;
    constexpr int VH = S::VH, NW = S::NW, WAVES = S::WAVES, NB = S::NB, NBV = S::NBV, TRK = S::TRK, NT = WAVES * 64;
    constexpr bool SHARE = VH == 2;
    touch_lane_params(p);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = wave % NW, vhalf = wave / NW;
    const int col = lane & 15, q4 = lane >> 4, head = col & 7, is_lo = col >> 3;
    const uint32_t odd_mask = 0u - (uint32_t)(q4 & 1);       // all ones in the lane groups whose accumulator rows are heads 4..7
    uint32_t nib_mask = 0x03C003C0u, nib_one = 0x4C004C00u;  // a nibble's place in an f16 mantissa; 16.0 twice
    asm volatile("" : "+s"(nib_mask), "+v"(nib_one));
    const uint32_t drop = is_lo ? 0xFFFFE000u : 0u;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds_raw, at_lds = lds0 + (uint32_t)(wave * S::kStrip);
    constexpr uint32_t kScK = 2 * S::kTile, kScV = kScK + TRK * NB * 4, kAtQ = WAVES * S::kStrip, kAtTrade = kAtQ + T * S::kQ;
    constexpr int KB = 64 / TRK;                             // blocks whose K scales a pass of the wave turns over
    const uint32_t kcode = lds_base(at_lds + col * S::KPITCH + 4 * q4 + 2), kscale = lds_base(at_lds + kScK + 16 * q4);
    const uint32_t vcode = lds_base(at_lds + S::kTile + 4 * q4 * S::ROWBV + col + 2), vscale = lds_base(at_lds + kScV + 16 * q4);
    const uint32_t kraw = lds_base(at_lds + (lane % TRK) * S::KPITCH + 18 * (lane / TRK)), kout = lds_base(at_lds + kScK + 4 * lane);
    const uint32_t vraw = lds_base(at_lds + S::kTile + (lane & 31) * S::ROWBV + 18 * (lane >> 5)), vout = lds_base(at_lds + kScV + 4 * lane);
    const uint32_t qop_at = lds_base(lds0 + kAtQ + 16 * lane), qsum_at = lds_base(lds0 + kAtQ + NB * 1024 + 4 * lane);

    const int kvh = blockIdx.y, groups = p.groups, head0 = kvh * groups;
    const size_t row_stride = (size_t)p.n_kv * S::ROWB;
    const size_t slot_bytes = p.kv_shared ? 0 : p.slot_stride ? p.slot_stride : (size_t)p.max_t * p.n_kv * S::ROWB;
    struct Token { int tok, len, start; size_t slot; };
    auto token = [&](int tok) __attribute__((always_inline)) {
        Token t;
        t.tok = tok;
        if (p.kv_shared) {
            // (crates/ksearch_codegen/src/lower.rs:4961-4983): meta = {rows attended by token 0, -, window}
            const int abs_t = (int)p.meta[0] + tok;
            t.len = min(abs_t, (int)p.meta[2]);
            t.start = abs_t - t.len;
            t.slot = 0;
        } else {
            t.len = (int)p.meta[(size_t)tok * p.meta_stride];
            t.start = (int)p.meta[(size_t)tok * p.meta_stride + 1];
            t.slot = p.slot_ids ? (size_t)max((int)p.slot_ids[tok], 0) : (size_t)tok;
        }
        return t;
    };
    // T = 2: workgroups 0 .. pairs - 1 have a pair's tokens, where the tiles of one are tiles of the other, else the first of
    // them, and workgroup `pairs` on has the second
    Token A, B;
    bool joint = false;
    if (T == 2) {
        const int pairs = (int)gridDim.z / 2, pair = (int)blockIdx.z % pairs, tok0 = (pair >> 5) * 64 + (pair & 31);
        if (tok0 >= n_tok) return;
        A = token(tok0);
        B = token(min(tok0 + 32, n_tok - 1));
        const int apart = B.start - A.start;
        const bool two = tok0 + 32 < n_tok, together = two && B.slot == A.slot && (apart == 0 || apart == 32);
        if ((int)blockIdx.z >= pairs) {
            if (together || !two) return;
            A = B;
        } else
            joint = together;
    } else
        A = B = token((int)blockIdx.z);
    const int delta = joint ? (B.start - A.start) / 32 : 0;   // B's first tile among A's
    int len[T];
    len[0] = A.len;
    if (T == 2) len[T - 1] = joint ? B.len : 0;

    // this lane's pieces of a wave's K and V rows
    constexpr int KPR = S::KPITCH / 16;                       // (with the padding: asked for again, never read)
    uint32_t koff[5], voff[SHARE ? 5 : 1];
    auto k_row = [&](int i, int l) __attribute__((always_inline)) { return min((64 * i + l) / KPR, TRK - 1) + TRK * vhalf; };
    auto k_piece = [&](int i, int l) __attribute__((always_inline)) { return 16u * (uint32_t)min((64 * i + l) % KPR, S::ROWB / 16 - 1); };
    auto v_row = [&](int i, int l) __attribute__((always_inline)) { return min((64 * i + l) / 9, 31); };
    auto v_piece = [&](int i, int l) __attribute__((always_inline)) { return 16u * (uint32_t)((64 * i + l) % 9); };
#pragma unroll
    for (int i = 0; i < 5; i++) {
        koff[i] = (uint32_t)k_row(i, lane) * (uint32_t)row_stride + k_piece(i, lane);
        if (SHARE) voff[i] = (uint32_t)v_row(i, lane) * (uint32_t)row_stride + v_piece(i, lane);
    }

    {
        const int rows = T == 2 && len[T - 1] ? max(len[0], 32 * delta + len[T - 1]) : len[0];
        const uint8_t *kbase = p.k + A.slot * slot_bytes + (size_t)kvh * S::ROWB + (size_t)A.start * row_stride;
        const uint8_t *vbase = p.v + A.slot * slot_bytes + (size_t)kvh * S::ROWB + (size_t)A.start * row_stride + (size_t)vhalf * S::ROWBV;
        const int ntiles = (rows + 31) / 32, nsteps = (ntiles + NW - 1) / NW;    // the same for every wave: the barriers below are uniform

        // a wave's tile R, straight into LDS: five requests each (rows past the end: the last row again; always issued, since
        // arrivals are known by the number of younger requests)
        auto ask = [&](const uint8_t *base, const uint32_t *off, bool k, int R, uint32_t dst) __attribute__((always_inline)) {
            const int r0 = 32 * min(R, ntiles - 1);
            const uint8_t *b = base + (size_t)r0 * row_stride;
            if (r0 + 32 <= rows) {
#pragma unroll
                for (int i = 0; i < 5; i++) to_lds16(b, off[i], dst + 1024u * i);
            } else {
                int l = lane;
                asm volatile("" : "+v"(l));                   // (worked out here, not kept in registers through the loop)
#pragma unroll
                for (int i = 0; i < 5; i++) {
                    const uint32_t o = k ? (uint32_t)min(k_row(i, l), rows - 1 - r0) * (uint32_t)row_stride + k_piece(i, l)
                                         : (uint32_t)min(v_row(i, l), rows - 1 - r0) * (uint32_t)row_stride + v_piece(i, l);
                    to_lds16(b, o, dst + 1024u * i);
                }
            }
        };
        auto ask_k = [&](int R) __attribute__((always_inline)) { ask(kbase, koff, true, R, at_lds); };
        auto ask_v = [&](int R) __attribute__((always_inline)) { ask(vbase, SHARE ? voff : koff, SHARE ? false : true, R, at_lds + S::kTile); };

        if (ntiles > 0) {
            ask_k(tile);
            ask_v(tile);
        }
        // ---- q: the B operands of the score products and 24 * sum_b(q), as in sdpa_mfma_kernel; wave w prepares blocks w, w + WAVES, ...
        {
            constexpr int QPW = NB / WAVES;
            const bool have = head < groups;
#pragma unroll
            for (int k = 0; k < T; k++) {
                const float *qh = p.q + ((size_t)(k && joint ? B.tok : A.tok) * p.n_q + head0 + min(head, groups - 1)) * HD;
                float4 qlo[QPW], qhi[QPW];
#pragma unroll
                for (int u = 0; u < QPW; u++) {
                    const int b = wave + WAVES * u;
                    qlo[u] = *reinterpret_cast<const float4 *>(qh + 32 * b + 4 * q4);
                    qhi[u] = *reinterpret_cast<const float4 *>(qh + 32 * b + 16 + 4 * q4);
                }
#pragma unroll
                for (int u = 0; u < QPW; u++) {
                    const int b = wave + WAVES * u;
                    const float4 lo4 = qlo[u], hi4 = qhi[u];
                    const float x[8] = {lo4.x, lo4.z, hi4.x, hi4.z, lo4.y, lo4.w, hi4.y, hi4.w};       // slot order (mfma_k_elem)
                    h8v op;
                    float sum = 0.f;
#pragma unroll
                    for (int s2 = 0; s2 < 8; s2++) {
                        const float xs = pinned(have ? x[s2] * p.scale : 0.f);
                        const _Float16 hi = (_Float16)xs;
                        const _Float16 lo = (_Float16)(xs - (float)hi);
                        const _Float16 v = is_lo ? lo : hi;
                        op[s2] = v;
                        sum += (float)v;
                    }
                    sum = xor32_sum(xor16_sum(sum));
                    lds_put<h8v>(qop_at + k * S::kQ + b * 1024, op);
                    lds_put<float>(qsum_at + k * S::kQ + b * 256, 24.f * sum);
                }
            }
            __syncthreads();
        }

        f4v O[T][2 * NBV];
        float Tl[T][NBV], m_run[T], l_run[T];
#pragma unroll
        for (int k = 0; k < T; k++) {
#pragma unroll
            for (int c = 0; c < 2 * NBV; c++) O[k][c] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int b = 0; b < NBV; b++) Tl[k][b] = 0.f;
            m_run[k] = -1.0e30f;
            l_run[k] = 0.f;
        }
        float sv[T][8];                                       // scores, then probabilities, of a lane's eight rows

        // ---- scores of the wave's rows: lane (col, q4) ends up with rows 4*q4 + r of each half
        auto scores = [&](const int (&kvalid)[T], bool second_too) __attribute__((always_inline)) {
            float acc[T][TRK / 16][4];
#pragma unroll
            for (int k = 0; k < T; k++)
#pragma unroll
                for (int t = 0; t < TRK / 16; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[k][t][r] = 0.f;
            struct Operands { f4v dk[TRK / 16]; uint32_t lo[TRK / 16], hi[TRK / 16]; h8v q[T]; float q24[T]; } op[2];
            // (a block's operands are on their way while the last block's are worked on: the compiler, left to itself, asks for
            // everything at once and keeps it in memory or, held to a block at a time, for a block's operands when it needs them)
            constexpr int ASKS = 3 * (TRK / 16) + T + 1;    // (q24 of two tokens is one operation)
            auto ask_block = [&](auto btag) __attribute__((always_inline)) {
                constexpr int b = decltype(btag)::value;
                Operands &o = op[b & 1];
                auto half = [&](auto ttag) __attribute__((always_inline)) {
                    constexpr int t = decltype(ttag)::value;
                    lds_ask_wide<16 * t * S::KPITCH + 18 * b, uint16_t>(o.lo[t], kcode);
                    lds_ask_wide<16 * t * S::KPITCH + 18 * b + 2, uint16_t>(o.hi[t], kcode);
                    lds_ask<(b * TRK + 16 * t) * 4>(o.dk[t], kscale);
                };
                each<0, TRK / 16>(half);
                lds_ask<b * 1024>(o.q[0], qop_at);
                lds_ask<b * 256>(o.q24[0], qsum_at);
                if constexpr (T == 2) {
                    lds_ask<S::kQ + b * 1024>(o.q[T - 1], qop_at);
                    lds_ask<S::kQ + b * 256>(o.q24[T - 1], qsum_at);
                }
            };
            ask_block(std::integral_constant<int, 0>{});
            auto block = [&](auto btag) __attribute__((always_inline)) {
                constexpr int b = decltype(btag)::value;
                if constexpr (b + 1 < NB) ask_block(std::integral_constant<int, b + 1>{});
                lds_left<b + 1 < NB ? ASKS : 0>();
                Operands &o = op[b & 1];
                h8v codes[TRK / 16];
#pragma unroll
                for (int t = 0; t < TRK / 16; t++) arrived(o.dk[t]);
#pragma unroll
                for (int k = 0; k < T; k++) { arrived(o.q[k]); arrived(o.q24[k]); }
#pragma unroll
                for (int t = 0; t < TRK / 16; t++) codes[t] = nibbles_f16(o.lo[t] | (o.hi[t] << 16), nib_mask, nib_one);
#pragma unroll
                for (int k = 0; k < T; k++) {
                    if (k && !second_too) break;
#pragma unroll
                    for (int t = 0; t < TRK / 16; t++) {
                        const f4v c = __builtin_amdgcn_mfma_f32_16x16x32_f16(codes[t], o.q[k], f4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[k][t][r] = fmaf(o.dk[t][r], c[r] - o.q24[k], acc[k][t][r]);
                        // (taken here: put off to behind the branches, sixteen products wait in registers)
                        asm volatile("" : "+v"(acc[k][t][0]), "+v"(acc[k][t][1]), "+v"(acc[k][t][2]), "+v"(acc[k][t][3]));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);      // (blocks run into each other cost registers that two tokens' states need)
            };
            each<0, NB>(block);
#pragma unroll
            for (int k = 0; k < T; k++)
#pragma unroll
                for (int t = 0; t < TRK / 16; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float tot = acc[k][t][r] + dpp_f32<0x128>(acc[k][t][r]);        // hi + lo column (row_ror:8)
                        sv[k][4 * t + r] = (16 * t + 4 * q4 + r) < kvalid[k] ? tot : -1.0e30f;
                    }
        };
        // ---- V's block scales, 0 past the end
        auto v_scales = [&](int nvalid) __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < 32 * NBV / 64; u++) {
                const float d = pinned(half_bits_to_f32(lds_at<uint16_t>(vraw + 36 * u)));
                lds_put<float>(vout + 256 * u, (lane & 31) < nvalid ? d : 0.f);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        // ---- online softmax of a token's tile
        auto softmax = [&](auto ktag, int nvalid) __attribute__((always_inline)) {
            constexpr int k = decltype(ktag)::value;
            float mt = sv[k][0];
#pragma unroll
            for (int i = 1; i < 8; i++) mt = fmaxf(mt, sv[k][i]);
            mt = xor32_max(xor16_max(mt));
            const float m_new = fmaxf(m_run[k], mt);
            const float alpha = __expf(m_run[k] - m_new);
            float ls = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int row = 16 * (i >> 2) + 4 * q4 + (i & 3);
                sv[k][i] = row < nvalid ? __expf(sv[k][i] - m_new) : 0.f;
                ls += sv[k][i];
            }
            l_run[k] = fmaf(l_run[k], alpha, ls);
            m_run[k] = m_new;
            float ah[8];
#pragma unroll
            for (int h = 0; h < 8; h++) ah[h] = as_f32((uint32_t)__builtin_amdgcn_readlane((int)as_u32(alpha), h));
            bool rescale = false;
#pragma unroll
            for (int h = 0; h < 8; h++) rescale = rescale || ah[h] != 1.0f;
            if (rescale) {
                float ar[4];
#pragma unroll
                for (int r = 0; r < 4; r++) ar[r] = as_f32((as_u32(ah[r]) & ~odd_mask) | (as_u32(ah[4 + r]) & odd_mask));
#pragma unroll
                for (int c = 0; c < 2 * NBV; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) O[k][c][r] *= ar[r];
            }
#pragma unroll
            for (int b = 0; b < NBV; b++) Tl[k][b] *= alpha;
        };
        // ---- P.V per block, for the tokens of the mask
        auto products = [&](int of) __attribute__((always_inline)) {
            struct Operands { f4v d[2]; uint32_t a[4], b[4]; } op[2];
            constexpr int ASKS = 10;
            auto ask_block = [&](auto btag) __attribute__((always_inline)) {
                constexpr int b = decltype(btag)::value;
                Operands &o = op[b & 1];
                auto rows2 = [&](auto itag) __attribute__((always_inline)) {
                    constexpr int i = decltype(itag)::value, at = (16 * ((2 * i) >> 2) + ((2 * i) & 3)) * S::ROWBV + 18 * b;
                    lds_ask_wide<at, uint8_t>(o.a[i], vcode);
                    lds_ask_wide<at + S::ROWBV, uint8_t>(o.b[i], vcode);
                };
                each<0, 4>(rows2);
                lds_ask<b * 128>(o.d[0], vscale);
                lds_ask<b * 128 + 64>(o.d[1], vscale);
            };
            ask_block(std::integral_constant<int, 0>{});
            auto block = [&](auto btag) __attribute__((always_inline)) {
                constexpr int b = decltype(btag)::value;
                if constexpr (b + 1 < NBV) ask_block(std::integral_constant<int, b + 1>{});
                lds_left<b + 1 < NBV ? ASKS : 0>();
                Operands &o = op[b & 1];
                arrived(o.d[0]); arrived(o.d[1]);
                const float dv[8] = {o.d[0][0], o.d[0][1], o.d[0][2], o.d[0][3], o.d[1][0], o.d[1][1], o.d[1][2], o.d[1][3]};
                uint32_t vlo[4], vhi[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t t2 = o.a[i] | (o.b[i] << 16);
                    vlo[i] = ((t2 << 6) & nib_mask) | nib_one;
                    vhi[i] = ((t2 << 2) & nib_mask) | nib_one;
                }
                const u32x4_t lo4 = {vlo[0], vlo[1], vlo[2], vlo[3]}, hi4 = {vhi[0], vhi[1], vhi[2], vhi[3]};
#pragma unroll
                for (int k = 0; k < T; k++) {
                    if (T == 2 && !(of & (1 << k))) continue;
                    uint32_t pa[4];
                    float tsum = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; i += 2) {
                        const float x0 = sv[k][i] * dv[i], x1 = sv[k][i + 1] * dv[i + 1];
                        const float y0 = x0 - as_f32(as_u32(x0) & drop), y1 = x1 - as_f32(as_u32(x1) & drop);
                        pa[i / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(y0, y1));
                        tsum += x0 + x1;
                    }
                    Tl[k][b] += tsum;
                    asm volatile("" : "+v"(Tl[k][b]));
                    const h8v pa8 = __builtin_bit_cast(h8v, u32x4_t{pa[0], pa[1], pa[2], pa[3]});
                    O[k][2 * b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa8, __builtin_bit_cast(h8v, lo4), O[k][2 * b], 0, 0, 0);
                    O[k][2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa8, __builtin_bit_cast(h8v, hi4), O[k][2 * b + 1], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            each<0, NBV>(block);
        };
        constexpr std::integral_constant<int, 0> n0{};
        constexpr std::integral_constant<int, 1> n1{};

        for (int it = 0; it < nsteps; it++) {
            const int R = it * NW + tile;
            int nv[T], kv[T];                                  // rows of the tile a token attends; of those whose scores are this wave's
            nv[0] = max(0, min(32, len[0] - 32 * R));
            if (T == 2) nv[T - 1] = R < delta ? 0 : max(0, min(32, len[T - 1] - 32 * (R - delta)));
            const int nvmax = T == 2 ? max(nv[0], nv[T - 1]) : nv[0];
#pragma unroll
            for (int k = 0; k < T; k++) kv[k] = SHARE ? max(0, min(TRK, nv[k] - TRK * vhalf)) : nv[k];
            asm volatile("s_waitcnt vmcnt(5)" ::: "memory");    // K is there (V may be on its way)
            if (nvmax > 0) {
#pragma unroll
                for (int u = 0; u < TRK * NB / 64; u++) {
                    lds_put<float>(kout + 256 * u, half_bits_to_f32(lds_at<uint16_t>(kraw + 18 * KB * u)));    // [block][row]
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                scores(kv, T == 2 && nv[T - 1] > 0);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (K has been read)
            ask_k(R + NW);
            if constexpr (SHARE) {
                // (two buffers: the other wave may still be reading the last step's)
                const uint32_t xch = lds0 + kAtTrade + ((it & 1) * NW + tile) * 1024 + 128 * q4 + 16 * head;
#pragma unroll
                for (int k = 0; k < T; k++)
                    if (nv[k] && !is_lo) lds_put<f4v>(xch + k * S::kTrade + 512 * vhalf, f4v{sv[k][0], sv[k][1], sv[k][2], sv[k][3]});
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int k = 0; k < T; k++)
                    if (nv[k]) {
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const f4v s4 = lds_at<f4v>(xch + k * S::kTrade + 512 * h);
                            sv[k][4 * h] = s4[0]; sv[k][4 * h + 1] = s4[1]; sv[k][4 * h + 2] = s4[2]; sv[k][4 * h + 3] = s4[3];
                        }
                    }
            }
            if (nv[0]) softmax(n0, nv[0]);
            if constexpr (T == 2) {
                if (nv[T - 1]) softmax(n1, nv[T - 1]);
            }
            asm volatile("s_waitcnt vmcnt(5)" ::: "memory");    // V is there (the next K may be on its way)
            // (a tile that ends for one token only is taken for one after the other, each with its own end)
            const int passes = T == 2 && nv[0] && nv[T - 1] && nv[0] != nv[T - 1] ? 2 : nvmax ? 1 : 0;
            for (int pass = 0; pass < passes; pass++) {
                const int of = T == 1 ? 1 : passes == 2 ? 1 << pass : (nv[0] ? 1 : 0) | (nv[T - 1] ? 2 : 0);
                v_scales(T == 2 && passes == 2 ? (pass ? nv[T - 1] : nv[0]) : nvmax);
                products(of);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (V has been read)
            ask_v(R + NW);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // (nothing is on its way into what the states are written over)

        // (worked out again from nothing: kept through the loop, these would be in memory)
        uint32_t all = ~0u;
        asm volatile("" : "+s"(all));
        const int elane = (int)__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u)), ecol = elane & 15, eq4 = elane >> 4;
        const uint32_t eodd_mask = 0u - (uint32_t)(eq4 & 1);

        // ---- the waves' states meet in LDS, one head's dimension a thread folds them in the order of a workgroup of one token:
        // tile t of B is tile t + delta here
        __syncthreads();
#pragma unroll
        for (int k = 0; k < T; k++) {
            if (k && !joint) break;
            float *ow = reinterpret_cast<float *>(lds_raw + k * S::kState);   // [V half][NW][8][256]
            float *mlw = ow + WAVES * 8 * 256;                              // [NW][8][2]
            const float l_tot = xor32_sum(xor16_sum(l_run[k]));
            const int odd = eq4 >> 1;
#pragma unroll
            for (int b = 0; b < NBV; b++) {
                const uint32_t tcol = as_u32(24.f * xor32_sum(xor16_sum(Tl[k][b])));
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const uint32_t t_lo = (uint32_t)__builtin_amdgcn_readlane((int)tcol, r), t_hi = (uint32_t)__builtin_amdgcn_readlane((int)tcol, 4 + r);
                    const float t24 = as_f32((t_lo & ~eodd_mask) | (t_hi & eodd_mask));
                    const auto sw = __builtin_amdgcn_permlane32_swap(as_u32(O[k][2 * b][r]), as_u32(O[k][2 * b + 1][r]), false, false);
                    ow[((size_t)wave * 8 + 4 * (eq4 & 1) + r) * 256 + ecol + 16 * odd + 32 * b] = (as_f32(sw[0]) - t24) + as_f32(sw[1]);
                }
            }
            if (elane < 8 && wave < NW) { mlw[(wave * 8 + elane) * 2] = m_run[k]; mlw[(wave * 8 + elane) * 2 + 1] = l_tot; }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < T; k++) {
            if (k && !joint) break;
            const float *ow = reinterpret_cast<const float *>(lds_raw + k * S::kState), *mlw = ow + WAVES * 8 * 256;
            static_assert(NT == HD, "a thread has one dimension of every head");
            const int turn = k ? delta : 0, tok = k ? B.tok : A.tok, d = wave * 64 + elane;
#pragma unroll
            for (int h = 0; h < 8; h++) {
                const int hq = head0 + h;
                if (h >= groups) break;
                float M = -1.0e30f;
#pragma unroll
                for (int w = 0; w < NW; w++) M = fmaxf(M, mlw[(((w + turn) & (NW - 1)) * 8 + h) * 2]);
                float L = 0.f, a = 0.f;
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    const int pw = (w + turn) & (NW - 1);
                    const float wt = __expf(mlw[(pw * 8 + h) * 2] - M);
                    L = fmaf(wt, mlw[(pw * 8 + h) * 2 + 1], L);
                    a = fmaf(wt, ow[((size_t)(d / 256 * NW + pw) * 8 + h) * 256 + d % 256], a);
                }
                p.out[((size_t)tok * p.n_q + hq) * HD + d] = a / L;
            }
        }
    }
}

}  // namespace
}  // namespace ksh
