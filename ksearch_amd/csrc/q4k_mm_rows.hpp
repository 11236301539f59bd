// The prompt GEMM over Q4_K weights and f32 rows (two f16 parts at the row's own scale, mm_prep_rows_kernel) or bf16 rows (one
// part, mm_prep_x_kernel): every wave
// converts its own weights in registers and multiplies them with fragments that the workgroup shares in LDS.
//
// What bounds it: the matrix pipe and the chip's power.  With two workgroups on every compute unit (gate | up of 12288 x 1536, 2048
// tokens) the pipe is busy 60 % of the chip's cycles, at 1.7 GHz, and with one (1536 x 12288, 192 workgroups) 44 %; a launch of nothing but its matrix instructions holds 1.6 GHz.  In its place was a tile of four waves
// that loaded and converted, handing weights to four that multiplied through LDS, and of fragments from memory to registers:
// at 32 x 64 a wave the fragments alone keep the path from L1 busy for as long as the matrix instructions take, and the roles
// waited for each other at every step (pipe busy 44 %).  Here a wave has 64 tokens x 64 rows (or 32 x 64, or 32 x 32), a
// converted weight meets four fragments (or two), a fragment comes from memory once a workgroup, and nobody waits for a
// converted weight.  With its preparation (64 x 64 a wave): 2048 tokens, gate | up of 12288 x 1536 380 -> 298 us, 1536 x 12288
// 252 -> 208, 4096 x 1536 82 -> 60; (32 x 32) 952 tokens, 1536 x 12288 152 -> 134, 700 tokens, 2048 x 8192 99 -> 87; rows cut
// as in launches of their own, 1989 tokens, 1536 x 12288 285 -> 245.
//
// With bf16 rows there are half as many matrix instructions to a converted weight, and a wave has 64 tokens x 32 rows, or 128 x
// 32 where the chip is full: 2048 tokens, 12288 x 4096 257 -> 221 us, 300 tokens, 12288 x 1536 29.7 -> 24.1, 65 tokens, 12288 x
// 8192 46 -> 40; 512 tokens, 8192 x 2048 in 64 x 128 30.5 -> 30.2.  That launch takes 128 x 128 now (28.5 -> 27.7 with its
// preparation), one wave to a SIMD, whose matrix pipe is busy for 36 % of the cycles and its vector ALU for 29; the wave waits for 18
// %, the rest lies between its instructions.  (In 64 x 128, two waves to a SIMD, the two take 18 and 23 of 45 thousand cycles, yet neither
// fragments read two units ahead, nor eight half steps on their way, nor a conversion of 11 % fewer instructions changed its time.)
//
// A product's order is fixed, so its bits do not depend on the shape that does it: per 16 columns the hi and the lo part against
// the same weights into a superblock's own accumulator, then F = (bias and mins, two short products) + F and F = d * C + F.
//
// CUT: the rows belong to prompts that would each have had a launch of their own, whose K slices depend on its length; the
// workgroup takes all of K, and where a row's slice ends its sum goes to a second accumulator and starts again from zero (the
// bits of those launches; through memory, as the tile has it, a slice end was a round trip of the results).
// PAIR: a gate and an up matrix of one size: a wave has a gate tile beside its up tile and stores gelu(gate) * up.
#pragma once
#include "ksh_device.hpp"
#include "ksh_internal.hpp"

namespace ksh {
namespace {

// Shape of a launch's workgroups: WM x WN = 4 waves, each MT x NT tiles of 32 tokens x 32 weight rows; LO: rows of f32, in two
// parts (else bf16, one part).
template <int MT_, int NT_, int WM_, int WN_, bool LO_ = true>
struct MmRows {
    static constexpr int MT = MT_, NT = NT_, WM = WM_, WN = WN_, PARTS = LO_ ? 2 : 1;
    static constexpr bool LO = LO_;
    static constexpr int TT = WM * MT, TM = 32 * TT, TN = 32 * WN * NT, kThreads = 64 * WM * WN;
    static constexpr int TF = TT * PARTS / 2;         // fragments of a half step that a wave fetches
    static constexpr bool kNeighbours = NT == 1 && LO;   // an L2's workgroups are neighbours
    static constexpr int SUMS = TT == 4 ? 2 : 1;      // ... and fragments of a superblock's sums
    static constexpr int kStage = TT * 2 * PARTS * 1024;   // bytes of the fragments of 32 columns: [token tile][hi | lo][k slice][lane][16]
    static constexpr int kSums = TT * 2 * 1024;       // bytes of a superblock's sums of x: [token tile][k slice][lane][16]
    static constexpr int kTile = 5 * 1024;            // bytes of a superblock of 32 weight rows: [row][144], whole kilobytes
    static constexpr int kInv = 256;                  // the tokens' 1 / s
    static constexpr int kLds = 4 * kStage + kSums + WM * WN * NT * kTile + kInv;
    static_assert(WM * WN == 4 && TT * PARTS <= 4 && MT * PARTS >= 2 && NT <= 2, "a wave fetches TF fragments of a half step, from one part of one token tile");
    // (a half step has MT PARTS units; the second half of them ask for a superblock's sums, one each)
    static_assert((MT * PARTS == 2 && SUMS == 1) || MT * PARTS == 4, "every request that the loop's waits count has its place");
    static_assert(!LO || TM * 4 <= kInv, "the tokens' 1 / s have their place");
};

// What comes from memory into LDS is not counted by the compiler, which would wait for all of it in front of every read of LDS: it
// is waited for by the number of younger operations, so every one of them is issued whatever the sizes (addresses are clamped
// instead).

template <class S, bool CUT, bool PAIR>
__global__ __launch_bounds__(S::kThreads, 2) void q4k_mm_rows_kernel(MmParams p)
{
    constexpr int MT = S::MT, NT = S::NT, TT = S::TT, TF = S::TF, PARTS = S::PARTS;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_rows[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::WN, wn = wave % S::WN, lm = lane & 31, h = lane >> 5;

    // Shapes for launches that do not fill the chip: consecutive workgroups go round the eight L2s, so as they are numbered each
    // L2 would fetch most of X and of W.  Here an L2's workgroups are neighbours, all weight rows of a few token tiles (and of a
    // K slice): 952 tokens, 1536 x 2048 30.6 -> 28.9 us, 700 tokens, 2048 x 2048 29.6 -> 27.9, 2048 tokens, 2560 x 1536 52.2 -> 49.6.
    // Where the chip is full the walk along the tokens is the better one (2048 tokens, gate | up 12288 x 1536 312 or 318), and with
    // bf16 rows, half the bytes, it is so mostly (1024 tokens, 4096 x 4096 50.1 or 51.8; 700, 2048 x 8192 53 or 47).
    // (The quotients come from the host's reciprocals: divided here, they are 0.5 us in front of the first request.)
    uint32_t bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if constexpr (S::kNeighbours) {
        if (p.wgs) {
            const uint32_t n = bx + p.gx * (by + p.gy * bz), l2 = n & 7;
            const uint32_t at = l2 * (p.wgs >> 3) + min(l2, p.wgs & 7) + (n >> 3), column = __umulhi(at, p.per_gy);
            bz = __umulhi(column, p.per_gx);
            by = at - column * p.gy;
            bx = column - bz * p.gx;
        }
    }

    // which matrix this row tile belongs to (the copy of the arguments is this workgroup's own)
    int ycol = 0;
    const int rows_all = p.rows + p.rows1 + p.rows2;
    const int rows_of[3] = {p.rows, p.rows1, p.rows2};
    if (!PAIR && p.rows1) {
        const int ty0 = (p.rows + S::TN - 1) / S::TN, ty1 = (p.rows1 + S::TN - 1) / S::TN;
        if ((int)by >= ty0 + ty1) { by -= ty0 + ty1; ycol = p.rows + p.rows1; p.W = p.W2; p.Y = p.Y2; p.rows = p.rows2; }
        else if ((int)by >= ty0) { by -= ty0; ycol = p.rows; p.W = p.W1; p.Y = p.Y1; p.rows = p.rows1; }
    }
    const int t0 = (int)bx * S::TM, r0 = (int)by * (PAIR ? S::TN / 2 : S::TN);
    const int nsb_row = p.cols / 256;
    int nsb = nsb_row, sb0 = 0;
    size_t ystride = (size_t)p.rows;
    if (p.ksplit) {
        const int slice = (int)bz;
        sb0 = nsb_row * slice / p.ksplit;
        nsb = nsb_row * (slice + 1) / p.ksplit - sb0;
        p.Y = p.Y_parts + (size_t)slice * p.batch * rows_all + ycol;   // partial sums: all matrices' columns side by side
        ystride = (size_t)rows_all;
    }

    // ---- everything the loop reads comes straight from memory into LDS: of the 4 TF kilobytes of a half step this wave asks for
    // TF; the sums of a superblock; and its own weight rows, a row's 144 bytes in nine lanes.  (Asked for in the order the
    // matrix instruction wants them, a row a lane, weights are 64 pieces of 16 bytes to an instruction: 2048 tokens, 12288 x
    // 1536, gate | up 312 us instead of 294.)
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds_rows;
    constexpr uint32_t kAtSums = 4 * S::kStage, kAtW = kAtSums + S::kSums, kAtInv = kAtW + 4 * NT * S::kTile;
    const int f0 = wave * TF, ntt = (p.batch + 31) / 32, fsum = wave * S::SUMS % (2 * TT);
    const uint8_t *xsrc = reinterpret_cast<const uint8_t *>(S::LO && ((f0 >> 1) & 1) ? p.Xf_lo : p.Xf) +
                          ((size_t)min(t0 / 32 + f0 / (2 * PARTS), ntt - 1) * nsb_row + sb0) * 16384 + (f0 & 1) * 1024;
    const uint8_t *sxsrc = reinterpret_cast<const uint8_t *>(p.SxA) + (((size_t)min(t0 / 32 + (fsum >> 1), ntt - 1) * nsb_row + sb0) * 2 + (fsum & 1)) * 1024;
    const uint32_t lane16 = 16u * (uint32_t)lane, lw = l0 + kAtW + (uint32_t)(wave * NT * S::kTile);
    auto ask_rows = [&](int hs, int stage, int i) __attribute__((always_inline)) {
        to_lds16(xsrc + (size_t)min(hs, 8 * nsb - 1) * 2048 + i * 1024, lane16, l0 + (uint32_t)(stage * S::kStage + (f0 + i) * 1024));
    };
    auto ask_sums = [&](int sb, int i) __attribute__((always_inline)) { to_lds16(sxsrc + (size_t)min(sb, nsb - 1) * 2048 + i * 1024, lane16, l0 + kAtSums + (uint32_t)((fsum + i) * 1024)); };
    const size_t row_bytes = (size_t)nsb_row * 144;
    const uint8_t *wbase[2];
    wbase[0] = p.W + (size_t)r0 * row_bytes + (size_t)sb0 * 144;
    wbase[1] = PAIR ? p.W1 + (size_t)r0 * row_bytes : wbase[0];
    uint32_t woff[NT][5];                             // piece 64 i + lane of a tile's rows (past the tile: its last row again)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int c = 64 * i + lane, row = min(c / 9, 31), r = PAIR ? wn * 32 + row : (wn * NT + nt) * 32 + row;
            woff[nt][i] = (uint32_t)min(r, p.rows - 1 - r0) * (uint32_t)row_bytes + 16u * (uint32_t)(c % 9);
        }
    auto ask_weights = [&](int sb, int j) __attribute__((always_inline)) {
        to_lds16(wbase[j / 5] + (size_t)min(sb, nsb - 1) * 144, woff[j / 5][j % 5], lw + (uint32_t)(j / 5 * S::kTile + j % 5 * 1024));
    };

    f16v F[MT][NT], C[MT][NT];
    const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) F[mt][nt] = C[mt][nt] = kZero16;
    // lane (lm, h) has row lm of each of its tiles: the header and bytes 16 h .. 16 h + 15 of every group's 32
    u32x4_t q[4][NT], hdr[NT];
    uint32_t scA[NT], scB[NT], s_lo[NT], s_hi[NT];   // the eight scales of a superblock; the two of the group being converted
    float dn[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) dn[nt] = 0.f;
    h8 b[2][NT];                                      // converted weights of a k slice, and of the next
    h8 a[2][2];                                       // a unit's fragments, and the next one's
    u32x4_t b2[NT];
    h8 s2[2];

    auto scales = [&]() __attribute__((always_inline)) {   // of the superblock whose header has arrived
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            scA[nt] = hdr[nt].y & 0x3F3F3F3Fu;
            scB[nt] = (hdr[nt].w & 0x0F0F0F0Fu) | ((hdr[nt].y & 0xC0C0C0C0u) >> 2);
        }
    };
    auto open_group = [&](auto gtag, int nt) __attribute__((always_inline)) {
        constexpr int g = decltype(gtag)::value;
        const uint32_t s = (g < 2 ? scA : scB)[nt];
        s_lo[nt] = (s >> (16 * (g & 1))) & 0xFFu;
        s_hi[nt] = (s >> (16 * (g & 1) + 8)) & 0xFFu;
        // bytes 8h .. 8h+7 and 16+8h .. 16+8h+7 of the group, which is what the matrix instruction wants of lane (lm, h)
        const auto x = __builtin_amdgcn_permlane32_swap(q[g][nt].x, q[g][nt].z, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(q[g][nt].y, q[g][nt].w, false, false);
        q[g][nt] = u32x4_t{x[0], y[0], x[1], y[1]};
    };
    auto convert = [&](auto gtag, auto ktag, int nt) __attribute__((always_inline)) {
        constexpr int g = decltype(gtag)::value, ks = decltype(ktag)::value;
        const uint32_t w0 = q[g][nt][2 * (ks & 1)], w1 = q[g][nt][2 * (ks & 1) + 1], sc = ks < 2 ? s_lo[nt] : s_hi[nt];
        constexpr int sh = ks < 2 ? 0 : 4;
        const u32x4_t o = {pair_f16((w0 >> sh) & 0x000F000Fu, sc), pair_f16((w0 >> (8 + sh)) & 0x000F000Fu, sc), pair_f16((w1 >> sh) & 0x000F000Fu, sc),
                           pair_f16((w1 >> (8 + sh)) & 0x000F000Fu, sc)};
        b[ks & 1][nt] = __builtin_bit_cast(h8, o);
    };
    // the row's eight coefficients -(dmin*m_j + 1024*d) as f16: hi[8] in lanes h = 0, lo[8] in lanes h = 1; two of this lane's
    // four at a time
    auto min_operand = [&](int nt, int i) __attribute__((always_inline)) {
        const float d = half_bits_to_f32(hdr[nt].x & 0xFFFFu), dmin = half_bits_to_f32(hdr[nt].x >> 16);
        if (i == 0) dn[nt] = d;
        const uint32_t mA = hdr[nt].z & 0x3F3F3F3Fu, mB = ((hdr[nt].w >> 4) & 0x0F0F0F0Fu) | ((hdr[nt].z & 0xC0C0C0C0u) >> 2);
        const uint32_t m = h ? mB : mA;
        const float c0 = pinned(-(dmin * (i ? ubyte_f32<2>(m) : ubyte_f32<0>(m)) + 1024.f * d)), c1 = pinned(-(dmin * (i ? ubyte_f32<3>(m) : ubyte_f32<1>(m)) + 1024.f * d));
        const _Float16 h0 = (_Float16)c0, h1 = (_Float16)c1;
        const _Float16 l0_ = (_Float16)(c0 - (float)h0), l1_ = (_Float16)(c1 - (float)h1);
        const auto x = __builtin_amdgcn_permlane32_swap((uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16),
                                                        (uint32_t)__builtin_bit_cast(uint16_t, l0_) | ((uint32_t)__builtin_bit_cast(uint16_t, l1_) << 16), false, false);
        b2[nt][i] = x[0];
        b2[nt][2 + i] = x[1];
    };
    auto fold = [&](int mt, int nt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; i++) F[mt][nt][i] = fmaf(dn[nt], C[mt][nt][i], F[mt][nt][i]);
    };

    // CUT: lane t % 32 keeps the superblocks per slice of the tile's row t and what is left of the current one; finished slices
    // add up in T
    static_assert(!PAIR || (S::LO && NT == 2), "a gate tile beside an up tile, of f32 rows");
    static_assert(!CUT || MT == 1, "one token tile to a wave leaves registers for T");
    f16v T[NT];
    int cut_len = nsb, cut_left = nsb;
    if (CUT) {
        const int row_tiles = (rows_of[0] + BN - 1) / BN + (rows_of[1] + BN - 1) / BN + (rows_of[2] + BN - 1) / BN;
        cut_len = cut_left = nsb / mm_k_slices(false, row_tiles, nsb, (int)p.cut_as[min(t0 + wm * 32 + lm, p.batch - 1)]);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) T[nt] = kZero16;
    }
    auto cut_ends = [&]() __attribute__((always_inline)) {   // behind a superblock's fold
        cut_left -= 1;
        uint32_t ends = (uint32_t)__ballot(cut_left == 0);
        if (cut_left == 0) cut_left = cut_len;
        if (!ends) return;
        ends >>= 4 * h;
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (ends & (1u << (8 * (i / 4) + (i & 3)))) {
                    T[nt][i] += F[0][nt][i];
                    F[0][nt][i] = 0.f;
                }
    };

    // A unit of the loop is 2 NT matrix instructions for two fragments: one part of a k slice for two token tiles (the parts, if
    // there are two, in turn), or both parts of it for one.  U units to a half step.
    constexpr int U = MT * PARTS;
    constexpr uint32_t kTokens = PARTS * 2048;                         // bytes of a token tile's fragments
    const uint32_t la = l0 + (uint32_t)(wm * MT) * kTokens + lane16;   // + stage, token tile, part, k slice
    const uint32_t lsum = l0 + kAtSums + (uint32_t)(wm * MT) * 2048u + lane16;
    const uint32_t lh = lw + 144u * (uint32_t)lm, lq = lh + 16u * (uint32_t)h;
    auto read_rows = [&](auto htag, auto utag, h8 (&v)[2]) __attribute__((always_inline)) {   // of unit U of a half step
        constexpr int hs = decltype(htag)::value & 3, u = decltype(utag)::value;
        constexpr int off = hs * S::kStage + (U == 4 ? (u >> 1) * 1024 + (u & 1) * (PARTS == 2 ? 2048 : 2 * kTokens) : u * 1024);
        lds_ask<off>(v[0], la);
        lds_ask<off + (MT == 1 ? 2048 : kTokens)>(v[1], la);
    };
    auto read_group = [&](auto gtag) __attribute__((always_inline)) {
        constexpr int o = 16 + 32 * decltype(gtag)::value;
        lds_ask<o>(q[decltype(gtag)::value][0], lq);
        if constexpr (NT == 2) lds_ask<o + S::kTile>(q[decltype(gtag)::value][1], lq);
    };
    auto read_header = [&]() __attribute__((always_inline)) {
        lds_ask<0>(hdr[0], lh);
        if constexpr (NT == 2) lds_ask<S::kTile>(hdr[1], lh);
    };
    auto settle = [&](auto &v) __attribute__((always_inline)) {
        for (auto &e : v) arrived(e);
    };
    constexpr std::integral_constant<int, 0> n0{};
    constexpr std::integral_constant<int, 1> n1{};
    constexpr std::integral_constant<int, 2> n2{};
    constexpr std::integral_constant<int, 3> n3{};

    // ---- in front of the loop: the first superblock's weights, three half steps of fragments; the first slice converted
    if (S::LO) to_lds4(reinterpret_cast<const uint8_t *>(p.inv_s), 4u * (uint32_t)min(t0 + lane, p.batch - 1), l0 + kAtInv);   // (every wave the same)
#pragma unroll
    for (int j = 0; j < 5 * NT; j++) ask_weights(0, j);
#pragma unroll
    for (int i = 0; i < S::SUMS; i++) ask_sums(0, i);
#pragma unroll
    for (int hs = 0; hs < 3; hs++)
#pragma unroll
        for (int i = 0; i < TF; i++) ask_rows(hs, hs, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * TF) : "memory");
    read_group(n0);
    read_group(n1);
    read_group(n2);
    read_group(n3);
    read_header();
    read_rows(n0, n0, a[0]);
    lds_left<0>();
    settle(q[0]); settle(q[1]); settle(q[2]); settle(q[3]); settle(hdr); settle(a[0]);
    scales();
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        open_group(n0, nt);
        convert(n0, n0, nt);
    }

    // Unit `place` of half step `half` of a superblock.  Under its matrix instructions the next unit's fragments come from LDS
    // and the next slice's weights are converted, spread evenly (the compiler's own order issues most matrix instructions back
    // to back and leaves their pipe idle under the rest).
    auto unit = [&](int sb, auto htag, auto utag) __attribute__((always_inline)) {
        constexpr int half = decltype(htag)::value, place = decltype(utag)::value;
        constexpr int g = half >> 1, ks = 2 * (half & 1) + place / (U / 2), part = U == 4 ? place & 1 : 0, set = place & 1;
        constexpr int gn = ks == 3 ? (g + 1) & 3 : g, kn = (ks + 1) & 3;               // the next slice
        constexpr bool last = place == U - 1;
        // Memory operations of a half step: its first units ask for the fragments of three half steps on; the last two (the
        // last, U = 2) of half steps 0 .. 4 for a piece of the next superblock's weights a tile, of half step 5 for its sums.
        constexpr auto extra = [](int hh) { return hh < 5 ? NT : hh == 5 ? S::SUMS : 0; };
        __builtin_amdgcn_sched_barrier(0);
        constexpr bool opens = half == 0 && place == 0;
        if constexpr (opens && CUT) {
            if (sb > 0) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) fold(mt, nt);
                cut_ends();
            }
        }
        constexpr int mins = MT == 4 ? (half == 2 ? place : -1) : U == 4 ? (g == 1 && part == 0 && ks < 2 ? ks : -1) : (g == 1 && ks >= 1 && ks <= MT ? ks - 1 : -1);
        constexpr bool take0 = half == 7 && place == 0, take3 = half == 7 && last;
        // (behind the first matrix instruction, whose 32 cycles cover part of it: a request to memory takes some 40 to issue)
        auto ask = [&]() __attribute__((always_inline)) {
            if constexpr (last) {
                // every wave has this half step's fragments in registers; the next one's, which this wave has asked for two half
                // steps ago, are in LDS (and at the end of half step 6 the weights, which are SUMS + 2 TF operations back)
                constexpr int pending = half == 6 ? S::SUMS + 2 * TF : extra((half + 6) & 7) + TF + extra((half + 7) & 7) + TF + (U == 4 && (half == 5 || (half < 5 && NT == 2)) ? 1 : 0);
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(pending) : "memory");
            }
            read_rows(std::integral_constant<int, (last ? half + 1 : half) & 7>{}, std::integral_constant<int, last ? 0 : place + 1>{}, a[set ^ 1]);
            // the short second product's: the sums of x of a token tile
            if constexpr (mins >= 0) {
                lds_ask<mins * 2048>(s2[0], lsum);
                lds_ask<mins * 2048 + 1024>(s2[1], lsum);
            }
            // the next superblock's weights, into the registers whose group has been converted
            if constexpr (take0) { read_group(n0); read_header(); }
            if constexpr (take3) { read_group(n1); read_group(n2); read_group(n3); }
            if constexpr (U == 4) {
                if constexpr (place < TF) ask_rows(8 * sb + half + 3, (half + 3) & 3, place);
                if constexpr (place >= 4 - NT && half < 5) ask_weights(sb + 1, NT * half + place - (4 - NT));
            } else if constexpr (place == 0) {
#pragma unroll
                for (int i = 0; i < TF; i++) ask_rows(8 * sb + half + 3, (half + 3) & 3, i);
            } else if constexpr (half < 5) {
#pragma unroll
                for (int i = 0; i < NT; i++) ask_weights(sb + 1, NT * half + i);
            }
            if constexpr (place >= U / 2 && place < U / 2 + S::SUMS && half == 5) ask_sums(sb + 1, place - U / 2);
        };
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int mt = MT == 4 ? 2 * part + i : MT == 2 ? i : 0;
                const bool first = MT == 4 ? half == 0 && ks == 0 : opens && (MT == 2 || i == 0);   // (a superblock's first product starts from the constant zero)
                if (first && !CUT) fold(mt, nt);
                C[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[set][i], b[ks & 1][nt], first ? kZero16 : C[mt][nt], 0, 0, 0);
                if (i == 0 && nt == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    ask();
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        std::integral_constant<int, gn> gnext{};
        std::integral_constant<int, kn> knext{};
        std::integral_constant<int, (g + 1) & 3> gopen{};
        // (groups are opened a unit ahead of their first conversion, U = 2: in front of it; the short product's operand in the
        // quiet units of the first steps)
        constexpr bool op0 = U == 4 ? ks == 2 && part == 1 : ks == 3, op1 = NT == 2 && (U == 4 ? ks == 3 && part == 0 : ks == 3), sc = op0 && g == 3;
        constexpr int mu = (half * U + place) - (U == 4 ? 1 : 0), mn = NT == 1 ? (mu < 2 ? mu : -1) : U == 4 ? (mu < 4 ? mu : -1) : (mu < 3 ? mu : mu == 4 ? 3 : -1);
        constexpr int converted = U == 2 ? NT : part < NT ? 1 : 0;
        if constexpr (sc) scales();
        if constexpr (U == 2) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                if constexpr (op0) open_group(gopen, nt);
                convert(gnext, knext, nt);
            }
        } else {
            if constexpr (converted) convert(gnext, knext, part);
            if constexpr (op0) open_group(gopen, 0);
            if constexpr (op1) open_group(gopen, 1);
        }
        if constexpr (mn >= 0) min_operand(mn >> 1, mn & 1);
        constexpr int valu = 11 * converted + (op0 ? 8 : 0) + (op1 ? 8 : 0) + (sc ? 5 * NT : 0) + (mn >= 0 ? 22 : 0), gaps = 2 * NT - 1;
        if constexpr (!opens) {
#pragma unroll
            for (int i = 0; i < gaps; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (valu + gaps - 1) / gaps, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        lds_left<0>();
        settle(a[set ^ 1]);
        if constexpr (take0) { settle(q[0]); settle(hdr); }
        if constexpr (take3) { settle(q[1]); settle(q[2]); settle(q[3]); }
        if constexpr (mins >= 0) {
            settle(s2);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) F[mins][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(s2[0], __builtin_bit_cast(h8, b2[nt]), F[mins][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const u32x4_t o = {h ? 0u : b2[nt].x, h ? 0u : b2[nt].y, h ? 0u : b2[nt].z, h ? 0u : b2[nt].w};
                F[mins][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(s2[1], __builtin_bit_cast(h8, o), F[mins][nt], 0, 0, 0);
            }
        }
    };
    for (int sb = 0; sb < nsb; sb++) {
#define KSH_HALF(H)                                                 \
    do {                                                            \
        constexpr std::integral_constant<int, H> hh{};              \
        unit(sb, hh, n0);                                           \
        unit(sb, hh, n1);                                           \
        if constexpr (U == 4) { unit(sb, hh, n2); unit(sb, hh, n3); } \
    } while (0)
        KSH_HALF(0); KSH_HALF(1); KSH_HALF(2); KSH_HALF(3); KSH_HALF(4); KSH_HALF(5); KSH_HALF(6); KSH_HALF(7);
#undef KSH_HALF
    }
    // (what is still on its way into LDS arrives before the workgroup gives it back)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) fold(mt, nt);
    if (CUT) {
        cut_ends();
#pragma unroll
        for (int nt = 0; nt < NT; nt++) F[0][nt] = T[nt];
    }
    // accumulator layout of the 32x32 tile: column = lane % 32, row = 8*(i/4) + 4*(lane/32) + i%4
    // (bf16 rows: stored past the L2s where mm_keeps does not say otherwise, since what those hold of it at the kernel's end is
    // written out before the next kernel starts; 512 tokens, 8192 x 2048 30.8 -> 29.5 us, 300 tokens, 12288 x 1536 24.1 -> 22.9.  In a
    // prompt's chain of launches it is even, 700 tokens 10.09 ms.)
    auto store = [&](auto keep) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int tb = t0 + (wm * MT + mt) * 32 + 4 * h, left = p.batch - tb;
            f32x4_t inv[4];
            if (S::LO) {
#pragma unroll
                for (int i4 = 0; i4 < 4; i4++) lds_ask<0>(inv[i4], l0 + kAtInv + 4u * (uint32_t)(tb - t0 + 8 * i4));
                lds_left<0>();
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt += PAIR ? 2 : 1) {
                const int r = r0 + (PAIR ? wn : wn * NT + nt) * 32 + lm;
                if (r >= p.rows) continue;
                float *y = p.Y + (size_t)tb * ystride + r;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int t = 8 * (i / 4) + (i & 3);
                    float v = S::LO ? F[mt][nt][i] * inv[i / 4][i & 3] : F[mt][nt][i];
                    if constexpr (PAIR) v = gelu_mul_f32(pinned(v), pinned(F[mt][1][i] * inv[i / 4][i & 3]));
                    if (t < left) mm_store<decltype(keep)::value>(&y[(size_t)t * ystride], v);
                }
            }
        }
    };
    if (S::LO || p.keep) store(std::true_type{});
    else store(std::false_type{});
}

}  // namespace
}  // namespace ksh
