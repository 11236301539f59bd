// The form of one launch (q4k_mm_few.hpp) over Q6_K, whose blocks of 210 bytes begin at any two-byte address and have a scale for every
// 16 columns: pieces from the 16-byte address in front of a block, the lane's words shifted as they leave LDS; 64 + q as bf16, from -96
// sum(x) on.  Error 0.70 to 0.91e-7 of the result for 512 to 8192 columns, 0.71 to 1.04e-7 in the form with slices, whose products of
// scale and weight are f16 (with scales of all eight bits 1.0e-7 and 1.4e-4).  2 tokens of 2048 x 2048
// 7.5 -> 4.0 us, 16 of 4096 x 4096 11.8 -> 6.9, 2 of 12288 x 8192 29.7 -> 19.8; some 285 vector instructions a tile and superblock.
#pragma once
#include "q4k_mm_few.hpp"

namespace ksh {
namespace {

typedef short s16x4_t __attribute__((ext_vector_type(4)));

template <int MT, int RH, int NW>
__global__ __launch_bounds__(NW * 64) void q6k_mm_few_kernel(FewParams p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t few[];
    p.mine();
    constexpr int WAVE = RH * 16 * kFewRow6, PIECES = RH * 16 * 14, ASKS = (PIECES + 63) / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, kg = lane >> 4;
    const int r0 = blockIdx.x * (16 * RH), nsb = p.cols / 256;
    const uint32_t row_bytes = (uint32_t)nsb * 210u;
    const int last = p.rows - 1 - r0;
    uint8_t *mine = few + wave * WAVE, *mx = few + NW * WAVE + wave * few_x_bytes(p.batch);
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mine;
    const uint32_t lx = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mx;
    // places from the 16-byte address at or in front of the workgroup's first row; the last piece that holds a byte of the matrix
    const uint8_t *W = p.W + (size_t)r0 * row_bytes;
    const uint32_t lead = (uint32_t)(uintptr_t)W & 15u;
    W -= lead;
    const uint32_t end = (lead + (uint32_t)(min(16 * RH - 1, last) + 1) * row_bytes - 1u) & ~15u;
    uint32_t at[ASKS], piece[ASKS];
#pragma unroll
    for (int i = 0; i < ASKS; i++) {
        const int c = 64 * i + lane, row = c / 14;
        at[i] = lead + (uint32_t)min(row, last) * row_bytes;
        piece[i] = 16u * (uint32_t)(c - 14 * row);
    }
    const uint8_t *xr[MT];
    int turn[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int t = min(16 * mt + n, p.batch - 1);
        xr[mt] = mx + t * 512 + 8 * (kg & 1);
        turn[mt] = t & 15;
    }

    f32x4_t F[MT][RH];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int rh = 0; rh < RH; rh++) F[mt][rh] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const f32x4_t kZero = {0.f, 0.f, 0.f, 0.f};
    const s16x4_t offset = {(short)0xC2C0, (short)0xC2C0, (short)0xC2C0, (short)0xC2C0};      // -96

    for (int sb = wave; sb < nsb; sb += NW) {
#pragma unroll
        for (int i = 0; i < ASKS; i++)
            if (64 * (i + 1) <= PIECES || lane < PIECES - 64 * i)
                to_lds16(W, min(((at[i] + (uint32_t)sb * 210u) & ~15u) + piece[i], end), l0 + (uint32_t)(i * 1024));
        few_ask_x(p, sb, lane, lx);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // the lane's bytes of its rows: columns 4 kg .. + 3 and 16 + 4 kg .. + 3 of every 32
        uint32_t ql[RH][8], qh[RH][4], sc[RH][4];
        float d[RH];
#pragma unroll
        for (int rh = 0; rh < RH; rh++) {
            const uint32_t sh = (lead + (uint32_t)min(16 * rh + n, last) * row_bytes + (uint32_t)sb * 210u) & 15u;
            const uint8_t *blk = mine + (16 * rh + n) * kFewRow6 + (sh & 12u);
            const uint32_t bits = sh & 2u;
            auto word = [&](int o) __attribute__((always_inline)) {
                const uint32_t *w = reinterpret_cast<const uint32_t *>(blk + o);
                return __builtin_amdgcn_alignbyte(w[1], w[0], bits);
            };
#pragma unroll
            for (int i = 0; i < 8; i++) ql[rh][i] = word(16 * i + 4 * kg);
#pragma unroll
            for (int i = 0; i < 4; i++) qh[rh][i] = word(128 + 16 * i + 4 * kg);
#pragma unroll
            for (int i = 0; i < 4; i++) sc[rh][i] = word(192 + 4 * i);
            d[rh] = half_bits_to_f32(*reinterpret_cast<const uint16_t *>(blk + 208 + bits));
        }
        u32x2v_t a[MT][16];
#pragma unroll
        for (int g = 0; g < 16; g++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) a[mt][g] = *reinterpret_cast<const u32x2v_t *>(xr[mt] + 16 * ((2 * g + (kg >> 1)) ^ turn[mt]));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the next superblock's come to the same place)
        f32x4_t P[MT][RH];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int rh = 0; rh < RH; rh++) P[mt][rh] = kZero;
#pragma unroll
        for (int g = 0; g < 16; g++) {
            // columns 16 g .. + 15: half g / 8 of the block, quarter g / 2 % 4 of that, its words g % 2
            const int half = g / 8, quarter = (g / 2) % 4, e = g % 2;
            f32x4_t S[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) S[mt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, a[mt][g]), offset, kZero, 0, 0, 0);
#pragma unroll
            for (int rh = 0; rh < RH; rh++) {
                // 64 + q as bf16: 64 .. 127 in steps of 1/2, the upper byte always 0x42
                const uint32_t l = ql[rh][4 * half + 2 * (quarter & 1) + e], h = qh[rh][2 * half + e];
                const uint32_t lo = quarter < 2 ? l << 1 : l >> 3;
                const uint32_t hi = quarter == 0 ? h << 5 : quarter == 1 ? h << 3 : quarter == 2 ? h << 1 : h >> 1;
                const uint32_t w = (hi & 0x60606060u) | ((lo & 0x1E1E1E1Eu) | 0x80808080u);
                const u32x2v_t b = {__builtin_amdgcn_perm(0x42424242u, w, 0x04010400u), __builtin_amdgcn_perm(0x42424242u, w, 0x04030402u)};
                const float c = (float)(int8_t)(sc[rh][g / 4] >> (8 * (g % 4)));
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    const f32x4_t C = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, a[mt][g]), __builtin_bit_cast(s16x4_t, b), S[mt], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) P[mt][rh][i] = fmaf(c, C[i], P[mt][rh][i]);
                }
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int rh = 0; rh < RH; rh++)
#pragma unroll
                for (int i = 0; i < 4; i++) F[mt][rh][i] = fmaf(d[rh], P[mt][rh][i], F[mt][rh][i]);
    }
    few_fold<MT, RH, NW, WAVE>(F, reinterpret_cast<float *>(few), p, r0, min(NW, nsb), tid);
}

}  // namespace
}  // namespace ksh
