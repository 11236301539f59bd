// GEMM of bf16 tokens, up to 32 to a workgroup, in one launch: the activations go into the matrix cores as they are.
//
// The forms that this stands in front of prepare the rows (q4k_mm_skinny_kernel: f16, in fragment order, with their sums) or fold slices
// (q6k_mm_rows_kernel) in a launch of their own, 2.3 us and a boundary of a call of 7.  Here the first operand is the rows' bf16 itself and
// the second 16 + nibble, exact in bf16 (a byte of 0x80 | nibble << 3 under one of 0x41); -16 sum(x) of a sub-block, from the matrix cores
// too, is what its product starts from, so that it ends as sum(x n):
//   y += d sum_s sc_s sum(x n) - dmin sum_s m_s sum(x)
// Nothing of x is rounded, where f16 lost what lies below its range, and a superblock's sums begin anew: the error is 0.6 to 1.0e-7 of the
// result, 3.5 to 6e-7 there.
//
// A workgroup is RH tiles of 16 weight rows and a group of the tokens; its eight waves deal a row's superblocks out and add their sums up through LDS
// in their order.  Weights and tokens come as whole 16-byte pieces straight into LDS: from registers' loads, 16 rows an instruction at half a
// line each, 16 tokens of 2048 x 2048 took 4.8 us, so 3.7.  What bounds it: up to some 256 workgroups the launch and one round trip (3.4
// us), then the vector instructions, some 215 a tile and superblock (half of them the products with the scales), and, from 17 tokens on,
// the LDS that lets one workgroup on a compute unit.  (Asking for the next superblock in front of the products: even.)
#pragma once
#include "ksh_device.hpp"

namespace ksh {
namespace {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2v_t __attribute__((ext_vector_type(2)));

struct FewParams {
    const uint8_t *W;
    const uint16_t *X;
    float *Y;
    int rows, cols, batch, tokens;      // tokens: of a workgroup (blockIdx.y)

    // the workgroup's own tokens
    __device__ __forceinline__ void mine()
    {
        const int t0 = (int)blockIdx.y * tokens;
        X += (size_t)t0 * cols;
        Y += (size_t)t0 * rows;
        batch = min(tokens, batch - t0);
    }
};

constexpr int kFewTokens = 32, kFewMost = 1024;      // of a workgroup, of a launch
// LDS of a wave: its weight rows of a superblock, whose place its sums take in the end, and the tokens' columns of it
// (a Q6_K block is 14 pieces wherever it begins)
constexpr int kFewRow4 = 144, kFewRow6 = 224;
__host__ __device__ constexpr int few_x_bytes(int batch) { return (batch + 1) / 2 * 1024; }
constexpr int few_lds(bool q6, int batch, int rh) { return 8 * (rh * 16 * (q6 ? kFewRow6 : kFewRow4) + few_x_bytes(batch)); }
// tiles of 16 weight rows a workgroup takes: one with more than 16 tokens, and what a compute unit's LDS holds
constexpr bool few_fits(bool q6, int batch, int rh) { return rh == 1 || ((rh == 2 || rh == 4) && batch <= 16 && few_lds(q6, batch, rh) <= 163840); }

__device__ __forceinline__ float byte_f32(uint32_t w, int i) { return i == 0 ? ubyte_f32<0>(w) : i == 1 ? ubyte_f32<1>(w) : i == 2 ? ubyte_f32<2>(w) : ubyte_f32<3>(w); }

// A wave's request for all tokens' columns of a superblock, two tokens an instruction.  (A token's pieces turned, so that the reads of 16
// tokens are of 16 places.)
__device__ __forceinline__ void few_ask_x(const FewParams &p, int sb, int lane, uint32_t dst)
{
    for (int j = 0; 2 * j < p.batch; j++) {
        const int t = 2 * j + (lane >> 5), piece = (lane & 31) ^ (t & 15);
        to_lds16(reinterpret_cast<const uint8_t *>(p.X) + (size_t)sb * 512, (uint32_t)min(t, p.batch - 1) * (uint32_t)(p.cols * 2) + 16u * (uint32_t)piece,
                 dst + (uint32_t)(j * 1024));
    }
}

// The waves' shares in their order: register i of lane (n, kg) is token 4 kg + i of the tile, weight row n.  `red`: WAVE bytes a wave.
template <int MT, int RH, int NW, int WAVE>
__device__ __forceinline__ void few_fold(const f32x4_t (&F)[MT][RH], float *red, const FewParams &p, int r0, int waves, int tid)
{
    constexpr int WF = WAVE / 4;
    static_assert(MT * RH * 1024 <= WAVE, "a wave's sums in the place of its rows");
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int rh = 0; rh < RH; rh++)
#pragma unroll
            for (int i = 0; i < 4; i++) red[wave * WF + ((mt * RH + rh) * 4 + i) * 64 + lane] = F[mt][rh][i];
    __syncthreads();
    for (int o = tid; o < MT * RH * 256; o += NW * 64) {
        float sum = red[o];
        for (int w = 1; w < waves; w++) sum += red[w * WF + o];
        const int mt = o / (RH * 256), rh = (o / 256) % RH, i = (o / 64) & 3, l = o & 63;
        const int t = 16 * mt + 4 * (l >> 4) + i, r = r0 + 16 * rh + (l & 15);
        if (t < p.batch && r < p.rows) p.Y[(size_t)t * p.rows + r] = sum;
    }
}

// MT: tiles of 16 tokens.  RH: tiles of 16 weight rows.  NW: waves, to which a row's superblocks are dealt.
template <int MT, int RH, int NW>
__global__ __launch_bounds__(NW * 64) void q4k_mm_few_kernel(FewParams p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t few[];
    p.mine();
    constexpr int WAVE = RH * 16 * kFewRow4, PIECES = RH * 16 * 9, ASKS = (PIECES + 63) / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, kg = lane >> 4;
    const int r0 = blockIdx.x * (16 * RH), nsb = p.cols / 256;
    const uint32_t row_bytes = (uint32_t)nsb * 144u;
    const int last = p.rows - 1 - r0;
    uint8_t *mine = few + wave * WAVE, *mx = few + NW * WAVE + wave * few_x_bytes(p.batch);
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mine;
    uint32_t off[ASKS];
#pragma unroll
    for (int i = 0; i < ASKS; i++) {
        const int c = 64 * i + lane, row = c / 9;
        off[i] = (uint32_t)min(row, last) * row_bytes + 16u * (uint32_t)(c - 9 * row);
    }
    const uint8_t *W = p.W + (size_t)r0 * row_bytes;
    const uint32_t lx = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mx;
    const uint8_t *xr[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) xr[mt] = mx + min(16 * mt + n, p.batch - 1) * 512;

    f32x4_t F[MT][RH];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int rh = 0; rh < RH; rh++) F[mt][rh] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const f32x4_t kZero = {0.f, 0.f, 0.f, 0.f};
    const bf8_t offset = __builtin_bit_cast(bf8_t, u32x4_t{0xC180C180u, 0xC180C180u, 0xC180C180u, 0xC180C180u});      // -16

    for (int sb = wave; sb < nsb; sb += NW) {
#pragma unroll
        for (int i = 0; i < ASKS; i++)
            if (64 * (i + 1) <= PIECES || lane < PIECES - 64 * i) to_lds16(W + (size_t)sb * 144, off[i], l0 + (uint32_t)(i * 1024));
        few_ask_x(p, sb, lane, lx);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u32x4_t hdr[RH], a[MT][8];
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int t = min(16 * mt + n, p.batch - 1);
                a[mt][s] = *reinterpret_cast<const u32x4_t *>(xr[mt] + 16 * ((4 * s + kg) ^ (t & 15)));
            }
        u32x2v_t q[RH][4];
#pragma unroll
        for (int rh = 0; rh < RH; rh++) {
            const uint8_t *blk = mine + (16 * rh + n) * 144;
            hdr[rh] = *reinterpret_cast<const u32x4_t *>(blk);
#pragma unroll
            for (int g = 0; g < 4; g++) q[rh][g] = *reinterpret_cast<const u32x2v_t *>(blk + 16 + 32 * g + 8 * kg);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the next superblock's come to the same place)
        // the rows' six-bit scales and minimums, a byte each
        uint32_t sc[RH][2], mn[RH][2];
        f32x4_t P[MT][RH], N[MT][RH];
#pragma unroll
        for (int rh = 0; rh < RH; rh++) {
            const uint32_t sy = hdr[rh].y, sz = hdr[rh].z, sw = hdr[rh].w;
            sc[rh][0] = sy & 0x3F3F3F3Fu; sc[rh][1] = (sw & 0x0F0F0F0Fu) | ((sy >> 2) & 0x30303030u);
            mn[rh][0] = sz & 0x3F3F3F3Fu; mn[rh][1] = ((sw >> 4) & 0x0F0F0F0Fu) | ((sz >> 2) & 0x30303030u);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) P[mt][rh] = N[mt][rh] = kZero;
        }
#pragma unroll
        for (int g = 0; g < 4; g++) {
            // sub-blocks 2g and 2g + 1: columns 8 kg .. 8 kg + 7 of each are the low and the high nibbles of the same bytes
            f32x4_t S[MT][2];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int u = 0; u < 2; u++) S[mt][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a[mt][2 * g + u]), offset, kZero, 0, 0, 0);
#pragma unroll
            for (int rh = 0; rh < RH; rh++) {
                // 16 + nibble as bf16: 16 .. 31 in steps of 1/8, the upper byte always 0x41
                u32x4_t lo, hi;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t w = q[rh][g][i], l = ((w << 3) & 0x78787878u) | 0x80808080u, h = ((w >> 1) & 0x78787878u) | 0x80808080u;
                    lo[2 * i] = __builtin_amdgcn_perm(0x41414141u, l, 0x04010400u); lo[2 * i + 1] = __builtin_amdgcn_perm(0x41414141u, l, 0x04030402u);
                    hi[2 * i] = __builtin_amdgcn_perm(0x41414141u, h, 0x04010400u); hi[2 * i + 1] = __builtin_amdgcn_perm(0x41414141u, h, 0x04030402u);
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int s = 2 * g + u;
                    const float c = byte_f32(sc[rh][s / 4], s % 4), m = byte_f32(mn[rh][s / 4], s % 4);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        const f32x4_t C = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a[mt][s]), __builtin_bit_cast(bf8_t, u ? hi : lo), S[mt][u], 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            P[mt][rh][i] = fmaf(c, C[i], P[mt][rh][i]);
                            N[mt][rh][i] = fmaf(m, S[mt][u][i], N[mt][rh][i]);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int rh = 0; rh < RH; rh++) {
            const float d = half_bits_to_f32(hdr[rh].x & 0xFFFFu), dmin = half_bits_to_f32(hdr[rh].x >> 16) * 0.0625f;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) F[mt][rh][i] = fmaf(d, P[mt][rh][i], fmaf(dmin, N[mt][rh][i], F[mt][rh][i]));
        }
    }
    few_fold<MT, RH, NW, WAVE>(F, reinterpret_cast<float *>(few), p, r0, min(NW, nsb), tid);
}

}  // namespace
}  // namespace ksh
