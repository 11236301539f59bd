// Batched prefill GEMM over Q4_K weights on the gfx950 matrix cores:
//   Y[t, r] = sum_c deq(W[r, c]) * X[t, c]      X bf16 [batch, cols], Y f32 [batch, rows]
//
// Takes the place of KirStmt::Q4kMulMm / ksearch_q4k_mul_mm
// (crates/ksearch_codegen/src/lower.rs:404-424, 788-818,
// crates/ksearch_codegen/src/render.rs:1073-1191), which dequantizes a 64x32
// weight tile to half (rounding every weight) and runs 8x8 simdgroup MMAs.
//
// Here no weight is rounded.  With w = d*sc_j*n - dmin*m_j (n the 4-bit code,
// j the 32-wide sub-block):
//
//   sum_c w*x = sum_sb [ d * sum_k (sc_j*n_k) x_k  -  sum_j dmin*m_j * Sx_j ],   Sx_j = sum_{k in j} x_k
//
// sc_j*n_k is an integer <= 945, exact in f16, and is produced two at a time
// by one 24-bit multiply-add that also ORs it into the mantissa of half 1024.0:
// (q & 0x000F000F) * sc + 0x64006400 = (1024 + sc*n_a, 1024 + sc*n_b).  The
// matrix cores accumulate C' = sum_k (1024 + sc*n) x_k per superblock in f32;
// the per-row f16 scale d is applied once per superblock (F += d * C'), and
// the bias and the mins go through a second, short matrix product against the
// per-sub-block sums of x:  F -= sum_j (dmin*m_j + 1024*d) * Sx_j, with both
// factors split into f16 hi + lo parts so that this term keeps f32 accuracy.
// X is bf16, which converts to f16 without loss for |x| >= 2^-17 (smaller
// values lose at most 2^-25 absolutely).
//
// Tiling: q4k_mm_rows.hpp (prompts), q4k_mm_skinny_kernel (up to 64 tokens); M = tokens, N = weight
// rows, so a lane's accumulator column is one weight row (one d per lane) and
// stores are contiguous along Y's row index.  Q6_K weights: q6k_mul_mm_kernel.
#include <algorithm>
#include <type_traits>

#include "ksh_device.hpp"
#include "ksh_internal.hpp"
#include "q4k_lane.hpp"
#include "q4k_mm_few.hpp"
#include "q6k_mm_few.hpp"
#include "round_operand.hpp"

namespace ksh {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int BM = 128, BN = 128, KS = 64;
constexpr int PITCH = KS + 8;      // halves per LDS row of the main tiles (144 B: conflict-free 16 B reads)

// X bf16 -> f16 (permuted) in the order the matrix instruction wants its A operand, plus the min-term
// operand per (token, superblock): 32 halves = Sx_hi[8] | Sx_hi[8] | Sx_lo[8] | 0[8].
// Xf[token / 32][k / 16][lane][8] with lane = token % 32 + 32 * ((k / 8) % 2): one 32 x 16 fragment is 1 KB,
// lane after lane: a whole kilobyte that goes straight into LDS (q4k_mm_rows.hpp) or, with a single 128-bit load
// per lane, into a multiplying wave's registers (the others).
// A wave takes 32 tokens x one 32-column sub-block: lane (token % 32, h) converts the 8-element runs h and 2 + h
// of the sub-block and is lane token % 32 + 32 h of the sub-block's two fragments, so both leave as whole
// kilobytes, lane after lane (with a thread per run in row order, the eight 16-byte pieces of a 128-byte line of
// Xf came from eight workgroups: 5.7 us for 2 MB).  The four waves of a workgroup take neighbouring sub-blocks, so
// that together they read whole lines of X.  The sub-block's sum is (run 0 + run 1) + (run 2 + run 3), the two
// halves of the wave trading their runs' sums.
template <bool IN_ORDER>
__global__ __launch_bounds__(256) void mm_prep_x_kernel(const uint16_t *__restrict__ X, _Float16 *__restrict__ Xf,
                                                        _Float16 *__restrict__ SxA, int batch, int cols)
{
    const int lane = threadIdx.x & 63, wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int nsub = cols / 32, tb = wave / nsub, s = wave - tb * nsub;
    const int t = tb * 32 + (lane & 31), h = lane >> 5;
    if (tb * 32 >= batch) return;
    const bool live = t < batch;
    const u32x4_t *row = reinterpret_cast<const u32x4_t *>(X + (size_t)min(t, batch - 1) * cols);   // (rows past the batch: read a real row, store nothing)
    float c[2];
    h8 o[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const u32x4_t in = row[4 * s + 2 * r + h];
        const uint32_t w[4] = {in.x, in.y, in.z, in.w};
        float f[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f[2 * i] = as_f32(w[i] << 16);
            f[2 * i + 1] = as_f32(w[i] & 0xFFFF0000u);
        }
        c[r] = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
#pragma unroll
        for (int i = 0; i < 8; i++) o[r][kperm(i)] = (_Float16)f[i];
    }
    // the other half's runs: (run 0 + run 1) and (run 2 + run 3), the same in both halves
    const auto x0 = __builtin_amdgcn_permlane32_swap(as_u32(c[0]), as_u32(c[0]), false, false);
    const auto x1 = __builtin_amdgcn_permlane32_swap(as_u32(c[1]), as_u32(c[1]), false, false);
    float sum = (as_f32(x0[0]) + as_f32(x0[1])) + (as_f32(x1[0]) + as_f32(x1[1]));
    if (!live) return;
    h8 *frag = reinterpret_cast<h8 *>(Xf) + ((size_t)tb * (cols / 16) + 2 * s) * 64 + lane;
    frag[0] = o[0];
    frag[64] = o[1];
    if (h == 0) {
        sum = pinned(sum);
        const _Float16 hi = (_Float16)sum;
        const _Float16 lo = (_Float16)(sum - (float)hi);
        const int jj = s % 8;
        constexpr int step = IN_ORDER ? 256 : 8;
        _Float16 *a2 = IN_ORDER ? SxA + ((size_t)tb * (cols / 256) + s / 8) * 1024 + lane * 8 : SxA + ((size_t)t * (cols / 256) + s / 8) * 32;
        a2[jj] = hi;
        a2[step + jj] = hi;
        a2[2 * step + jj] = lo;
        a2[3 * step + jj] = (_Float16)0.f;
    }
}

// The same for f32 activations (the decode loops' prompt chunks): x = hi + 2^-11 lo with hi = f16(x) and
// lo = f16(2^11 (x - hi)), 22 bits of x, each part with its own fragments and its own sums.  The product then runs
// twice, the second pass adding 2^-11 times its result to the first.
__global__ __launch_bounds__(256) void mm_prep_x_f32_kernel(const float *__restrict__ X, _Float16 *__restrict__ Xf_hi,
                                                            _Float16 *__restrict__ Xf_lo, _Float16 *__restrict__ SxA_hi,
                                                            _Float16 *__restrict__ SxA_lo, int batch, int cols)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= batch * (cols / 8)) return;   // (whole quads: cols is a multiple of 32)
    const f32x4_t in0 = reinterpret_cast<const f32x4_t *>(X)[2 * (size_t)idx], in1 = reinterpret_cast<const f32x4_t *>(X)[2 * (size_t)idx + 1];
    const float f[8] = {in0.x, in0.y, in0.z, in0.w, in1.x, in1.y, in1.z, in1.w};
    h8 oh, ol;
    float fh[8], fl[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const _Float16 hi = (_Float16)f[i];
        const _Float16 lo = (_Float16)((f[i] - (float)hi) * 2048.0f);   // kept 2^11 up, in the normal range wherever hi is
        oh[kperm(i)] = hi;
        ol[kperm(i)] = lo;
        fh[i] = (float)hi;
        fl[i] = (float)lo;
    }
    float sh = ((fh[0] + fh[1]) + (fh[2] + fh[3])) + ((fh[4] + fh[5]) + (fh[6] + fh[7]));
    float sl = ((fl[0] + fl[1]) + (fl[2] + fl[3])) + ((fl[4] + fl[5]) + (fl[6] + fl[7]));
    sh += dpp_f32<0xB1>(sh);
    sh += dpp_f32<0x4E>(sh);
    sl += dpp_f32<0xB1>(sl);
    sl += dpp_f32<0x4E>(sl);
    const int k8 = cols / 8, t = idx / k8, j = idx - t * k8;
    const size_t frag = ((size_t)(t >> 5) * (cols / 16) + (j >> 1)) * 64 + (t & 31) + 32 * (j & 1);
    reinterpret_cast<h8 *>(Xf_hi)[frag] = oh;
    reinterpret_cast<h8 *>(Xf_lo)[frag] = ol;
    if ((threadIdx.x & 3) == 0) {
        const int s = j / 4, jj = s % 8;
        const size_t o = ((size_t)t * (cols / 256) + s / 8) * 32;
        const float sums[2] = {sh, sl};
        _Float16 *dst[2] = {SxA_hi + o, SxA_lo + o};
#pragma unroll
        for (int part = 0; part < 2; part++) {
            const float sum = pinned(sums[part]);
            const _Float16 hi = (_Float16)sum;
            const _Float16 lo = (_Float16)(sum - (float)hi);
            dst[part][jj] = hi;
            dst[part][8 + jj] = hi;
            dst[part][16 + jj] = lo;
            dst[part][24 + jj] = (_Float16)0.f;
        }
    }
}

// The same preparation with the producer of the rows folded in (f32 activations), one workgroup per row, cols / 8
// threads (1024 at most) with 8 consecutive elements each per trip:
//   MODE 0  x = X
//   MODE 1  x = rmsnorm(X, w)                                  (rmsnorm_rows, crates/ksearch_kernels/src/lib.rs:1478-1500)
//   MODE 2  x_new = res + rmsnorm(X, w_post), stored; x = rmsnorm(x_new, w_norm)   (rmsnorm_add_then_rmsnorm_rows)
//   MODE 3  x = gelu(X) * up                                   (gelu_mul on rows, gemma_prim.rs:1516-1538)
// in the operation order of the kernels that do these alone (every product and sum rounded by itself).
//
// inv_s = nullptr: the two parts as above (lo kept 2^11 up, each part with its own sums), for the small-batch form.
// inv_s != nullptr (the tile): the row is first scaled by the power of two s that puts its largest magnitude into
// [2^9, 2^10) -- exact, and any f32 row fits f16 then, sums of 32 elements included -- and x s = hi + lo with BOTH
// parts at that scale, so that one accumulator takes hi * w and lo * w of the same converted weight.  lo is a
// subnormal f16 for elements below 2^-13 of the row's largest; what that costs is below 2^-35 of the largest.  The
// sums of a sub-block are those of hi + lo, split in two halves as for bf16 rows; 1 / s goes to inv_s[row] for the
// tile's last step.
// Which row workgroup b prepares.  Eight neighbouring rows share every 128-byte line of the fragments, 16 bytes each, and
// workgroups go to the eight dies in turn: taken as they come, a line was written in eight pieces from eight L2s.  Eight
// rows in turn on one die meet in its L2 (2048 rows: 12288 columns 133 -> 102 us, 1536 columns 13.7 -> 11.2; 82 with the row kept instead of produced twice).
__device__ __forceinline__ int prep_row(int b, int rows)
{
    const int turn = b >> 3;
    return b < rows / 64 * 64 ? ((turn >> 3) * 8 + (b & 7)) * 8 + (turn & 7) : b;
}

template <int MODE>
__global__ __launch_bounds__(1024) void mm_prep_rows_kernel(const float *__restrict__ X, const float *__restrict__ P0, const float *P1,
                                                             const float *__restrict__ P2, float *x_out, _Float16 *__restrict__ Xf_hi,
                                                             _Float16 *__restrict__ Xf_lo, _Float16 *__restrict__ SxA_hi,
                                                             _Float16 *__restrict__ SxA_lo, int cols, float eps, int x_slices,
                                                             float *__restrict__ inv_s)
{
    // x_slices != 0: X is the unfolded partial sums of the GEMM that produced it, [slice][row][stride] with stride =
    // cols (MODE 3: 2 * cols, gate | up side by side, and `up` is read from there); the slices are added here in the
    // fold's order
    __shared__ float red[3][16];
    const int t = prep_row(blockIdx.x, gridDim.x), lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    auto ld8 = [](const float *p, float (&v)[8]) __attribute__((always_inline)) {
        const f32x4_t a = reinterpret_cast<const f32x4_t *>(p)[0], b = reinterpret_cast<const f32x4_t *>(p)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    };
    auto row_sum = [&](float v, int which) __attribute__((always_inline)) {
        v = wave_sum(v);
        if (lane == 0) red[which][wave] = v;
        __syncthreads();
        float s = 0.f;
        for (int i = 0; i < nw; i++) s += red[which][i];
        return s;
    };
    const size_t x_stride = MODE == 3 ? 2 * (size_t)cols : (size_t)cols, x_plane = (size_t)gridDim.x * x_stride;
    auto ldx = [&](int j, size_t col0, float (&v)[8]) __attribute__((always_inline)) {
        const float *src = X + (size_t)t * x_stride + col0 + 8 * (size_t)j;
        ld8(src, v);
        for (int k = 1; k < x_slices; k++) {
            float a[8];
            ld8(src + (size_t)k * x_plane, a);
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] += a[i];
        }
    };
    // the row's elements 8j .. 8j+7 (the norms run with cols / 8 threads, one trip; plain rows and gelu * up of longer
    // rows take several)
    auto produce = [&](int j, float (&f)[8]) __attribute__((always_inline)) {
        const size_t e0 = (size_t)t * cols + 8 * (size_t)j;
        if (x_slices) ldx(j, 0, f);
        else ld8(X + e0, f);
        if (MODE == 1 || MODE == 2) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) ss += f[i] * f[i];
            const float inv = 1.0f / sqrtf(row_sum(ss, 0) / (float)cols + eps);
            float w[8];
            ld8(P0 + 8 * j, w);
#pragma unroll
            for (int i = 0; i < 8; i++) f[i] = __fmul_rn(__fmul_rn(f[i], inv), w[i]);
            if (MODE == 2) {
                float r[8], wn[8];
                ld8(P1 + e0, r);
                float ss2 = 0.f;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    f[i] = __fadd_rn(r[i], f[i]);
                    ss2 += f[i] * f[i];
                }
                reinterpret_cast<f32x4_t *>(x_out + e0)[0] = f32x4_t{f[0], f[1], f[2], f[3]};
                reinterpret_cast<f32x4_t *>(x_out + e0)[1] = f32x4_t{f[4], f[5], f[6], f[7]};
                const float inv2 = 1.0f / sqrtf(row_sum(ss2, 1) / (float)cols + eps);
                ld8(P2 + 8 * j, wn);
#pragma unroll
                for (int i = 0; i < 8; i++) f[i] = __fmul_rn(__fmul_rn(f[i], inv2), wn[i]);
            }
        }
        if (MODE == 3) {
            float u[8];
            if (x_slices) ldx(j, (size_t)cols, u);
            else ld8(P0 + e0, u);
#pragma unroll
            for (int i = 0; i < 8; i++) f[i] = gelu_mul_f32(f[i], u[i]);
        }
    };
    const int octets = cols / 8;
    // (rows of up to KEEP octets a thread are produced once and kept; the norms' sums want one)
    constexpr int KEEP = MODE == 1 || MODE == 2 ? 1 : 2;
    const bool keep = octets <= KEEP * (int)blockDim.x;
    float kept[KEEP][8];
    float s = 1.0f;
    if (inv_s) {
        // the row's largest magnitude (rows too long to keep are produced again below)
        float m = 0.f;
        if (keep) {
#pragma unroll
            for (int u = 0; u < KEEP; u++) {
                const int j = threadIdx.x + u * blockDim.x;
                if (j < octets) {
                    produce(j, kept[u]);
#pragma unroll
                    for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(kept[u][i]));
                }
            }
        } else {
            for (int j = threadIdx.x; j < octets; j += blockDim.x) {
                float f[8];
                produce(j, f);
#pragma unroll
                for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(f[i]));
            }
        }
        m = wave_max(m);
        if (lane == 0) red[2][wave] = m;
        __syncthreads();
        for (int i = 0; i < nw; i++) m = fmaxf(m, red[2][i]);
        // s = 2^(9 - floor(log2 m)); rows of zeros (and anything below 2^-112) take 2^121, infinities and NaNs 2^-118
        const uint32_t e = (uint32_t)max((int)((as_u32(m) >> 23) & 0xFFu), 15);
        s = as_f32((263u - e) << 23);
        if (threadIdx.x == 0) inv_s[t] = as_f32((e - 9u) << 23);
    }
    auto write = [&](int j, const float (&f)[8]) __attribute__((always_inline)) {
        h8 oh, ol;
        float fh[8], fl[8];
        const float lo_up = inv_s ? 1.0f : 2048.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float x = pinned(f[i]) * s;
            const _Float16 hi = (_Float16)x;
            const _Float16 lo = (_Float16)((x - (float)hi) * lo_up);
            oh[kperm(i)] = hi;
            ol[kperm(i)] = lo;
            fh[i] = (float)hi;
            fl[i] = (float)lo;
        }
        float sh = ((fh[0] + fh[1]) + (fh[2] + fh[3])) + ((fh[4] + fh[5]) + (fh[6] + fh[7]));
        float sl = ((fl[0] + fl[1]) + (fl[2] + fl[3])) + ((fl[4] + fl[5]) + (fl[6] + fl[7]));
        sh += dpp_f32<0xB1>(sh);
        sh += dpp_f32<0x4E>(sh);
        sl += dpp_f32<0xB1>(sl);
        sl += dpp_f32<0x4E>(sl);
        const size_t frag = ((size_t)(t >> 5) * (cols / 16) + (j >> 1)) * 64 + (t & 31) + 32 * (j & 1);
        reinterpret_cast<h8 *>(Xf_hi)[frag] = oh;
        reinterpret_cast<h8 *>(Xf_lo)[frag] = ol;
        if ((threadIdx.x & 3) == 0) {
            const int sbk = j / 4, jj = sbk % 8;
            const size_t o = ((size_t)t * (cols / 256) + sbk / 8) * 32;
            const float sums[2] = {inv_s ? sh + sl : sh, sl};
            _Float16 *dst[2] = {SxA_hi + o, SxA_lo + o};
#pragma unroll
            for (int part = 0; part < 2; part++) {
                if (part && inv_s) break;       // (one set of sums; the other operand's place holds inv_s)
                const float sum = pinned(sums[part]);
                const _Float16 hi = (_Float16)sum;
                const _Float16 lo = (_Float16)(sum - (float)hi);
                // (the tile's: fragments of 32 tokens too, hi | hi and lo | 0)
                _Float16 *a2 = inv_s ? SxA_hi + (((size_t)(t >> 5) * (cols / 256) + sbk / 8) * 128 + (t & 31)) * 8 : dst[part];
                const int h1 = inv_s ? 256 : 8, k1 = inv_s ? 512 : 16;
                a2[jj] = hi;
                a2[h1 + jj] = hi;
                a2[k1 + jj] = lo;
                a2[k1 + h1 + jj] = (_Float16)0.f;
            }
        }
    };
    if (inv_s && keep) {
#pragma unroll
        for (int u = 0; u < KEEP; u++)
            if ((int)(threadIdx.x + u * blockDim.x) < octets) write(threadIdx.x + u * blockDim.x, kept[u]);
    } else {
        for (int j = threadIdx.x; j < octets; j += blockDim.x) {
            float f[8];
            produce(j, f);
            write(j, f);
        }
    }
}

// eight bf16 of a row as f16, in the order of the weights beside them (kperm)
__device__ __forceinline__ h8 from_bf16(h8 raw)
{
    const u32x4_t w = __builtin_bit_cast(u32x4_t, raw);
    h8 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o[kperm(2 * i)] = (_Float16)as_f32(w[i] << 16);
        o[kperm(2 * i + 1)] = (_Float16)as_f32(w[i] & 0xFFFF0000u);
    }
    return o;
}

struct MmParams {
    const uint8_t *W;
    const _Float16 *Xf, *SxA;   // fragment-ordered f16 activations (mm_prep_x_kernel), sums of x
    float *Y;
    int rows, cols, batch;
    // Small grids (few tokens x few weight rows): blockIdx.z = K slice.  A workgroup then takes the superblocks of
    // its slice only and every z stores its own batch x rows partial sums behind Y_parts for the fold (ksplit = 0:
    // full K, results in Y).
    int ksplit;
    float *Y_parts;
    // Up to three matrices that share the activations (q | k | v of a prompt chunk) in one launch of the
    // tile: blockIdx.y counts the row tiles of W, then of W1, then of W2, each with its own result.
    const uint8_t *W1, *W2;
    float *Y1, *Y2;
    int rows1, rows2;
    // f32 activations (the kernel's LO form): the lo parts' fragments and 1 / s per token row (see mm_prep_rows_kernel)
    const _Float16 *Xf_lo;
    const float *inv_s;
    // the kernel's CUT form: per row, the tokens of the launch whose K slices its sums are to be cut into
    const float *cut_as;
    // q4k_mm_rows_kernel's numbering of the workgroups: how many there are, in x and in y, ceil(2^32 / gx) and ceil(2^32 / gy)
    // (exact quotients where wgs * gx and wgs * gy stay below 2^32; wgs = 0: as the launch numbers them)
    uint32_t wgs, gx, gy, per_gx, per_gy;
    // bf16 rows: results go through the L2s as usual (mm_keeps)
    int keep;
};

template <bool KEEP>
__device__ __forceinline__ void mm_store(float *y, float v)
{
    if (KEEP) *y = v;
    else __builtin_nontemporal_store(v, y);
}

// F32 activations: the tokens and weight rows (BN) of the tiles that the rule of the K slices counts.  How a row's sum is cut
// decides its bits, so the rule stays when the tiles that do the work change (q4k_mm_rows_kernel's are others).
__host__ __device__ constexpr int mm_tile_tokens(bool q6) { return q6 ? 128 : 64; }

// F32 activations, few tiles (a prompt of a few hundred tokens, or a narrow matrix): the nsb superblocks of a row are split
// into this many K slices, until the grid is about one workgroup per compute unit; every slice has its own sum and the
// sums are added in a fixed order.  (A slice of one superblock is all prologue; the workgroups are counted with the token
// tile they will have, and rows of more than half a prompt pass as that many: how a row's sum is cut does not depend on
// which pass of its prompt the row is in.)
__host__ __device__ constexpr int mm_k_slices(bool q6, int row_tiles, int nsb, int batch)
{
    const int counted = batch > kPrefillPass / 2 ? kPrefillPass / 2 : batch;
    int ks = 1;
    while (nsb % (ks * 2) == 0 && nsb / (ks * 2) >= 2) {
        const int tm = mm_tile_tokens(q6);
        if ((int64_t)((counted + tm - 1) / tm) * row_tiles * ks * 2 > 256) break;
        ks *= 2;
    }
    return ks;
}

// Results of bf16 rows go past the L2s, since what those hold of them at the kernel's end is written out before the next kernel starts
// (figures at the kernels' ends).  Not so:
// - Small partial sums, which the fold reads at once, and waits the longer for the more slices there are: 10 tokens of 297 x 7424 in 29
//   slices (0.3 MB) 10.9 us past the L2s or 9.9 kept, 39 of 580 x 5120 in 20 (1.8 MB) 11.8 or 11.1, 11 of 3832 x 3328 in 13 (2.2
//   MB) even, 153 of 495 x 7680 in 15 (4.5 MB) 16.4 or 17.0, 36 of 3288 x 2304 in 9 (4.3 MB) 11.5 or 12.0; Q6_K alike.  (Whole results
//   of that size 1 % shorter.)
// - Few slices of large results, whose fold is bound by what it moves (two slices of Q6_K, 733 tokens of 2549 x 3072 34.6 or 31.9 us, 315
//   of 4905 x 2560 29.2 or 28.0; 4.9 MB a slice 27.1 or 26.2, 3.7 even).
// - Results of the tile of two roles (one workgroup a compute unit, nobody works while it stores) whose rows are not whole pieces of 64
//   bytes: 1785 tokens of 4311 x 1024 46.1 or 36.4 us, 573 of 11713 x 1024 45.7 or 39.6, 463 of 3272 x 768 14.3 or 14.0, 339 of 5959 x 2816
//   even; in whole pieces 338 of 9616 x 1792 25.9 or 27.4, 512 of 8192 x 2048 30.8 or 32.8.  (The others' within 5 % either way.)
// 344 shapes with slices: 0.04 % over the better of the two on average and 1.6 % at most, all past 3.0 % on average, all kept 1.2 %.
bool mm_keeps(int ks, int64_t batch, int64_t rows_all, bool two_roles, int64_t rows, int64_t rows1, int64_t rows2)
{
    const int64_t slice = batch * rows_all * 4;
    if (ks * slice <= 1000000 + (int64_t)ks * 160000) return true;
    return ks > 1 ? slice >= 3600000 : two_roles && ((rows | rows1 | rows2) & 15);
}

// Bf16 activations: token tile and K slices (of any number of superblocks) by what the launches are made of, in us:
//   preparation (Q4_K), launches, what rows and results cost; per round of workgroups over the compute units; per superblock of
//   the slice in one round, in two, in more (each), more as the chip fills; the fold and its round trips, eight slices each
// Fitted to 525 shapes of 200 .. 16384 rows of 512 .. 8192 columns, 2 .. 2048 tokens, with every slice count that shortens a slice,
// called one after the other as a program calls them.  Against the best (tile, slices) of 420 others: Q4_K 0.8 % over it on average,
// 5 % at 19 in 20, 17 % at most, Q6_K 0.2 %, 1 %, 10 % (the figures of the kernels before these 1.4, 9, 22 and 1.1, 8, 21).  224 tokens of
// 1653 x 4608 20.3 us, with 64 tokens a workgroup 17.9; 512 of 8192 x 2048 27.7, so 28.5.
struct MmPlan {
    int tm, ks;
    float us;
};
MmPlan mm_plan_bf16(bool q6, int row_tiles, int nsb, int64_t batch, int64_t rows_all, int ks_given)
{
    struct Cost {
        int tm;
        float launch, round, one, two, more, fill, out, out_more, fold, trip, part;
    };
    constexpr Cost kQ4[] = {{64, 5.765f, 0.035f, 1.236f, 1.626f, 0.812f, 0.156f, 1.178f, 1.056f, 1.674f, 0.501f, 1.744f},
                            {128, 6.168f, 0.041f, 1.767f, 2.606f, 1.338f, 0.124f, 1.19f, 1.26f, 1.919f, 0.584f, 1.408f}};
    constexpr Cost kQ6[] = {{32, 2.974f, 0.424f, 1.888f, 2.881f, 1.306f, 0.081f, 1.314f, 0.f, 1.712f, 0.479f, 1.474f},
                            {64, 3.872f, 0.06f, 2.121f, 3.147f, 1.582f, 0.076f, 0.962f, 0.913f, 1.885f, 0.43f, 1.564f},
                            {128, 2.364f, 1.164f, 2.378f, 4.471f, 2.11f, 0.074f, 1.241f, 1.701f, 1.968f, 0.515f, 1.813f}};
    MmPlan best{128, 1, 1e30f};
    const int ks_max = std::min(nsb, 64);
    const float m = (float)(batch * rows_all) * 1e-6f;
    for (const Cost *c = q6 ? kQ6 : kQ4, *end = c + (q6 ? 3 : 2); c < end; c++)
        for (int ks = ks_given ? ks_given : 1; ks <= (ks_given ? ks_given : ks_max); ks++) {
            const int64_t wgs = (batch + c->tm - 1) / c->tm * row_tiles * ks;
            const float sb = (float)((nsb + ks - 1) / ks), w = std::min((float)wgs / 256.f, 2.f), rounds = (float)((wgs + 255) / 256);
            const float each = rounds <= 1.f ? c->one : rounds <= 2.f ? c->two : c->more * rounds;
            const float us = c->launch + c->round * rounds + each * (1.f + c->fill * w) * sb + (rounds <= 2.f ? c->out : c->out_more) * m +
                             (q6 ? 0.f : (float)(batch * nsb) * 256e-6f) + (ks > 1 ? c->fold + c->trip * (float)((ks + 6) / 8) + c->part * (float)ks * m : 0.f);
            if (us < best.us) best = MmPlan{c->tm, ks, us};
        }
    return best;
}

// (the small-batch form's way of loading, see the figures at q4k_mm_skinny_kernel)
constexpr bool skinny_pieces(int mt, bool lo, int nsb)
{
    if (mt == 1) return lo ? nsb % 8 == 0 || nsb > 12 : nsb > 4;
    return !lo && nsb % 8 == 0;
}

// The small-batch form beside it (Q4_K, bf16), with its preparation: a workgroup of eight waves per 32 rows, superblocks dealt to
// the waves, the fullest of which has `turns` (fitted to 230 of those shapes, 2 to 5 % off; where it is chosen 18 % over the best at most: 59
// tokens of 9510 x 512 10.8 us, 9.2 in the tile).  50 tokens of 10158 x 4352 28.3 us here, 19.2 in the tile; 5 of 1442 x 6144 9.9 and 10.8.
float mm_skinny_us(int64_t rows, int nsb, int64_t batch)
{
    const float turns = (float)((nsb + 7) / 8), each = (float)nsb / 8.f, x = (float)(batch * nsb) * 1e-3f, more = (float)((rows + 8191) / 8192 - 1);
    if (batch <= 32) return 4.99f + 0.84f * turns + each * (0.73f + 1.57f * more) + 1.99f * x;
    if (skinny_pieces(2, false, nsb)) return 5.01f + each * (3.97f + 4.22f * more) + 1.67f * x;
    return 4.75f + 2.13f * turns + each * (1.8f + 5.41f * more) + 2.42f * x;
}

// The form of one launch beside both (mm_few: bf16 tokens in groups of up to 32, Q4_K and Q6_K): workgroups of a group's tokens and rh tiles
// of 16 weight rows, as many to a compute unit at a time as its LDS takes, in rounds; `turns` superblocks to the fullest wave.  Fitted to
// 780 shapes of 200 .. 16384 rows, 512 .. 8192 columns, 1 .. 800 tokens (4 % off, 10 % at 19 in 20; the shortest of it and the others is
// 0.4 % over the best of all on average, 18 % at most).  In those up to 32 tokens the others take 1.64 times as long, beyond 1.27: Q4_K, 2
// tokens of 2048 x 2048 6.3 -> 3.4 us, 16 of 4096 x 4096 9.0 -> 5.6, 32 9.5 -> 7.7, 5 of 2048 x 8192 12.4 -> 7.1, 246 of 428 x 2048 12.0 ->
// 4.9; Q6_K 7.5 -> 4.0, 11.8 -> 6.9, 12.9 -> 9.1, 11.4 -> 8.8, 333 of 280 x 1280 11.1 -> 4.3.  32 of 8192 x 2048 Q4_K stay where they are (7.4;
// 9.1 so).  It is taken where it is estimated 4 % shorter.
struct FewPlan {
    int rh, tokens;
    float us;
    int64_t wgs;
};
// Whether a call that leaves the schedule open may take it: where the estimate holds (of 405 further shapes inside the fit's range at which it is
// taken the others are the shorter ones at 4, by 21 % at most).  Not rows of more than 8192 columns, where a wave has five superblocks and more one behind
// the other (19 x 24576, 5 tokens 11.5 us and 15.2 so, 64 x 16384, 1000 tokens 16.8 and 24.8); more than 256 tokens of more than 4096
// columns (128 x 8192, 1000 tokens 15.9 and 28.3, 512 13.0 and 14.2); Q4_K of 256 columns in more workgroups than compute units (65536 rows, 1
// token 12.0 and 15.0, 14412, 21 tokens 6.7 and 8.6, 2048, 192 tokens 7.4 and 8.2).  Q4_K beyond 192 tokens, left open, stays the
// tile, whose handles report its K slices (300 rows of 1536 columns, 200 tokens: 11 us, 4 in this form).
bool mm_few_open(bool q6, int nsb, int64_t batch, const FewPlan &few)
{
    return nsb <= 32 && batch <= (q6 ? kFewMost : 192) && (nsb <= 16 || batch <= 256) && (q6 || nsb > 1 || few.wgs <= 256);
}
FewPlan mm_few_plan(bool q6, int64_t rows, int nsb, int64_t batch)
{
    struct Cost {
        float launch, round, turn, each, tile, rows16, token;
    };
    constexpr Cost kCost[2][2] = {{{1.848f, 1.301f, 0.118f, 0.016f, -0.388f, 0.909f, 0.03f}, {1.495f, 0.944f, 0.583f, 0.362f, 0.f, 0.299f, 0.038f}},
                                  {{1.639f, 1.406f, 0.098f, 0.106f, -0.536f, 1.522f, 0.029f}, {1.302f, 0.114f, 0.254f, 1.71f, 0.f, 1.198f, 0.032f}}};
    FewPlan best{1, 1, 1e30f, 0};
    const float turns = (float)((nsb + 7) / 8), each = (float)nsb / 8.f;
    for (int most : {32, 16})
        for (int rh : {1, 2, 4}) {
            const int64_t groups = (batch + most - 1) / most;
            const int tokens = (int)((batch + groups - 1) / groups);
            if (!few_fits(q6, tokens, rh)) break;
            const Cost &c = kCost[q6][tokens > 16];
            const int64_t wgs = (rows + 16 * rh - 1) / (16 * rh) * groups, load = (wgs + 255) / 256, fit = 163840 / few_lds(q6, tokens, rh);
            const float us = c.launch + (float)((load + fit - 1) / fit) * (c.round + c.turn * turns) +
                             (float)load * (c.each + each * (c.tile + c.rows16 * (float)rh + c.token * (float)tokens));
            if (us < best.us) best = FewPlan{rh, tokens, us, wgs};
        }
    return best;
}

// Bf16 rows of Q6_K products as they are (the kernel's ROWS form): the conversion between the matrix instructions costs 0.25
// us per superblock and round, the preparation a launch (2.5 us) and its pass over X (316 tokens of 3005 x 2048 28.2 us prepared, 26.0
// as they are, 1211 of 8949 x 1280 73.9 and 68.6, 677 of 12177 x 8192 247 and 263).  At those shapes and their slice counts 0.1 % over
// the better of the two on average, 7 % at most.
bool mm_rows_direct(int64_t workgroups, int sb_per_slice, int64_t batch, int64_t cols)
{
    return 0.25f * (float)((workgroups + 255) / 256 * sb_per_slice) < 2.5f + (float)(batch * cols) * 1.1e-6f;
}

__device__ __forceinline__ uint32_t pair_f16(uint32_t masked, uint32_t sc)
{
    return __umul24(masked, sc) + 0x64006400u;     // half 1024.0 twice
}

constexpr int kThreadsMM = 512;
constexpr int kLdsMain = BN * PITCH;             // halves per main stage (the dequantized weight tile)

// A wave's way to 32 rows of a Q6_K superblock: 16-byte pieces at 16-byte addresses, 14 of them around a row's 210 bytes (which
// begin at any even one), lane after lane along the rows, and by way of LDS to the lanes that want them.  A row a lane, at those
// odd addresses, takes L1 186 cycles a load of 16 bytes (of 8 bytes 72), and L1 was busy for as long as the kernels ran.
// (A piece holds a byte of the matrix at least: what else it reads lies in the same 16 bytes.)
struct Q6Way {
    static constexpr int kPitch = 240, kBytes = 32 * kPitch;
    struct Pieces { u32x4_t v[7]; };
    const uint8_t *tile;
    uint8_t *lds;
    uint32_t row_bytes, off[7];
    int last, slot[7], at[7], nsb;

    __device__ __forceinline__ Q6Way(const uint8_t *W, int r0, int rows, int nsb_row, int sb0, int nsb_, uint8_t *lds_, int lane)
        : tile(W + ((size_t)min(r0, rows - 1) * nsb_row + sb0) * 210), lds(lds_), row_bytes((uint32_t)nsb_row * 210u), last(min(32, max(1, rows - r0)) - 1), nsb(nsb_)
    {
#pragma unroll
        for (int i = 0; i < 7; i++) {
            const int c = 64 * i + lane, row = c / 14;
            off[i] = (uint32_t)min(row, last) * row_bytes;
            slot[i] = 16 * (c % 14);
            at[i] = row * kPitch + slot[i];
        }
    }
    __device__ __forceinline__ void fetch(int sb, Pieces &w) const
    {
        const uint8_t *b = tile + (size_t)min(sb, nsb - 1) * 210;
        const uint32_t low = (uint32_t)(uintptr_t)b & 15u;
        b -= low;
#pragma unroll
        for (int i = 0; i < 7; i++) w.v[i] = *reinterpret_cast<const u32x4_t *>(b + (((off[i] + low) & ~15u) + (uint32_t)slot[i]));
    }
    // (a wave's LDS operations complete in order: the fences keep the compiler from moving them)
    __device__ __forceinline__ void put(const Pieces &w) const
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
#pragma unroll
        for (int i = 0; i < 7; i++) *reinterpret_cast<u32x4_t *>(lds + at[i]) = w.v[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // the words that row r's block begins in, and the bits of the first that come before it
    __device__ __forceinline__ const uint32_t *row(int sb, int r, uint32_t &bits) const
    {
        const uint32_t a = (uint32_t)(uintptr_t)(tile + (size_t)min(sb, nsb - 1) * 210 + (uint32_t)min(r, last) * row_bytes) & 15u;
        bits = (a & 2u) * 8u;
        return reinterpret_cast<const uint32_t *>(lds + r * kPitch + (a & 12u));
    }
};
// A code as it stands, the bits of a half, is code * 2^-24; with a scale 2^8 up, fma(code, scale, -32 * scale) is q * sc * 2^-16 in
// one instruction, rounded as the product q * sc of halves is, and d takes the 2^16 back (f16 of any size counts in full here, the
// subnormal ones too).
constexpr float kQ6Unit = 65536.f;
constexpr _Float16 kQ6Offset = (_Float16)(-32.f / 16777216.f);
__device__ __forceinline__ h2 q6_scale(int8_t sc)
{
    const _Float16 s = (_Float16)(float)((int)sc * 256);
    return h2{s, s};
}
// N words of a block from word `at` on
template <int N>
__device__ __forceinline__ void q6_words(const uint32_t *row, uint32_t bits, int at, uint32_t *v)
{
    uint32_t raw[N + 1];
#pragma unroll
    for (int i = 0; i <= N; i++) raw[i] = row[at + i];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = __builtin_amdgcn_alignbit(raw[i + 1], raw[i], bits);
}
constexpr size_t kLdsBytes = 2 * (size_t)kLdsMain * 2 + 2 * BN * 4 + 4 * Q6Way::kBytes;

// The GEMM over Q6_K weights (K3b of the reference's plan: Q6_K tensors in prefill): 128 tokens x 128 weight rows a workgroup,
// eight waves in two roles, one of each per SIMD.  Waves 0..3 only multiply:
// each owns 32 tokens x 128 columns (1 x 4 MFMA tiles) and works on LDS stage s&1.  Waves 4..7 only
// load and convert: during the same step they request the activations of step
// s+4 (and, when a superblock opens, the next superblock's weights) and write
// step s+1 into stage (s+1)&1.  One barrier per K step joins them, so the
// conversions and the LDS writes of one role run in the shadow of the other
// role's matrix instructions.
//
// w = d * sc_j * q with q = code - 32 in [-32, 31] and sc_j an int8 per 16 columns; the loaders build sc_j * q two at a time,
// as a packed fma of halves (q6_scale).
// What bounds it: the vector instructions, which here add to the matrix instructions' time (one loading and one multiplying wave
// on a SIMD; pipe busy a third of the cycles).  Hence words by alignbit and perm and one fma a pair, 9 instructions to four
// weights where 11.5 were, and the weights by pieces (Q6Way): 2048 tokens, 12288 x 4096 309 -> 279 us, 512 tokens, 8192 x 2048
// 35.4 -> 32.5, 333 tokens, 1536 x 6144 in six slices 25.3 -> 23.3.
// sc_j * q is exact in f16 up to 2048; beyond that (needs |sc_j| > 64) it rounds to the nearest even integer, a
// relative 2^-11 at most and on those weights only (the reference's tile rounds every weight to half, the same
// bound).  There is no min term; d is applied per superblock as for Q4_K.
// LO = true: f32 activations as two f16 parts at the row's own scale.  Every converted weight meets the hi and the lo
// fragment of a token tile in the same accumulator (twice the matrix instructions per conversion, and the
// conversions are what a step waits for), and the finished sums are multiplied by 1 / s of their token.
// CUT = true (f32 activations): the rows belong to prompts that would each have had a launch of their own, whose K slices
// depend on its length.  The workgroup takes all of K, and where a row's slice ends its sum is added to Y and starts
// again from zero: the bits of those launches from one that fills the chip (a read and a write of the tile's results
// per slice end, from L2).
// ROWS = true (bf16 activations; no sums of x are wanted): the A operands come from the rows of X as they are
// and the multiplying waves convert them, eight values of a row a lane, between their matrix instructions -- no
// preparation launch (mm_rows_direct; 333 tokens, 1536 x 6144 in six slices: 28.9 -> 25.4 us).
template <bool LO, bool CUT = false, bool ROWS = false>
__global__ __launch_bounds__(kThreadsMM, 1) void q6k_mul_mm_kernel(MmParams p)
{
    extern __shared__ __attribute__((aligned(16))) _Float16 lds[];
    auto main_stage = [&](int i) { return lds + (i & 1) * kLdsMain; };
    auto dsc_stage = [&](int i) { return reinterpret_cast<float *>(lds + 2 * kLdsMain) + (i & 1) * BN; };

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // which matrix this row tile belongs to (the copy of the arguments is this workgroup's own)
    int by = blockIdx.y, ycol = 0;
    const int rows_all = p.rows + p.rows1 + p.rows2;
    const int rows_of[3] = {p.rows, p.rows1, p.rows2};
    if (p.rows1) {
        const int ty0 = (p.rows + BN - 1) / BN, ty1 = (p.rows1 + BN - 1) / BN;
        if (by >= ty0 + ty1) { by -= ty0 + ty1; ycol = p.rows + p.rows1; p.W = p.W2; p.Y = p.Y2; p.rows = p.rows2; }
        else if (by >= ty0) { by -= ty0; ycol = p.rows; p.W = p.W1; p.Y = p.Y1; p.rows = p.rows1; }
    }
    const int t0 = blockIdx.x * BM, r0 = by * BN;
    const int nsb_row = p.cols / 256;                            // superblocks per weight row
    int nsb = nsb_row, sb0 = 0;                                  // this workgroup's share of them
    size_t ystride = (size_t)p.rows;
    if (p.ksplit) {
        const int slice = blockIdx.z;
        sb0 = nsb_row * slice / p.ksplit;
        nsb = nsb_row * (slice + 1) / p.ksplit - sb0;
        p.Y = p.Y_parts + (size_t)blockIdx.z * p.batch * rows_all + ycol;   // partial sums: all matrices' columns side by side
        ystride = (size_t)rows_all;
    }
    const int nsteps = nsb * 4;

    if (wave >= 4) {
        // ------------------------------------------------------------------ loaders
        // thread lh of a row's pair converts columns 32*lh .. 32*lh+31 of every 64-column step: step (h, part)
        // of a superblock = ql bytes 64h + 32lh .. +31 (nibble `part`), qh bytes 32h .. +31 (bit pair
        // 4*part + 2*lh), scales 8h + 4*part + 2*lh and the next one.  Blocks are 2-byte aligned.
        const int lt = tid - 256, lrow = lt >> 1, lh = lt & 1;
        const Q6Way rows(p.W, r0 + 32 * (wave - 4), p.rows, nsb_row, sb0, nsb, reinterpret_cast<uint8_t *>(lds + 2 * kLdsMain) + 2 * BN * 4 + (wave - 4) * Q6Way::kBytes, lane);
        struct Sb6Regs {
            uint32_t ql[16];  // [8h + i]: ql bytes 64h + 32lh + 4i .. +3
            uint32_t qh[16];  // all 64 qh bytes
            uint32_t sc[4];   // the 16 int8 scales
            uint32_t d;
        };
        auto take = [&](int sb, Sb6Regs &r) __attribute__((always_inline)) {
            uint32_t bits;
            const uint32_t *q = rows.row(sb, lane >> 1, bits);
            q6_words<8>(q, bits, 8 * lh, r.ql);
            q6_words<8>(q, bits, 16 + 8 * lh, r.ql + 8);
            q6_words<16>(q, bits, 32, r.qh);
            q6_words<4>(q, bits, 48, r.sc);
            r.d = (q[52] >> bits) & 0xFFFFu;
        };
        auto stage = [&](int step, auto gtag, const Sb6Regs &w) __attribute__((always_inline)) {
            constexpr int G = decltype(gtag)::value, H = G >> 1, P = G & 1;
            _Float16 *Bs = main_stage(step);
            const uint32_t s16 = (w.sc[2 * H + P] >> (16 * lh)) & 0xFFFFu;
            const h2 sc2[2] = {q6_scale((int8_t)(s16 & 0xFFu)), q6_scale((int8_t)(s16 >> 8))};
            const h2 off2[2] = {sc2[0] * kQ6Offset, sc2[1] * kQ6Offset};
            const int hsh = 4 * P + 2 * lh;
            uint32_t o[16];
#pragma unroll
            for (int j = 0; j < 8; j++) {   // 4 columns per dword; dwords 0..3 take the first scale, 4..7 the second
                const uint32_t L = w.ql[8 * H + j], Q = w.qh[8 * H + j];
                const uint32_t nib = (P ? (L >> 4) : L) & 0x0F0F0F0Fu;
                const uint32_t c = nib | (__builtin_amdgcn_alignbit(Q, Q, (uint32_t)(hsh - 4) & 31u) & 0x30303030u);   // four 6-bit codes (turned: only whole bytes' bits stay)
                // columns (0, 2) and (1, 3), as halves
                const h2 va = __builtin_elementwise_fma(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, c, 0x0C020C00u)), sc2[j >> 2], off2[j >> 2]);
                const h2 vb = __builtin_elementwise_fma(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, c, 0x0C030C01u)), sc2[j >> 2], off2[j >> 2]);
                o[2 * j] = __builtin_bit_cast(uint32_t, va);
                o[2 * j + 1] = __builtin_bit_cast(uint32_t, vb);
            }
            uint4 *dst = reinterpret_cast<uint4 *>(&Bs[lrow * PITCH + 32 * lh]);
#pragma unroll
            for (int i = 0; i < 4; i++) dst[i] = make_uint4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
            if (G == 0 && lh == 0) dsc_stage(step >> 2)[lrow] = half_bits_to_f32(w.d) * kQ6Unit;
        };
        Q6Way::Pieces next;
        Sb6Regs w;
        rows.fetch(0, next);
        rows.put(next);
        take(0, w);
        stage(0, std::integral_constant<int, 0>{}, w);
        __syncthreads();
        auto step_body = [&](int sb, auto gtag) __attribute__((always_inline)) {
            constexpr int g = decltype(gtag)::value;
            const int step = 4 * sb + g;
            if (g == 0) {
                rows.fetch(sb + 1, next);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (step + 1 < nsteps) {
                if (g == 3) {
                    rows.put(next);
                    take(sb + 1, w);
                }
                stage(step + 1, std::integral_constant<int, (g + 1) & 3>{}, w);
            }
            __syncthreads();
        };
        for (int sb = 0; sb < nsb; sb++) {
            step_body(sb, std::integral_constant<int, 0>{});
            step_body(sb, std::integral_constant<int, 1>{});
            step_body(sb, std::integral_constant<int, 2>{});
            step_body(sb, std::integral_constant<int, 3>{});
        }
        return;
    }

    // ---------------------------------------------------------------------- multipliers
    // A multiplying wave owns 32 tokens x all 128 columns instead of 64 x 64 -- one A fragment per k slice serves four
    // products, so the activations cross the vector-memory path once per workgroup instead of twice, and all four waves read
    // every B operand from LDS (twice the LDS reads, which the operands requested a slice ahead hide).
    constexpr int NW_ = 4;
    const int wm = wave;
    f16v F[NW_], Cp[NW_];
#pragma unroll
    for (int b = 0; b < NW_; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) { F[b][i] = 0.f; Cp[b][i] = 0.f; }
    const int lm = lane & 31, lk = (lane >> 5) * 8;
    const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // A operands straight from memory: fragment (token tile, k / 16) is 64 lanes x 16 bytes, 1 KB apart along k.
    // Two register sets, each refilled for two steps ahead as soon as its own step's instructions are issued (LO: one
    // set of hi and lo fragments, refilled for the next step -- a step is long against the way to the cache).
    const int ntt = (p.batch + 31) / 32;
    const uint16_t *xrow = reinterpret_cast<const uint16_t *>(p.Xf) + (size_t)min(t0 + wm * 32 + lm, p.batch - 1) * p.cols + (size_t)sb0 * 256 + lk;   // ROWS
    const h8 *xa = reinterpret_cast<const h8 *>(p.Xf) + ((size_t)min(t0 / 32 + wm, ntt - 1) * (p.cols / 16) + (size_t)sb0 * 16) * 64 + lane;
    const ptrdiff_t lo_delta = LO ? reinterpret_cast<const h8 *>(p.Xf_lo) - reinterpret_cast<const h8 *>(p.Xf) : 0;
    auto afrag = [&](int step, int ks) __attribute__((always_inline)) {
        if (ROWS) return *reinterpret_cast<const h8 *>(xrow + step * KS + 16 * ks);      // (bf16 as yet)
        return xa[(ptrdiff_t)(step * (KS / 16) + ks) * 64];
    };
    auto afrag_lo = [&](int step, int ks) __attribute__((always_inline)) { return xa[(ptrdiff_t)(step * (KS / 16) + ks) * 64 + lo_delta]; };
    constexpr int AHEAD = LO ? 1 : 2;
    struct ARegs { h8 a[KS / 16], al[LO ? KS / 16 : 1]; };
    auto fetch_a = [&](int step, ARegs &r) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < KS / 16; ks++) {
            r.a[ks] = afrag(step, ks);
            if (LO) r.al[ks] = afrag_lo(step, ks);
        }
    };
    // CUT: lane t % 32 keeps the superblocks per slice of the tile's row t and what is left of the current one
    int cut_len = nsb, cut_left = nsb;
    if (CUT) {
        const int row_tiles = (rows_of[0] + BN - 1) / BN + (rows_of[1] + BN - 1) / BN + (rows_of[2] + BN - 1) / BN;
        cut_len = cut_left = nsb / mm_k_slices(true, row_tiles, nsb, (int)p.cut_as[min(t0 + wm * 32 + lm, p.batch - 1)]);
    }
    ARegs a0, a1;
    fetch_a(0, a0);
    if (!LO) fetch_a(min(1, nsteps - 1), a1);
    __syncthreads();   // stage 0 is written
    auto mul_step = [&](int sb, auto gtag, ARegs &A) __attribute__((always_inline)) {
        constexpr int g = decltype(gtag)::value;
        const int step = 4 * sb + g;
        const _Float16 *Bs = main_stage(step);
        // B operands a k slice ahead: left to itself the compiler reads a slice's operands into the registers the previous
        // slice's products have just released, so every slice begins with an LDS round trip in front of its four matrix
        // instructions.
        h8 b[2][NW_];
#pragma unroll
        for (int nt = 0; nt < NW_; nt++) b[0][nt] = *reinterpret_cast<const h8 *>(&Bs[(nt * 32 + lm) * PITCH + lk]);
#pragma unroll
        for (int ks = 0; ks < KS / 16; ks++) {
            if (ks + 1 < KS / 16) {
#pragma unroll
                for (int nt = 0; nt < NW_; nt++)
                    b[(ks + 1) & 1][nt] = *reinterpret_cast<const h8 *>(&Bs[(nt * 32 + lm) * PITCH + 16 * (ks + 1) + lk]);
            }
            __builtin_amdgcn_sched_barrier(0);   // (the requests stay in front of this slice's products)
#pragma unroll
            for (int nt = 0; nt < NW_; nt++)
                // a superblock's first product starts from the constant zero: no pass over the accumulators to clear them
                Cp[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ROWS ? from_bf16(A.a[ks]) : A.a[ks], b[ks & 1][nt], (g == 0 && ks == 0) ? kZero16 : Cp[nt], 0, 0, 0);
            if (LO) {
#pragma unroll
                for (int nt = 0; nt < NW_; nt++) Cp[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A.al[ks], b[ks & 1][nt], Cp[nt], 0, 0, 0);
            }
            // this k slice's fragments are spent: ask for the ones of AHEAD steps on right away
            A.a[ks] = afrag(min(step + AHEAD, nsteps - 1), ks);
            if (LO) A.al[ks] = afrag_lo(min(step + AHEAD, nsteps - 1), ks);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (g == 3) {
            // ---- end of the superblock: the row scale
            const float *dsc = dsc_stage(sb);
#pragma unroll
            for (int nt = 0; nt < NW_; nt++) {
                const float dn = dsc[nt * 32 + lm];
#pragma unroll
                for (int i = 0; i < 16; i++) F[nt][i] = fmaf(dn, Cp[nt][i], F[nt][i]);
            }
            if (CUT) {
                cut_left -= 1;
                // (rows past the batch never end.  1 / s is a power of two: it can wait for the last slice)
                const bool last = sb + 1 == nsb;
                const bool live = t0 + wm * 32 + lm < p.batch;
                uint32_t ends = (uint32_t)__ballot(live && cut_left == 0), first = (uint32_t)__ballot(sb + 1 == cut_len);
                if (cut_left == 0) cut_left = cut_len;
                if (ends) {
                    // (opaque copies: what follows from them is worked out here, not kept in registers through the loop)
                    const int h4 = 4 * (lane >> 5);
                    int row = t0 + wm * 32 + h4;
                    asm volatile("" : "+v"(row));
                    ends >>= h4;
                    first >>= h4;
#pragma unroll
                    for (int nt = 0; nt < NW_; nt++) {
                        int r = r0 + nt * 32 + lm;
                        asm volatile("" : "+v"(r), "+v"(row));
                        if (r < p.rows) {
                            float *y = p.Y + (size_t)row * ystride + r;
#pragma unroll
                            for (int i0 = 0; i0 < 16; i0 += 8) {
                                float sum[8];
#pragma unroll
                                for (int i = 0; i < 8; i++) {
                                    const int tr = 2 * i0 + 8 * (i / 4) + (i & 3);
                                    sum[i] = 0.f;
                                    if ((ends & ~first) & (1u << tr)) sum[i] = y[(size_t)tr * ystride];
                                }
#pragma unroll
                                for (int i = 0; i < 8; i++) {
                                    const int tr = 2 * i0 + 8 * (i / 4) + (i & 3);
                                    sum[i] += F[nt][i0 + i];
                                    if (last) sum[i] *= p.inv_s[min(row + tr, p.batch - 1)];
                                    if (ends & (1u << tr)) y[(size_t)tr * ystride] = sum[i];
                                }
                            }
                        }
#pragma unroll
                        for (int i = 0; i < 16; i++)
                            if (ends & (1u << (8 * (i / 4) + (i & 3)))) F[nt][i] = 0.f;
                    }
                }
            }
        }
        __syncthreads();
    };
    for (int sb = 0; sb < nsb; sb++) {
        mul_step(sb, std::integral_constant<int, 0>{}, a0);
        mul_step(sb, std::integral_constant<int, 1>{}, LO ? a0 : a1);
        mul_step(sb, std::integral_constant<int, 2>{}, a0);
        mul_step(sb, std::integral_constant<int, 3>{}, LO ? a0 : a1);
    }

    if (CUT) return;   // (the last slices' ends have stored everything)
    // accumulator layout of the 32x32 tile: column = lane % 32, row = 8*(i/4) + 4*(lane/32) + i%4
    auto store = [&](auto keep) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < NW_; nt++) {
            const int r = r0 + nt * 32 + lm;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = t0 + wm * 32 + 8 * (i / 4) + 4 * (lane >> 5) + (i & 3);
                if (t < p.batch && r < p.rows) mm_store<decltype(keep)::value>(&p.Y[(size_t)t * ystride + r], LO ? F[nt][i] * p.inv_s[t] : F[nt][i]);
            }
        }
    };
    if (LO || p.keep) store(std::true_type{});
    else store(std::false_type{});
}

}  // namespace
}  // namespace ksh

#include "q4k_mm_rows.hpp"
#include "q6k_mm_rows.hpp"

namespace ksh {
namespace {

// A wave's request for its 32 rows of a Q4_K superblock, as pieces of 16 bytes, lane after lane along the rows, straight into LDS
// at `dst` ([row][144]).  (A row a lane, an instruction is 64 places of L1 instead of some 20, and that path is what launches of a
// few tokens are busy with.)  `blk`: row 0's superblock; `last`: the last row there is.
constexpr int kRoundTile = 32 * 144 / 4;      // floats
__device__ __forceinline__ void ask_q4k_tile(const uint8_t *blk, uint32_t row_bytes, int last, int lane, uint32_t dst)
{
#pragma unroll
    for (int i = 0; i < 5; i++) {
        const int c = 64 * i + lane, row = c / 9;
        if (i < 4 || lane < 32) to_lds16(blk, (uint32_t)min(row, last) * row_bytes + 16u * (uint32_t)(c % 9), dst + (uint32_t)(i * 1024));
    }
}

// ---- small batches (up to 64 tokens): a GEMV-shaped launch on the matrix cores ---------------------------------
// A prompt remainder or a round of decoding slots is a few dozen tokens: the tiles then leave most of the
// chip idle (rows / 128 workgroups) and half of every tile empty.  Here a workgroup owns 32 weight rows and all
// tokens; its 8 waves split the row's superblocks between them (K-split inside the workgroup, folded through LDS at
// the end, so the sum order is fixed) and every wave reads its weights, from memory or LDS, in the order the matrix
// instruction wants its B operand: lane (n, h) = (lane % 32, lane / 32) owns row n and, in every 16-column slice,
// columns 8h .. 8h+7 -- per 64-column group the low and the high nibbles of bytes 8h .. 8h+7 and 16+8h .. 16+8h+7,
// two 8-byte loads.  Conversion (sc*n as exact f16, biased by 1024), the per-superblock scale and the bias / min
// product are those of the big tile; the activations come as the same fragments, hi and lo part in the same pass
// (each converted weight is used for both), so f32 activations cost one launch.
//
// PIECES: the weights come as pieces of 16 bytes by way of LDS, which costs a second round trip and saves most of the time in L1.
// Measured (us, rows a lane -> pieces, 3045 rows; 500 and 8192 rows are alike):
// up to 32 tokens, one part: 1280 columns 7.0 -> 6.5, 2048 8.3 -> 6.8, 6144 15.3 -> 10.9; where four waves or fewer do everything
// it is even within what runs differ by (512 5.8 -> 5.7 .. 6.1).  Two parts, whose matrix instructions are as many again and hide more
// of L1: where all eight waves have the same number of superblocks (2048 9.8 -> 8.9, 4096 14.9 -> 13.2, 6144 20.1 -> 17.5) and on
// longer rows (3584 13.2 -> 12.9, 5120 17.3 -> 16.8), not between (1280 8.2 -> 8.6, 1792 8.8 -> 8.9, 2304 11.3 -> 12.0, 2560 11.9 ->
// 12.1, 3072 12.3 -> 12.6).
// 33 .. 64 tokens, one part: the same number to every wave (40 tokens: 2048 10.2 -> 9.5, 4096 15.3 -> 13.8, 6144 20.6 -> 18.0), else
// even or slower (512 7.5 -> 8.1, 1280 8.4 -> 8.7, 2304 11.7 -> 12.2, 3584 13.3 -> 13.3, 5120 17.5 -> 17.2).  Two parts of 64 tokens
// have no registers left for it.
constexpr int skinny_wave(int mt, bool pieces) { return pieces && mt == 1 ? kRoundTile : mt * 16 * 64; }      // floats of LDS
struct SkinnyParams {      // (its own: arguments are copied at every launch, and two launches of 3 us are what such a call is)
    const uint8_t *W;
    const _Float16 *Xf, *SxA, *Xf_lo, *SxA_lo;
    float *Y;
    int rows, cols, batch;
    float lo_scale;
};
template <int MT, bool HAS_LO, bool PIECES>
__global__ __launch_bounds__(512) void q4k_mm_skinny_kernel(SkinnyParams p)
{
    extern __shared__ __attribute__((aligned(16))) float red[];   // [8][WAVE]: a wave's weight rows, then its [MT][16][64]
    constexpr int WAVE = skinny_wave(MT, PIECES);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int r0 = blockIdx.x * 32, nsb = p.cols / 256;
    const size_t row_bytes = (size_t)nsb * 144;
    const uint8_t *wrow = p.W + (size_t)min(r0 + n, p.rows - 1) * row_bytes;
    const float *mine = red + wave * WAVE;
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)(red + wave * WAVE);
    const int ntt = (p.batch + 31) / 32;
    const h8 *xa[MT], *xl[MT];
    const _Float16 *sxa[MT], *sxl[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const size_t frag0 = (size_t)min(mt, ntt - 1) * (p.cols / 16) * 64 + lane;
        xa[mt] = reinterpret_cast<const h8 *>(p.Xf) + frag0;
        xl[mt] = reinterpret_cast<const h8 *>(HAS_LO ? p.Xf_lo : p.Xf) + frag0;
        const size_t so = (size_t)min(mt * 32 + n, p.batch - 1) * nsb * 32 + 8 * h;   // + sb * 32 + 16 * ks
        sxa[mt] = p.SxA + so;
        sxl[mt] = (HAS_LO ? p.SxA_lo : p.SxA) + so;
    }
    f16v F[MT], Fl[MT];
    const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < MT; mt++) { F[mt] = kZero16; Fl[mt] = kZero16; }

    for (int sb = wave; sb < nsb; sb += 8) {
        if constexpr (PIECES) {
            ask_q4k_tile(p.W + (size_t)r0 * row_bytes + (size_t)sb * 144, (uint32_t)row_bytes, p.rows - 1 - r0, lane, l0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        const uint8_t *blk = PIECES ? reinterpret_cast<const uint8_t *>(mine) + 144 * n : wrow + (size_t)sb * 144;
        const u32x4_t hdr = *reinterpret_cast<const u32x4_t *>(blk);
        u32x2_t q[4][2];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            q[g][0] = *reinterpret_cast<const u32x2_t *>(blk + 16 + 32 * g + 8 * h);
            q[g][1] = *reinterpret_cast<const u32x2_t *>(blk + 16 + 32 * g + 16 + 8 * h);
        }
        if constexpr (PIECES) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the next superblock's rows come to the same place)
        f16v C[MT], Cl[MT];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            // this group's activation fragments: slices 4g .. 4g+3 of the superblock
            h8 a[MT][4], al[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const size_t o = (size_t)(sb * 16 + 4 * g + j) * 64;
                    a[mt][j] = xa[mt][o];
                    if (HAS_LO) al[mt][j] = xl[mt][o];
                }
            const uint4 s = q4k_group_scales(hdr.y, hdr.z, hdr.w, g);   // sc_lo, mn_lo, sc_hi, mn_hi
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // slice j: bytes (j & 1 ? 16 + 8h : 8h) .. +7, low nibbles for j < 2, high nibbles after
                const u32x2_t qq = q[g][j & 1];
                const uint32_t sc = j < 2 ? s.x : s.z;
                uint32_t o[4];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t d = j < 2 ? qq[i] : qq[i] >> 4;
                    o[2 * i] = pair_f16(d & 0x000F000Fu, sc);
                    o[2 * i + 1] = pair_f16((d >> 8) & 0x000F000Fu, sc);
                }
                const u32x4_t ov = {o[0], o[1], o[2], o[3]};
                const h8 b = __builtin_bit_cast(h8, ov);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    C[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][j], b, (g == 0 && j == 0) ? kZero16 : C[mt], 0, 0, 0);
                    if (HAS_LO) Cl[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[mt][j], b, (g == 0 && j == 0) ? kZero16 : Cl[mt], 0, 0, 0);
                }
            }
        }
        // bias + mins of the superblock: the row's eight coefficients -(dmin*m_j + 1024*d) as f16 hi | lo, against the
        // tokens' sums of x (hi[8] hi[8] lo[8] 0[8] per token and superblock): hi*hi + hi*lo + lo*hi
        const float d = half_bits_to_f32(hdr.x & 0xFFFFu), dmin = half_bits_to_f32(hdr.x >> 16);
        _Float16 chi[8], clo[8];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint4 s = q4k_group_scales(hdr.y, hdr.z, hdr.w, g);
            const float c0 = pinned(-(dmin * (float)s.y + 1024.f * d)), c1 = pinned(-(dmin * (float)s.w + 1024.f * d));
            chi[2 * g] = (_Float16)c0; chi[2 * g + 1] = (_Float16)c1;
            clo[2 * g] = (_Float16)(c0 - (float)chi[2 * g]); clo[2 * g + 1] = (_Float16)(c1 - (float)chi[2 * g + 1]);
        }
        h8 b2[2];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            b2[0][i] = h ? clo[i] : chi[i];                 // columns 0..7: hi, 8..15: lo
            b2[1][i] = h ? (_Float16)0.f : chi[i];          // columns 16..23: hi, 24..31: zero
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const h8 a2 = *reinterpret_cast<const h8 *>(sxa[mt] + (size_t)sb * 32 + 16 * ks);
                F[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, b2[ks], F[mt], 0, 0, 0);
                if (HAS_LO) {
                    const h8 a2l = *reinterpret_cast<const h8 *>(sxl[mt] + (size_t)sb * 32 + 16 * ks);
                    Fl[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2l, b2[ks], Fl[mt], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 16; i++) {
                F[mt][i] = fmaf(d, C[mt][i], F[mt][i]);
                if (HAS_LO) Fl[mt][i] = fmaf(d, Cl[mt][i], Fl[mt][i]);
            }
        }
    }
    // fold the eight waves' shares (fixed order), then store: accumulator i of lane (n, h) is token
    // 8*(i/4) + 4*h + i%4 of the tile, weight row n
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            red[wave * WAVE + (mt * 16 + i) * 64 + lane] = HAS_LO ? fmaf(p.lo_scale, Fl[mt][i], F[mt][i]) : F[mt][i];
    __syncthreads();
    for (int o = tid; o < MT * 16 * 64; o += 512) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < 8; w++) sum += red[w * WAVE + o];
        const int mt = o / (16 * 64), i = (o / 64) & 15, l = o & 63;
        const int t = mt * 32 + 8 * (i / 4) + 4 * (l >> 5) + (i & 3), r = r0 + (l & 31);
        if (t < p.batch && r < p.rows) p.Y[(size_t)t * p.rows + r] = sum;
    }
}

// ---- decode rounds (up to 16 tokens) --------------------------------------------------------------------------
// A round of decoding slots is at most 16 rows, and several GEMMs read the same rows (q | k | v, gate | up).  Two
// kinds serve it (neither has a counterpart in the reference, whose round is one decode step per request):
//   KSH_ROUND_PREP    x f32[batch, cols] -> a prepared operand: the fragments of the 32 x 32 x 16 matrix instruction
//                     with x = hi + 2^-11 lo in ONE tile -- rows 0..15 the tokens' hi parts, rows 16..31 their lo
//                     parts -- so that one instruction per weight slice serves both parts, and the sums of x per
//                     sub-block for the bias / min product, hi and lo.  Written once per distinct input.
//   KSH_MATVEC_ROUND  up to three Q4_K matrices of the same width against one prepared operand in one launch, or a
//                     gate | up pair whose workgroups hold the same 32 rows of both and store gelu(gate) * up.
// A workgroup owns 32 weight rows of one matrix and 8 superblocks of columns, one per wave: every load of the
// workgroup (80 bytes of weights and 288 of activations per lane) goes out before anything is used, so the launch is
// one memory round trip where the small-batch form above walks a wave's superblocks one round trip at a time.  Rows
// longer than 2048 columns split over blockIdx.y; the slices' sums go to a scratch buffer and a second launch adds
// them in a fixed order.  Conversion, scales and the bias / min product are those of the forms above.

// what one thread does with 8 consecutive elements (8 j .. 8 j + 7) of token row t; whole quads call it together
// (the four threads of a sub-block add their sums up over the quad)
__device__ __forceinline__ void round_prep_write(const float (&f)[8], int t, int j, int cols, _Float16 *__restrict__ Xp)
{
    h8 oh, ol;
    float sh, sl;
    round_split8(f, oh, ol, sh, sl);
    sh += dpp_f32<0xB1>(sh);
    sh += dpp_f32<0x4E>(sh);
    sl += dpp_f32<0xB1>(sl);
    sl += dpp_f32<0x4E>(sl);
    // fragment of 16 columns: lane = row + 32 * ((k / 8) % 2); row t is the token's hi part, row 16 + t its lo part
    const size_t frag = (size_t)(j >> 1) * 64 + t + 32 * (j & 1);
    reinterpret_cast<h8 *>(Xp)[frag] = oh;
    reinterpret_cast<h8 *>(Xp)[frag + 16] = ol;
    if ((threadIdx.x & 3) == 0) round_store_sums(Xp, cols, t, j / 4, sh, sl);
}

// one thread per 8 elements of the 16 token rows (rows past the batch are written as zeros)
__global__ __launch_bounds__(256) void mm_round_prep_kernel(const float *__restrict__ X, _Float16 *__restrict__ Xp, int batch, int cols)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int k8 = cols / 8;
    if (idx >= kRoundTokens * k8) return;   // (whole quads: cols is a multiple of 32)
    const int t = idx / k8, j = idx - t * k8;
    f32x4_t in0 = {0.f, 0.f, 0.f, 0.f}, in1 = in0;
    if (t < batch) {
        in0 = reinterpret_cast<const f32x4_t *>(X)[2 * ((size_t)t * k8 + j)];
        in1 = reinterpret_cast<const f32x4_t *>(X)[2 * ((size_t)t * k8 + j) + 1];
    }
    const float f[8] = {in0.x, in0.y, in0.z, in0.w, in1.x, in1.y, in1.z, in1.w};
    round_prep_write(f, t, j, cols, Xp);
}

// The rows forms of the norms (rmsnorm_rows, rmsnorm_add_then_rmsnorm rows: crates/ksearch_kernels/src/lib.rs:1478-1560)
// with the prepared operand as their output: one workgroup per token row, the same sums in the same order as the
// kernels that write f32 rows (explicitly rounded products and sums: nothing is contracted).
//   MODE 1:  v = (x * inv) * w                                                     -> xp
//   MODE 2:  x_new = [scale *] (res + (y * inv) * w_post);  v = (x_new * inv2) * w_norm   -> xp, x_new (may be res)
//   MODE 3:  x_new = res + (y * inv) * w_post;  v = x_new                          -> xp, x_new (may be res)
__device__ __forceinline__ float round_block_sum(float v, float *red)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();                       // (red may still be read from the previous sum)
    if (lane == 0) red[wave] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

template <int MODE>
__global__ __launch_bounds__(256) void mm_round_prep_norm_kernel(const float *__restrict__ x, const float *__restrict__ w_first, const float *res,
                                                                 const float *__restrict__ w_norm, float *x_new, _Float16 *__restrict__ Xp,
                                                                 int batch, int cols, float eps, float scale)
{
    __shared__ float red[4];
    extern __shared__ float mid[];      // MODE 2: the row between the two norms
    const int t = blockIdx.x, k8 = cols / 8;
    if (t >= batch) {
        const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int j = threadIdx.x; j < k8; j += 256) round_prep_write(zero, t, j, cols, Xp);
        return;
    }
    x += (size_t)t * cols;
    float ss = 0.f;
    for (int i = threadIdx.x; i < cols; i += 256) ss = __fadd_rn(ss, __fmul_rn(x[i], x[i]));
    ss = round_block_sum(ss, red);
    float inv = 1.0f / sqrtf(__fadd_rn(ss / (float)cols, eps));
    if (MODE >= 2) {
        res += (size_t)t * cols;
        x_new += (size_t)t * cols;
        float ss2 = 0.f;
        for (int i = threadIdx.x; i < cols; i += 256) {
            float v = __fadd_rn(__fmul_rn(__fmul_rn(x[i], inv), w_first[i]), res[i]);
            if (scale != 0.f) v = __fmul_rn(scale, v);
            mid[i] = v;
            x_new[i] = v;
            ss2 = __fadd_rn(ss2, __fmul_rn(v, v));
        }
        if (MODE == 2) {
            ss2 = round_block_sum(ss2, red);
            inv = 1.0f / sqrtf(__fadd_rn(ss2 / (float)cols, eps));
        } else {
            __syncthreads();   // the row is read across threads below
        }
    }
    const float *src = MODE >= 2 ? mid : x, *w = MODE == 2 ? w_norm : w_first;
    for (int j = threadIdx.x; j < k8; j += 256) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = MODE == 3 ? src[8 * j + i] : pinned(__fmul_rn(__fmul_rn(src[8 * j + i], inv), w[8 * j + i]));
        round_prep_write(f, t, j, cols, Xp);
    }
}

// The same for rows of up to 2048 columns (the widths of the models this serves): thread j owns elements 8 j .. 8 j + 7
// from the first load to the fragment it writes, every input is requested up front, and the row never passes through
// LDS -- the launch is one round trip and two block sums where the form above is three dependent passes.  (The sums
// of squares are taken in a different order than the kernels that write f32 rows: equal to the last bit or two.)
template <int MODE>
__global__ __launch_bounds__(256) void mm_round_prep_norm8_kernel(const float *__restrict__ x, const float *__restrict__ w_first, const float *res,
                                                                  const float *__restrict__ w_norm, float *x_new, _Float16 *__restrict__ Xp,
                                                                  int batch, int cols, float eps, float scale, int slices)
{
    __shared__ float red[4];
    const int t = blockIdx.x, k8 = cols / 8, j = threadIdx.x;
    const bool has = j < k8;                  // (whole quads: cols is a multiple of 32)
    if (t >= batch) {
        const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (has) round_prep_write(zero, t, j, cols, Xp);
        return;
    }
    const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
    const size_t e = (size_t)t * cols + 8 * (size_t)min(j, k8 - 1), ew = 8 * (size_t)min(j, k8 - 1);
    auto ld8 = [&](const float *p, size_t off, float (&o)[8]) {
        const f32x4_t a = has ? *reinterpret_cast<const f32x4_t *>(p + off) : z4, b = has ? *reinterpret_cast<const f32x4_t *>(p + off + 4) : z4;
        o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
    };
    float y[8], w1[8], r[8], w2[8];
    ld8(x, e, y);
    // x as the column slices' partial sums of a split GEMM ([slices][batch][cols]): added here, slice after slice, in
    // the order the GEMM's own second launch adds them
    for (int sl = 1; sl < slices; sl++) {
        float ys[8];
        ld8(x, (size_t)sl * batch * cols + e, ys);
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = __fadd_rn(y[i], ys[i]);
    }
    ld8(w_first, ew, w1);
    if (MODE >= 2) ld8(res, e, r);
    if (MODE == 2) ld8(w_norm, ew, w2);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) ss = __fadd_rn(ss, __fmul_rn(y[i], y[i]));
    ss = round_block_sum(ss, red);
    float inv = 1.0f / sqrtf(__fadd_rn(ss / (float)cols, eps));
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = __fmul_rn(__fmul_rn(y[i], inv), w1[i]);
    if (MODE >= 2) {
        float ss2 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            f[i] = __fadd_rn(f[i], r[i]);
            if (scale != 0.f) f[i] = __fmul_rn(scale, f[i]);
            ss2 = __fadd_rn(ss2, __fmul_rn(f[i], f[i]));
        }
        if (has) {
            *reinterpret_cast<f32x4_t *>(x_new + e) = f32x4_t{f[0], f[1], f[2], f[3]};
            *reinterpret_cast<f32x4_t *>(x_new + e + 4) = f32x4_t{f[4], f[5], f[6], f[7]};
        }
        if (MODE == 2) {
            ss2 = round_block_sum(ss2, red);
            inv = 1.0f / sqrtf(__fadd_rn(ss2 / (float)cols, eps));
#pragma unroll
            for (int i = 0; i < 8; i++) f[i] = __fmul_rn(__fmul_rn(f[i], inv), w2[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = pinned(f[i]);
    if (has) round_prep_write(f, t, j, cols, Xp);
}

struct RoundParams {
    const uint8_t *W0, *W1, *W2;
    float *Y0, *Y1, *Y2;
    int rows0, rows1, rows2, tiles0, tiles1;
    int cols, batch;
    const _Float16 *Xp;
    float *part;                 // [slices][batch][rows0] when the columns are split
    const float *mul;            // NM = 1: y = gelu(W0 x) * mul[t * mul_stride + r] (the per-layer-embedding gate)
    int mul_stride;
    _Float16 *emit;              // not null: the result goes out as the prepared operand of the next GEMM (rows0 columns)
};

// NM = 2: the gate | up pair (W0, W1 of rows0 rows each; gelu(W0 x) * (W1 x) to Y0)
// PIECES: the weights come as pieces of 16 bytes, lane after lane along the rows, straight into LDS.  (A row a lane, an instruction is
// 64 places of L1 instead of some 20, and L1's path was the busy unit; read back matrix by matrix they also leave registers for a
// second workgroup on the compute unit.  16 rows: gate | up of 12288 x 1536 17.1 -> 14.3 us, 1536 x 12288 11.9 -> 9.7, 1536 x 2048
// 5.6 -> 4.9.)  Else a row a lane, which saves the way through LDS where that path is not busy (round_pieces).
template <int NM, bool PIECES>
__global__ __launch_bounds__(512, PIECES ? 4 : 2) void q4k_mm_round_kernel(RoundParams p)
{
    // a wave's weight rows per matrix, and over them its shares of the results, [8][64]: kRoundTile floats each
    extern __shared__ __attribute__((aligned(16))) float red[];   // [8][NM][kRoundTile]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    // the workgroup's matrix: a choice between arguments already fetched, not an indexed read of them
    int tile = blockIdx.x;
    const bool in1 = NM == 1 && tile >= p.tiles0, in2 = in1 && tile - p.tiles0 >= p.tiles1;
    if (in1) tile -= p.tiles0;
    if (in2) tile -= p.tiles1;
    const uint8_t *W = in2 ? p.W2 : in1 ? p.W1 : p.W0;
    float *Y = in2 ? p.Y2 : in1 ? p.Y1 : p.Y0;
    const int rows = in2 ? p.rows2 : in1 ? p.rows1 : p.rows0;
    const int r0 = tile * 32, nsb = p.cols / 256;
    const int sb = blockIdx.y * 8 + wave;
    const bool active = sb < nsb;                        // (wave-uniform: a row of 1536 columns leaves two waves idle)
    const int sbc = min(sb, nsb - 1);

    // (the other waves ask for nothing: a quarter of the requests were for a row's last superblock again, and the vector-memory
    // path is what the launch is busy with -- gate | up of 12288 x 1536 for 16 rows 18.8 -> 16.8 us)
    if (active) {
        // ---- every load of the wave, up front
        float *mine = red + wave * NM * kRoundTile;
        const int last = rows - 1 - r0;
        const uint32_t row_bytes = (uint32_t)nsb * 144u;
        u32x4_t hdr[NM];
        u32x2_t q[NM][4][2];
        auto take = [&](int m, const uint8_t *blk) __attribute__((always_inline)) {
            hdr[m] = *reinterpret_cast<const u32x4_t *>(blk);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                q[m][g][0] = *reinterpret_cast<const u32x2_t *>(blk + 16 + 32 * g + 8 * h);
                q[m][g][1] = *reinterpret_cast<const u32x2_t *>(blk + 16 + 32 * g + 16 + 8 * h);
            }
        };
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const uint8_t *blk = (m ? p.W1 : W) + (size_t)r0 * row_bytes + (size_t)sbc * 144;
            if constexpr (PIECES) ask_q4k_tile(blk, row_bytes, last, lane, (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)mine + (uint32_t)(m * kRoundTile * 4));
            else take(m, blk + (size_t)min(n, last) * row_bytes);
        }
        const h8 *xa = reinterpret_cast<const h8 *>(p.Xp) + (size_t)sbc * 16 * 64 + lane;
        h8 a[16];
#pragma unroll
        for (int j = 0; j < 16; j++) a[j] = xa[(size_t)j * 64];
        // sums of x: rows 0..15 the tokens' hi parts, rows 16..31 their lo parts
        const _Float16 *sx = p.Xp + round_xf_halves(p.cols) + (n >= 16 ? round_sx_halves(p.cols) : 0) + ((size_t)(n & 15) * nsb + sbc) * 32 + 8 * h;
        const h8 a2[2] = {*reinterpret_cast<const h8 *>(sx), *reinterpret_cast<const h8 *>(sx + 16)};
        if constexpr (PIECES) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

        const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; m++) {
            if constexpr (PIECES) take(m, reinterpret_cast<const uint8_t *>(mine + m * kRoundTile) + 144 * n);
            f16v C = kZero16;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint4 s = q4k_group_scales(hdr[m].y, hdr[m].z, hdr[m].w, g);   // sc_lo, mn_lo, sc_hi, mn_hi
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    // slice j: bytes (j & 1 ? 16 + 8h : 8h) .. +7, low nibbles for j < 2, high nibbles after
                    const u32x2_t qq = q[m][g][j & 1];
                    const uint32_t sc = j < 2 ? s.x : s.z;
                    uint32_t o[4];
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const uint32_t d = j < 2 ? qq[i] : qq[i] >> 4;
                        o[2 * i] = pair_f16(d & 0x000F000Fu, sc);
                        o[2 * i + 1] = pair_f16((d >> 8) & 0x000F000Fu, sc);
                    }
                    const u32x4_t ov = {o[0], o[1], o[2], o[3]};
                    C = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[4 * g + j], __builtin_bit_cast(h8, ov), C, 0, 0, 0);
                }
            }
            // bias + mins of the superblock: the row's eight coefficients -(dmin*m_j + 1024*d) as f16 hi | lo, against the
            // sums of x (hi[8] hi[8] lo[8] 0[8] per row and superblock): hi*hi + hi*lo + lo*hi
            const float d = half_bits_to_f32(hdr[m].x & 0xFFFFu), dmin = half_bits_to_f32(hdr[m].x >> 16);
            _Float16 chi[8], clo[8];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint4 s = q4k_group_scales(hdr[m].y, hdr[m].z, hdr[m].w, g);
                const float c0 = pinned(-(dmin * (float)s.y + 1024.f * d)), c1 = pinned(-(dmin * (float)s.w + 1024.f * d));
                chi[2 * g] = (_Float16)c0; chi[2 * g + 1] = (_Float16)c1;
                clo[2 * g] = (_Float16)(c0 - (float)chi[2 * g]); clo[2 * g + 1] = (_Float16)(c1 - (float)chi[2 * g + 1]);
            }
            h8 b2[2];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                b2[0][i] = h ? clo[i] : chi[i];                 // columns 0..7: hi, 8..15: lo
                b2[1][i] = h ? (_Float16)0.f : chi[i];          // columns 16..23: hi, 24..31: zero
            }
            f16v F = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2[0], b2[0], kZero16, 0, 0, 0);
            F = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2[1], b2[1], F, 0, 0, 0);
            // accumulator i of lane (n, h) is row 8*(i/4) + 4*h + i%4 of the tile: i < 8 a token's hi part, i + 8 its lo part
#pragma unroll
            for (int i = 0; i < 8; i++)
                mine[m * kRoundTile + i * 64 + lane] = fmaf(1.0f / 2048.0f, fmaf(d, C[i + 8], F[i + 8]), fmaf(d, C[i], F[i]));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8 * NM; i++) red[(wave * NM + i / 8) * kRoundTile + (i & 7) * 64 + lane] = 0.f;
    }
    __syncthreads();
    // one output per thread: the eight waves' shares in a fixed order
    const int i = tid >> 6, t = 8 * (i >> 2) + 4 * h + (i & 3), r = r0 + n;
    float v[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        v[m] = 0.f;
#pragma unroll
        for (int w = 0; w < 8; w++) v[m] += red[(w * NM + m) * kRoundTile + i * 64 + lane];
    }
    const bool in = t < p.batch && r < rows;
    float y = NM == 2 ? gelu_mul_f32(v[0], v[NM - 1]) : v[0];
    if (NM == 1 && p.mul) y = gelu_mul_f32(y, p.mul[(size_t)min(t, p.batch - 1) * p.mul_stride + min(r, rows - 1)]);
    if (!p.emit) {
        if (in) {
            if (gridDim.y == 1) Y[(size_t)t * rows + r] = y;
            else p.part[((size_t)blockIdx.y * p.batch + t) * rows + r] = y;
        }
        return;
    }
    // The tile's 16 x 32 results are 32 columns of the next GEMM's input: two fragments' worth of every token row and
    // exactly one sub-block of sums, so the workgroup writes its share of the prepared operand itself (rows0 is a
    // multiple of 256 and the columns are not split: host-checked).  Rows past the batch are written as zeros.
    float *T = red + 8 * NM * kRoundTile;         // [16][33]
    T[t * 33 + n] = in ? y : 0.f;
    __syncthreads();
    if (tid < 64) {
        const int tt = tid & 15, ks = (tid >> 4) & 1, kh = tid >> 5;
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = T[tt * 33 + 16 * ks + 8 * kh + e];
        h8 oh, ol;
        float sh, sl;
        round_split8(f, oh, ol, sh, sl);
        const size_t frag = (size_t)(r0 / 16 + ks) * 64 + tt + 32 * kh;
        reinterpret_cast<h8 *>(p.emit)[frag] = oh;
        reinterpret_cast<h8 *>(p.emit)[frag + 16] = ol;
    } else if (tid < 80) {
        const int tt = tid - 64;
        float sh4[4], sl4[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; e++) f[e] = T[tt * 33 + 8 * g + e];
            h8 oh, ol;
            round_split8(f, oh, ol, sh4[g], sl4[g]);
        }
        round_store_sums(p.emit, rows, tt, r0 / 32, (sh4[0] + sh4[1]) + (sh4[2] + sh4[3]), (sl4[0] + sl4[1]) + (sl4[2] + sl4[3]));
    }
}

// y[i] = the slices' partial sums of element i, slice after slice
__global__ __launch_bounds__(256) void mm_round_fold_kernel(const float *__restrict__ part, float *__restrict__ y, int n, int slices)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float s = part[i];
    for (int k = 1; k < slices; k++) s += part[(size_t)k * n + i];
    y[i] = s;
}

// y[i] = the K slices' partial sums of element i, slice after slice; the slices of the low parts of f32 activations
// (parts = 2) come in scaled.  The partial sums hold the columns of up to three matrices side by side (rows0 | rows1 |
// rows2 per token), each with a result buffer of its own.
__global__ __launch_bounds__(256) void mm_parts_fold_kernel(const float *__restrict__ part, float *__restrict__ y0, float *__restrict__ y1, float *__restrict__ y2,
                                                             int batch, int rows0, int rows1, int rows2, int slices)
{
    const int rows_all = rows0 + rows1 + rows2, n = batch * rows_all;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    // (eight slices in flight: one at a time, 29 slices of 8 x 517 took 8 us)
    float s = part[i];
    for (int k0 = 1; k0 < slices; k0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = part[(size_t)min(k0 + u, slices - 1) * n + i];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + u < slices) s += v[u];
    }
    if (!rows1) { y0[i] = s; return; }
    const int t = i / rows_all, c = i - t * rows_all;
    if (c < rows0) y0[(size_t)t * rows0 + c] = s;
    else if (c < rows0 + rows1) y1[(size_t)t * rows1 + c - rows0] = s;
    else y2[(size_t)t * rows2 + c - rows0 - rows1] = s;
}

// The same round against a Q6_K matrix with row-grouped fields (KSH_Q6K_ROWS: the LM head as the decode loops keep it;
// rows of up to 2048 columns).  The B operand is the 6-bit code minus 32 as an exact f16 integer (the code OR-ed into
// the mantissa of 1024.0, minus 1056 with one packed subtraction per two weights); Q6_K has one int8 scale per 16
// columns, which is the K depth of the matrix instruction, so the scale is applied in f32 to the instruction's
// result: nothing is rounded (folded into the f16 operand as the tile of two roles does it, sc * q above 2048 loses
// its last bit).  A workgroup keeps the activations of the whole row in registers -- wave w the 16 fragments of
// superblock w -- and walks tiles of 32 weight rows, the next tile's bytes in flight under the current one; the waves'
// shares of a tile meet in LDS (two buffers, one barrier per tile).
constexpr int kQ6rRowAlign = 16;
__host__ __device__ inline size_t round_q6r_row_bytes(int bpr) { return ((size_t)bpr * 210 + kQ6rRowAlign - 1) / kQ6rRowAlign * kQ6rRowAlign; }

struct Round6Params {
    const uint8_t *W;
    float *Y;
    int rows, cols, batch, tiles, tiles_per_wg;
    const _Float16 *Xp;
};

struct Q6Tile {
    u32x2_t ql[2][2][2];   // [half][quadrant parity][low / high 16 positions]: bytes 8h .. 8h+7 of them
    u32x2_t qh[2][2];      // [half][low / high 16 positions]
    u32x4_t sc;            // the superblock's 16 int8 scales
    uint32_t d;
};

__global__ __launch_bounds__(512) void q6r_mm_round_kernel(Round6Params p)
{
    extern __shared__ __attribute__((aligned(16))) float red[];   // [2][8 waves][8][64]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int bpr = p.cols / 256;
    const bool active = wave < bpr;                       // (wave-uniform: a row of 1536 columns leaves two waves idle)
    const int sbc = min(wave, bpr - 1);
    const size_t row_bytes = round_q6r_row_bytes(bpr);
    const h8 *xa = reinterpret_cast<const h8 *>(p.Xp) + (size_t)sbc * 16 * 64 + lane;
    h8 a[16];
#pragma unroll
    for (int j = 0; j < 16; j++) a[j] = xa[(size_t)j * 64];
    auto load_tile = [&](Q6Tile &dst, int tile) {
        const uint8_t *rp = p.W + (size_t)min(tile * 32 + n, p.rows - 1) * row_bytes;
#pragma unroll
        for (int ip = 0; ip < 2; ip++)
#pragma unroll
            for (int lh = 0; lh < 2; lh++) {
#pragma unroll
                for (int par = 0; par < 2; par++)
                    dst.ql[ip][par][lh] = *reinterpret_cast<const u32x2_t *>(rp + (size_t)sbc * 128 + 64 * ip + 32 * par + 16 * lh + 8 * h);
                dst.qh[ip][lh] = *reinterpret_cast<const u32x2_t *>(rp + (size_t)bpr * 128 + (size_t)sbc * 64 + 32 * ip + 16 * lh + 8 * h);
            }
        dst.sc = *reinterpret_cast<const u32x4_t *>(rp + (size_t)bpr * 192 + (size_t)sbc * 16);
        dst.d = *reinterpret_cast<const uint16_t *>(rp + (size_t)bpr * 208 + (size_t)sbc * 2);
    };
    const int tile0 = blockIdx.x * p.tiles_per_wg, tile1 = min(tile0 + p.tiles_per_wg, p.tiles);
    if (tile0 >= tile1) return;
    uint32_t byte_mask = 0x00FF00FFu, bias = 0x64006400u;   // in registers: the and-or is then one instruction
    asm volatile("" : "+v"(byte_mask), "+v"(bias));
    const h8 k1056 = {(_Float16)1056.f, (_Float16)1056.f, (_Float16)1056.f, (_Float16)1056.f,
                      (_Float16)1056.f, (_Float16)1056.f, (_Float16)1056.f, (_Float16)1056.f};
    const f16v kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    Q6Tile cur, nxt;
    load_tile(cur, tile0);
    int buf = 0;
    for (int tile = tile0; tile < tile1; tile++) {
        load_tile(nxt, min(tile + 1, tile1 - 1));
        f16v G = kZero16;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            // group j: half ip, quadrant q, positions 16 lh .. +15; element 16 j of the superblock onwards
            const int ip = j >> 3, q = (j >> 1) & 3, lh = j & 1;
            const u32x2_t ql2 = cur.ql[ip][q & 1][lh], qh2 = cur.qh[ip][lh];
            uint32_t o[4];
#pragma unroll
            for (int dw = 0; dw < 2; dw++) {
                const uint32_t lo4 = (ql2[dw] >> (4 * (q >> 1))) & 0x0F0F0F0Fu, hi2 = (qh2[dw] >> (2 * q)) & 0x03030303u;
                const uint32_t code = lo4 | (hi2 << 4);
                o[2 * dw] = (code & byte_mask) | bias;              // codes of bytes 0 and 2 as 1024 + c
                o[2 * dw + 1] = ((code >> 8) & byte_mask) | bias;   // bytes 1 and 3: the order the fragments keep
            }
            const u32x4_t ov = {o[0], o[1], o[2], o[3]};
            const h8 b = __builtin_bit_cast(h8, ov) - k1056;
            const f16v C = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[j], b, kZero16, 0, 0, 0);
            const float sc = (float)(int)(int8_t)(cur.sc[j >> 2] >> (8 * (j & 3)));
#pragma unroll
            for (int i = 0; i < 16; i++) G[i] = fmaf(sc, C[i], G[i]);
        }
        // accumulator i of lane (n, h) is row 8*(i/4) + 4*h + i%4 of the tile: i < 8 a token's hi part, i + 8 its lo part
        const float d = active ? half_bits_to_f32(cur.d) : 0.f;
        float *mine = red + (size_t)(buf * 8 + wave) * 8 * 64 + lane;
#pragma unroll
        for (int i = 0; i < 8; i++) mine[i * 64] = d * fmaf(1.0f / 2048.0f, G[i + 8], G[i]);
        __syncthreads();
        {
            const int i = wave, t = 8 * (i >> 2) + 4 * h + (i & 3), r = tile * 32 + n;
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < 8; w++) sum += red[(size_t)((buf * 8 + w) * 8 + i) * 64 + lane];
            if (t < p.batch && r < p.rows) p.Y[(size_t)t * p.rows + r] = sum;
        }
        buf ^= 1;
        cur = nxt;
    }
}

int launch_round_prep(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    const int cols = (int)k.desc.dims[0], batch = (int)k.desc.dims[1], mode = (int)k.desc.dims[2];
    const int n = kRoundTokens * (cols / 8);
    const float *in1 = mode ? (const float *)a.in[1] : nullptr, *in2 = mode >= 2 ? (const float *)a.in[2] : nullptr,
                *in3 = mode == 2 ? (const float *)a.in[3] : nullptr;
    float *x_new = mode >= 2 ? (float *)a.out[1] : nullptr;
    const float scale = mode == 2 ? k.desc.params[1] : 0.f;
    const int slices = (int)std::max<int64_t>(1, k.desc.dims[3]);
#define KSH_PN(KERNEL, M, LDS) \
    hipLaunchKernelGGL(KERNEL<M>, dim3(kRoundTokens), dim3(256), LDS, st, (const float *)a.in[0], in1, in2, in3, x_new, (_Float16 *)a.out[0], batch, cols, \
                       k.desc.params[0], scale)
#define KSH_PN8(M) \
    hipLaunchKernelGGL(mm_round_prep_norm8_kernel<M>, dim3(kRoundTokens), dim3(256), 0, st, (const float *)a.in[0], in1, in2, in3, x_new, \
                       (_Float16 *)a.out[0], batch, cols, k.desc.params[0], scale, slices)
    if (mode && cols <= 2048) {
        if (mode == 1) KSH_PN8(1);
        else if (mode == 2) KSH_PN8(2);
        else KSH_PN8(3);
    } else if (mode == 1) {
        KSH_PN(mm_round_prep_norm_kernel, 1, 0);
    } else if (mode == 2) {
        KSH_PN(mm_round_prep_norm_kernel, 2, (size_t)cols * 4);
    } else if (mode == 3) {
        KSH_PN(mm_round_prep_norm_kernel, 3, (size_t)cols * 4);
    }
#undef KSH_PN
#undef KSH_PN8
    else
        hipLaunchKernelGGL(mm_round_prep_kernel, dim3((n + 255) / 256), dim3(256), 0, st, (const float *)a.in[0], (_Float16 *)a.out[0], batch, cols);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "round_prep launch");
}

// The weights by pieces, or a row a lane: where all eight waves work, or two workgroups share a compute unit, the path of L1 is
// busy; else the way through LDS is what counts.  16 rows, us, a row a lane | pieces: 1536 x 256 3.00 | 3.27, 4096 x 1024 3.65 | 4.00,
// 2048 x 1536 with two of 256 rows 4.34 | 4.54, 8192 x 1792 5.37 | 5.58, 12288 x 768 4.92 | 5.20; 8448 x 1024 5.44 | 5.36, 8448 x
// 1536 7.54 | 7.05, 256 x 2048 5.43 | 4.58, 8192 x 2048 6.53 | 5.82; gate | up 1024 x 256 3.67 | 4.08, 3072 x 768 4.33 | 4.46, 6144 x
// 1536 even, 9000 x 512 6.32 | 5.82.
bool round_pieces(bool pair, int nsb, int tiles) { return pair ? nsb >= 6 || tiles > 256 : nsb >= 8 || (nsb >= 4 && tiles > 256); }

int launch_matvec_round(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    const int64_t *d = k.desc.dims;
    if (k.desc.dtypes[0] == KSH_Q6K_ROWS) {
        Round6Params p6{};
        p6.W = (const uint8_t *)a.in[0];
        p6.Xp = (const _Float16 *)a.in[1];
        p6.Y = (float *)a.out[0];
        p6.rows = (int)d[0]; p6.cols = (int)d[1]; p6.batch = (int)d[2];
        p6.tiles = (p6.rows + 31) / 32;
        p6.tiles_per_wg = (p6.tiles + (int)k.info.grid[0] - 1) / (int)k.info.grid[0];
        hipLaunchKernelGGL(q6r_mm_round_kernel, dim3(k.info.grid[0]), dim3(512), k.info.lds_bytes, st, p6);
        const hipError_t e6 = hipGetLastError();
        return e6 == hipSuccess ? 0 : hip_fail(e6, "matvec_round (Q6_K rows) launch");
    }
    const bool pair = d[5] != 0;
    const int n_mat = pair ? 2 : d[4] ? 3 : d[3] ? 2 : 1;
    RoundParams p{};
    p.W0 = (const uint8_t *)a.in[0];
    p.Xp = (const _Float16 *)a.in[1];
    p.W1 = n_mat > 1 ? (const uint8_t *)a.in[2] : p.W0;
    p.W2 = n_mat > 2 ? (const uint8_t *)a.in[3] : p.W0;
    p.Y0 = (float *)a.out[0];
    p.Y1 = (!pair && n_mat > 1) ? (float *)a.out[1] : p.Y0;
    p.Y2 = n_mat > 2 ? (float *)a.out[2] : p.Y0;
    p.rows0 = (int)d[0]; p.rows1 = pair ? (int)d[0] : (int)d[3]; p.rows2 = (int)d[4];
    p.tiles0 = (p.rows0 + 31) / 32; p.tiles1 = pair ? 0 : (p.rows1 + 31) / 32;
    p.cols = (int)d[1]; p.batch = (int)d[2];
    p.part = (float *)k.scratch;
    if (d[7]) { p.mul = (const float *)a.in[2]; p.mul_stride = (int)d[7]; }
    if (d[6] == 1) { p.emit = (_Float16 *)a.out[0]; p.Y0 = p.Y1 = p.Y2 = nullptr; }
    if (d[6] == 2) p.part = (float *)a.out[0];     // the slices' partial sums are the result
    const dim3 grid(k.info.grid[0], k.info.grid[1]);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(512), k.info.lds_bytes, st, p); };
    if (round_pieces(pair, p.cols / 256, (int)grid.x)) pair ? launch(q4k_mm_round_kernel<2, true>) : launch(q4k_mm_round_kernel<1, true>);
    else pair ? launch(q4k_mm_round_kernel<2, false>) : launch(q4k_mm_round_kernel<1, false>);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "matvec_round launch");
    if (grid.y > 1 && d[6] != 2) {
        const int n = p.batch * p.rows0;
        hipLaunchKernelGGL(mm_round_fold_kernel, dim3((n + 255) / 256), dim3(256), 0, st, (const float *)k.scratch, p.Y0, n, (int)grid.y);
        e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, "matvec_round fold launch");
    }
    return 0;
}

constexpr int kSkinnyMaxBatch = 64;
// k.variant: 1 the small-batch form; else 2 * the K slices where their sums are folded (0: one slice), and this bit where
// the tile reads bf16 rows as they are
constexpr int kRowsDirect = 1 << 24;
// ... and this one where the rows of Q4_K take the tall shape of q4k_mm_rows_kernel (of Q6_K, of q6k_mm_rows_kernel)
constexpr int kTall = 1 << 25;
constexpr int kRows6 = 1 << 26;             // bf16 rows of Q6_K: q6k_mm_rows_kernel
using MmRowsTall = MmRows<2, 2, 1, 4>;      // 64 tokens x 256 rows
using MmRowsShort = MmRows<1, 2, 1, 4>;     // 32 tokens x 256 rows: gate | up, and CUT
using MmRowsSmall = MmRows<1, 1, 1, 4>;     // 32 tokens x 128 rows: the others
// bf16 rows (mm_plan_bf16)
using MmRowsBfTall = MmRows<4, 1, 1, 4, false>;   // 128 tokens x 128 rows
using MmRowsBf = MmRows<2, 1, 1, 4, false>;       // 64 x 128
static_assert(MmRowsBfTall::TN == BN && MmRowsBf::TN == BN, "mm_plan_bf16 counts rows of tiles so");

// Workgroups of a launch of `tm` tokens and `tn` rows (gate | up: half as many of each) a workgroup
dim3 mm_rows_grid(const ksh_kernel_desc &d, int tm, int tn, bool pair, int64_t ks)
{
    const int64_t y = pair ? (d.dims[0] + tn / 2 - 1) / (tn / 2) : (d.dims[0] + tn - 1) / tn + (d.dims[3] + tn - 1) / tn + (d.dims[4] + tn - 1) / tn;
    return dim3((unsigned)((d.dims[2] + tm - 1) / tm), (unsigned)y, (unsigned)ks);
}

// Tall or not: us a superblock takes the busiest compute unit, fitted to 256 .. 24576 rows of 256 .. 12288 columns and 63 ..
// 2048 tokens.  A tall workgroup alone on its compute unit 3.1, two of them 6.5 (the chip is then at its power limit, and more
// take turns); a short one alone 2.45, each further one 2.2; a small one alone 1.75, two or more 1.18 each.  Either side of its
// line: 1536 x 12288, 952 tokens (90 tall workgroups or 360 small ones) 158 us or 134, 2048 tokens (192 or 768) 201 or 221;
// 4096 x 1536, 2048 tokens (512 or 2048) 61 or 74; gate | up of 12288 x 1536, 140 tokens (288 tall or 480 short) 51 or 41.
// (A wave of two row tiles alone on its SIMD leaves the matrix pipe idle for half of the time.  Small for short: 2048 x 8192,
// 700 tokens 93 -> 87 us, 2048 x 2048, 63 tokens in four slices 12.8 -> 10.2, 1536 x 12288, 140 tokens 41.8 -> 35.7.  CUT stays
// short: 1989 tokens, 1536 x 12288 240 or 243 us, 1536 x 6144 129 or 131, 1536 x 2048 52 or 49.)
bool mm_rows_tall(const ksh_kernel_desc &d, bool pair, int64_t ks)
{
    auto turns = [&](int tm, int tn) {
        const dim3 g = mm_rows_grid(d, tm, tn, pair, ks);
        return (float)(((int64_t)g.x * g.y * g.z + 255) / 256);
    };
    const float tall = turns(MmRowsTall::TM, MmRowsTall::TN);
    const float other = pair ? turns(MmRowsShort::TM, MmRowsShort::TN) : turns(MmRowsSmall::TM, MmRowsSmall::TN);
    return (tall == 1.f ? 3.1f : 3.25f * tall) < (pair ? (other == 1.f ? 2.45f : 2.2f * other) : (other == 1.f ? 1.75f : 1.18f * other));
}

int mm_row_tiles(const ksh_kernel_desc &d) { return (int)((d.dims[0] + BN - 1) / BN + (d.dims[3] + BN - 1) / BN + (d.dims[4] + BN - 1) / BN); }

int launch_mul_mm_few(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    const FewParams p{(const uint8_t *)a.in[0], (const uint16_t *)a.in[1], (float *)a.out[0], (int)k.desc.dims[0], (int)k.desc.dims[1], (int)k.desc.dims[2], (int)k.info.sched.lds_tile};
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(k.info.grid[0], k.info.grid[1]), dim3(512), k.info.lds_bytes, st, p); };
    const int rh = k.info.sched.unroll;
    if (k.desc.dtypes[0] == KSH_Q6K) {
        if (p.tokens > 16) launch(q6k_mm_few_kernel<2, 1, 8>);
        else if (rh == 1) launch(q6k_mm_few_kernel<1, 1, 8>);
        else if (rh == 2) launch(q6k_mm_few_kernel<1, 2, 8>);
        else launch(q6k_mm_few_kernel<1, 4, 8>);
    } else if (p.tokens > 16) launch(q4k_mm_few_kernel<2, 1, 8>);
    else if (rh == 1) launch(q4k_mm_few_kernel<1, 1, 8>);
    else if (rh == 2) launch(q4k_mm_few_kernel<1, 2, 8>);
    else launch(q4k_mm_few_kernel<1, 4, 8>);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "mul_mm (few tokens) launch");
}

int launch_mul_mm(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    const int rows = (int)k.desc.dims[0], cols = (int)k.desc.dims[1], batch = (int)k.desc.dims[2];
    const bool f32x = k.desc.dtypes[1] == KSH_F32;
    const size_t xf_halves = (size_t)((batch + 31) / 32 * 32) * cols, sx_halves = (size_t)((batch + 31) / 32 * 32) * (cols / 256) * 32;
    _Float16 *Xf = (_Float16 *)k.scratch;
    _Float16 *SxA = Xf + xf_halves;
    _Float16 *Xf_lo = SxA + sx_halves, *SxA_lo = Xf_lo + xf_halves;     // f32 activations only
    const int n = batch * (cols / 8);
    const int n_mat0 = 1 + (k.desc.dims[3] > 0) + (k.desc.dims[4] > 0), prologue = (int)k.desc.dims[5];
    // f32 activations of the tile: both parts at the row's own scale, 1 / s per row where the small-batch form keeps
    // the sums of the lo parts (which the tile does not use)
    const bool tile = k.variant != 1;
    float *inv_s = f32x && tile ? reinterpret_cast<float *>(SxA_lo) : nullptr;
    // whole waves: the row-wide reductions read every lane.  An octet of the row a thread, from 1024 octets on two (12288
    // columns: 768 threads) where the tile keeps them
    const int octets = cols / 8, pb1 = (octets + 63) / 64 * 64;
    const dim3 pg((unsigned)batch), pb((unsigned)std::min(pb1 > 1024 && inv_s ? (octets / 2 + 63) / 64 * 64 : pb1, 1024));
    const bool rows_direct = (k.variant & (kRowsDirect | kRows6)) != 0;
    const int slices = (k.variant & ~(kRowsDirect | kTall | kRows6)) >> 1;                  // 0: no fold
    if (prologue) {
        // the rows' producer runs inside the preparation: in = W, X, [W1, W2,] then the prologue's operands
        const int xs = (int)k.desc.dims[7];
        const int n_out0 = k.desc.dims[6] & 1 ? 1 : n_mat0;                    // (unfolded partial sums are one buffer)
        const float *X = (const float *)a.in[1], *q0 = (const float *)a.in[1 + n_mat0];
        const float eps = k.desc.params[0];
        if (prologue == 1)
            hipLaunchKernelGGL(mm_prep_rows_kernel<1>, pg, pb, 0, st, X, q0, nullptr, nullptr, nullptr, Xf, Xf_lo, SxA, SxA_lo, cols, eps, xs, inv_s);
        else if (prologue == 2)
            hipLaunchKernelGGL(mm_prep_rows_kernel<2>, pg, pb, 0, st, X, q0, (const float *)a.in[2 + n_mat0], (const float *)a.in[3 + n_mat0], (float *)a.out[n_out0],
                               Xf, Xf_lo, SxA, SxA_lo, cols, eps, xs, inv_s);
        else
            hipLaunchKernelGGL(mm_prep_rows_kernel<3>, pg, pb, 0, st, X, xs ? X : q0, nullptr, nullptr, nullptr, Xf, Xf_lo, SxA, SxA_lo, cols, eps, xs, inv_s);
    } else if (f32x && tile)
        hipLaunchKernelGGL(mm_prep_rows_kernel<0>, pg, pb, 0, st, (const float *)a.in[1], nullptr, nullptr, nullptr, nullptr, Xf, Xf_lo, SxA, SxA_lo, cols, 0.f, 0, inv_s);
    else if (f32x) hipLaunchKernelGGL(mm_prep_x_f32_kernel, dim3((n + 255) / 256), dim3(256), 0, st, (const float *)a.in[1], Xf, Xf_lo, SxA, SxA_lo, batch, cols);
    else if (!rows_direct) {
        const dim3 xg(((batch + 31) / 32 * (cols / 32) + 3) / 4);
        if (tile) hipLaunchKernelGGL(mm_prep_x_kernel<true>, xg, dim3(256), 0, st, (const uint16_t *)a.in[1], Xf, SxA, batch, cols);
        else hipLaunchKernelGGL(mm_prep_x_kernel<false>, xg, dim3(256), 0, st, (const uint16_t *)a.in[1], Xf, SxA, batch, cols);
    }
    if (k.variant == 1) {
        // the small-batch form: one launch, the low parts riding along
        const SkinnyParams sp{(const uint8_t *)a.in[0], Xf, SxA, Xf_lo, SxA_lo, (float *)a.out[0], rows, cols, batch, 1.0f / 2048.0f};
        const dim3 sg((rows + 31) / 32);
        const int mt = batch <= 32 ? 1 : 2;
        const bool pieces = skinny_pieces(mt, f32x, cols / 256);
        const size_t lds = (size_t)8 * skinny_wave(mt, pieces) * 4;
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, sg, dim3(512), lds, st, sp); };
        if (f32x && mt == 2) launch(q4k_mm_skinny_kernel<2, true, false>);
        else if (f32x) pieces ? launch(q4k_mm_skinny_kernel<1, true, true>) : launch(q4k_mm_skinny_kernel<1, true, false>);
        else if (mt == 2) pieces ? launch(q4k_mm_skinny_kernel<2, false, true>) : launch(q4k_mm_skinny_kernel<2, false, false>);
        else pieces ? launch(q4k_mm_skinny_kernel<1, false, true>) : launch(q4k_mm_skinny_kernel<1, false, false>);
        const hipError_t e2 = hipGetLastError();
        return e2 == hipSuccess ? 0 : hip_fail(e2, "mul_mm (small batch) launch");
    }
    MmParams p;
    p.W = (const uint8_t *)a.in[0];
    p.Y = (float *)a.out[0];
    p.rows = rows; p.cols = cols; p.batch = batch;
    const int rows1 = (int)k.desc.dims[3], rows2 = (int)k.desc.dims[4];
    p.rows1 = rows1; p.rows2 = rows2;
    p.W1 = rows1 ? (const uint8_t *)a.in[2] : p.W; p.W2 = rows2 ? (const uint8_t *)a.in[3] : p.W;
    const bool unfolded_out = k.desc.dims[6] == 1, pair = k.desc.dims[6] == 3;
    p.Y1 = rows1 && !unfolded_out && !pair ? (float *)a.out[1] : p.Y; p.Y2 = rows2 && !unfolded_out ? (float *)a.out[2] : p.Y;
    const bool cut = k.desc.dims[6] == 2;
    const dim3 grid(k.info.grid[0], k.info.grid[1], k.info.grid[2]);
    p.Xf = rows_direct ? (const _Float16 *)a.in[1] : Xf;
    p.SxA = SxA; p.Xf_lo = Xf_lo; p.inv_s = inv_s;
    p.ksplit = 0; p.Y_parts = nullptr;
    p.cut_as = cut ? (const float *)a.in[k.info.n_inputs - 1] : nullptr;
    const bool q6 = k.desc.dtypes[0] == KSH_Q6K;
    p.keep = mm_keeps(std::max(slices, 1), batch, rows + rows1 + rows2, q6 && !(k.variant & kRows6), rows, rows1, rows2);
    const uint64_t wgs = (uint64_t)grid.x * grid.y * grid.z;
    p.wgs = wgs * std::max(grid.x, grid.y) < (1ull << 32) && grid.x > 1 && grid.y > 1 ? (uint32_t)wgs : 0;
    p.gx = grid.x; p.gy = grid.y;
    p.per_gx = (uint32_t)(((1ull << 32) + grid.x - 1) / grid.x); p.per_gy = (uint32_t)(((1ull << 32) + grid.y - 1) / grid.y);
    auto launch_rows = [&]() {
#define KSH_ROWS(S, ...) hipLaunchKernelGGL((q4k_mm_rows_kernel<S, __VA_ARGS__>), grid, dim3(S::kThreads), S::kLds, st, p)
        if (!f32x) {
            if (k.variant & kTall) KSH_ROWS(MmRowsBfTall, false, false);
            else KSH_ROWS(MmRowsBf, false, false);
        } else if (cut) KSH_ROWS(MmRowsShort, true, false);
        else if (k.variant & kTall) {
            if (pair) KSH_ROWS(MmRowsTall, false, true);
            else KSH_ROWS(MmRowsTall, false, false);
        } else if (pair) KSH_ROWS(MmRowsShort, false, true);
        else KSH_ROWS(MmRowsSmall, false, false);
#undef KSH_ROWS
    };
    auto launch_tile = [&]() {
#define KSH_TILE(...) hipLaunchKernelGGL((q6k_mul_mm_kernel<__VA_ARGS__>), grid, dim3(kThreadsMM), kLdsBytes, st, p)
        if (!q6) launch_rows();
        else if (cut) KSH_TILE(true, true);
        else if (f32x) KSH_TILE(true);
        else if (k.variant & kRows6) {
            if (k.variant & kTall) hipLaunchKernelGGL(q6k_mm_rows_kernel<2>, grid, dim3(Mm6Rows<2>::kThreads), Mm6Rows<2>::kLds, st, p);
            else hipLaunchKernelGGL(q6k_mm_rows_kernel<1>, grid, dim3(Mm6Rows<1>::kThreads), Mm6Rows<1>::kLds, st, p);
        }
        else if (rows_direct) KSH_TILE(false, false, true);
        else KSH_TILE(false);
#undef KSH_TILE
    };
    if (slices) {
        // few tiles: K slices as blockIdx.z of one launch, then the fold
        const int ks = slices;
        p.ksplit = ks;
        const bool unfolded = k.desc.dims[6] == 1;                    // the partial sums are the result: the reader adds them
        p.Y_parts = unfolded ? (float *)a.out[0] : (float *)((f32x ? SxA_lo : SxA) + sx_halves);     // (else behind the prepared activations)
        launch_tile();
        hipError_t e3 = hipGetLastError();
        if (e3 != hipSuccess) return hip_fail(e3, "mul_mm (K slices) launch");
        if (unfolded) return 0;
        const int n2 = batch * (rows + rows1 + rows2);
        hipLaunchKernelGGL(mm_parts_fold_kernel, dim3((n2 + 255) / 256), dim3(256), 0, st, (const float *)p.Y_parts, p.Y, p.Y1, p.Y2, batch, rows, rows1, rows2,
                           ks);
        e3 = hipGetLastError();
        return e3 == hipSuccess ? 0 : hip_fail(e3, "mul_mm fold launch");
    }
    launch_tile();
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "mul_mm launch");
}

}  // namespace

// (f32 activations)
int matvec_batch_slices(const ksh_kernel_desc &d, int batch)
{
    return mm_k_slices(d.dtypes[0] == KSH_Q6K, mm_row_tiles(d), (int)(d.dims[1] / 256), batch);
}

bool gate_up_pair(int dt_gate, int dt_up, int64_t ffn, int64_t hidden, int64_t batch)
{
    const int row_tiles = (int)(2 * ((ffn + BN - 1) / BN));
    return dt_gate == KSH_Q4K && dt_up == KSH_Q4K && mm_k_slices(false, row_tiles, (int)(hidden / 256), (int)batch) == 1;
}

int bind_matvec_batch(ksh_kernel &k)
{
    const int64_t rows = k.desc.dims[0], cols = k.desc.dims[1], batch = k.desc.dims[2];
    const bool q6 = k.desc.dtypes[0] == KSH_Q6K;
    if (k.desc.dtypes[0] != KSH_Q4K && !q6) return set_error("matvec_batch: weight dtype %d is not built (Q4_K and Q6_K are)", k.desc.dtypes[0]);
    const bool f32x = k.desc.dtypes[1] == KSH_F32;
    if (k.desc.dtypes[1] != KSH_BF16 && !f32x) return set_error("matvec_batch: activation dtype %d is not built (BF16 and F32 are)", k.desc.dtypes[1]);
    if (rows <= 0 || batch <= 0 || rows > (1 << 24) || batch > (1 << 20)) return set_error("matvec_batch: rows=%lld batch=%lld", (long long)rows, (long long)batch);
    if (cols <= 0 || cols % 256 || cols > (1 << 20)) return set_error("matvec_batch: cols=%lld is not a positive multiple of 256", (long long)cols);
    // dims[3], dims[4]: the rows of a second and a third matrix over the same activations (q | k | v of a prompt
    // chunk), taken by the tiles in the same launch
    const int64_t rows1 = k.desc.dims[3], rows2 = k.desc.dims[4], rows_all = rows + rows1 + rows2;
    if (rows1 < 0 || rows2 < 0 || (rows2 && !rows1) || rows_all > (1 << 24)) return set_error("matvec_batch: rows of the further matrices %lld, %lld", (long long)rows1, (long long)rows2);
    const int n_mat = 1 + (rows1 > 0) + (rows2 > 0);
    k.info.n_inputs = 1 + n_mat;
    k.info.n_outputs = n_mat;
    const size_t row_bytes = (size_t)(cols / 256) * (q6 ? 210 : 144);
    k.in_bytes[0] = (size_t)rows * row_bytes; k.in_align[0] = q6 ? 2 : 16;
    k.in_bytes[1] = (size_t)batch * cols * (f32x ? 4 : 2); k.in_align[1] = 16;
    k.out_bytes[0] = (size_t)batch * rows * 4; k.out_align[0] = 4;
    if (rows1) { k.in_bytes[2] = (size_t)rows1 * row_bytes; k.in_align[2] = k.in_align[0]; k.out_bytes[1] = (size_t)batch * rows1 * 4; k.out_align[1] = 4; }
    if (rows2) { k.in_bytes[3] = (size_t)rows2 * row_bytes; k.in_align[3] = k.in_align[0]; k.out_bytes[2] = (size_t)batch * rows2 * 4; k.out_align[2] = 4; }
    // dims[5]: the producer of the rows, run inside the preparation of f32 activations (params[0] = eps):
    //   1 rmsnorm(X, w)                 in: ..., w[cols]
    //   2 add then norm                 in: ..., w_post[cols], res[batch, cols], w_norm[cols]   out: ..., x_new[batch, cols] (may be res)
    //   3 gelu(X) * up                  in: ..., up[batch, cols]
    const int64_t prologue = k.desc.dims[5];
    if (prologue < 0 || prologue > 3) return set_error("matvec_batch: prologue %lld (0 none, 1 rmsnorm, 2 add then norm, 3 gelu * up)", (long long)prologue);
    // dims[6] = 1: the K slices' partial sums are the result, unfolded: out[0] = f32[slices][batch][all rows] (the
    // matrices' columns side by side; slices = grid[2] of the bound kernel), for a reader that adds them itself --
    // dims[7] = the slices (grid[2]) of the GEMM whose unfolded result this one's X is (prologues 1 to 3; prologue 3
    // then reads gate | up from that one buffer and takes no `up` operand)
    // dims[6] = 2: the rows belong to several prompts, each to be summed as in a launch of its own: one more input,
    // f32[batch], the tokens of that launch for every row (more than 64).  For f32 activations.
    // dims[6] = 3: W and W1 are a gate and an up matrix of one size and the result is gelu(W x) * (W1 x), f32[batch][rows].
    // For f32 activations, Q4_K, and rows that are not cut into K slices (matvec_batch_slices = 1).
    const bool unfolded = k.desc.dims[6] == 1, cut = k.desc.dims[6] == 2, pair = k.desc.dims[6] == 3;
    const int64_t x_slices = k.desc.dims[7];
    if (k.desc.dims[6] < 0 || k.desc.dims[6] > 3)
        return set_error("matvec_batch: dims[6]=%lld (0, 1 for unfolded partial sums, 2 for rows summed as in launches of their own, 3 for gelu(gate) * up)", (long long)k.desc.dims[6]);
    if (pair && (!f32x || q6 || rows1 != rows || rows2 || k.desc.sched.nr0 == 32 ||
                 (k.desc.sched.k_split ? k.desc.sched.k_split != 1 : matvec_batch_slices(k.desc, (int)batch) != 1)))
        return set_error("matvec_batch: gelu(gate) * up (dims[6]=3) takes F32 activations, two Q4_K matrices of one size and rows in one K slice");
    if (cut && !f32x) return set_error("matvec_batch: rows summed as in launches of their own (dims[6]=2) take F32 activations");
    if (x_slices && (!prologue || x_slices < 1 || x_slices > 64))
        return set_error("matvec_batch: X as unfolded partial sums (dims[7]=%lld) takes a prologue and 1 to 64 slices", (long long)k.desc.dims[7]);
    if (prologue) {
        if (!f32x) return set_error("matvec_batch: a prologue takes F32 activations");
        if (prologue != 3 && (cols > 8192 || cols % 512)) return set_error("matvec_batch: a norm prologue takes rows of a multiple of 512 up to 8192 columns, got %lld", (long long)cols);
        int ni = 1 + n_mat;
        const size_t vec = (size_t)cols * 4, mat = (size_t)batch * cols * 4;
        auto add_in = [&](size_t bytes) { k.in_bytes[ni] = bytes; k.in_align[ni] = 16; ni++; };
        if (prologue == 1) add_in(vec);
        if (prologue == 2) { add_in(vec); add_in(mat); add_in(vec); k.out_bytes[n_mat] = mat; k.out_align[n_mat] = 16; k.info.n_outputs = n_mat + 1; }
        if (prologue == 3 && !x_slices) add_in(mat);
        k.info.n_inputs = ni;
        if (x_slices) k.in_bytes[1] = (size_t)x_slices * mat * (prologue == 3 ? 2 : 1);
    }
    if (pair) {
        if (prologue == 2) { k.out_bytes[1] = k.out_bytes[n_mat]; k.out_align[1] = 16; }
        k.info.n_outputs = prologue == 2 ? 2 : 1;
    }
    if (cut) {
        const int ni = k.info.n_inputs++;
        k.in_bytes[ni] = (size_t)batch * 4; k.in_align[ni] = 4;
    }
    // f16 copy of X plus the min-term operand (32 halves per token and superblock)
    const size_t batch32 = (size_t)((batch + 31) / 32 * 32);
    k.scratch_bytes = (batch32 * cols * 2 + batch32 * (cols / 256) * 64) * (f32x ? 2 : 1);
    // schedule: nr0 = weight rows per workgroup.  32 = the small-batch form (Q4_K, up to 64 tokens: the default
    // there), 128 = the tiles (their tokens and rows follow from the sizes).
    // 16: one launch of bf16 tokens, up to 32 to a workgroup and kFewMost in all (sched.unroll: tiles of 16 weight rows a workgroup), the
    // default where it is estimated the shortest (mm_few_open, mm_few_plan).
    const uint32_t want = k.desc.sched.nr0;
    if (want && want != 16 && want != 32 && want != BN) return set_error("matvec_batch: unsupported schedule nr0=%u (16, 32 or %d)", want, BN);
    const bool can_skinny = !q6 && batch <= kSkinnyMaxBatch && n_mat == 1 && !unfolded && !cut && !pair;
    if (want == 32 && !can_skinny) return set_error("matvec_batch: the small-batch form takes Q4_K weights and up to %d tokens", kSkinnyMaxBatch);
    // (long rows of a short matrix leave the small-batch form 64 workgroups with four superblocks per wave: f32, from 33
    // tokens on, the tile over K slices is faster there -- 2048 x 8192 at 63 tokens: 27.5 us against 41.0; bf16 rows take
    // whichever form is estimated shorter -- 1536 x 6144 at 50 tokens: 16.1 against 21.1)
    const bool long_rows = f32x ? batch > 32 && rows <= 2048 && cols >= 8192
                                : mm_plan_bf16(q6, mm_row_tiles(k.desc), (int)(cols / 256), batch, rows_all, (int)k.desc.sched.k_split).us < mm_skinny_us(rows, (int)(cols / 256), batch);
    k.variant = (want == 32 || (want == 0 && can_skinny && !long_rows)) ? 1 : 0;
    k.info.sched = k.desc.sched;
    const bool can_few = n_mat == 1 && !unfolded && !cut && !pair && !f32x && batch <= kFewMost;
    if (want == 16 && !can_few) return set_error("matvec_batch: the form of one launch takes bf16 rows, one matrix and up to %d tokens", kFewMost);
    if (can_few && (want == 16 || sched_is_zero(k.desc.sched))) {
        const int nsb = (int)(cols / 256);
        const FewPlan few = mm_few_plan(q6, rows, nsb, batch);
        const float tiles = mm_plan_bf16(q6, mm_row_tiles(k.desc), nsb, batch, rows_all, 0).us;
        if (want == 16 || (mm_few_open(q6, nsb, batch, few) && 1.04f * few.us < (q6 || batch > kSkinnyMaxBatch ? tiles : std::min(mm_skinny_us(rows, nsb, batch), tiles)))) {
            // (as a schedule names them, where they are a launch)
            const int u = (int)k.desc.sched.unroll, l = (int)std::min<uint32_t>(k.desc.sched.lds_tile, kFewTokens + 1);
            const int tokens = want == 16 && l >= 1 && l <= kFewTokens ? (int)std::min<int64_t>(l, batch) : few.tokens;
            const int rh = want == 16 && few_fits(q6, tokens, u) ? u : few_fits(q6, tokens, few.rh) ? few.rh : 1;
            k.scratch_bytes = 0;
            k.variant = 1;
            set_launch(k, (uint32_t)((rows + 16 * rh - 1) / (16 * rh)), (uint32_t)((batch + tokens - 1) / tokens), 1, 512, (uint32_t)few_lds(q6, tokens, rh));
            k.info.sched.tg = 512; k.info.sched.nsg = 8; k.info.sched.nr0 = 16; k.info.sched.unroll = (uint32_t)rh; k.info.sched.k_split = 8;
            k.info.sched.lds_tile = (uint32_t)tokens;
            set_name(k, "mul_mm_%s_few_%dxT%d", q6 ? "q6k" : "q4k", 16 * rh, tokens <= 16 ? 16 : 32);
            k.launch = launch_mul_mm_few;
            return 0;
        }
    }
    if (k.variant == 1) {
        const int mt = batch <= 32 ? 1 : 2;
        set_launch(k, (uint32_t)((rows + 31) / 32), 1, 1, 512, (uint32_t)(8 * skinny_wave(mt, skinny_pieces(mt, f32x, (int)(cols / 256))) * 4));
        k.info.sched.tg = 512; k.info.sched.nsg = 8; k.info.sched.nr0 = 32; k.info.sched.k_split = 8; k.info.sched.lds_tile = 16;
        set_name(k, "mul_mm_q4k_skinny_32xT%d%s", batch <= 32 ? 32 : 64, f32x ? "_f32x" : "");
        k.launch = launch_mul_mm;
        return 0;
    }
    // K slices: workgroups of one launch, every slice storing its partial sums, and a second launch that adds them
    // (mm_k_slices, mm_plan_bf16).  sched.k_split names the slice count (a divisor of cols / 256; 1 = none).  For bf16 rows
    // the plan takes any count, and a schedule that a bound kernel has reported (it names the tile too) takes it again.  (512
    // threads and 64 columns are what the tile of two roles reports; saved plans of Q4_K may hold them too, from when it was theirs.)
    const int64_t row_tiles = mm_row_tiles(k.desc), nsb = cols / 256;
    int64_t ks = cut ? 1 : k.desc.sched.k_split;
    const bool reported = !f32x && want == BN && ((k.desc.sched.tg == kThreadsMM && k.desc.sched.lds_tile == KS) || (k.desc.sched.tg == MmRowsBf::kThreads && k.desc.sched.lds_tile == (q6 ? KS : 32))) &&
                          ks <= std::min<int64_t>(nsb, 64);
    if (!cut && ks && nsb % ks && !reported) return set_error("matvec_batch: k_split=%lld does not divide the %lld superblocks of a row", (long long)ks, (long long)nsb);
    int tm = 0;
    if (f32x) {
        if (!ks) ks = mm_k_slices(q6, (int)row_tiles, (int)nsb, (int)batch);
        tm = mm_tile_tokens(q6);
    } else {
        const MmPlan plan = mm_plan_bf16(q6, (int)row_tiles, (int)nsb, batch, rows_all, (int)ks);
        ks = plan.ks;
        tm = plan.tm;
    }
    const bool z_form = unfolded || ks > 1;
    k.variant = z_form ? (int)(ks << 1) : 0;
    if (!f32x && q6 && tm < BM) k.variant |= kRows6 | (tm == Mm6Rows<2>::TM ? kTall : 0);
    else if (!f32x && q6 && mm_rows_direct((batch + tm - 1) / tm * row_tiles * ks, (int)((nsb + ks - 1) / ks), batch, cols)) k.variant |= kRowsDirect;
    if (z_form && !unfolded) k.scratch_bytes += (size_t)ks * batch * rows_all * 4;
    if (unfolded) {
        const int keep = prologue == 2 ? 1 : 0;                       // (the add-then-norm prologue's x_new stays an output)
        if (keep) { k.out_bytes[1] = k.out_bytes[n_mat]; k.out_align[1] = 16; }
        k.out_bytes[0] = (size_t)ks * batch * rows_all * 4; k.out_align[0] = 16;
        k.info.n_outputs = 1 + keep;
    }
    if (f32x && !q6) {
        const bool tall = !cut && mm_rows_tall(k.desc, pair, z_form ? ks : 1);
        if (tall) k.variant |= kTall;
        const bool small = !tall && !pair && !cut;
        const int tmr = tall ? MmRowsTall::TM : MmRowsShort::TM, tnr = small ? MmRowsSmall::TN : MmRowsTall::TN;
        const dim3 g = mm_rows_grid(k.desc, tmr, tnr, pair, z_form ? ks : 1);
        set_launch(k, g.x, g.y, g.z, MmRowsTall::kThreads, (uint32_t)(tall ? MmRowsTall::kLds : small ? MmRowsSmall::kLds : MmRowsShort::kLds));
        k.info.sched.tg = MmRowsTall::kThreads; k.info.sched.nsg = MmRowsTall::kThreads / 64; k.info.sched.nr0 = BN; k.info.sched.k_split = (uint32_t)ks; k.info.sched.lds_tile = 32;
        set_name(k, "mul_mm_q4k_%dx%dx32_f32x%s%s%s", tmr, tnr, z_form ? "_kz" : "", n_mat == 3 ? "_x3" : n_mat == 2 ? "_x2" : "",
                 prologue == 1 ? "_rms" : prologue == 2 ? "_addrms" : prologue == 3 ? "_gelu" : "");
    } else if (!q6) {
        if (tm == MmRowsBfTall::TM) k.variant |= kTall;
        set_launch(k, (uint32_t)((batch + tm - 1) / tm), (uint32_t)row_tiles, z_form ? (uint32_t)ks : 1, MmRowsBf::kThreads, (uint32_t)(tm == MmRowsBfTall::TM ? MmRowsBfTall::kLds : MmRowsBf::kLds));
        k.info.sched.tg = MmRowsBf::kThreads; k.info.sched.nsg = MmRowsBf::kThreads / 64; k.info.sched.nr0 = BN; k.info.sched.k_split = (uint32_t)ks; k.info.sched.lds_tile = 32;
        set_name(k, "mul_mm_q4k_%dx%dx32%s%s", tm, BN, z_form ? "_kz" : "", n_mat == 3 ? "_x3" : n_mat == 2 ? "_x2" : "");
    } else if (k.variant & kRows6) {
        const int lds = tm == Mm6Rows<2>::TM ? Mm6Rows<2>::kLds : Mm6Rows<1>::kLds;
        set_launch(k, (uint32_t)((batch + tm - 1) / tm), (uint32_t)row_tiles, z_form ? (uint32_t)ks : 1, Mm6Rows<2>::kThreads, (uint32_t)lds);
        k.info.sched.tg = Mm6Rows<2>::kThreads; k.info.sched.nsg = Mm6Rows<2>::kThreads / 64; k.info.sched.nr0 = BN; k.info.sched.k_split = (uint32_t)ks; k.info.sched.lds_tile = KS;
        set_name(k, "mul_mm_q6k_%dx%dx%d%s%s", tm, BN, KS, z_form ? "_kz" : "", n_mat == 3 ? "_x3" : n_mat == 2 ? "_x2" : "");
    } else {
        set_launch(k, (uint32_t)((batch + tm - 1) / tm), (uint32_t)row_tiles, z_form ? (uint32_t)ks : 1, kThreadsMM, (uint32_t)kLdsBytes);
        k.info.sched.tg = kThreadsMM; k.info.sched.nsg = kThreadsMM / 64; k.info.sched.nr0 = BN; k.info.sched.k_split = (uint32_t)ks; k.info.sched.lds_tile = KS;
        set_name(k, "mul_mm_q6k_%dx%dx%d%s%s%s%s", BM, BN, KS, f32x ? "_f32x" : "", z_form ? "_kz" : "", n_mat == 3 ? "_x3" : n_mat == 2 ? "_x2" : "",
                 prologue == 1 ? "_rms" : prologue == 2 ? "_addrms" : prologue == 3 ? "_gelu" : "");
    }
    if (pair) { char nm[64]; snprintf(nm, sizeof(nm), "%s", k.info.name); set_name(k, "%s_gate_up", nm); }
    if (cut) { char nm[64]; snprintf(nm, sizeof(nm), "%s", k.info.name); set_name(k, "%s_cut", nm); }
    if (unfolded) { char nm[64]; snprintf(nm, sizeof(nm), "%s", k.info.name); set_name(k, "%s_unfolded", nm); }
    k.launch = launch_mul_mm;
    return 0;
}

int bind_round_prep(ksh_kernel &k)
{
    const int64_t cols = k.desc.dims[0], batch = k.desc.dims[1], mode = k.desc.dims[2];
    if (cols <= 0 || cols % 256 || cols > (1 << 16)) return set_error("round_prep: cols=%lld is not a positive multiple of 256 up to 65536", (long long)cols);
    if (batch < 1 || batch > kRoundTokens) return set_error("round_prep: %lld rows (1 to %d)", (long long)batch, kRoundTokens);
    if (mode < 0 || mode > 3) return set_error("round_prep: mode %lld (0 plain, 1 rmsnorm, 2 add then rmsnorm, 3 rmsnorm add)", (long long)mode);
    if (mode >= 2 && cols > 8192) return set_error("round_prep: the add-then-norm form keeps a row in LDS (cols=%lld, up to 8192)", (long long)cols);
    const int64_t slices = std::max<int64_t>(1, k.desc.dims[3]);
    if (k.desc.dims[3] < 0 || slices > 64 || (slices > 1 && (!mode || cols > 2048)))
        return set_error("round_prep: an input in %lld column slices takes a norm (mode 1 to 3) and rows of up to 2048 columns", (long long)k.desc.dims[3]);
    k.info.n_inputs = mode == 2 ? 4 : mode == 3 ? 3 : mode == 1 ? 2 : 1;
    k.info.n_outputs = mode >= 2 ? 2 : 1;
    k.in_bytes[0] = (size_t)slices * batch * cols * 4; k.in_align[0] = 16;
    // (128-bit loads and stores of every operand)
    if (mode) { k.in_bytes[1] = (size_t)cols * 4; k.in_align[1] = 16; }
    if (mode >= 2) {
        k.in_bytes[2] = (size_t)batch * cols * 4; k.in_align[2] = 16;
        if (mode == 2) { k.in_bytes[3] = (size_t)cols * 4; k.in_align[3] = 16; }
        k.out_bytes[1] = (size_t)batch * cols * 4; k.out_align[1] = 16;
    }
    k.out_bytes[0] = (round_xf_halves((int)cols) + 2 * round_sx_halves((int)cols)) * 2; k.out_align[0] = 16;
    if (mode) set_launch(k, kRoundTokens, 1, 1, 256, mode >= 2 ? (uint32_t)cols * 4 : 0);
    else set_launch(k, (uint32_t)((kRoundTokens * (cols / 8) + 255) / 256), 1, 1, 256, 0);
    set_name(k, mode == 3 ? "round_prep_rmsnorm_add" : mode == 2 ? "round_prep_add_then_rmsnorm" : mode == 1 ? "round_prep_rmsnorm" : "round_prep_f32x");
    k.launch = launch_round_prep;
    return 0;
}

int bind_matvec_round(ksh_kernel &k)
{
    const int64_t *d = k.desc.dims;
    const int64_t rows0 = d[0], cols = d[1], batch = d[2], rows1 = d[3], rows2 = d[4];
    const bool pair = d[5] != 0;
    const bool q6r = k.desc.dtypes[0] == KSH_Q6K_ROWS;
    if (k.desc.dtypes[0] != KSH_Q4K && !q6r) return set_error("matvec_round: weight dtype %d is not built (Q4_K and row-grouped Q6_K are)", k.desc.dtypes[0]);
    if (cols <= 0 || cols % 256 || cols > (1 << 16)) return set_error("matvec_round: cols=%lld is not a positive multiple of 256 up to 65536", (long long)cols);
    if (batch < 1 || batch > kRoundTokens) return set_error("matvec_round: %lld rows (1 to %d)", (long long)batch, kRoundTokens);
    if (q6r) {
        if (rows1 || rows2 || pair) return set_error("matvec_round: row-grouped Q6_K takes one matrix per launch");
        if (cols > 2048) return set_error("matvec_round: row-grouped Q6_K rows of up to 2048 columns (cols=%lld)", (long long)cols);
        if (rows0 <= 0 || rows0 > (1 << 24)) return set_error("matvec_round: rows %lld", (long long)rows0);
        k.info.n_inputs = 2;
        k.info.n_outputs = 1;
        k.in_bytes[0] = (size_t)rows0 * round_q6r_row_bytes((int)(cols / 256)); k.in_align[0] = 16;
        k.in_bytes[1] = (round_xf_halves((int)cols) + 2 * round_sx_halves((int)cols)) * 2; k.in_align[1] = 16;
        k.out_bytes[0] = (size_t)batch * rows0 * 4; k.out_align[0] = 4;
        // one workgroup per compute unit (its registers hold the activations of a whole row), tiles shared out evenly
        const int64_t tiles = (rows0 + 31) / 32, per = (tiles + 255) / 256;
        set_launch(k, (uint32_t)((tiles + per - 1) / per), 1, 1, 512, (uint32_t)(2 * 8 * 8 * 64 * 4));
        k.info.sched = k.desc.sched;
        k.info.sched.tg = 512; k.info.sched.nsg = 8; k.info.sched.nr0 = 32; k.info.sched.k_split = 1; k.info.sched.lds_tile = 16;
        set_name(k, "matvec_round_q6krows");
        k.launch = launch_matvec_round;
        return 0;
    }
    if (rows0 <= 0 || rows1 < 0 || rows2 < 0 || (rows2 && !rows1) || rows0 + rows1 + rows2 > (1 << 24))
        return set_error("matvec_round: rows %lld / %lld / %lld", (long long)rows0, (long long)rows1, (long long)rows2);
    if (pair && (rows1 || rows2)) return set_error("matvec_round: a gate | up pair names one row count (both matrices have it)");
    const int slices = (int)((cols / 256 + 7) / 8);
    if (slices > 1 && (pair || rows1)) return set_error("matvec_round: rows longer than 2048 columns take one matrix per launch");
    const bool emit = d[6] == 1, unfolded = d[6] == 2;
    if (d[6] < 0 || d[6] > 2) return set_error("matvec_round: result form %lld (0 rows, 1 prepared operand, 2 the column slices' partial sums)", (long long)d[6]);
    const int64_t mul_stride = d[7];
    if (mul_stride && (pair || rows1 || mul_stride < rows0)) return set_error("matvec_round: the gate multiplier takes one matrix and a row stride of at least its rows");
    if (emit && (rows1 || slices > 1 || rows0 % 256))
        return set_error("matvec_round: the result as a prepared operand takes one matrix (or a pair) of up to 2048 columns whose rows are a multiple of 256");
    const int n_mat = pair ? 2 : rows2 ? 3 : rows1 ? 2 : 1;
    const int64_t rows[3] = {rows0, pair ? rows0 : rows1, rows2};
    k.info.n_inputs = 1 + n_mat;
    k.info.n_outputs = pair ? 1 : n_mat;
    k.in_bytes[0] = (size_t)rows0 * (cols / 256) * 144; k.in_align[0] = 16;
    k.in_bytes[1] = (round_xf_halves((int)cols) + 2 * round_sx_halves((int)cols)) * 2; k.in_align[1] = 16;
    for (int i = 1; i < n_mat; i++) { k.in_bytes[1 + i] = (size_t)rows[i] * (cols / 256) * 144; k.in_align[1 + i] = 16; }
    if (mul_stride) { k.info.n_inputs = 3; k.in_bytes[2] = ((size_t)(batch - 1) * mul_stride + rows0) * 4; k.in_align[2] = 4; }
    for (int i = 0; i < k.info.n_outputs; i++) { k.out_bytes[i] = (size_t)batch * rows[i] * 4; k.out_align[i] = 4; }
    if (emit) { k.out_bytes[0] = (round_xf_halves((int)rows0) + 2 * round_sx_halves((int)rows0)) * 2; k.out_align[0] = 16; }
    if (unfolded && (rows1 || pair)) return set_error("matvec_round: partial sums as the result take one matrix");
    k.scratch_bytes = slices > 1 && !unfolded ? (size_t)slices * batch * rows0 * 4 : 0;
    if (unfolded) k.out_bytes[0] = (size_t)slices * batch * rows0 * 4;
    const int64_t tiles = pair ? (rows0 + 31) / 32 : (rows0 + 31) / 32 + (rows1 + 31) / 32 + (rows2 + 31) / 32;
    set_launch(k, (uint32_t)tiles, (uint32_t)slices, 1, 512, (uint32_t)(8 * (pair ? 2 : 1) * kRoundTile * 4 + (emit ? 16 * 33 * 4 : 0)));
    k.info.sched = k.desc.sched;
    k.info.sched.tg = 512; k.info.sched.nsg = 8; k.info.sched.nr0 = 32; k.info.sched.k_split = (uint32_t)slices; k.info.sched.lds_tile = 16;
    set_name(k, "matvec_round_q4k_%s%s%s", pair ? "gate_up_gelu" : mul_stride ? "gelu_mul" : n_mat == 3 ? "x3" : n_mat == 2 ? "x2" : "x1",
             slices > 1 ? "_ksplit" : "", emit ? "_prepared" : "");
    k.launch = launch_matvec_round;
    return 0;
}

// Schedules of the prefill GEMM beside the library's own, which a search times first, as the bound kernels report them: whole
// rows, for bf16 tokens the form of one launch (Q4_K beyond 192 tokens: where it is estimated the shorter), for Q4_K weights and up to 64 tokens 32
// weight rows per workgroup with the K range split over its 8 waves, and K slices where half as many leave the chip short of workgroups.  (The shape of a workgroup follows from the sizes, for bf16 rows from the
// slice count too; counts that do not divide a row come from the library's own schedule only.)
int mul_mm_candidates(const ksh_kernel_desc &d, ksh_sched *out, int cap)
{
    int n = 0;
    const bool q6 = d.dtypes[0] == KSH_Q6K, f32x = d.dtypes[1] == KSH_F32;
    const int row_tiles = mm_row_tiles(d), nsb = (int)(d.dims[1] / 256);
    if (nsb <= 0 || row_tiles <= 0 || d.dims[2] <= 0) return 0;
    int tm = BM;                       // tokens a workgroup
    auto tile = [&](uint32_t ks) {
        if (!f32x) tm = mm_plan_bf16(q6, row_tiles, nsb, d.dims[2], d.dims[0] + d.dims[3] + d.dims[4], (int)ks).tm;
        const bool two_roles = q6 && tm == BM;
        ksh_sched s{};
        s.tg = two_roles ? kThreadsMM : MmRowsBf::kThreads; s.nsg = s.tg / 64; s.nr0 = BN; s.lds_tile = q6 ? KS : 32; s.unroll = 1; s.vec = 0; s.k_split = ks;
        return s;
    };
    if (n < cap) out[n++] = tile(1);
    // workgroups of whole rows, and the number that fills the chip: one to a compute unit of 128 tokens, two of the others (two of the
    // large ones take turns on what the chip's power allows, see mm_rows_tall)
    int64_t wgs = (d.dims[2] + tm - 1) / tm * row_tiles;
    int64_t full = tm == BM ? 256 : 512;
    if (f32x && !q6) {
        const bool tall = mm_rows_tall(d, false, 1);
        const dim3 g = tall ? mm_rows_grid(d, MmRowsTall::TM, MmRowsTall::TN, false, 1) : mm_rows_grid(d, MmRowsSmall::TM, MmRowsSmall::TN, false, 1);
        wgs = (int64_t)g.x * g.y;
        full = tall ? 256 : 512;
    }
    if (!f32x && d.dims[2] <= kFewMost && !d.dims[3] && !d.dims[6]) {
        const FewPlan few = mm_few_plan(q6, d.dims[0], nsb, d.dims[2]);
        const int tokens = few.tokens;
        const bool timed = d.dims[2] <= (q6 ? kFewMost : 192) || few.us < mm_plan_bf16(q6, row_tiles, nsb, d.dims[2], d.dims[0], 0).us;
        for (uint32_t rh : {1u, 2u, 4u}) {
            if (!timed || n >= cap || !few_fits(q6, tokens, (int)rh)) break;
            ksh_sched s{};
            s.tg = 512; s.nsg = 8; s.nr0 = 16; s.lds_tile = (uint32_t)tokens; s.unroll = rh; s.vec = 0; s.k_split = 8;
            out[n++] = s;
        }
    }
    if (n < cap && !q6 && d.dims[2] <= kSkinnyMaxBatch && !d.dims[3]) {
        ksh_sched s{};
        s.tg = 512; s.nsg = 8; s.nr0 = 32; s.lds_tile = 16; s.unroll = 1; s.vec = 0; s.k_split = 8;
        out[n++] = s;
    }
    for (uint32_t ks : {2u, 4u, 8u, 16u}) {
        if (n >= cap || nsb % ks || wgs * (ks / 2) >= full) continue;
        out[n++] = tile(ks);
    }
    return n;
}

}  // namespace ksh
