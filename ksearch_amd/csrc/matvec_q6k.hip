// Q6_K packed-weight GEMV for gfx950 (the LM head: 262144 x 2048).
//
// Takes the place of lower_matvec_q6k_coop
// (crates/ksearch_codegen/src/lower.rs:2086-2472) and
// ksearch_q6k_coop_frag_nr4_dev (crates/ksearch_codegen/src/render.rs:886-930),
// which give 2 lanes x 16 positions per superblock with byte loads on a
// 32-lane simdgroup.  Here:
//
//   - a superblock (210 B: ql[128] qh[64] sc[16] d) is owned by 8 lanes: lane j
//     has ql bytes 16j .. 16j+15, i.e. in half ip = j / 4 the positions
//     l0 = 16 * (j % 2) .. +15 of the quadrants part (low nibbles) and part + 2
//     (high nibbles), part = (j / 2) % 2, and the 16 qh bytes of those;
//   - a wave sweeps 8 superblocks (2048 columns) per step; the activation
//     vector is staged once per workgroup in LDS as three int8 digit planes of
//     X = rint(x / s), s = max|x| / (2^20 - 1) per 128 elements (optionally
//     after an RMSNorm / add-then-RMSNorm computed by the workgroup itself,
//     gemv_prologue.hpp), and a lane keeps its 32 positions' digits in
//     registers across every row it owns;
//   - the 6-bit values are assembled four at a time with dword logic and meet
//     the digit planes in v_dot4_i32_i8 (exact integer sums per quadrant); the
//     -32 offset is applied through the pre-summed X of each run:
//       y += d * s * sum_k sc_k * (sum(v*X) - 32*SX_k)
//     |x - s X| <= s/2 = 2^-21 of the run's largest magnitude, below the f32
//     summation noise of a 2048-term dot;
//   - a workgroup walks a long run of rows (x staged once).  Two byte orders:
//     the file's (q6k_stream_kernel) and rows regrouped by field
//     (q6r_gemv_kernel).
//
// The result differs from dequant-then-dot (gguf_impl.rs:761-791 +
// check_mul_mm.rs:60-71) by reassociation and by that rounding of x.
#include <algorithm>
#include <type_traits>

#include "gemv_prologue.hpp"
#include "ksh_internal.hpp"

KSH_STAMP_BUFFER
KSH_STAMP_READER(ksh_stamps_matvec_q6k)

namespace ksh {
namespace {

constexpr int kQ6kBytes = 210;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int dot4_start(int a, int b)
{
    int r;
    asm("v_dot4_i32_i8 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

struct Q6kParams {
    const uint8_t *W;
    float *y;
    Prologue pro;
    int rows, bpr;
    int rows_per_wave;    // regrouped rows
    int wgs;              // file order: workgroups (gridDim would come with arguments of its own)
};
static_assert(sizeof(Q6kParams) <= kArgBytes, "a launch's arguments");

// ---- Q6K_ROWS: the same weights with every row regrouped by field ------------
// Row of bpr superblocks: ql [bpr][128] | qh [bpr][64] | sc [bpr][16] | d [bpr][2], each section 16-byte
// aligned, the row padded to a multiple of 16 bytes (q6r_row_bytes: 1264 for the 1260 bytes of a 1536-column
// row; nothing for 2048 or 4096 columns).  A step covers 8 superblocks with ONE 128-bit load per lane over 1 KB of ql, lane
// after lane: lane j = lane % 8 of superblock b = lane / 8 holds ql bytes 16j .. 16j+15, i.e. in half ip = j / 4
// the positions l0 = 16 * (j % 2) .. +15 of the quadrants k = part (low nibbles) and part + 2 (high nibbles),
// part = (j / 2) % 2.  It fetches the 16 qh bytes of those positions (lanes j and j ^ 2 the same ones), the
// half's 8 scale bytes and d.  A row is then fetched through the fewest cache lines it spans (14) instead of
// the ~80 that the per-field loads of the 210-byte superblocks touch.
__host__ __device__ constexpr size_t q6r_row_bytes(int bpr) { return ((size_t)bpr * 210 + 15) / 16 * 16; }

struct Q6rLane {
    u32x4_t ql, qh;
    u32x2 sc;
    uint32_t d;
};

__device__ __forceinline__ Q6rLane q6r_load(const uint8_t *row, int bpr, int blk, int lane)
{
    const int j = lane & 7, ip = j >> 2;
    Q6rLane r;
    // (streamed once per launch and never reused: loads marked non-temporal, 88.6 -> 85.8 us on 262144 x 2048; the same
    // mark on the Q4_K GEMVs' weights costs them 5 %)
    r.ql = __builtin_nontemporal_load((const KSH_GLOBAL u32x4_t *)(row + (size_t)blk * 128 + 16 * j));
    r.qh = __builtin_nontemporal_load((const KSH_GLOBAL u32x4_t *)(row + (size_t)bpr * 128 + (size_t)blk * 64 + 32 * ip + 16 * (j & 1)));
    r.sc = *(const KSH_GLOBAL u32x2 *)(row + (size_t)bpr * 192 + (size_t)blk * 16 + 8 * ip);
    r.d = *(const KSH_GLOBAL uint16_t *)(row + (size_t)bpr * 208 + (size_t)blk * 2);
    return r;
}

// the lane's share of the staged vector: digit planes of its 16 positions in its two quadrants, minus 32 times
// the sum of X over each 16, and the scale of its 128-element half
struct XQ6r {
    u32x4_t H[2], M[2], L[2];
    int nsx5[2];
    float s;
    __device__ __forceinline__ void load(const uint8_t *lds, int blk, int lane, bool valid)
    {
        const int j = lane & 7, ip = j >> 2, part = (j >> 1) & 1, l0 = 16 * (j & 1);
        const uint8_t *half = lds + (blk * 2 + ip) * kQ6HalfBytes;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int k = part + 2 * q, o = 32 * k + l0;
            H[q] = *reinterpret_cast<const u32x4_t *>(half + o);
            M[q] = *reinterpret_cast<const u32x4_t *>(half + 128 + o);
            L[q] = *reinterpret_cast<const u32x4_t *>(half + 256 + o);
            const int *nsx = reinterpret_cast<const int *>(half + 384) + 4 * k + 2 * (j & 1);   // runs of 8
            nsx5[q] = (nsx[0] + nsx[1]) * 32;
        }
        s = valid ? *reinterpret_cast<const float *>(half + 448) : 0.f;
    }
};

__device__ __forceinline__ float q6r_lane_dot(const Q6rLane &B, int lane, const XQ6r &X)
{
    const int j = lane & 7, part = (j >> 1) & 1;
    int hs[2], ms[2], ls[2];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const uint32_t t = B.qh[w] >> (2 * part);
        const uint32_t a[2] = {(B.ql[w] & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u), ((B.ql[w] >> 4) & 0x0F0F0F0Fu) | (t & 0x30303030u)};
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (w == 0) {
                hs[q] = dot4_start((int)a[q], (int)X.H[q][0]);
                ms[q] = dot4_start((int)a[q], (int)X.M[q][0]);
                ls[q] = __builtin_amdgcn_sdot4((int)a[q], (int)X.L[q][0], X.nsx5[q], false);   // starts at -32*sum(X)
            } else {
                hs[q] = __builtin_amdgcn_sdot4((int)a[q], (int)X.H[q][w], hs[q], false);
                ms[q] = __builtin_amdgcn_sdot4((int)a[q], (int)X.M[q][w], ms[q], false);
                ls[q] = __builtin_amdgcn_sdot4((int)a[q], (int)X.L[q][w], ls[q], false);
            }
        }
    }
    // scales of the half: index 2k + l0/16 for k = part and part + 2: byte 2*part + (j&1) of each dword
    const int sh = 8 * (2 * part + (j & 1));
    const float c0 = (float)(int8_t)(B.sc.x >> sh), c1 = (float)(int8_t)(B.sc.y >> sh);
    const int x0 = (((hs[0] << 7) + ms[0]) << 7) + ls[0], x1 = (((hs[1] << 7) + ms[1]) << 7) + ls[1];
    return (half_bits_to_f32(B.d) * X.s) * fmaf(c1, (float)x1, c0 * (float)x0);
}

template <int R, int NW, int STEPS>
__global__ __launch_bounds__(NW * 64) void q6r_gemv_kernel(Q6kParams p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // timeline build (tag 0): slots 0 entry, 1 loads issued, 2 vector staged, 3 barrier passed, 4 first row done, 5 last row stored, 6 acknowledged
    // (every fourth workgroup leaves records: 2048 workgroups of 8 waves are more than the buffer holds)
    const int sw = (blockIdx.x & 3) ? kStampWaves : (int)(blockIdx.x >> 2) * NW + wave;
    (void)sw;
    KSH_STAMP_BEGIN
    const int bl = lane >> 3;
    const int cols = p.bpr * 256;
    const size_t row_bytes = q6r_row_bytes(p.bpr);
    const int w0 = (blockIdx.x * NW + wave) * p.rows_per_wave;
    const int w1 = min(w0 + p.rows_per_wave, p.rows);

    Q6rLane cur[STEPS][R], nxt[STEPS][R];
    auto load_rows = [&](Q6rLane (&dst)[STEPS][R], int row0) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint8_t *rp = p.W + (size_t)min(row0 + r, p.rows - 1) * row_bytes;
#pragma unroll
            for (int s = 0; s < STEPS; s++) dst[s][r] = q6r_load(rp, p.bpr, min(s * 8 + bl, p.bpr - 1), lane);   // past the row's end: the last superblock again, against a zero scale
        }
    };
    constexpr int KMAX = (STEPS * 512 + NW * 64 - 1) / (NW * 64);   // float4 of the vector per thread: cols == STEPS * 2048
    StageRegs sr;
    stage_fetch<NW * 64, false, KMAX>(p.pro, cols, sr);
    load_rows(cur, min(w0, p.rows - 1));
    KSH_STAMP(1);
    stage_finish<kXQ6, NW * 64, false, KMAX>(p.pro, xs, cols, sr);
    KSH_STAMP(2);
    __syncthreads();
    KSH_STAMP(3);
    if (w0 >= w1) return;

    XQ6r X[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; s++) X[s].load(xs, min(s * 8 + bl, p.bpr - 1), lane, s * 8 + bl < p.bpr);

    for (int row0 = w0; row0 < w1; row0 += R) {
        load_rows(nxt, min(row0 + R, p.rows - 1));
#pragma unroll
        for (int r = 0; r < R; r++) {
            float acc = 0.f;
#pragma unroll
            for (int s = 0; s < STEPS; s++) acc += q6r_lane_dot(cur[s][r], lane, X[s]);
            acc = wave_sum(acc);
            if (lane == 0 && row0 + r < w1) p.y[row0 + r] = acc;
        }
        if (row0 == w0) KSH_STAMP(4);
#pragma unroll
        for (int s = 0; s < STEPS; s++)
#pragma unroll
            for (int r = 0; r < R; r++) cur[s][r] = nxt[s][r];
    }
    KSH_STAMP(5);
    KSH_STAMP_FLUSH(0, sw, 6);
}

// ---- Q6_K: blocks in file order (210 bytes, at 2-byte addresses) --------------
// Streamed by way of LDS: a wave asks for G rows' bytes as whole 16-byte pieces at 16-byte addresses, NBUF such groups ahead,
// and reads its lanes' fields from there.  What bounds it: the stream of the weights, 6.3 TB/s at 440 MB in a trace, which is what flat
// 16-byte loads reach, with 85 vector instructions a step of eight superblocks (half of the stream's time) beside it.  Before,
// lanes loaded their fields from memory: 80 cache lines touched a row instead of 14, a row of 1280 bytes or of 512 paid
// for whole steps of eight superblocks, and the registers for a row's loads held rows of more than 4096 columns to one wave a
// SIMD.  (Before -> now, cold, us) 262144 x 2048 99.7 -> 69.5, 262144 x 1536 94.5 -> 63.1, 200000 x 2560 143.6 -> 69.7, 100000 x
// 4096 84.8 -> 55.8, 16384 x 8192 59.6 -> 23.2, 14682 x 512 9.4 -> 3.9; below some 5 MB both are the rate of launches.
//
// Regrouped rows of 1536, 2048 and 4096 columns go the same way (ROWS): their fields lie at aligned places, 16 bytes a lane side by side.
//
// Superblocks past the last whole step (TAIL): G rows share one more step, which bpr % 8 groups of lanes each fill with their row's.

// A lane's share of one superblock in LDS, as it lies there: 16 bytes of ql and of qh with the two behind them, two scales, d.
struct Q6sLane {
    uint32_t a[5], b[5], d;
    uint32_t ash, bsh;      // bits in front of the lane's bytes, and in front of its quadrants' pair of bits
    int c0, c1;
};

__device__ __forceinline__ Q6sLane q6s_take(uint32_t at, int lane)
{
    typedef const __attribute__((address_space(3))) uint32_t *W32;
    const int j = lane & 7, ip = j >> 2;
    const uint32_t w = at & ~3u;
    const W32 q = (W32)(uintptr_t)(w + 16 * j), h = (W32)(uintptr_t)(w + (128 + 32 * ip + 16 * (j & 1)));
    Q6sLane r;
#pragma unroll
    for (int i = 0; i < 5; i++) { r.a[i] = q[i]; r.b[i] = h[i]; }
    const uint32_t sc = at + (uint32_t)(8 * ip + 2 * ((j >> 1) & 1) + (j & 1));
    lds_ask_signed<192>(r.c0, sc);
    lds_ask_signed<196>(r.c1, sc);
    r.d = *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)(at + 208);
    r.ash = at << 3;                                      // (the shift takes its low five bits: 16 at the odd places)
    r.bsh = (at << 3) + (uint32_t)(lane & 2);
    return r;
}

// the low nibble of every byte of a, the high one of b: one instruction (the compiler makes two of the expression)
__device__ __forceinline__ uint32_t low_nibbles_of(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(0x0F0F0F0Fu), "v"(a), "v"(b));
    return r;
}
// of 16 bytes of ql and of qh, the quadrants' pairs in bits 0..1 and 4..5 of the latter
__device__ __forceinline__ float q6s_dot_of(const uint32_t (&ql)[4], const uint32_t (&qh)[4], int c0, int c1, uint32_t d, const XQ6r &X)
{
    uint32_t v[2][4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const uint32_t l = ql[w], t = qh[w] & 0x33333333u;
        v[0][w] = low_nibbles_of(l, t << 4);      // low nibbles with the bits 0..1 of every byte's two pairs, high ones with 4..5
        v[1][w] = low_nibbles_of(l >> 4, t);
    }
    // the digits' sums one behind the other, each begun from 128 times the one before: 128 (128 h + m) + l - 32 sum(X)
    int x[2] = {0, 0};
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
        for (int q = 0; q < 2; q++) x[q] = __builtin_amdgcn_sdot4((int)v[q][w], (int)X.H[q][w], x[q], false);
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
        for (int q = 0; q < 2; q++) x[q] = __builtin_amdgcn_sdot4((int)v[q][w], (int)X.M[q][w], w ? x[q] : x[q] << 7, false);
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
        for (int q = 0; q < 2; q++) x[q] = __builtin_amdgcn_sdot4((int)v[q][w], (int)X.L[q][w], w ? x[q] : (x[q] << 7) + X.nsx5[q], false);
    const int x0 = x[0], x1 = x[1];
    return (half_bits_to_f32(d) * X.s) * fmaf((float)c1, (float)x1, (float)c0 * (float)x0);
}
__device__ __forceinline__ float q6s_dot(const Q6sLane &B, const XQ6r &X)
{
    uint32_t l[4], t[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        l[w] = __builtin_amdgcn_alignbit(B.a[w + 1], B.a[w], B.ash);
        t[w] = __builtin_amdgcn_alignbit(B.b[w + 1], B.b[w], B.bsh);
    }
    return q6s_dot_of(l, t, B.c0, B.c1, B.d, X);
}
// The same of superblock blk of a regrouped row at `row` in LDS, whose fields are aligned
__device__ __forceinline__ float q6s_dot_rows(uint32_t row, int bpr, int blk, int lane, const XQ6r &X)
{
    typedef const __attribute__((address_space(3))) u32x4_t *V;
    const int j = lane & 7, ip = j >> 2;
    const u32x4_t a = *(V)(uintptr_t)(row + (uint32_t)(blk * 128 + 16 * j)), b = *(V)(uintptr_t)(row + (uint32_t)(bpr * 128 + blk * 64 + 32 * ip + 16 * (j & 1)));
    const uint32_t sc = row + (uint32_t)(bpr * 192 + blk * 16 + 8 * ip + 2 * ((j >> 1) & 1) + (j & 1));
    int c0, c1;
    lds_ask_signed<0>(c0, sc);
    lds_ask_signed<4>(c1, sc);
    const uint32_t d = *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)(row + (uint32_t)(bpr * 208 + blk * 2));
    uint32_t l[4], t[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        l[w] = a[w];
        t[w] = b[w] >> (lane & 2);
    }
    return q6s_dot_of(l, t, c0, c1, d, X);
}

// bytes of LDS in front of the waves' rings: the vector's image and its sums over up to 16 waves
__host__ __device__ constexpr uint32_t q6s_image_bytes(int cols) { return ((uint32_t)xs_image_bytes<kXQ6>(cols) + 256u + 15u) & ~15u; }

// A: whole steps of eight superblocks a row.  TAIL: a rest behind them.  G: rows taken together.  NL: requests of 1 KB that hold
// G rows.  NBUF: groups on their way.  NW: waves, one workgroup a compute unit.  NT: the weights marked as read once.
// ROWS: regrouped rows, at 16-byte addresses.
template <int A, bool TAIL, int G, int NL, int NBUF, int NW, bool NT, bool ROWS>
__global__ __launch_bounds__(NW * 64) void q6k_stream_kernel(Q6kParams p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sw = (int)blockIdx.x * NW + wave;      // timeline build: as q6r_gemv_kernel's slots
    (void)sw;
    KSH_STAMP_BEGIN
    const int bl = lane >> 3, cols = p.bpr * 256;
    const uint32_t row_bytes = ROWS ? (uint32_t)q6r_row_bytes(p.bpr) : (uint32_t)p.bpr * kQ6kBytes;
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)xs;
    const uint32_t ring = l0 + q6s_image_bytes(cols) + (uint32_t)wave * (NBUF * NL * 1024u);
    // groups of G rows: a run of them to a workgroup, its waves taking them in turn
    const int groups = (p.rows + G - 1) / G;
    const int g0 = (int)((int64_t)groups * blockIdx.x / p.wgs), g1 = (int)((int64_t)groups * (blockIdx.x + 1) / p.wgs);
    const int n = max(0, (g1 - g0 - wave + NW - 1) / NW);
    auto source = [&](int it) __attribute__((always_inline)) { return p.W + (size_t)(g0 + it * NW + wave) * (G * row_bytes); };
    // (the first and the last 16 bytes may begin before the group's first and end behind its last byte)
    auto ask = [&](int it, int buf) __attribute__((always_inline)) {
        const uint8_t *src = source(it);
        const uint32_t low = (uint32_t)(uintptr_t)src & 15u;
        const uint32_t last = (low + (uint32_t)min(G, p.rows - (g0 + it * NW + wave) * G) * row_bytes - 1u) & ~15u;
#pragma unroll
        for (int i = 0; i < NL; i++)
            to_lds16_stream<NT>(src - low, min((uint32_t)(i * 1024) + 16u * (uint32_t)lane, last), ring + (uint32_t)((buf * NL + i) * 1024));
    };

    constexpr int KMAX = ((A + TAIL) * 512 + NW * 64 - 1) / (NW * 64);   // float4 of the vector per thread
    static_assert(KMAX <= kStageP, "the norms' operands of the whole row in registers");
    StageRegs sr;
    stage_fetch<NW * 64, false, KMAX>(p.pro, cols, sr);
    // One group is asked for behind the vector, and the others behind the barrier: a compute unit takes a limited number of requests,
    // and a wave that waits to issue its last keeps all of them from the barrier.  (All groups here -> now, cold, us) 16384 x 2048
    // 8.5 -> 7.25, 8192 x 2048 5.6 -> 4.95, 16384 x 4096 12.9 -> 11.9, 16384 x 8192 25.8 -> 24.6, 60000 x 8192 70.7 -> 68.2, 262144 x
    // 2048 and 1536 the same within a hundredth; 1500 x 8192, whose waves have a row each, 6.6 -> 7.05.
    stage_arrived<KMAX>(sr);
    if (n > 0) ask(0, 0);
    KSH_STAMP(1);
    stage_finish<kXQ6, NW * 64, false, KMAX>(p.pro, xs, cols, sr);
    KSH_STAMP(2);
    __syncthreads();
    KSH_STAMP(3);
#pragma unroll
    for (int i = 1; i < NBUF; i++)
        if (i < n) ask(i, i);
    if (n == 0) return;

    // TAIL: the lane's row of the group and its superblock there.  (Lanes behind the last row take that row's again and are left out.)
    const int rest = TAIL ? p.bpr - 8 * A : 1, trow = bl / rest, tblk = 8 * A + bl % rest;
    const uint32_t tail_row = (uint32_t)min(trow, G - 1) * row_bytes, tail_off = tail_row + (uint32_t)tblk * kQ6kBytes;
    XQ6r X[A + TAIL];
#pragma unroll
    for (int s = 0; s < A; s++) X[s].load(xs, 8 * s + bl, lane, true);
    if (TAIL) X[A].load(xs, tblk, lane, true);

    // results, kept until there is one for every lane: pairs of rows in half a wave each, single rows in all of it
    constexpr int P = (G + 1) / 2, kHold = G > 1 ? 32 : 64;
    const int slot = lane & (kHold - 1);
    float out = 0.f;
    int held = 0, stored = 0, buf = 0;
    for (int it = 0; it < n; it++) {
        // (a store on its way counts among the younger requests: the wait is then for more than this group)
        static_assert(NBUF <= 4, "one case for every number of younger groups");
        switch (min(NBUF - 1, n - 1 - it)) {
        case 0: memory_left<0>(); break;
        case 1: memory_left<NL>(); break;
        case 2: memory_left<2 * NL>(); break;
        default: memory_left<3 * NL>(); break;
        }
        const uint32_t at = ring + (uint32_t)(buf * NL * 1024) + (ROWS ? 0u : (uint32_t)(uintptr_t)source(it) & 15u);
        float acc[G], tail = 0.f;
#pragma unroll
        for (int r = 0; r < G; r++) {
            acc[r] = 0.f;
#pragma unroll
            for (int s = 0; s < A; s++) {
                const float d = ROWS ? q6s_dot_rows(at + (uint32_t)r * row_bytes, p.bpr, 8 * s + bl, lane, X[s])
                                     : q6s_dot(q6s_take(at + (uint32_t)r * row_bytes + (uint32_t)((8 * s + bl) * kQ6kBytes), lane), X[s]);
                acc[r] = s ? acc[r] + d : d;
            }
        }
        if (TAIL) tail = ROWS ? q6s_dot_rows(at + tail_row, p.bpr, tblk, lane, X[A]) : q6s_dot(q6s_take(at + tail_off, lane), X[A]);
        lds_left<0>();               // the group's bytes are in registers: its place can be asked for again
        if (it + NBUF < n) ask(it + NBUF, buf);
        buf = buf + 1 == NBUF ? 0 : buf + 1;
        if (TAIL) {
#pragma unroll
            for (int r = 0; r < G; r++) acc[r] += trow == r ? tail : 0.f;
        }
        float v[P];
        rows_sum<G>(acc, v);
#pragma unroll
        for (int k = 0; k < P; k++) {
            out = slot == held ? v[k] : out;
            held++;
        }
        if (held == kHold || it + 1 == n) {
            const int q = stored + slot, row = (g0 + (q / P) * NW + wave) * G + (G > 1 ? 2 * (q % P) + (lane >> 5) : 0);
            if (slot < held && row < p.rows) p.y[row] = out;
            stored += kHold;
            held = 0;
        }
        if (it == 0) KSH_STAMP(4);
    }
    KSH_STAMP(5);
    KSH_STAMP_FLUSH(0, sw, 6);
}

// The form for rows of bpr superblocks: 16 waves where four groups of up to 2 KB, or two of 4, fit beside the vector's image;
// 12 and 8 where the groups are larger (2560 columns: 12 waves 28.6 us, 8 with three groups 29.8, 16 with single rows of 3 KB
// 29.5; 53147 rows, with the argmax).
struct Q6sForm {
    int G, NL, NBUF, NW;
    size_t lds(int cols) const { return q6s_image_bytes(cols) + (size_t)NBUF * NL * 1024 * NW; }
};
template <class F>
auto q6s_with_form(int bpr, F f)
{
#define KSH_FORM(a, t, g, nl, nbuf, nw) \
    f(std::integral_constant<int, a>{}, std::integral_constant<bool, t>{}, std::integral_constant<int, g>{}, std::integral_constant<int, nl>{}, std::integral_constant<int, nbuf>{}, std::integral_constant<int, nw>{})
    if (bpr == 1) return KSH_FORM(0, true, 8, 2, 4, 16);
    if (bpr == 2) return KSH_FORM(0, true, 4, 2, 4, 16);
    if (bpr < 5) return KSH_FORM(0, true, 2, 2, 4, 16);
    if (bpr < 8) return KSH_FORM(0, true, 1, 2, 4, 16);
    if (bpr == 8) return KSH_FORM(1, false, 2, 4, 2, 16);
    if (bpr < 13) return KSH_FORM(1, true, 2, 5, 2, 12);
    if (bpr < 16) return KSH_FORM(1, true, 1, 4, 2, 16);
    if (bpr == 16) return KSH_FORM(2, false, 1, 4, 2, 16);
    if (bpr < 24) return KSH_FORM(2, true, 1, 5, 2, 12);
    if (bpr == 24) return KSH_FORM(3, false, 1, 5, 2, 12);
    if (bpr < 32) return KSH_FORM(3, true, 1, 7, 2, 8);
    return KSH_FORM(4, false, 1, 7, 2, 8);
#undef KSH_FORM
}
Q6sForm q6s_form(int bpr)
{
    return q6s_with_form(bpr, [](auto, auto, auto g, auto nl, auto nbuf, auto nw) { return Q6sForm{g, nl, nbuf, nw}; });
}
// Marked as read once from 128 MB on.  A matrix that the memory-side cache (256 MB) keeps from one call to the next is better off
// there: 32768 x 2048 (55 MB), three in turn, 11.2 us or, marked, 13.7; 65536 x 2048 (110 MB) 22.0 or 20.5 with three in turn and
// 19.0 or 22.3 alone; 131072 x 2048 (220 MB) 41.8 or 36.3, alone 33.9 or 35.2; 262144 x 2048 80.4 or 69.5, alone 80.0 or 68.6.
constexpr size_t kQ6sReadOnce = (size_t)128 << 20;

int launch_q6k_stream(const Q6kParams &p, bool by_rows, unsigned grid, size_t lds, hipStream_t st)
{
    const bool once = (size_t)p.rows * p.bpr * kQ6kBytes >= kQ6sReadOnce;
    q6s_with_form(p.bpr, [&](auto a, auto t, auto g, auto nl, auto nbuf, auto nw) {
        auto go = [&](auto nt) {
            // (regrouped rows: of 6, 8 and 16 superblocks)
            if constexpr (t ? a == 0 && g == 1 : a <= 2) {
                if (by_rows) {
                    hipLaunchKernelGGL((q6k_stream_kernel<a, t, g, nl, nbuf, nw, nt, true>), dim3(grid), dim3(nw * 64), lds, st, p);
                    return;
                }
            }
            hipLaunchKernelGGL((q6k_stream_kernel<a, t, g, nl, nbuf, nw, nt, false>), dim3(grid), dim3(nw * 64), lds, st, p);
        };
        if (once) go(std::true_type{});
        else go(std::false_type{});
        return 0;
    });
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "q6k_stream launch");
}

// Whether regrouped rows whose schedule is left open are streamed.  (q6r_gemv_kernel and here, cold, us) 262144 x 2048 75.7 and 68.9, x 4096
// 155.5 and 134.9; 65536 x 2048 28.0 and 23.3, 32768 x 1536 14.9 and 12.0, 16384 x 2048 12.2 and 7.7, x 4096 28.1 and 12.9, 8192 x 2048 6.6
// and 5.3, x 1536 6.2 and 5.1, 4096 x 2048 4.5 and 4.1, x 4096 7.7 and 6.2, x 1536 4.4 and 4.1, 3000 x 2048 4.4 and 3.9; below, where a
// workgroup has few rows to stage the vector for, 2048 x 4096 4.5 and 4.9, x 1536 3.3 and 3.7, 1000 x 2048 3.15 and 3.4.  Rows of 1536 columns,
// six of eight lane groups at work and requests of 2048 bytes for 1264, gain less the longer the stream: 65536 rows 22.2 and 19.7, 131072
// 34.0 and 31.7, 200000 51.6 and 46.6, 262144 62.4 and 60.8 (64.2 and 61.1 behind a norm).
bool q6r_streams(int64_t rows) { return rows >= 3000; }

struct Q6kGeom {
    int R, NW, rpw;
};

Q6kGeom pick_geom6(const ksh_sched &s, int rows)
{
    Q6kGeom G;
    G.NW = s.nsg ? (int)s.nsg : 4;
    G.R = s.nr0 ? (int)s.nr0 : 2;
    // rows a wave walks: long enough to amortise the x staging, short enough
    // to leave >= 8 workgroups per CU
    int rpw = s.unroll ? (int)s.unroll * G.R : 16;
    if (!s.unroll) while (rpw > G.R && rows / (rpw * G.NW) < 2048) rpw >>= 1;   // (an explicit count is taken as given)
    if (rpw < G.R) rpw = G.R;
    G.rpw = rpw;
    return G;
}

template <int R, int NW>
int launch_steps(int steps, const Q6kParams &p, unsigned grid, size_t lds, hipStream_t st)
{
    switch (steps) {
    case 1: hipLaunchKernelGGL((q6r_gemv_kernel<R, NW, 1>), dim3(grid), dim3(NW * 64), lds, st, p); break;
    case 2: hipLaunchKernelGGL((q6r_gemv_kernel<(R > 2 ? 2 : R), NW, 2>), dim3(grid), dim3(NW * 64), lds, st, p); break;
    default: return set_error("matvec_q6k: cols=%d is not built for row-grouped weights (1536, 2048 and 4096 are)", p.bpr * 256);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "q6k_gemv launch");
}

int launch_matvec_q6k(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    Q6kParams p{};
    p.W = (const uint8_t *)a.in[0];
    p.y = (float *)a.out[0];
    p.pro.x = (const float *)a.in[1];
    p.pro.eps = k.desc.params[0];
    p.pro.kind = k.desc.kind == KSH_MATVEC ? kPlain : (k.desc.dims[2] ? kAddThenRms : kRms);
    if (p.pro.kind != kPlain) p.pro.w_norm = (const float *)a.in[2];
    if (p.pro.kind == kAddThenRms) {
        p.pro.nwg = __builtin_bit_cast(int, k.desc.params[1] != 0.f ? k.desc.params[1] : 1.0f);   // the stream scale
        p.pro.w_post = (const float *)a.in[3];
        p.pro.res = (const float *)a.in[4];
        p.pro.x_out = (float *)a.out[1];
    }
    p.rows = (int)k.desc.dims[0];
    p.bpr = (int)(k.desc.dims[1] / 256);
    const unsigned grid = k.info.grid[0];
    const size_t lds = k.info.lds_bytes;
    p.wgs = (int)grid;
    if (!k.variant) return launch_q6k_stream(p, k.desc.dtypes[0] == KSH_Q6K_ROWS, grid, lds, st);
    const int R = k.variant & 0xFF, NW = (k.variant >> 8) & 0xFF;
    p.rows_per_wave = k.variant >> 16;
    const int steps = (p.bpr + 7) / 8;
#define KSH_CASE(r, w) \
    if (R == r && NW == w) return launch_steps<r, w>(steps, p, grid, lds, st);
    KSH_CASE(1, 4) KSH_CASE(2, 4) KSH_CASE(4, 4)
    KSH_CASE(1, 2) KSH_CASE(2, 2) KSH_CASE(4, 2)
    KSH_CASE(1, 8) KSH_CASE(2, 8) KSH_CASE(4, 8)
#undef KSH_CASE
    return set_error("matvec_q6k: no instance for nr0=%d nsg=%d", R, NW);
}

}  // namespace

int bind_matvec_q6k(ksh_kernel &k)
{
    const int64_t rows = k.desc.dims[0], cols = k.desc.dims[1];
    const bool pro = k.desc.kind == KSH_RMSNORM_MATVEC, has_res = pro && k.desc.dims[2] != 0;
    if (k.desc.kind != KSH_MATVEC && !pro) return set_error("matvec_q6k: kind %d is not built for Q6_K weights", k.desc.kind);
    if (rows <= 0 || rows > (1 << 30)) return set_error("matvec: rows=%lld", (long long)rows);
    if (cols <= 0 || cols % 256 || cols > 8192)
        return set_error("matvec_q6k: cols=%lld is not a positive multiple of 256 up to 8192", (long long)cols);
    const bool by_rows = k.desc.dtypes[0] == KSH_Q6K_ROWS;
    if (by_rows && cols != 1536 && cols != 2048 && cols != 4096)
        return set_error("matvec_q6k: row-grouped weights are built for 1536, 2048 and 4096 columns (got %lld)", (long long)cols);
    const int bpr = (int)(cols / 256);
    const Q6sForm form = q6s_form(bpr);
    // (file order has one kernel for a row length: a schedule that names it, as its handle reports it, or one of those that are
    // built for regrouped rows is taken for it; regrouped rows are streamed by a schedule that names it)
    ksh_sched sched = k.desc.sched;
    const bool named = sched.nsg == (uint32_t)form.NW && sched.nr0 == (uint32_t)form.G && sched.unroll == (uint32_t)form.NBUF;
    if (named) sched = ksh_sched{};
    Q6kGeom G = pick_geom6(sched, (int)rows);
    const bool stream = !by_rows || named || (sched_is_zero(sched) && q6r_streams(rows));
    if (by_rows && sched_is_zero(sched)) {   // measured best on 262144 x 2048
        G.NW = 8;
        G.R = 1;
        G.rpw = 16;
        while (G.rpw > 1 && rows / (G.rpw * G.NW) < 2048) G.rpw >>= 1;
    }
    // keeps the double buffer and the digit planes in registers
    if (cols > 4096) { G.rpw = G.rpw / G.R; G.R = 1; }
    else if (cols > 2048 && G.R > 2) { G.rpw = G.rpw / G.R * 2; G.R = 2; }
    if (!((G.R == 1 || G.R == 2 || G.R == 4) && (G.NW == 2 || G.NW == 4 || G.NW == 8)) || G.rpw % G.R || G.rpw > 32767)
        return set_error("matvec_q6k: unsupported schedule nr0=%d nsg=%d unroll=%u", G.R, G.NW, k.desc.sched.unroll);
    // (the streaming kernel holds the norms' operands of every length in registers, whatever the schedule that stands for it)
    if (pro && !stream && cols > (int64_t)4 * G.NW * 64 * kStageP)
        return set_error("rmsnorm_matvec requires LOCAL staging of the vector (cols=%lld too large)", (long long)cols);
    k.info.n_inputs = pro ? (has_res ? 5 : 3) : 2;
    k.info.n_outputs = has_res ? 2 : 1;
    k.in_bytes[0] = by_rows ? (size_t)rows * q6r_row_bytes(bpr) : (size_t)rows * bpr * kQ6kBytes;
    k.in_align[0] = by_rows ? 16 : 2;
    for (int i = 1; i < k.info.n_inputs; i++) { k.in_bytes[i] = (size_t)cols * 4; k.in_align[i] = 16; }
    k.out_bytes[0] = (size_t)rows * 4;
    k.out_align[0] = 4;
    if (has_res) { k.out_bytes[1] = (size_t)cols * 4; k.out_align[1] = 16; }
    k.info.sched = k.desc.sched;
    k.info.sched.vec = 3;
    k.info.sched.k_split = 1;
    const char *pre = pro ? (has_res ? "addrms_" : "rms_") : "";
    if (!stream) {
        const int rows_per_wg = G.rpw * G.NW;
        set_launch(k, (uint32_t)((rows + rows_per_wg - 1) / rows_per_wg), 1, 1, (uint32_t)G.NW * 64, (uint32_t)xs_bytes<kXQ6>((int)cols));
        k.info.sched.nsg = (uint32_t)G.NW;
        k.info.sched.nr0 = (uint32_t)G.R;
        k.info.sched.unroll = (uint32_t)(G.rpw / G.R);
        set_name(k, "%smatvec_q6krows_r%d_w%d_u%d", pre, G.R, G.NW, G.rpw / G.R);
        k.variant = G.R | (G.NW << 8) | (G.rpw << 16);
    } else {
        set_launch(k, (uint32_t)std::min<int64_t>(256, (rows + form.G - 1) / form.G), 1, 1, (uint32_t)form.NW * 64, (uint32_t)form.lds((int)cols));
        k.info.sched.nsg = (uint32_t)form.NW;
        k.info.sched.nr0 = (uint32_t)form.G;
        k.info.sched.unroll = (uint32_t)form.NBUF;
        set_name(k, "%smatvec_q6k%s_stream_g%d_w%d_n%d", pre, by_rows ? "rows" : "", form.G, form.NW, form.NBUF);
    }
    k.info.sched.tg = 64ull * k.info.sched.nsg;
    k.launch = launch_matvec_q6k;
    return 0;
}

int matvec_q6k_candidates(const ksh_kernel_desc &d, ksh_sched *out, int cap)
{
    int n = 0;
    const int64_t cols = d.dims[1];
    // the streaming kernel: file order's one form, and one of regrouped rows'
    if (n < cap && cols > 0 && cols % 256 == 0 && cols <= 8192) {
        const Q6sForm form = q6s_form((int)(cols / 256));
        ksh_sched s{};
        s.nsg = (uint32_t)form.NW; s.tg = 64ull * s.nsg; s.vec = 3; s.unroll = (uint32_t)form.NBUF; s.nr0 = (uint32_t)form.G; s.k_split = 1;
        out[n++] = s;
    }
    if (d.dtypes[0] == KSH_Q6K) return n;
    for (uint32_t nsg : {2u, 4u, 8u})
        for (uint32_t nr0 : {1u, 2u, 4u})
            for (uint32_t unroll : {2u, 8u}) {
                if (n >= cap) return n;
                ksh_sched s{};
                s.tg = 64ull * nsg; s.vec = 3; s.unroll = unroll; s.nsg = nsg; s.nr0 = nr0; s.k_split = 1;
                out[n++] = s;
            }
    return n;
}

}  // namespace ksh
