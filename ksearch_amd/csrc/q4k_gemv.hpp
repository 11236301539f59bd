// The kernels of the Q4_K GEMV family and their launches (matvec_q4k.hip explains them); a header because they are
// built twice: over f32 activations there, over the caller's half buffers (H) in matvec_q4k_half.hip.
#pragma once
#include "gemv_prologue.hpp"
#include "ksh_internal.hpp"
#include "q4k_lane.hpp"

KSH_STAMP_BUFFER

namespace ksh {

// One launch covers up to three weight matrices that share the input vector.
//   mode 0: the matrices are independent row ranges (plain GEMV: one; QKV:
//           three).  Every wave owns RPW consecutive rows of ONE matrix.
//   mode 1: gate || up: every wave owns the same RPW rows of W[0] and W[1] and
//           stores gelu(W0.x) * (W1.x).
// (Named fields, not arrays: a run-time index into a by-value kernel argument
// makes the compiler copy the whole struct to scratch memory.)
struct MatvecParams {
    const uint8_t *W0, *W1, *W2;
    float *y0, *y1, *y2;
    int rows0, rows1, rows2;
    int waves0, waves1, waves2;   // waves assigned to each matrix (mode 0)
    Prologue pro;
    int bpr;                      // superblocks per row (cols / 256)
    int mode;
};

// ... as the launch passes them: a launch from a stream costs the host 2.7 us while its arguments take no more than 112 bytes, 3.4
// beyond, in a loop of launches that do nothing (4096 x 4096, a call after the other: 3.7 to 4.1 us by the process with the 136 bytes of the
// fields one by one, so 3.6 to 3.9).  What follows from the rest is left out: the second and the third matrix have the same rows, and a matrix's waves
// follow from its rows.
struct MatvecArgs {
    const uint8_t *W0, *W1, *W2;
    float *y0, *y1, *y2;
    const float *x, *w_norm, *w_post, *res;
    float *x_out;
    int rows0, rows1;
    float eps;
    int nwg;
    uint32_t shape;               // bpr | prologue kind << 16 | hd_log2 << 20 | mode << 28
    int wgs;                      // q4k_stream_kernel: workgroups
};
static_assert(sizeof(MatvecArgs) <= kArgBytes, "a launch's arguments");
inline MatvecArgs pack_params(const MatvecParams &p)
{
    return MatvecArgs{p.W0, p.W1, p.W2, p.y0, p.y1, p.y2, p.pro.x, p.pro.w_norm, p.pro.w_post, p.pro.res, p.pro.x_out, p.rows0, p.rows1, p.pro.eps, p.pro.nwg,
                      (uint32_t)p.bpr | (uint32_t)p.pro.kind << 16 | (uint32_t)p.pro.hd_log2 << 20 | (uint32_t)p.mode << 28, 0};
}

struct Q4kGeom {
    int R, NW, var;
    bool half, stream = false;    // stream: q4k_stream_kernel (the other fields are then not its)
    int rpw() const { return R * (half ? 2 : 1); }   // rows per wave
};

// the same launch over half activations (matvec_q4k_half.hip); false: no half instance for the schedule
bool q4k_gemv_half_built(const Q4kGeom &G);
int launch_q4k_gemv_half(const Q4kGeom &G, int nm, const MatvecParams &p, int total_waves, hipStream_t st);
int launch_q4k_stream_half(int nm, const MatvecParams &p, unsigned grid, hipStream_t st);

namespace {

// timeline build: one record set per decode-step shape -- tag = prologue kind * 2 + (two matrices per wave)
// slots: 0 entry, 1 every load issued, 2 vector staged, 3 barrier passed, 4 inner products done, 5 stores issued, 6 stores acknowledged,
//        7 (half-wave form) the vector's loads issued, in front of the barrier that holds the weight loads back
#define KSH_GEMV_TAG(p, NM) ((p).pro.kind * 2 + ((NM) - 1))

// Kernel arguments are fetched with scalar loads where they are first used;
// left alone the compiler sinks each into the branch that needs it, and a wave
// then pays one scalar-cache round trip after another before its first weight
// load.  Copying the fields through two opaque statements at the top turns
// that into a few wide loads and two waits.
// RPW: rows per wave.
template <int RPW>
__device__ __forceinline__ MatvecParams fetch_params(const MatvecArgs &p)
{
    const uint8_t *W0 = p.W0, *W1 = p.W1, *W2 = p.W2;
    float *y0 = p.y0, *y1 = p.y1, *y2 = p.y2;
    int rows0 = p.rows0, rows1 = p.rows1;
    const float *x = p.x, *w_norm = p.w_norm, *w_post = p.w_post, *res = p.res;
    float *x_out = p.x_out;
    int eps = __float_as_int(p.eps), nwg = p.nwg;
    uint32_t shape = p.shape;
    asm volatile("" : "+s"(W0), "+s"(W1), "+s"(W2), "+s"(y0), "+s"(y1), "+s"(y2), "+s"(rows0), "+s"(rows1));
    asm volatile("" : "+s"(x), "+s"(w_norm), "+s"(w_post), "+s"(res), "+s"(x_out), "+s"(eps), "+s"(nwg), "+s"(shape));
    MatvecParams q;
    q.W0 = W0; q.W1 = W1; q.W2 = W2;
    q.y0 = y0; q.y1 = y1; q.y2 = y2;
    q.rows0 = rows0; q.rows1 = q.rows2 = rows1;
    q.waves0 = (rows0 + RPW - 1) / RPW;
    q.waves1 = q.waves2 = (rows1 + RPW - 1) / RPW;
    q.pro.x = x; q.pro.w_norm = w_norm; q.pro.w_post = w_post; q.pro.res = res; q.pro.x_out = x_out;
    q.pro.eps = __int_as_float(eps); q.pro.nwg = nwg;
    q.bpr = (int)(shape & 0xFFFFu);
    q.pro.kind = (int)(shape >> 16 & 0xFu);
    q.pro.hd_log2 = (int)(shape >> 20 & 0xFFu);
    q.mode = (int)(shape >> 28);
    return q;
}

struct WaveTask {
    const uint8_t *W0, *W1;
    float *y;
    int row0, rows;    // first row of this wave (or half-wave), rows in its matrix
    bool active;
};

// (by-value arguments: all three are read before the choice, so nothing turns
// this into a choice of address followed by a dependent load)
template <class T>
__device__ __forceinline__ T sel3(bool in1, bool in2, T a0, T a1, T a2)
{
    return in2 ? a2 : in1 ? a1 : a0;
}

// maps a global wave index onto (matrix, first row).  rpw = rows per wave.  The
// index must live in scalar registers (readfirstlane): the matrix is then
// picked with scalar loads of the kernel arguments instead of a per-lane
// gather from them, which would put a memory round trip in front of every load.
template <int NM>
__device__ __forceinline__ WaveTask wave_task(const MatvecParams &p, int wv, int rpw)
{
    WaveTask t;
    // one matrix, or a gate | up pair whose waves all own rows of both: nothing to choose between (a scalar branch
    // instead of thirty selects in front of the first weight load)
    if (NM == 2 || (p.waves1 == 0 && p.waves2 == 0)) {
        t.W0 = p.W0;
        t.W1 = p.W1;
        t.y = p.y0;
        t.rows = p.rows0;
        t.row0 = wv * rpw;
        t.active = t.row0 < t.rows;
        if (!t.active) t.row0 = 0;
        return t;
    }
    // selects between already-fetched arguments rather than indexing them
    const bool in1 = p.mode == 0 && wv >= p.waves0;
    const bool in2 = in1 && wv - p.waves0 >= p.waves1;
    if (in1) wv -= p.waves0;
    if (in2) wv -= p.waves1;
    t.W0 = sel3(in1, in2, p.W0, p.W1, p.W2);
    t.W1 = p.W1;
    t.y = sel3(in1, in2, p.y0, p.y1, p.y2);
    t.rows = sel3(in1, in2, p.rows0, p.rows1, p.rows2);
    const int nw = sel3(in1, in2, p.waves0, p.waves1, p.waves2);
    t.row0 = wv * rpw;
    t.active = t.row0 < t.rows && (p.mode == 1 || wv < nw);
    if (!t.active) {   // keeps its loads (so that every wave issues the same number) but points them at row 0
        t.W0 = p.W0;
        t.rows = p.rows0;
        t.row0 = 0;
    }
    return t;
}

// Full-wave form: a wave owns R rows and sweeps 16 superblocks per step.
// NM = 1 (mode 0) or 2 (mode 1).  The weight loads of step s+1 are issued
// before step s is consumed, and step 0's before the input is staged, so the
// first HBM round trip overlaps the prologue.
// MERGE: built with the partition-merging prologue (kept out of every other instance: a longer program in front
// of the first weight load costs 0.1 us at 4096 x 4096)
// CB: superblocks per row when the instance is built for one row length (0: p.bpr); KIND: its prologue kind (-1:
// p.pro.kind).  The instances with both (the plain GEMV over 4096 and 8192 columns) reach their weight loads in a
// fraction of the instructions the general form needs.
template <int R, int NW, int NM, int XF, bool MULTI, bool MERGE, bool H, int CB = 0, int KIND = -1>
__global__ __launch_bounds__(NW * 64) void q4k_gemv_kernel(MatvecArgs p_in)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];
    const MatvecParams p = fetch_params<R>(p_in);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    KSH_STAMP_BEGIN
    const int g = lane & 3, bl = lane >> 2;
    const int bpr = CB ? CB : p.bpr, cols = bpr * 256;
    const size_t row_bytes = (size_t)bpr * kQ4kBytes;
    constexpr int KMAX = CB ? (CB * 64 + NW * 64 - 1) / (NW * 64) : kStageX;   // float4 of the vector per thread
    const WaveTask t = wave_task<NM>(p, blockIdx.x * NW + wave, R);

    const uint8_t *rowp[NM][R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        // rows past the end re-read the last row; their sums are never stored
        const size_t off = (size_t)min(t.row0 + r, t.rows - 1) * row_bytes;
        rowp[0][r] = t.W0 + off;
        if (NM == 2) rowp[NM - 1][r] = t.W1 + off;
    }

    // Every wave and lane issues the same loads, unconditionally (lanes past the
    // row's end re-read its last superblock and drop the product): the wait for
    // the staged vector can then be an exact count that leaves the weight loads
    // in flight, where a conditional load would force a wait for everything.
    // MULTI: rows longer than 16 superblocks take several steps and double-buffer.
    Q4kLane cur[NM][R], nxt[MULTI ? NM : 1][MULTI ? R : 1];
    StageRegs sr;
    constexpr int RPRE = R;   // (splitting the issue as the half-wave form does costs 0.5 us at 4096 x 4096)
    stage_fetch<NW * 64, MERGE, KMAX, KIND, H>(p.pro, cols, sr);
    // The short front reaches its weight loads a few dozen instructions behind the vector's, and loads of different
    // waves share one in-order path per compute unit: without this barrier a wave's vector loads queue behind another
    // wave's HBM-cold weights (vector staged in the slowest wave at 2.3 us instead of 1.7).  The general form's long
    // front keeps the two apart by itself.
    if (CB) __syncthreads();
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int r = 0; r < RPRE; r++) cur[m][r] = q4k_load(rowp[m][r] + (size_t)min(bl, bpr - 1) * kQ4kBytes, g);
    KSH_STAMP(1);
    stage_finish<XF, NW * 64, MERGE, KMAX, KIND, H>(p.pro, xs, cols, sr);
    KSH_STAMP(2);
    __syncthreads();
    KSH_STAMP(3);
    if (!t.active) return;
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int r = RPRE; r < R; r++) cur[m][r] = q4k_load(rowp[m][r] + (size_t)min(bl, bpr - 1) * kQ4kBytes, g);

    float acc[NM][R];
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[m][r] = 0.f;

    for (int b0 = 0; b0 < bpr; b0 += 16) {
        const int b = min(b0 + bl, bpr - 1);
        const bool mine = b0 + bl < bpr;
        if (MULTI) {
            const int bn = min(b0 + 16 + bl, bpr - 1);
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int r = 0; r < R; r++) nxt[m][r] = q4k_load(rowp[m][r] + (size_t)bn * kQ4kBytes, g);
        }
        XGroup<XF> X;
        X.load(xs, cols, b, g);
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float v = q4k_group_dot<XF>(cur[m][r], g, X);
                acc[m][r] += mine ? v : 0.f;
            }
        if (MULTI) {
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int r = 0; r < R; r++) cur[m][r] = nxt[m][r];
        }
    }

    KSH_STAMP_USE(acc[NM - 1][R - 1]);
    KSH_STAMP(4);
    // every row is reduced before the first is stored: a store in front of a later row's wait makes that wait one for
    // the store's acknowledgement as well (loads and stores retire in order)
    float res[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        float s[NM];
#pragma unroll
        for (int m = 0; m < NM; m++) s[m] = wave_sum(acc[m][r]);
        res[r] = (NM == 2) ? gelu_mul_f32(s[0], s[NM - 1]) : s[0];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int row = t.row0 + r;
        if (lane == 0 && row < t.rows) act_st<H>(t.y, row, res[r]);
    }
    KSH_STAMP(5);
    KSH_STAMP_FLUSH(KSH_GEMV_TAG(p, NM), blockIdx.x * NW + wave, 6);
}

// Half-wave form for rows of at most 8 superblocks (BPR = 8: 2048 columns, no lane idles; BPR = 6: 1536 columns,
// a quarter of the lanes re-read the row's last superblock and drop the product): lanes 0..31 and 32..63 work
// on different rows, so a wave covers 2R rows in a single step.
template <int R, int NW, int NM, int XF, bool MERGE, int BPR, bool H>
__global__ __launch_bounds__(NW * 64) void q4k_gemv_half_kernel(MatvecArgs p_in)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];
    const MatvecParams p = fetch_params<2 * R>(p_in);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    KSH_STAMP_BEGIN
    const int g = lane & 3, slot = (lane >> 2) & 7, hw = lane >> 5;
    constexpr int bpr = BPR;
    const int bl = BPR == 8 ? slot : min(slot, BPR - 1);
    const bool mine = BPR == 8 || slot < BPR;
    constexpr size_t row_bytes = (size_t)bpr * kQ4kBytes;
    WaveTask t = wave_task<NM>(p, blockIdx.x * NW + wave, 2 * R);
    const int row0 = t.row0 + hw * R;

    Q4kLane L[NM][R];
    StageRegs sr;
    // (the instances that merge attention partitions are launched for that prologue alone: the other kinds' loads
    // and arithmetic are not compiled into them)
    constexpr int KIND = MERGE ? kMergeParts : -1;
    stage_fetch<NW * 64, MERGE, kStageX, KIND, H>(p.pro, bpr * 256, sr);
    // With a normalising prologue every wave's vector loads are queued before any wave's weight loads: behind
    // another wave's HBM-cold weights in the compute unit's memory pipeline they came back up to 1.3 us late, and
    // the prologue's reduction waits for the slowest wave.
    KSH_STAMP(7);
    if (MERGE || p.pro.kind != kPlain) __syncthreads();
    auto load_r = [&](int r) {
        const size_t off = (size_t)min(row0 + r, t.rows - 1) * row_bytes + (size_t)bl * kQ4kBytes;
        L[0][r] = q4k_load(t.W0 + off, g);
        if (NM == 2) L[NM - 1][r] = q4k_load(t.W1 + off, g);
    };
    // Only the first row's loads go out before the input is staged: a compute
    // unit's memory queue is finite, a wave that cannot issue cannot reach the
    // staging barrier either, and one row per half-wave already covers the HBM
    // round trips that the staging takes.  The other rows follow the barrier
    // and stream in while the first is being multiplied (gate || up, 2048 ->
    // 8192 with the add-then-norm prologue: 8.1 -> 7.1 us).
    load_r(0);
    KSH_STAMP(1);
    stage_finish<XF, NW * 64, MERGE, kStageX, KIND, H>(p.pro, xs, bpr * 256, sr);
    KSH_STAMP(2);
    __syncthreads();
    KSH_STAMP(3);
    if (!t.active) return;
#pragma unroll
    for (int r = 1; r < R; r++) load_r(r);

    XGroup<XF> X;
    X.load(xs, bpr * 256, bl, g);

    // (every row is multiplied and reduced before the first is stored, as in the full-wave form)
    float res[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        float s[NM];
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const float v = q4k_group_dot<XF>(L[m][r], g, X);
            const float2 hs = wave_half_sums(mine ? v : 0.f);
            s[m] = hw ? hs.y : hs.x;
        }
        res[r] = (NM == 2) ? gelu_mul_f32(s[0], s[NM - 1]) : s[0];
    }
    KSH_STAMP_USE(res[R - 1]);
    KSH_STAMP(4);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int row = row0 + r;
        if ((lane & 31) == 0 && row < t.rows) act_st<H>(t.y, row, res[r]);
    }
    KSH_STAMP(5);
    KSH_STAMP_FLUSH(KSH_GEMV_TAG(p, NM), blockIdx.x * NW + wave, 6);
}

int waves_for(int rows, int rpw) { return (rows + rpw - 1) / rpw; }

size_t lds_for(int var, int cols) { return var == kXI8 ? xs_bytes<kXI8>(cols) : var == kXI2 ? xs_bytes<kXI2>(cols) : xs_bytes<kXF32>(cols); }

template <int R, int NW, int NM, int XF, bool MERGE, bool H>
void launch_pro(bool half, const MatvecParams &p, unsigned grid, size_t lds, hipStream_t st)
{
    if (half && p.bpr == 8)
        hipLaunchKernelGGL((q4k_gemv_half_kernel<R, NW, NM, XF, MERGE, 8, H>), dim3(grid), dim3(NW * 64), lds, st, pack_params(p));
    else if (half)
        hipLaunchKernelGGL((q4k_gemv_half_kernel<R, NW, NM, XF, MERGE, 6, H>), dim3(grid), dim3(NW * 64), lds, st, pack_params(p));
    // the plain GEMV over 4096 columns, built for that row length (4.25 against 4.35 us at 4096 x 4096; the same for 8192
    // columns -- the down projection -- was slower inside the decode loop, 1111 against 1123 tok/s, and is not built)
    else if (NM == 1 && !MERGE && NW == 8 && R <= 2 && p.pro.kind == kPlain && p.bpr == 16)
        hipLaunchKernelGGL((q4k_gemv_kernel<(R <= 2 ? R : 1), 8, 1, XF, false, false, H, 16, kPlain>), dim3(grid), dim3(NW * 64), lds, st, pack_params(p));
    else if (p.bpr > 16)
        hipLaunchKernelGGL((q4k_gemv_kernel<R, NW, NM, XF, true, MERGE, H>), dim3(grid), dim3(NW * 64), lds, st, pack_params(p));
    else
        hipLaunchKernelGGL((q4k_gemv_kernel<R, NW, NM, XF, false, MERGE, H>), dim3(grid), dim3(NW * 64), lds, st, pack_params(p));
}

template <int R, int NW, int NM, int XF, bool H>
int launch_inst(bool half, const MatvecParams &p, int total_waves, hipStream_t st)
{
    const unsigned grid = (unsigned)((total_waves + NW - 1) / NW);
    const size_t lds = xs_bytes<XF>(p.bpr * 256);
    if (NM == 1 && p.pro.kind == kMergeParts) launch_pro<R, NW, 1, XF, true, H>(half, p, grid, lds, st);
    else launch_pro<R, NW, NM, XF, false, H>(half, p, grid, lds, st);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "q4k_gemv launch");
}

}  // namespace
}  // namespace ksh
