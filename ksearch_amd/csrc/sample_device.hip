// The device half of the sampled decode step: what the host sampler (sample.cpp) needs of a row of logits.
//
// sample_softcap_min_p (crates/ksearch_gemma/src/sample.rs:9-77) walks the whole vocabulary three times with a tanh
// and an exp per entry, on the host: 3.2 ms for 262144 logits, and the row has to be read back first.  After its
// min-p filter only entries within temperature * ln(1 / min_p) of the best one can be drawn, a handful of a real
// model's distribution.  So the device finds those (with a margin that covers the rounding of its tanh), sums the
// softmax's denominator, and hands the host a few hundred bytes; the host does the reference's arithmetic on them.
//   pass 1  one read of the logits: 128 workgroups per row, each with its own list and its own partial denominator
//   pass 2  one workgroup per row joins the lists behind one another (sums in a fixed order) and writes the row's
//           record straight into pinned host memory; of a row with more candidates than the host takes (sample_most)
//           only the count
// Bound: launch latency (a row is one megabyte at the real vocabulary).  Sixteen requests served with sampling, prompts
// of about 150 tokens and ten tokens of answer each: 552 ms with the whole rows read back and walked on the host, 146 ms
// with the candidates (72 since their prompts share a pass).
#include "ksh_device.hpp"
#include "ksh_internal.hpp"

namespace ksh {
namespace {

constexpr int kParts = kSampleParts, kThreads = 256, kJoinThreads = 512;

struct Rows {
    SampleRow r[kSampleMaxRows];
};

__global__ __launch_bounds__(kThreads) void sample_scan_kernel(const float *__restrict__ logits, int n, float cap, const float *best_ids, Rows rows,
                                                               uint2 *lists, uint32_t *counts, float *sums)
{
    __shared__ uint32_t s_count;
    __shared__ float s_sum[kThreads / 64];
    const int row = blockIdx.y, part = blockIdx.x;
    const SampleRow p = rows.r[row];
    if (!(p.temperature > 0.0f)) {   // a greedy row: its id is the argmax's
        if (threadIdx.x == 0) { counts[row * kParts + part] = 0; sums[row * kParts + part] = 0.0f; }
        return;
    }
    if (threadIdx.x == 0) s_count = 0;
    __syncthreads();
    logits += (size_t)row * n;
    const uint32_t id = (uint32_t)best_ids[row];
    const float xb = logits[id < (uint32_t)n ? id : 0u];
    const float best = cap > 0.0f ? cap * tanhf(xb / cap) : xb, inv_t = 1.0f / p.temperature, cut = best - p.below;
    const int per = (n + kParts - 1) / kParts, i0 = part * per, i1 = min(n, i0 + per);
    uint2 *list = lists + (size_t)row * n + i0;
    float sum = 0.0f;
    for (int i = i0 + threadIdx.x; i < i1; i += kThreads) {
        const float x = logits[i], y = cap > 0.0f ? cap * tanhf(x / cap) : x;
        sum += expf((y - best) * inv_t);
        if (y >= cut) list[atomicAdd(&s_count, 1u)] = make_uint2((uint32_t)i, __float_as_uint(x));
    }
    for (int d = 32; d; d >>= 1) sum += __shfl_xor(sum, d);
    if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        counts[row * kParts + part] = s_count;
        float t = 0.0f;
        for (int w = 0; w < kThreads / 64; w++) t += s_sum[w];
        sums[row * kParts + part] = t;
    }
}

__global__ __launch_bounds__(kJoinThreads) void sample_join_kernel(const float *best_ids, int n, uint32_t most, const uint2 *lists, const uint32_t *counts,
                                                                   const float *sums, uint2 *joined, SampleHead *heads)
{
    __shared__ uint32_t s_at[kParts];
    __shared__ float s_sum[kParts];
    const int row = blockIdx.x, t = threadIdx.x;
    if (t < kParts) {
        s_at[t] = counts[row * kParts + t];
        s_sum[t] = sums[row * kParts + t];
    }
    __syncthreads();
    for (int d = 1; d < kParts; d <<= 1) {   // inclusive prefix sum
        const uint32_t v = t < kParts && t >= d ? s_at[t - d] : 0u;
        __syncthreads();
        if (t < kParts) s_at[t] += v;
        __syncthreads();
    }
    const uint32_t total = s_at[kParts - 1];
    for (int d = kParts / 2; d; d >>= 1) {
        if (t < d) s_sum[t] += s_sum[t + d];
        __syncthreads();
    }
    const int per = (n + kParts - 1) / kParts;
    SampleHead *h = heads + row;
    // entry j of the joined list: in the first part whose prefix sum lies above it
    for (uint32_t j = t; total <= most && j < total; j += kJoinThreads) {
        int part = 0;
        for (int d = kParts / 2; d; d >>= 1)
            if (s_at[part + d - 1] <= j) part += d;
        const uint2 c = lists[(size_t)row * n + (size_t)part * per + (j - (part ? s_at[part - 1] : 0u))];
        if (j < (uint32_t)kSampleInline) { h->cand[j].id = c.x; h->cand[j].logit = __uint_as_float(c.y); }
        if (total > (uint32_t)kSampleInline) joined[(size_t)row * n + j] = c;
    }
    if (t == 0) {
        h->count = total;
        h->best_id = (uint32_t)best_ids[row];
        h->sum = s_sum[0];
    }
}

}  // namespace

// Candidates of `rows` rows of n logits on the stream; best_ids: the rows' argmax (f32, on the device).  The records
// are in s.heads once the stream has been waited for.
int launch_sample_candidates(SampleScratch &s, const float *logits, int n, int rows, float cap, const float *best_ids, const SampleRow *params,
                             hipStream_t st)
{
    if (rows < 1 || rows > kSampleMaxRows || n < 1) return set_error("sample: %d rows of %d logits", rows, n);
    if (s.reserve(rows, n, st)) return 1;
    uint2 *lists = (uint2 *)s.lists;
    s.joined = lists + (size_t)s.rows * n;
    uint32_t *counts = (uint32_t *)((char *)s.lists + (size_t)s.rows * s.n * 16);
    float *sums = (float *)(counts + (size_t)s.rows * kParts);
    Rows r{};
    for (int i = 0; i < rows; i++) r.r[i] = params[i];
    hipLaunchKernelGGL(sample_scan_kernel, dim3(kParts, rows), dim3(kThreads), 0, st, logits, n, cap, best_ids, r, lists, counts, sums);
    hipLaunchKernelGGL(sample_join_kernel, dim3(rows), dim3(kJoinThreads), 0, st, best_ids, n, sample_most(n), lists, counts, sums, (uint2 *)s.joined, s.heads);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "sample launch");
}

}  // namespace ksh
