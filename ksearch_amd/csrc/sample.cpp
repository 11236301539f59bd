// Host-side logit sampling for the non-greedy branch of forward_token: soft
// cap, temperature, min-p filter, one multinomial draw.
//
// Mirrors sample_softcap_min_p (crates/ksearch_gemma/src/sample.rs:9-77)
// operation for operation on f32 logits (the reference reads them as f16): the
// same pass structure, the same f32 accumulators, the same splitmix32 draw, so
// that a seed picks the same id.
#include <algorithm>
#include <cmath>
#include <vector>

#include "ksh_internal.hpp"

namespace {

// sample.rs:79-85
uint32_t splitmix32(uint32_t &state)
{
    state += 0x9E3779B9u;
    uint32_t z = state;
    z = (z ^ (z >> 16)) * 0x7feb352du;
    z = (z ^ (z >> 15)) * 0x846ca68bu;
    return z ^ (z >> 16);
}

}  // namespace

namespace ksh {

bool sample_row_params(float temperature, float min_p, SampleRow *out)
{
    if (!(min_p > 0.0f) || !(temperature >= 1e-6f) || !std::isfinite(temperature)) return false;
    // An entry survives when exp((y - best) / temperature) >= min_p.  The margin is far above what the device's and the
    // host's tanh and exp can differ by (an ulp or two of y, of the order of 1e-5 at a soft cap of 30); entries inside
    // it that do not survive are dropped by the exact comparison below.
    out->temperature = temperature;
    out->below = std::fmax(-temperature * std::log(min_p), 0.0f) * 1.001f + 1e-3f + 1e-3f * temperature;
    return true;
}

// Room for `rows` rows of n logits: two lists of (id, logit) per row, then a count and a sum per part.  The sizes say what
// is allocated: after a failure nothing is, and the next call asks again.
int SampleScratch::reserve(int want_rows, int want_n, hipStream_t st)
{
    if (!heads) KSH_HIP(hipHostMalloc((void **)&heads, sizeof(SampleHead) * kSampleMaxRows, hipHostMallocDefault));
    if (rows >= want_rows && n >= want_n) return 0;
    const int r = want_rows > rows ? want_rows : rows, m = want_n > n ? want_n : n;
    if (lists) {
        KSH_HIP(hipStreamSynchronize(st));
        void *old = lists;
        lists = joined = nullptr;
        rows = n = 0;
        KSH_HIP(hipFree(old));
    }
    KSH_HIP(hipMalloc(&lists, (size_t)r * ((size_t)m * 2 * sizeof(SampleCand) + kSampleParts * 8)));
    rows = r;
    n = m;
    return 0;
}

SampleScratch::~SampleScratch()
{
    if (lists) (void)hipFree(lists);
    if (heads) (void)hipHostFree(heads);
}

// ksh_sample_softcap_min_p below on the entries that can survive its filter.  The rest of the vocabulary takes part in
// the result through the denominator alone, which scales every probability and the draw alike.
bool sample_from_candidates(SampleCand *cand, size_t count, float sum, size_t n, float cap, float temperature, float min_p, uint32_t seed,
                            uint32_t *out)
{
    if (!count || count > sample_most((int64_t)n) || !std::isfinite(sum)) return false;
    std::sort(cand, cand + count, [](const SampleCand &a, const SampleCand &b) { return a.id < b.id; });
    uint32_t best_i = 0;
    float best_v = -INFINITY;
    for (size_t i = 0; i < count; i++) {
        const float x = cand[i].logit;
        const float y = cap > 0.0f ? cap * std::tanh(x / cap) : x;
        cand[i].logit = y;
        if (y > best_v) { best_v = y; best_i = cand[i].id; }
    }
    *out = best_i;
    const float inv = 1.0f / std::fmax(sum, 1e-30f);
    float p_max = 0.0f;
    for (size_t i = 0; i < count; i++) {
        const float x = std::exp((cand[i].logit - best_v) / temperature) * inv;
        cand[i].logit = x;
        if (x > p_max) p_max = x;
    }
    const float threshold = p_max * std::fmax(min_p, 0.0f);
    float filtered = 0.0f;
    for (size_t i = 0; i < count; i++) {
        if (cand[i].logit < threshold) cand[i].logit = 0.0f;
        else filtered += cand[i].logit;
    }
    if (filtered <= 1e-9f) return true;
    uint32_t rng = seed | 1u;
    const float r = ((float)splitmix32(rng) / 4294967296.0f) * filtered;
    float cdf = 0.0f;
    for (size_t i = 0; i < count; i++) {
        cdf += cand[i].logit;
        if (r < cdf) { *out = cand[i].id; return true; }
    }
    *out = (uint32_t)(n - 1);
    return true;
}

}  // namespace ksh

extern "C" int ksh_sample_softcap_min_p(const float *logits, size_t n, float cap, float temperature, float min_p, uint32_t seed,
                                        uint32_t *out)
{
    using namespace ksh;
    if (!logits || !n || !out) return set_error("ksh_sample_softcap_min_p: bad arguments");
    uint32_t best_i = 0;
    float best_v = -INFINITY;
    std::vector<float> xs(n);
    for (size_t i = 0; i < n; i++) {
        const float x = logits[i];
        const float y = cap > 0.0f ? cap * std::tanh(x / cap) : x;
        xs[i] = y;
        if (y > best_v) { best_v = y; best_i = (uint32_t)i; }
    }
    *out = best_i;
    if (temperature < 1e-6f) return 0;   // greedy: argmax after the soft cap, lowest index on ties
    float sum = 0.0f;
    for (float &x : xs) {
        x = std::exp((x - best_v) / temperature);
        sum += x;
    }
    const float inv = 1.0f / std::fmax(sum, 1e-30f);
    float p_max = 0.0f;
    for (float &x : xs) {
        x *= inv;
        if (x > p_max) p_max = x;
    }
    const float threshold = p_max * std::fmax(min_p, 0.0f);
    float filtered = 0.0f;
    for (float &x : xs) {
        if (x < threshold) x = 0.0f;
        else filtered += x;
    }
    if (filtered <= 1e-9f) return 0;
    uint32_t rng = seed | 1u;
    const float r = ((float)splitmix32(rng) / 4294967296.0f) * filtered;
    float cdf = 0.0f;
    for (size_t i = 0; i < n; i++) {
        cdf += xs[i];
        if (r < cdf) { *out = (uint32_t)i; return 0; }
    }
    *out = (uint32_t)(n - 1);
    return 0;
}
