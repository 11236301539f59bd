// Shared internals of libksearch_hip: error plumbing, handle structs and the
// per-kind binder table.  Nothing here is part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <string>
#include <vector>

#include "../../include/ksearch_hip.h"

namespace ksh {

int set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
int hip_fail(hipError_t e, const char *what);

#define KSH_HIP(expr)                                            \
    do {                                                         \
        hipError_t _e = (expr);                                  \
        if (_e != hipSuccess) return ::ksh::hip_fail(_e, #expr); \
    } while (0)

// Tokens of one pass of a prompt through the layers (the reference's chunk length counts in the hundreds,
// gemma_prim.rs:16): 2048 while the prompt has as many left, then 1024, then the rest.  At 1024 rows a hidden-wide
// projection is 192 workgroups (1536 x 12288) and a quarter of the compute units has none; at 2048 a second workgroup
// shares half of them (3000 prompt tokens of the checkpoints' layout: 66.0 -> 61.4 ms).
constexpr int kPrefillPass = 2048;
inline int prefill_pass_tokens(int left)
{
    return left >= kPrefillPass ? kPrefillPass : left >= kPrefillPass / 2 ? kPrefillPass / 2 : left;
}

// The kinds of a prompt pass whose schedule says how a row's sums are cut.  The decode loops bind them by the library's own
// rules (schedule tg = all ones), whatever the plan cache holds: a prompt's caches depend neither on the passes its tokens
// were dealt to nor on a plan that a search has left for one of their lengths.
inline bool prompt_kind(int kind) { return kind == KSH_MATVEC_BATCH || kind == KSH_SDPA_BATCH; }

// The prompt tokens of several pool slots in one pass through the layers: n[i] tokens behind slot slots[i]'s sequence
// length, at most kPrefillPass in all, with the bits of passes of their own.  taken[i] tells which slots went along (the
// others, and every slot where fewer than two can, are left to the caller); nonzero with the error set when the pass of
// those failed (rows behind the slots' lengths may then have been written).  The scheduler finds the models' function here (null: no model code is linked in, every slot takes its
// own pass).
using PrefillSlotsFn = int (*)(ksh_gemma4 *m, ksh_kvpool *pool, const int32_t *slots, const uint32_t *const *tokens, const int *n, int count,
                               uint8_t *taken);
extern PrefillSlotsFn g_prefill_slots;

constexpr int kMaxIn = 8;
constexpr int kMaxOut = 4;

// device pointers with the caller's byte offsets already applied
struct LaunchArgs {
    const void *in[kMaxIn];
    void *out[kMaxOut];
};

}  // namespace ksh

struct ksh_buf {
    void *ptr = nullptr;
    size_t bytes = 0;
    std::atomic<int> rc{1};
    ksh_buf *parent = nullptr;   // a view: ptr lies inside the parent's allocation, which the view keeps alive
};

struct ksh_kernel {
    ksh_kernel_desc desc{};
    ksh_kernel_info info{};
    // bytes each binding must provide from its offset on (0 = not checked)
    size_t in_bytes[ksh::kMaxIn] = {};
    size_t out_bytes[ksh::kMaxOut] = {};
    // alignment each binding's device address must have
    uint32_t in_align[ksh::kMaxIn] = {};
    uint32_t out_align[ksh::kMaxOut] = {};
    int variant = 0;
    // device scratch the runtime allocates for the handle after a successful bind
    size_t scratch_bytes = 0;
    void *scratch = nullptr;
    int (*launch)(const ksh_kernel &, const ksh::LaunchArgs &, hipStream_t) = nullptr;
    // the same launch taking half buffers for its activations as they are, where the kernel is built for them
    int (*launch_half)(const ksh_kernel &, const ksh::LaunchArgs &, hipStream_t) = nullptr;
    // a handle with half activations at the boundary (half_boundary.hip): the f32 handle it wraps, which bindings are
    // half, and where their f32 staging lies in `scratch`
    const ksh_kernel *inner = nullptr;
    uint32_t half_in = 0, half_out = 0;
    size_t stage_in[ksh::kMaxIn] = {}, stage_out[ksh::kMaxOut] = {};
};

namespace ksh {
// what entry points outside the runtime's translation unit need of a context
hipStream_t ctx_stream(ksh_ctx *ctx);
int ctx_device(ksh_ctx *ctx);   // the ordinal of the device the context's stream belongs to
// a buffer object over bytes [off, off + bytes) of `parent` (retained until the view is released); nullptr + error when out of range
ksh_buf *buffer_view(ksh_buf *parent, size_t off, size_t bytes);
void ctx_mark_pending(ksh_ctx *ctx);
// half activations at the boundary: whether the kind takes them, and the wrapping of its bound f32 handle
bool half_boundary_kind(const ksh_kernel_desc &d);
int bind_half_boundary(ksh_kernel &k, const ksh_kernel &inner);
// resolves the device address of the static partial-result array of ksh_softcap_argmax_static for the current
// device (called when a context is created, with the context's device current; the entry point then uses the
// address kept for the context's device)
int argmax_static_setup();
// the end of a decode step (glue.hip): argmax over the logits, position update, the next token's embedding row
struct DecodeTail {
    const float *pv; const uint32_t *pi; int nparts;       // filled in by launch_decode_tail
    float *tok, *history; int max_hist;
    float *meta; const float *rope; float *rope_cur; int hd;
    const uint8_t *embd; int dtype; int64_t n_rows; int n; float scale; float *x_out;
};
int launch_decode_tail(const ksh_kernel &k_argmax, const float *logits, DecodeTail t, hipStream_t st);

// The sampled decode step (sample_device.hip, sample.cpp): the entries of a row of logits that can survive its min-p
// filter are gathered on the device, the reference's arithmetic runs on those on the host.
constexpr int kSampleMaxRows = 16, kSampleInline = 126, kSampleParts = 128;
// More candidates than this and the row is read back and walked whole: the host's sort and arithmetic on c of them take
// 0.05 / 1.0 / 2.2 / 10.2 ms at 4096 / 32768 / 65536 / 262144, the walk over all of 262144 entries 2.95.
inline uint32_t sample_most(int64_t n) { return n / 8 > 4096 ? (uint32_t)(n / 8) : 4096u; }
struct SampleRow {
    float temperature;   // 0: a greedy row
    float below;         // candidates lie at most this far below the best soft-capped logit
};
struct SampleCand { uint32_t id; float logit; };
struct SampleHead {
    uint32_t count, best_id;   // candidates (more than kSampleInline: in the device list, up to sample_most), the argmax
    float sum, pad;            // sum over the vocabulary of exp((y - best) / temperature)
    SampleCand cand[kSampleInline];   // in no particular order
};
struct SampleScratch {
    void *lists = nullptr, *joined = nullptr;   // device
    SampleHead *heads = nullptr;                // pinned host memory
    int rows = 0, n = 0;                        // what `lists` holds (0: nothing)
    int reserve(int want_rows, int want_n, hipStream_t st);
    ~SampleScratch();
};
int launch_sample_candidates(SampleScratch &s, const float *logits, int n, int rows, float cap, const float *best_ids, const SampleRow *params,
                             hipStream_t st);
// false: the row takes the whole vocabulary (no min-p filter)
bool sample_row_params(float temperature, float min_p, SampleRow *out);
// one draw; false: the logits are not finite or the candidates too many, and the row takes the whole vocabulary
bool sample_from_candidates(SampleCand *cand, size_t count, float sum, size_t n, float cap, float temperature, float min_p, uint32_t seed,
                            uint32_t *out);
}  // namespace ksh

// a pool's identity for whoever caches things per pool (HIP graphs captured over its buffers): unlike its address,
// never handed out twice
extern "C" uint64_t ksh_kvpool_uid(const ksh_kvpool *p);

// hands a buffer's reference over to a model, which releases it when it is destroyed (the GGUF loader's uploads)
extern "C" void ksh_gemma4_adopt(ksh_gemma4 *m, ksh_buf *b);

namespace ksh {

// block geometry: crates/ksearch_ir/src/lib.rs:52-74, gguf_impl.rs:50-64
inline bool block_spec(int dtype, size_t &elems, size_t &bytes)
{
    switch (dtype) {
    case KSH_F32: elems = 1; bytes = 4; return true;
    case KSH_F16: case KSH_BF16: elems = 1; bytes = 2; return true;
    case KSH_Q40: elems = 32; bytes = 18; return true;
    case KSH_Q4K: elems = 256; bytes = 144; return true;
    case KSH_Q5K: elems = 256; bytes = 176; return true;
    case KSH_Q6K: case KSH_Q6K_ROWS: elems = 256; bytes = 210; return true;
    }
    return false;
}

inline size_t packed_bytes(int dtype, size_t n)
{
    size_t e, b;
    if (!block_spec(dtype, e, b) || n % e) return 0;
    return n / e * b;
}

// Buffers that are there together or not at all: where one cannot be allocated the others are given back and every
// pointer stays null, so that a later call asks for all of them again.  `owned` releases them in the end.
struct BufWant {
    size_t bytes;
    ksh_buf **out;
};
inline int alloc_together(ksh_ctx *ctx, std::vector<ksh_buf *> &owned, std::initializer_list<BufWant> wants)
{
    const size_t had = owned.size();
    for (const BufWant &w : wants) {
        ksh_buf *b = nullptr;
        if (ksh_buffer_alloc(ctx, w.bytes ? w.bytes : 16, nullptr, &b)) {
            for (; owned.size() > had; owned.pop_back()) ksh_buffer_release(owned.back());
            for (const BufWant &u : wants) *u.out = nullptr;
            return 1;
        }
        owned.push_back(b);
        *w.out = b;
    }
    return 0;
}

// A buffer of at least `bytes` that only some calls need: made, or made larger (in steps of 16 MiB), by the first that does.
// Its contents do not survive; nothing that keeps its address (a captured graph) may use it.
inline int grow_buffer(ksh_ctx *ctx, std::vector<ksh_buf *> &owned, size_t bytes, ksh_buf **b)
{
    if (*b && ksh_buffer_size(*b) >= bytes) return 0;
    if (*b) {
        if (ksh_synchronize(ctx)) return 1;
        for (size_t i = 0; i < owned.size(); i++)
            if (owned[i] == *b) { owned.erase(owned.begin() + (long)i); break; }
        ksh_buffer_release(*b);
        *b = nullptr;
    }
    const size_t step = (size_t)16 << 20;
    return alloc_together(ctx, owned, {{(bytes + step - 1) / step * step, b}});
}

inline bool sched_is_zero(const ksh_sched &s)
{
    return s.tg == 0 && s.vec == 0 && s.unroll == 0 && s.nsg == 0 && s.nr0 == 0 && s.k_split == 0 &&
           s.lds_tile == 0;
}

// per-kind binders: validate the descriptor, pick a template instance, fill
// info / sizes / launch.  Return non-zero (with the error set) to refuse.
int bind_matvec(ksh_kernel &k);
int bind_matvec_q4k(ksh_kernel &k);
int bind_matvec_q6k(ksh_kernel &k);
int bind_matvec_q4k_family(ksh_kernel &k);
int bind_matvec_qkv(ksh_kernel &k);
int bind_matvec_gate_up_gelu(ksh_kernel &k);
int bind_matvec_batch(ksh_kernel &k);
int matvec_batch_slices(const ksh_kernel_desc &d, int batch);   // K slices of the tile over `batch` tokens (F32 activations)
// whether a gate and an up matrix of ffn x hidden take the GEMM that leaves gelu(gate) * up (KSH_MATVEC_BATCH, dims[6] = 3)
bool gate_up_pair(int dt_gate, int dt_up, int64_t ffn, int64_t hidden, int64_t batch);
int bind_round_prep(ksh_kernel &k);
int bind_matvec_round(ksh_kernel &k);
int bind_dequant(ksh_kernel &k);
int bind_repack_rows(ksh_kernel &k);
int bind_quantize_k(ksh_kernel &k);
int bind_quantize_q40(ksh_kernel &k);
int bind_sdpa(ksh_kernel &k);
bool sdpa_lanes_supports(int64_t n_q, int64_t n_kv, int64_t hd);
int bind_sdpa_lanes(ksh_kernel &k, int nwg, int n_slots);
int bind_attend_decode(ksh_kernel &k);          // NAIVE, MWG_PART, MWG_REDUCE, SLOTS
int bind_rmsnorm(ksh_kernel &k);       // RMSNORM, RMSNORM_ADD_THEN_RMSNORM
int bind_per_head_qkv_q40(ksh_kernel &k);
int bind_glue(ksh_kernel &k);          // COPY_SCALE_INDEXED, GELU_MUL, COPY_SLICE
int bind_softcap_argmax(ksh_kernel &k);
int bind_ple_ops(ksh_kernel &k);       // RMSNORM_PER_HEAD, ADD_SCALE, MATVEC_GELU_MUL
int bind_read_floor(ksh_kernel &k);

int plan_dims(const ksh_kernel_desc &d);   // how many leading dims take part in a plan's key
// candidate schedules per kind (BEAM)
int matvec_candidates(const ksh_kernel_desc &d, ksh_sched *out, int cap);

inline void set_name(ksh_kernel &k, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(k.info.name, sizeof(k.info.name), fmt, ap);
    va_end(ap);
}

inline void set_launch(ksh_kernel &k, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, uint32_t lds)
{
    k.info.grid[0] = gx; k.info.grid[1] = gy; k.info.grid[2] = gz;
    k.info.block[0] = bx; k.info.block[1] = 1; k.info.block[2] = 1;
    k.info.lds_bytes = lds;
}

}  // namespace ksh
