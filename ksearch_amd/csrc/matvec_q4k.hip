// Q4_K packed-weight GEMV family for gfx950: y = W x, the fused QKV triple and
// the fused gate||up + GELU.
//
// Takes the place of lower_matvec_q4k_coop / lower_matvec_qkv_q4k_coop /
// lower_matvec_gate_up_q4k_coop (crates/ksearch_codegen/src/lower.rs:1763-2082,
// 3343-3462, 2673-2968) and the ksearch_q4k_coop_frag_nr4* bodies
// (crates/ksearch_codegen/src/render.rs:459-607).  Those are 32-lane maps with
// 8 lanes per superblock and 2-byte loads; this one is laid out for wave64 and
// 128-bit loads:
//
//   - a superblock (144 B = 9 x 16 B) is owned by 4 lanes; lane g of the four
//     takes the 64-element group g: its 32 quant bytes (two dwordx4) plus the
//     16-byte header (broadcast across the four lanes by the memory system);
//   - a wave therefore sweeps 16 superblocks (4096 columns) per step, and keeps
//     the matching 64 activations per lane in registers across R rows, so x is
//     read once per R rows;
//   - the activation vector is staged once per workgroup in LDS, either as
//     padded f32 or as three int8 digit planes (gemv_prologue.hpp), optionally
//     after an RMSNorm / add-then-RMSNorm computed by the workgroup itself;
//   - every row's loads are issued before the first use, so one workgroup
//     keeps R * 192 B per lane in flight;
//   - the 6-bit scales/mins are unpacked in registers, the mins are applied
//     through per-sub-block sums of x, and rows are reduced with DPP;
//   - inner product variant 0: nibble -> f32 byte converts + FMAs; variant 3:
//     nibbles unpacked to bytes and v_dot4_i32_i8 against the digit planes
//     (exact integer sums per 32-wide sub-block, one f32 scale per sub-block).
//
// Arithmetic per (row, superblock, group), all f32:
//   acc += d*sc_lo * sum(n_lo*x) + d*sc_hi * sum(n_hi*x) - dmin*(m_lo*Sx_lo + m_hi*Sx_hi)
// which is the reference's coop form (render.rs:506-511) and differs from the
// CPU dequant-then-dot (gguf_impl.rs:690-721 + check_mul_mm.rs:60-71) by
// reassociation only.
#include "q4k_gemv.hpp"
#include "q4k_stream.hpp"

KSH_STAMP_READER(ksh_stamps_matvec_q4k)

namespace ksh {
namespace {

template <int NM, int XF>
int launch_rn(const Q4kGeom &G, const MatvecParams &p, int total_waves, hipStream_t st)
{
#define KSH_CASE(r, w) \
    if (G.R == r && G.NW == w) return launch_inst<r, w, NM, XF, false>(G.half, p, total_waves, st);
    KSH_CASE(1, 4) KSH_CASE(2, 4) KSH_CASE(4, 4)
    KSH_CASE(1, 8) KSH_CASE(2, 8) KSH_CASE(4, 8)
#undef KSH_CASE
    return set_error("q4k gemv: no instance for nr0=%d nsg=%d", G.R, G.NW);
}

template <int NM>
int launch_q4k(const Q4kGeom &G, const MatvecParams &p, int total_waves, hipStream_t st)
{
    return G.var == kXI8 ? launch_rn<NM, kXI8>(G, p, total_waves, st)
         : G.var == kXI2 ? launch_rn<NM, kXI2>(G, p, total_waves, st) : launch_rn<NM, kXF32>(G, p, total_waves, st);
}

// default schedule, from cold-cache timings of the candidate set on the decode
// shapes and the 4096 x 4096 case: 8 waves per workgroup and 2 rows per wave
// where that still leaves ~150 workgroups, else fewer rows, else smaller
// workgroups; int8 dot, except for rows longer than one 16-superblock step,
// where the f32 form is the faster one.
Q4kGeom pick_geom(const ksh_sched &s, int n_mat, int total_rows, int bpr)
{
    Q4kGeom G;
    G.half = (bpr == 8 || bpr == 6);
    G.var = sched_is_zero(s) ? (bpr > 16 ? kXF32 : kXI8) : (s.vec == 3 ? kXI8 : s.vec == 2 ? kXI2 : kXF32);
    if (s.nsg && s.nr0) {
        G.NW = (int)s.nsg;
        G.R = (int)s.nr0;
        return G;
    }
    // 1536-column matrices of 12288 rows and more (the wide feed-forward of the cache-reading layers): 4-wave
    // workgroups, twice as many of them (in the decode loop 1.398 against 1.410 ms per token)
    if (bpr == 6 && total_rows >= 12288 && !s.nsg && !s.nr0) {
        G.NW = 4;
        G.R = 2;
        return G;
    }
    // rows of more than one sweep: a wave's registers hold one of them and what follows it, and two in turn leave the last workgroups
    // alone (r = 2 -> 1, the median of three in turn: 6000 x 4352 10.7 -> 8.6 us, x 8192 10.9 -> 9.8, 16384 x 5120 20.5 -> 18.8, q | k | v of
    // 4096 + 2 x 1024 x 8192 11.7 -> 9.7, gate | up 8192 x 5120, whose two rows of two matrices do not fit the registers, 182 -> 21).  One
    // matrix of 7680 columns and more is a little faster in two rows a wave where their workgroups are a turn over the compute units
    // or fill the last one (r = 1 against 2: 1.01 to 1.06 at 2304 to 4096 rows of 7680 to 15360 columns, 1.02 to 1.035 at 8192, 12288,
    // 16384 and 24576 x 8192).
    const int64_t two = (total_rows + 15) / 16;
    const bool pairs = n_mat == 1 && bpr >= 30 && (two <= 256 || full_turns(two));
    for (int nw : {8, 4})
        for (int r : {2, 1}) {
            if (sched_is_zero(s) && bpr > 16 && r == 2 && !pairs) continue;
            if (s.nsg && (int)s.nsg != nw) continue;
            if (s.nr0 && (int)s.nr0 != r) continue;
            G.NW = nw;
            G.R = r;
            if (total_rows / (nw * G.rpw()) >= 144) return G;
        }
    G.NW = s.nsg ? (int)s.nsg : 4;
    G.R = s.nr0 ? (int)s.nr0 : 1;
    return G;
}

bool geom_ok(const Q4kGeom &G) { return (G.R == 1 || G.R == 2 || G.R == 4) && (G.NW == 4 || G.NW == 8); }

void fill_info(ksh_kernel &k, const Q4kGeom &G, int total_waves, int bpr, const char *base)
{
    set_launch(k, (uint32_t)((total_waves + G.NW - 1) / G.NW), 1, 1, (uint32_t)G.NW * 64,
               (uint32_t)lds_for(G.var, bpr * 256));
    k.info.sched = k.desc.sched;
    k.info.sched.tg = (uint64_t)G.NW * 64;
    k.info.sched.nsg = (uint32_t)G.NW;
    k.info.sched.nr0 = (uint32_t)G.R;
    k.info.sched.vec = (uint32_t)G.var;
    k.info.sched.unroll = 1;
    k.info.sched.k_split = 1;
    set_name(k, "%s_q4k_r%d_w%d_v%d%s", base, G.R, G.NW, G.var, G.half ? "_h" : "");
    k.variant = G.R | (G.NW << 8) | (G.var << 16) | ((int)G.half << 24) | ((int)G.stream << 25);
}

Q4kGeom geom_of(const ksh_kernel &k)
{
    Q4kGeom G;
    G.R = k.variant & 0xFF;
    G.NW = (k.variant >> 8) & 0xFF;
    G.var = (k.variant >> 16) & 0xFF;
    G.half = (k.variant >> 24) & 1;
    G.stream = (k.variant >> 25) & 1;
    return G;
}

// The three shapes (plain / QKV / gate-up), each with an optional normalising
// prologue.  Binding order of inputs: weight matrices, the vector, then for a
// prologue w_norm, and with a residual w_post, res; outputs: the GEMV results,
// then with a residual the new residual stream.
struct Shape {
    int n_mat;        // weight matrices bound
    int nm;           // matrices per wave (2 for gate||up)
    int64_t rows[3];
    int64_t cols;
    int prologue;     // kPlain / kRms / kAddThenRms / kMergeParts
    float eps;
    int nwg, hd;      // kMergeParts
};

Shape shape_of(const ksh_kernel_desc &d)
{
    Shape s{};
    const int64_t *D = d.dims;
    switch (d.kind) {
    case KSH_MATVEC: s.n_mat = 1; s.nm = 1; s.rows[0] = D[0]; s.cols = D[1]; break;
    case KSH_RMSNORM_MATVEC: s.n_mat = 1; s.nm = 1; s.rows[0] = D[0]; s.cols = D[1]; s.prologue = D[2] ? kAddThenRms : kRms; break;
    case KSH_MATVEC_QKV: s.n_mat = 3; s.nm = 1; s.rows[0] = D[0]; s.rows[1] = s.rows[2] = D[1]; s.cols = D[2]; break;
    case KSH_RMSNORM_MATVEC_QKV:
        s.n_mat = 3; s.nm = 1; s.rows[0] = D[0]; s.rows[1] = s.rows[2] = D[1]; s.cols = D[2];
        s.prologue = D[3] ? kAddThenRms : kRms;
        break;
    case KSH_MATVEC_GATE_UP_GELU: s.n_mat = 2; s.nm = 2; s.rows[0] = s.rows[1] = D[0]; s.cols = D[1]; break;
    case KSH_RMSNORM_MATVEC_GATE_UP_GELU:
        s.n_mat = 2; s.nm = 2; s.rows[0] = s.rows[1] = D[0]; s.cols = D[1];
        s.prologue = D[2] ? kAddThenRms : kRms;
        break;
    case KSH_ATTN_MERGE_MATVEC:
        s.n_mat = 1; s.nm = 1; s.rows[0] = D[0]; s.cols = D[1] * D[2]; s.prologue = kMergeParts;
        s.hd = (int)D[2]; s.nwg = (int)D[3];
        break;
    }
    s.eps = d.params[0];
    return s;
}

template <bool H>
int launch_any(const ksh_kernel &k, const LaunchArgs &a, hipStream_t st)
{
    const Q4kGeom G = geom_of(k);
    const Shape s = shape_of(k.desc);
    MatvecParams p{};
    int total = 0;
    const int n_y = s.nm == 2 ? 1 : s.n_mat;
    const uint8_t **W[3] = {&p.W0, &p.W1, &p.W2};
    float **y[3] = {&p.y0, &p.y1, &p.y2};
    int *rows[3] = {&p.rows0, &p.rows1, &p.rows2}, *waves[3] = {&p.waves0, &p.waves1, &p.waves2};
    for (int m = 0; m < s.n_mat; m++) {
        *W[m] = (const uint8_t *)a.in[m];
        *rows[m] = (int)s.rows[m];
        *waves[m] = waves_for(*rows[m], G.rpw());
        if (s.nm == 1) total += *waves[m];
    }
    for (int m = 0; m < n_y; m++) *y[m] = (float *)a.out[m];
    if (s.nm == 2) total = p.waves0;
    p.mode = s.nm == 2 ? 1 : 0;
    p.bpr = (int)(s.cols / 256);
    p.pro.kind = s.prologue;
    p.pro.eps = s.eps;
    p.pro.x = (const float *)a.in[s.n_mat];
    if (s.prologue == kMergeParts) {
        p.pro.w_norm = p.pro.x + (size_t)s.cols * s.nwg;   // the (m, l) pairs follow the values
        p.pro.nwg = s.nwg;
        p.pro.hd_log2 = __builtin_ctz((unsigned)s.hd);
        return H ? launch_q4k_gemv_half(G, 1, p, total, st) : launch_q4k<1>(G, p, total, st);
    }
    if (s.prologue != kPlain) p.pro.w_norm = (const float *)a.in[s.n_mat + 1];
    if (s.prologue == kAddThenRms) {
        p.pro.nwg = __builtin_bit_cast(int, k.desc.params[1] != 0.f ? k.desc.params[1] : 1.0f);   // the stream scale
        p.pro.w_post = (const float *)a.in[s.n_mat + 2];
        p.pro.res = (const float *)a.in[s.n_mat + 3];
        p.pro.x_out = (float *)a.out[n_y];
    }
    if (G.stream) return H ? launch_q4k_stream_half(s.nm, p, k.info.grid[0], st) : launch_q4k_stream<false>(s.nm, p, k.info.grid[0], st);
    if (H) return launch_q4k_gemv_half(G, s.nm, p, total, st);
    return s.nm == 2 ? launch_q4k<2>(G, p, total, st) : launch_q4k<1>(G, p, total, st);
}

}  // namespace

int bind_matvec_q4k_family(ksh_kernel &k)
{
    const Shape s = shape_of(k.desc);
    if (!s.n_mat) return set_error("q4k gemv: kind %d", k.desc.kind);
    if (k.desc.dtypes[0] != KSH_Q4K) return set_error("%d: only Q4_K weights are built for this kind", k.desc.kind);
    if (k.desc.dtypes[1] != KSH_F32 && k.desc.dtypes[1] != 0)
        return set_error("matvec: activation dtype %d is not built (f32 only)", k.desc.dtypes[1]);
    int64_t total_rows = 0;
    for (int m = 0; m < s.n_mat; m++) {
        if (s.rows[m] <= 0 || s.rows[m] > (1 << 30)) return set_error("matvec: rows=%lld", (long long)s.rows[m]);
        total_rows += s.rows[m];
    }
    if (s.cols <= 0 || s.cols % 256) return set_error("Q4_K matvec: cols=%lld is not a positive multiple of 256", (long long)s.cols);
    if (s.cols > 32768) return set_error("Q4_K matvec: cols=%lld does not fit the LDS staging buffer", (long long)s.cols);
    const int bpr = (int)(s.cols / 256);
    // (a schedule that names the streaming form, as its handle reports it, or one that is left open)
    const Q4sForm f = q4s_form(s.nm, bpr);
    ksh_sched sched = k.desc.sched;
    const bool named = s.prologue != kMergeParts && bpr <= kQ4sMost && sched.nsg == (uint32_t)f.NW && sched.nr0 == (uint32_t)f.G &&
                       sched.unroll == (uint32_t)f.NBUF && sched.vec == kXI8;
    if (named) sched = ksh_sched{};
    const int64_t sized_by = s.nm == 2 ? s.rows[0] : total_rows;
    Q4kGeom G = pick_geom(sched, s.n_mat, (int)sized_by, bpr);
    const int64_t half_wgs = (sized_by + G.rpw() * G.NW - 1) / (G.rpw() * G.NW);
    G.stream = named || (sched_is_zero(sched) && s.prologue != kMergeParts && q4s_pays(s.n_mat, sized_by, bpr, half_wgs, G.NW));
    // QKV at one row per half-wave: one dot per lane does not pay for turning the vector into digit planes (3.86 vs 4.08 us)
    if (sched_is_zero(sched) && s.n_mat == 3 && G.half && G.R == 1) G.var = kXF32;
    if (s.prologue == kMergeParts) {
        if (s.hd < 4 || (s.hd & (s.hd - 1)) || s.nwg < 1 || s.nwg > kMergeMaxParts)
            return set_error("attn_merge_matvec: hd=%d must be a power of two, nwg=%d at most %d", s.hd, s.nwg, kMergeMaxParts);
        if (!k.desc.sched.nsg) { G.NW = 8; if (!k.desc.sched.nr0) G.R = 1; }   // one float4 of the merged vector per thread
        if (s.cols > (int64_t)4 * G.NW * 64)
            return set_error("attn_merge_matvec: n_q*hd=%lld exceeds one float4 per thread (%d)", (long long)s.cols, 4 * G.NW * 64);
    }
    if (lds_for(G.var, (int)s.cols) > 65536)
        return set_error("Q4_K matvec: cols=%lld does not fit the LDS staging buffer", (long long)s.cols);
    if (!geom_ok(G)) return set_error("matvec_q4k: unsupported schedule nr0=%d nsg=%d (nr0 in 1,2,4; nsg in 4,8)", G.R, G.NW);
    if (s.prologue != kPlain && s.prologue != kMergeParts && s.cols > (int64_t)4 * G.NW * 64 * kStageP)
        return set_error("rmsnorm_matvec requires LOCAL staging of the vector (cols=%lld too large)", (long long)s.cols);
    const size_t rb = (size_t)bpr * kQ4kBytes, vb = (size_t)s.cols * 4;
    const int n_y = s.nm == 2 ? 1 : s.n_mat;
    int ni = 0, no = 0;
    for (int m = 0; m < s.n_mat; m++) { k.in_bytes[ni] = (size_t)s.rows[m] * rb; k.in_align[ni++] = 16; }
    k.in_bytes[ni] = s.prologue == kMergeParts ? (size_t)s.nwg * (s.cols + 2 * (s.cols / s.hd)) * 4 : vb; k.in_align[ni++] = 16;
    if (s.prologue == kRms || s.prologue == kAddThenRms) { k.in_bytes[ni] = vb; k.in_align[ni++] = 16; }
    if (s.prologue == kAddThenRms) {
        k.in_bytes[ni] = vb; k.in_align[ni++] = 16;
        k.in_bytes[ni] = vb; k.in_align[ni++] = 16;
    }
    for (int m = 0; m < n_y; m++) { k.out_bytes[no] = (size_t)s.rows[m] * 4; k.out_align[no++] = 4; }
    if (s.prologue == kAddThenRms) { k.out_bytes[no] = vb; k.out_align[no++] = 16; }
    k.info.n_inputs = ni;
    k.info.n_outputs = no;
    int waves = 0;
    if (s.nm == 2) waves = waves_for((int)s.rows[0], G.rpw());
    else for (int m = 0; m < s.n_mat; m++) waves += waves_for((int)s.rows[m], G.rpw());
    static const char *pre[] = {"", "rms_", "addrms_", "attn_merge_"};
    char base[48];
    snprintf(base, sizeof(base), "%smatvec%s", pre[s.prologue], s.n_mat == 3 ? "_qkv" : s.nm == 2 ? "_gate_up_gelu" : "");
    fill_info(k, G, waves, bpr, base);
    if (G.stream) {
        int groups = 0;
        if (s.nm == 2) groups = (int)((s.rows[0] + f.G / 2 - 1) / (f.G / 2));
        else for (int m = 0; m < s.n_mat; m++) groups += (int)((s.rows[m] + f.G - 1) / f.G);
        set_launch(k, (uint32_t)std::min(256, groups), 1, 1, (uint32_t)f.NW * 64, (uint32_t)q4s_lds(s.nm, bpr));
        k.info.sched.tg = (uint64_t)f.NW * 64;
        k.info.sched.nsg = (uint32_t)f.NW;
        k.info.sched.nr0 = (uint32_t)f.G;
        k.info.sched.unroll = (uint32_t)f.NBUF;
        k.info.sched.vec = kXI8;
        set_name(k, "%s_q4k_stream_g%d_w%d_n%d", base, f.G, f.NW, f.NBUF);
    }
    k.launch = launch_any<false>;
    if (q4k_gemv_half_built(G)) k.launch_half = launch_any<true>;
    return 0;
}

int bind_matvec_q4k(ksh_kernel &k) { return bind_matvec_q4k_family(k); }
int bind_matvec_qkv(ksh_kernel &k) { return bind_matvec_q4k_family(k); }
int bind_matvec_gate_up_gelu(ksh_kernel &k) { return bind_matvec_q4k_family(k); }

int matvec_q4k_candidates(const ksh_kernel_desc &d, ksh_sched *out, int cap)
{
    (void)d;
    int n = 0;
    // (vec = 2, the two-plane form, is built and can be asked for by schedule, but the search does not offer it: its
    // error is 2^-16 of a 32-element sub-block's largest magnitude, which is 1e-3 of an element next to an outlier
    // sixty times its size -- the three-plane form has 2^-21)
    for (uint32_t var : {3u, 1u})
        for (uint32_t nsg : {4u, 8u})
            for (uint32_t nr0 : {1u, 2u, 4u}) {
                if (n >= cap) return n;
                ksh_sched s{};
                s.tg = 64ull * nsg; s.vec = var; s.unroll = 1; s.nsg = nsg; s.nr0 = nr0; s.k_split = 1;
                out[n++] = s;
            }
    return n;
}

}  // namespace ksh
