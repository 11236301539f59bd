"""The work that a user of this library has it do, as cases that can be timed.

Every case goes through the public entry points of ``ksearch_amd.hip``: the operator calls of ``Eng`` / ``Context``
(a caller with a model of its own), the two decode loops (``Gemma``, ``Gemma4``) and the slot scheduler (``Serve``).

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare(case, seed)`` makes what a
program has in hand before the call, ``run(state)`` is one pass, ``work(case)`` what a pass cannot do without and
``tolerance(case)`` how far another correct implementation may be off.
"""
import math
import os
import random
import tempfile

import numpy as np
import torch

# Kernels by the library's defaults: no schedule search at load, and no plan file an earlier search left behind.
os.environ.setdefault("KSEARCH_SKIP_BEAM", "1")
os.environ.setdefault("KSEARCH_BEAM_CACHE", tempfile.mkdtemp(prefix="ksearch_cases_plans_"))

from ksearch_amd import hip  # noqa: E402
from ksearch_amd.hip import DType, Kind  # noqa: E402
from ksearch_amd.synth import GEMMA_E2B_SYNTH  # noqa: E402

EPS = 1e-6
DTYPES = {"q4k": DType.Q4K, "q6k": DType.Q6K}
BLOCK = {"q4k": 144, "q6k": 210, "q5k": 176}          # bytes of 256 weights

# The layer layout of the real checkpoints, as in the repository's own benchmark: 35 layers, four sliding-window
# layers per full-attention layer, the last 20 reading earlier layers' caches, per-layer embeddings.
LAYOUT = dict(n_layers=35, hidden=1536, n_q=8, n_kv=1, vocab=262144, max_seq=4096, hd_swa=256, hd_full=512,
              sliding_window=512, shared_kv_layers=20, ple_dim=256, eps=EPS, softcap=30.0, rope_theta_swa=1e4,
              rope_theta_full=1e6, partial_rotary=0.25, attn_scale=1.0)
LAYOUT_FFN = [6144] * 15 + [12288] * 20
LAYOUT_SWA = [(i + 1) % 5 != 0 for i in range(35)]


def listed():
    return [
        # one projection called by itself by a program with its own model code: launch and call overhead count
        dict(name="gemv_q4k", op="gemv", dtype="q4k", rows=4096, cols=4096),
        # the tied LM head of the checkpoints' vocabulary with its soft-capped argmax, on GGUF-order Q6_K
        dict(name="lm_head_q6k", op="head", rows=262144, cols=2048),
        # a prompt chunk's feed-forward projection
        dict(name="gemm_q4k", op="gemm", dtype="q4k", rows=8192, cols=2048, tokens=512),
        # the same kind on a Q6_K tensor (files keep attn_v / ffn_down so), with a ragged prompt
        dict(name="gemm_q6k_ragged", op="gemm", dtype="q6k", rows=1536, cols=6144, tokens=333),
        # attention of one decode step of several sequences of unequal length
        dict(name="attention_slots", op="slots", n_q=8, n_kv=1, hd=256, max_t=16384, slots=4),
        # one decode layer, operator by operator, on the half activation buffers that the reference's runtime keeps
        dict(name="half_layer", op="layer", hidden=2048, ffn=8192, n_q=8, n_kv=1, hd=256, attn_t=700, max_t=4096),
        # loading a file: a Q6_K tensor is requantized to Q4_K on the device (ffn_down of the checkpoints)
        dict(name="requantize", op="requantize", rows=2048, cols=8192),
        # a short chat turn: 64 tokens of prompt, 64 of answer
        dict(name="chat", op="generate", model="e2b", prompt=64, new=64),
        # time to the first token of a medium prompt
        dict(name="first_token", op="generate", model="e2b", prompt=700, new=1),
        # ... and of a document, at the checkpoints' layout; odd, more than two chunks
        dict(name="first_token_long", op="generate", model="layout", prompt=3001, new=1),
        # an answer streamed token by token, deep in a conversation; the caller chooses the tokens
        dict(name="stream_long", op="stream", model="layout", context=2500, new=32),
        # sixteen requests under the scheduler, sampled
        dict(name="serve_sampled", op="serve", model="layout", requests=16, prompt=200, new=10, temperature=0.8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "head", "gemm", "gemm", "slots", "slots", "layer", "layer", "requantize",
                     "generate", "generate", "stream", "serve"])
    if op == "gemv":
        dtype = rng.choice(["q4k", "q6k"])
        return dict(op=op, dtype=dtype, rows=_log(rng, 200, 16384), cols=256 * _log(rng, 2, 32))
    if op == "head":
        return dict(op=op, rows=_log(rng, 30000, 262144), cols=rng.choice([1536, 2048, 2560, 4096]))
    if op == "gemm":
        return dict(op=op, dtype=rng.choice(["q4k", "q6k"]), rows=_log(rng, 256, 12288), cols=256 * _log(rng, 2, 32),
                    tokens=_log(rng, 2, 2048))
    if op == "slots":
        n_q, n_kv, hd = rng.choice([(8, 1, 256), (8, 1, 256), (8, 1, 512), (4, 1, 256), (16, 2, 256), (8, 4, 128),
                                    (32, 8, 128)])
        return dict(op=op, n_q=n_q, n_kv=n_kv, hd=hd, max_t=_log(rng, 300, 16384), slots=_log(rng, 1, 16))
    if op == "layer":
        n_q, n_kv, hd = rng.choice([(8, 1, 256), (8, 1, 512), (16, 2, 128), (8, 2, 256)])
        max_t = rng.choice([2048, 4096])
        return dict(op=op, hidden=256 * rng.randint(4, 16), ffn=256 * rng.randint(16, 48), n_q=n_q, n_kv=n_kv, hd=hd,
                    attn_t=_log(rng, 130, max_t), max_t=max_t)
    if op == "requantize":
        return dict(op=op, rows=_log(rng, 256, 16384), cols=256 * rng.randint(2, 32))
    if op == "generate":
        new = rng.choice([1, rng.randint(8, 80)])
        return dict(op=op, model=rng.choice(["e2b", "layout"]), prompt=_log(rng, 8, 3900 if new == 1 else 600), new=new)
    if op == "stream":
        return dict(op=op, model="layout", context=_log(rng, 30, 4000), new=rng.randint(16, 40))
    return dict(op=op, model="layout", requests=rng.randint(2, 16), prompt=_log(rng, 16, 300), new=rng.randint(5, 12),
                temperature=rng.choice([0.0, 0.7, 1.0]))


# -- state ------------------------------------------------------------------

_ctx = None


def _context():
    """One context for the process, as a program keeps it."""
    global _ctx
    if _ctx is None:
        torch.zeros(1, device="cuda")
        _ctx = hip.Context()
    return _ctx


class _Span:
    """Device memory of the library, as torch takes it."""

    def __init__(self, ptr, n, typestr, keep):
        self.keep = keep
        self.__cuda_array_interface__ = dict(shape=(n,), typestr=typestr, data=(ptr, False), version=3, strides=None)


def _view(buf, dtype=torch.float32, n=None):
    size, typestr = {torch.float32: (4, "<f4"), torch.float16: (2, "<f2"), torch.uint8: (1, "|u1"),
                     torch.bfloat16: (2, "<i2")}[dtype]
    t = torch.as_tensor(_Span(buf.device_ptr, buf.nbytes // size if n is None else n, typestr, buf), device="cuda")
    return t.view(dtype) if dtype == torch.bfloat16 else t


class _State:
    """What run() works on.  Models and schedulers are closed when the state goes."""

    def __init__(self, case, seed):
        self.case, self.ctx, self.eng = case, _context(), hip.Eng()
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.rng = random.Random(seed)
        self.closing = []

    def __del__(self):
        try:
            for x in self.closing:
                x.close()
        except Exception:
            pass

    def put(self, t):
        """A device buffer with the tensor's bytes."""
        t = t.contiguous()
        b = self.ctx.buffer_empty_bytes(t.numel() * t.element_size())
        _view(b, torch.uint8).copy_(t.view(-1).view(torch.uint8))
        return b

    def normal(self, n, std=1.0, dtype=torch.float32, mean=0.0):
        return self.put((torch.randn(n, generator=self.gen, device="cuda") * std + mean).to(dtype))

    def scratch(self, n):
        if getattr(self, "_scratch", None) is None or self._scratch.nbytes < 4 * n:
            self._scratch = self.ctx.buffer_empty_f32(n)
        return self._scratch

    def packed(self, n, dtype, std=0.02):
        """n weights ~N(0, std), packed on the device as the loader packs them."""
        dst = self.ctx.buffer_empty_bytes(n // 256 * BLOCK[dtype])
        step = 1 << 26
        src = self.scratch(min(n, step))
        for at in range(0, n, step):
            m = min(step, n - at)
            _view(src, n=m).normal_(0.0, std, generator=self.gen)
            torch.cuda.synchronize()
            k = self.eng._k(self.ctx, Kind.QUANTIZE_K, (m,), (DTYPES[dtype],))
            self.ctx.encode_offsets_multi(k, [src], [0], [dst], [at // 256 * BLOCK[dtype]])
            self.ctx.synchronize()
        return dst

    def kv_rows(self, n_blocks):
        """Q4_0 blocks: scales of half precision, uniform nibbles."""
        t = torch.randint(0, 256, (n_blocks, 18), generator=self.gen, device="cuda", dtype=torch.uint8)
        d = torch.rand(n_blocks, generator=self.gen, device="cuda") * 0.09 + 0.01
        t[:, 0:2] = d.to(torch.float16).view(torch.uint8).view(n_blocks, 2)
        return self.put(t)


def _e2b(s):
    """The repository's synthetic benchmark model.  The norms that close a block have weights around 0.3: a block adds a
    fraction of the residual stream, which keeps the next-token distribution as peaked as a trained model's."""
    c = GEMMA_E2B_SYNTH
    h, f, qd, kvd = c["hidden"], c["ffn"], c["n_q"] * c["hd"], c["n_kv"] * c["hd"]
    shapes = dict(wq=qd * h, wk=kvd * h, wv=kvd * h, wo=h * qd, wgate=f * h, wup=f * h, wdown=h * f)
    norms = dict(attn_norm=(h, 1.0), q_norm=(c["hd"], 1.0), k_norm=(c["hd"], 1.0), post_attn_norm=(h, 0.3),
                 ffn_norm=(h, 1.0), post_ffw_norm=(h, 0.3))
    layers = []
    for _ in range(c["n_layers"]):
        lw = {k: s.packed(n, "q4k") for k, n in shapes.items()}
        lw.update({k: s.normal(n, 0.1 * m, mean=m) for k, (n, m) in norms.items()})
        layers.append(lw)
    w = dict(layers=layers, token_embd=s.packed(c["vocab"] * h, "q6k"), output_norm=s.normal(h, 0.1, mean=1.0))
    torch.cuda.synchronize()
    return hip.Gemma(s.ctx, c, w)


def _layout(s):
    """Synthetic weights at the checkpoints' layer layout, Q4_K with a Q6_K tied embedding and a Q5_K per-layer table."""
    c, h, pd = LAYOUT, LAYOUT["hidden"], LAYOUT["ple_dim"]
    layers = []
    for i in range(c["n_layers"]):
        hd = c["hd_swa"] if LAYOUT_SWA[i] else c["hd_full"]
        qd, kvd, f = c["n_q"] * hd, c["n_kv"] * hd, LAYOUT_FFN[i]
        shapes = dict(wq=qd * h, wo=h * qd, wgate=f * h, wup=f * h, wdown=h * f, inp_gate=pd * h, proj=h * pd)
        if i < c["n_layers"] - c["shared_kv_layers"]:
            shapes.update(wk=kvd * h, wv=kvd * h)
        lw = {k: s.packed(n, "q4k") for k, n in shapes.items()}
        norms = dict(attn_norm=(h, 1.0), q_norm=(hd, 0.3), k_norm=(hd, 0.3), post_attn_norm=(h, 0.3), ffn_norm=(h, 1.0),
                     post_ffw_norm=(h, 0.3), post_norm=(h, 0.3))
        lw.update({k: s.normal(n, 0.1 * m, mean=m) for k, (n, m) in norms.items()})
        lw.update(is_swa=int(LAYOUT_SWA[i]), ffn=f, layer_scale=s.rng.uniform(0.8, 1.2))
        layers.append(lw)
    pt = c["n_layers"] * pd
    table = torch.randint(0, 256, (c["vocab"] * pt // 256, BLOCK["q5k"]), generator=s.gen, device="cuda", dtype=torch.uint8)
    d = (torch.rand(2 * len(table), generator=s.gen, device="cuda") * 9e-4 + 1e-4).to(torch.float16)
    table[:, 0:4] = d.view(torch.uint8).view(len(table), 4)
    g = dict(token_embd=s.packed(c["vocab"] * h, "q6k"), dt_embd=DType.Q6K, output_norm=s.normal(h, 0.1, mean=1.0),
             ple_embd=s.put(table), dt_ple=DType.Q5K, ple_model_proj=s.packed(pt * h, "q4k"), dt_ple_proj=DType.Q4K,
             ple_proj_norm=s.normal(pd, 0.1, mean=1.0))
    torch.cuda.synchronize()
    return hip.Gemma4(s.ctx, c, dict(layers=layers, globals=g))


def _lengths(case):
    """Attended rows of every slot, from the case alone."""
    r = random.Random(case["slots"] * 7919 + case["max_t"])
    return [r.randint(max(1, case["max_t"] // 16), case["max_t"]) for _ in range(case["slots"])]


def prepare(case, seed):
    s = _State(case, seed)
    op = case["op"]
    if op in ("gemv", "head"):
        s.w = s.packed(case["rows"] * case["cols"], case.get("dtype", "q6k"))
        s.x, s.y, s.idx = s.normal(case["cols"]), s.ctx.buffer_empty_f32(case["rows"]), s.ctx.buffer_empty_f32(1)
        s.out = {"y": _view(s.y)}
        if op == "head":
            s.out["id"] = _view(s.idx)
    elif op == "gemm":
        s.w = s.packed(case["rows"] * case["cols"], case["dtype"])
        s.x = s.normal(case["tokens"] * case["cols"], dtype=torch.bfloat16)
        s.y = s.ctx.buffer_empty_f32(case["tokens"] * case["rows"])
        s.out = _view(s.y)
    elif op == "slots":
        n, n_q, n_kv, hd, max_t = (case[k] for k in ("slots", "n_q", "n_kv", "hd", "max_t"))
        k = s.ctx.compile(hip.make_desc(Kind.SDPA_SLOTS, (n_q, n_kv, hd, max_t, n, 0), (DType.Q40, DType.F32), (1.0 / 16.0,)))
        s.q, s.k, s.v = s.normal(n * n_q * hd), s.kv_rows(n * max_t * n_kv * hd // 32), s.kv_rows(n * max_t * n_kv * hd // 32)
        meta = np.zeros((n, 4), np.float32)
        meta[:, 0] = _lengths(case)
        s.meta = s.ctx.buffer_f32(meta)
        s.tmp = s.ctx.buffer_empty_f32(n * n_q * k.info.sched.k_split * (hd + 2))
        s.o = s.ctx.buffer_empty_f32(n * n_q * hd)
        s.out = _view(s.o)
    elif op == "layer":
        _prepare_layer(s)
    elif op == "requantize":
        n = case["rows"] * case["cols"]
        s.src, s.f32, s.dst = s.packed(n, "q6k"), s.ctx.buffer_empty_f32(n), s.ctx.buffer_empty_bytes(n // 256 * 144)
        s.out = {"f32": _view(s.f32), "q4k": _view(s.dst, torch.uint8)}
    else:
        s.model = _e2b(s) if case["model"] == "e2b" else _layout(s)
        s._scratch = None
        vocab = s.model.cfg["vocab"]
        s.tokens = lambda n: [s.rng.randrange(200, vocab) for _ in range(n)]
        if op == "serve":
            s.pool = hip.KvPool(s.ctx, 16, LAYOUT["max_seq"], LAYOUT["n_layers"] - LAYOUT["shared_kv_layers"],
                                LAYOUT["hd_full"], LAYOUT["n_kv"])
            s.serve = hip.Serve(s.model, s.pool, slots=case["requests"], eos=(1, 106))
            # prompts of unequal length, answers that end at different steps
            s.prompts = [s.tokens(max(2, case["prompt"] - case["prompt"] * (i % 5) // 6)) for i in range(case["requests"])]
            s.closing += [s.serve]
        elif op == "stream":
            s.model.prefill_chunk(s.tokens(case["context"]))
            s.given = s.tokens(case["new"])
        else:
            s.prompt = s.tokens(case["prompt"])
        s.closing += [s.model] + ([s.pool] if op == "serve" else [])
        s.logits = None
    torch.cuda.synchronize()
    return s


def _prepare_layer(s):
    """Kernel handles and buffers of one decode layer with half activations (descriptor dtypes[1] = F16)."""
    c = s.case
    h, f, n_q, n_kv, hd, max_t = (c[k] for k in ("hidden", "ffn", "n_q", "n_kv", "hd", "max_t"))
    qd, kvd, nwg, half = n_q * hd, n_kv * hd, hip.Eng.SDPA_MWG_NWG, torch.float16

    def kernel(kind, dims, w=0, params=()):
        return s.ctx.compile(hip.make_desc(kind, dims, (w, DType.F16), params))

    def empty(n):
        return s.ctx.buffer_empty_f16(n)

    wq, wk, wv = s.packed(qd * h, "q4k"), s.packed(kvd * h, "q4k"), s.packed(kvd * h, "q4k")
    wo, wg, wu, wd = (s.packed(n, "q4k") for n in (h * qd, f * h, f * h, h * f))
    x, y, x1, x2, ff, o = s.normal(h, dtype=half), empty(h), empty(h), empty(h), empty(f), empty(qd)
    q, k, v, q1 = empty(qd), empty(kvd), empty(kvd), empty(qd)
    n_attn, n_ffn, n_post, n_pffw = (s.normal(h, 0.1, half, 1.0) for _ in range(4))
    n_qh, n_kh = s.normal(hd, 0.1, half, 1.0), s.normal(hd, 0.1, half, 1.0)
    kc, vc = s.kv_rows(max_t * kvd // 32), s.kv_rows(max_t * kvd // 32)
    pos, row = c["attn_t"] - 1, kvd // 32 * 18
    ang = torch.arange(max_t, device="cuda")[:, None] * (1e4 ** (-torch.arange(hd // 2, device="cuda") / (hd // 2)))[None]
    rope = s.put(torch.cat([ang.cos(), ang.sin()], 1).float())
    meta, tmp = s.ctx.buffer_f32([c["attn_t"], 0, 0, pos]), s.ctx.buffer_empty_f32(n_q * nwg * (hd + 2))
    s.steps = [
        (kernel(Kind.RMSNORM_MATVEC_QKV, (qd, kvd, h, 0), DType.Q4K, (EPS,)), [wq, wk, wv, x, n_attn], None, [q, k, v], None),
        (kernel(Kind.RMSNORM_PER_HEAD_QKV_Q40, (n_q, n_kv, hd), 0, (EPS,)), [q, n_qh, rope, k, n_kh, v],
         [0, 0, pos * hd * 4, 0, 0, 0], [q1, kc, vc], [0, pos * row, pos * row]),
        (kernel(Kind.SDPA_MWG_PART, (n_q, n_kv, hd, max_t, nwg), DType.Q40, (1.0 / 16.0,)), [q1, kc, vc, meta], None, [tmp], None),
        (kernel(Kind.SDPA_MWG_REDUCE, (n_q, hd, nwg)), [tmp], None, [o], None),
        (kernel(Kind.MATVEC, (h, qd), DType.Q4K), [wo, o], None, [y], None),
        (kernel(Kind.RMSNORM_MATVEC_GATE_UP_GELU, (f, h, 1), DType.Q4K, (EPS,)), [wg, wu, y, n_ffn, n_post, x], None, [ff, x1], None),
        (kernel(Kind.MATVEC, (h, f), DType.Q4K), [wd, ff], None, [y], None),
        (kernel(Kind.RMSNORM, (h, 1, 0), 0, (EPS, 0.0)), [y, n_pffw, x1], None, [x2], None),
    ]
    s.out = {"x": _view(x2, half), "o": _view(o, half), "ff": _view(ff, half)}


def run(s):
    c, op = s.case, s.case["op"]
    if op == "gemv":
        s.eng.matvec_wd(s.ctx, c["rows"], c["cols"], DTYPES[c["dtype"]], s.w, s.x, s.y)
        return s.out
    if op == "head":
        s.eng.matvec_wd(s.ctx, c["rows"], c["cols"], DType.Q6K, s.w, s.x, s.y)
        s.eng.softcap_argmax(s.ctx, c["rows"], 30.0, s.y, s.idx)
        return s.out
    if op == "gemm":
        s.eng.matvec_batch(s.ctx, c["rows"], c["cols"], c["tokens"], DTYPES[c["dtype"]], s.w, s.x, s.y)
        return s.out
    if op == "slots":
        s.eng.sdpa_slots(s.ctx, c["n_q"], c["n_kv"], c["hd"], c["max_t"], c["slots"], s.q, s.k, s.v, s.meta, s.tmp, s.o,
                         scale=1.0 / 16.0)
        return s.out
    if op == "layer":
        for step in s.steps:
            s.ctx.encode_offsets_multi(*step)
        return s.out
    if op == "requantize":
        n = c["rows"] * c["cols"]
        s.eng.dequant(s.ctx, DType.Q6K, n, s.src, s.f32)
        s.eng.quantize_k(s.ctx, DType.Q4K, n, s.f32, s.dst)
        return s.out
    if op == "generate":
        s.model.reset()
        ids, _, _ = s.model.generate(s.prompt, c["new"])
        return {"ids": np.array(ids, np.int64), "logits": _logits(s)}
    if op == "stream":
        s.model.bind_slot(None, c["context"])
        ids = [s.model.forward_token(t, use_graph=True) for t in s.given]
        return {"ids": np.array(ids, np.int64), "logits": _logits(s)}
    order = [s.serve.submit(p, c["new"] - i % 3, c["temperature"], 0.05, 1000 + i) for i, p in enumerate(s.prompts)]
    got = {r: [] for r in order}
    for e in s.serve.run():
        if e[0] == "token":
            got[e[1]].append(e[2])
    return [np.array(got[r], np.int64) for r in order]


def _logits(s):
    """The last step's logits, where the model keeps them."""
    if s.logits is None:
        get = hip.lib().ksh_gemma_logits if s.case["model"] == "e2b" else hip.lib().ksh_gemma4_logits
        s.logits = _view(hip.Buffer(s.ctx, get(s.model.h), owned=False))
    return s.logits


# -- what a pass cannot do without -------------------------------------------

def _model_work(model):
    """(bytes of all weights of a token, weights of a token, bytes of one cached position, layers' head sizes)."""
    if model == "e2b":
        c = GEMMA_E2B_SYNTH
        h, hd = c["hidden"], c["hd"]
        layer = 2 * c["n_q"] * hd * h + 2 * c["n_kv"] * hd * h + 3 * c["ffn"] * h
        mats, head = c["n_layers"] * layer, c["vocab"] * h
        return mats, head, [(hd, c["max_seq"], True)] * c["n_layers"], c["n_q"]
    c, h, pd = LAYOUT, LAYOUT["hidden"], LAYOUT["ple_dim"]
    mats, att = c["n_layers"] * pd * h, []
    for i in range(c["n_layers"]):
        hd, owns = (c["hd_swa"] if LAYOUT_SWA[i] else c["hd_full"]), i < c["n_layers"] - c["shared_kv_layers"]
        mats += 2 * c["n_q"] * hd * h + (2 * c["n_kv"] * hd * h if owns else 0) + 3 * LAYOUT_FFN[i] * h + 2 * pd * h
        att.append((hd, c["sliding_window"] if LAYOUT_SWA[i] else c["max_seq"], owns))
    return mats, c["vocab"] * h, att, c["n_q"]


def _tokens_work(model, first, n, with_logits, passes):
    """n tokens of one sequence from position `first` on, the layers' weights read `passes` times, logits `with_logits` times."""
    mats, head, att, n_q = _model_work(model)
    b = passes * mats * 144 / 256 + with_logits * (head * 210 / 256 + 4 * 262144)
    f = 2.0 * mats * n + 2.0 * head * with_logits
    for hd, window, _ in att:
        seen = sum(min(t + 1, window) for t in range(first, first + n))
        f += 4.0 * n_q * hd * seen
        # a pass reads each cached row once: per token in decode, per chunk in a prompt
        b += 2 * hd * 18 / 32 * (seen if passes >= n else passes * min(first + n, window + n))
    return b, f


def work(case):
    op = case["op"]
    if op in ("gemv", "head"):
        n = case["rows"] * case["cols"]
        b = n // 256 * BLOCK[case.get("dtype", "q6k")] + 4 * (case["rows"] + case["cols"])
        return {"bytes": b, "flops": 2.0 * n}
    if op == "gemm":
        n = case["rows"] * case["cols"]
        return {"bytes": n // 256 * BLOCK[case["dtype"]] + case["tokens"] * (2 * case["cols"] + 4 * case["rows"]),
                "flops": 2.0 * n * case["tokens"]}
    if op == "slots":
        rows, n_q, n_kv, hd = sum(_lengths(case)), case["n_q"], case["n_kv"], case["hd"]
        return {"bytes": rows * n_kv * hd // 32 * 36 + 8 * case["slots"] * n_q * hd, "flops": 4.0 * rows * n_q * hd}
    if op == "layer":
        h, f, qd, kvd = case["hidden"], case["ffn"], case["n_q"] * case["hd"], case["n_kv"] * case["hd"]
        n = 2 * qd * h + 2 * kvd * h + 3 * f * h
        return {"bytes": n // 256 * 144 + case["attn_t"] * kvd // 32 * 36 + 2 * (6 * h + qd + f),
                "flops": 2.0 * n + 4.0 * case["attn_t"] * qd}
    if op == "requantize":
        n = case["rows"] * case["cols"]
        return {"bytes": n // 256 * 210 + 4 * n + n // 256 * 144, "flops": 0}
    if op == "generate":
        p, new = case["prompt"], case["new"]
        b0, f0 = _tokens_work(case["model"], 0, p - 1, 0, -(-(p - 1) // 1024)) if p > 1 else (0, 0)
        b1, f1 = _tokens_work(case["model"], p - 1, new, new, new)
        return {"bytes": b0 + b1, "flops": f0 + f1}
    if op == "stream":
        b, f = _tokens_work(case["model"], case["context"], case["new"], case["new"], case["new"])
        return {"bytes": b, "flops": f}
    b = f = 0.0
    for i in range(case["requests"]):
        p, new = max(2, case["prompt"] - case["prompt"] * (i % 5) // 6), case["new"] - i % 3
        b0, f0 = _tokens_work(case["model"], 0, p - 1, 0, 1)
        _, f1 = _tokens_work(case["model"], p - 1, new, new, new)
        b, f = b + b0, f + f0 + f1
    # the steps of all requests share the weights
    b1, _ = _tokens_work(case["model"], case["prompt"], case["new"], case["new"], case["new"])
    return {"bytes": b + b1, "flops": f}


def tolerance(case):
    op = case["op"]
    if op in ("gemv", "head"):
        return {"rel": 1e-5}                      # f32 sums of exact codes
    if op == "gemm":
        # f32 sums of exact codes; Q6_K codes times their scales are rounded to half
        return {"rel": 1e-4} if case["dtype"] == "q4k" else {"rel": 1e-3}
    if op == "slots":
        return {"rel": 2e-3}                      # half operands of the matrix cores
    if op == "layer":
        return {"rel": 5e-3, "max": 0.1}          # half results of every operator, a requantized cache row
    if op == "requantize":
        return "exact"                            # the host routine's bytes
    # f32 activations, but every token's keys and values are requantized to 4 bits: a last-digit difference can move a code
    return {"rel": 1e-2, "max": 0.2, "differ": 0.01}
