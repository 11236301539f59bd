"""The decode-before-prefill slot scheduler (crates/ksearch_cli/src/scheduler.rs:78-349) through the C ABI: each
request produces the tokens the model produces for it alone, admission / chunking / stop rules follow the
reference's rounds."""
import numpy as np
import pytest

import oracle
from ksearch_amd import hip, synth
from tests.test_gpu_gemma4 import FFN, PATTERN

pytestmark = pytest.mark.gpu

NO_EOS = (0xFFFFFFFF, 0xFFFFFFFE)   # ids no model emits: runs end by length


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context()
    yield c
    c.close()


@pytest.fixture(scope="module")
def model(ctx):
    cfg = dict(synth.GEMMA4_TINY)
    w = synth.gemma4_weights(cfg, 610, oracle.quantize_q4k, oracle.quantize_q6k, ffn=FFN, swa_pattern=PATTERN, std=0.05)
    m = hip.Gemma4(ctx, cfg, w)
    yield m, cfg
    m.close()


def make_pool(ctx, cfg, slots):
    owners = cfg["n_layers"] - cfg["shared_kv_layers"]
    return hip.KvPool(ctx, slots, cfg["max_seq"], owners, max(cfg["hd_swa"], cfg["hd_full"]), cfg["n_kv"])


def alone(m, prompt, n_new):
    m.bind_slot(None, 0)
    m.reset()
    return m.generate(prompt, n_new, use_graph=True)[0]


def prompts_of(cfg, lens, seed):
    rng = np.random.default_rng(seed)
    return [[int(t) for t in rng.integers(0, cfg["vocab"], n)] for n in lens]


def split(events):
    toks, done, errs = {}, {}, {}
    for e in events:
        if e[0] == "token":
            toks.setdefault(e[1], []).append(e[2])
        elif e[0] == "done":
            assert e[1] not in done
            done[e[1]] = e[2:]
        else:
            errs[e[1]] = e[2]
    return toks, done, errs


@pytest.mark.parametrize("use_graph,batched", [(True, 0), (False, 0), (True, 2)])
def test_three_requests_through_two_slots_equal_the_runs_alone(ctx, model, use_graph, batched):
    """batched = 2: whenever both slots decode, their step is one ksh_gemma4_decode_round (one pass over the weights
    for both); the tokens are still those of the runs alone."""
    m, cfg = model
    prompts = prompts_of(cfg, (5, 9, 3), 700)
    max_new = (10, 6, 8)
    want = [alone(m, p, n) for p, n in zip(prompts, max_new)]
    pool = make_pool(ctx, cfg, 2)
    sv = hip.Serve(m, pool, slots=2, prefill_chunk=4, prefill_tokens_per_tick=8, eos=NO_EOS, use_graph=use_graph, batched_decode=batched)
    ids = [sv.submit(p, n) for p, n in zip(prompts, max_new)]
    events = sv.tick()
    assert sv.pending() == (1, 2) and len(pool.active_batch()) == 2     # the third waits for a slot
    events += sv.run()
    toks, done, errs = split(events)
    assert not errs
    for i, rid in enumerate(ids):
        assert toks[rid] == want[i], i
        assert done[rid] == ("length", len(prompts[i]), max_new[i])
    assert pool.active_batch() == [] and sv.pending() == (0, 0)
    # the slots are clean for the next round of requests: same answers again
    ids2 = [sv.submit(p, n) for p, n in zip(prompts[::-1], max_new[::-1])]
    toks2, _, _ = split(sv.run())
    assert [toks2[r] for r in ids2] == want[::-1]
    sv.close()
    m.bind_slot(None, 0)
    pool.close()


def test_prefill_takes_small_chunks_while_something_decodes(ctx, model):
    """scheduler.rs:243-292: with nothing decoding a prefilling request eats the tick's budget, with a decoding
    request beside it only prefill_chunk tokens per tick; the prompt's last token is the first decode input."""
    m, cfg = model
    pa, pb = prompts_of(cfg, (2, 21), 701)
    pool = make_pool(ctx, cfg, 2)
    sv = hip.Serve(m, pool, slots=2, prefill_chunk=4, prefill_tokens_per_tick=8, eos=NO_EOS)
    ra, rb = sv.submit(pa, 12), sv.submit(pb, 3)
    seen_b, first_b_token_tick = [], None
    events = []
    for tick in range(1, 9):
        ev = sv.tick()
        events += ev
        seen_b.append(pool.seq_len(1))
        if first_b_token_tick is None and any(e[0] == "token" and e[1] == rb for e in ev):
            first_b_token_tick = tick
    # tick 1: A's one prefill token (budget 8 -> 7), B takes the 7 left; then 4 a tick while A decodes; 20 = the
    # prompt minus its last token; the decode tokens follow
    assert seen_b[:6] == [7, 11, 15, 19, 20, 21]
    assert first_b_token_tick == 6
    events += sv.run()
    toks, done, _ = split(events)
    assert toks[ra] == alone(m, pa, 12) and toks[rb] == alone(m, pb, 3)
    assert done[ra] == ("length", 2, 12) and done[rb] == ("length", 21, 3)
    sv.close()
    m.bind_slot(None, 0)
    pool.close()


def test_stop_rules_errors_and_cancellation(ctx, model):
    m, cfg = model
    # a prompt whose continuation has, at some position cut >= 2, a token that has not appeared before it (the tiny
    # random model repeats itself soon)
    for seed in range(702, 742):
        (p,) = prompts_of(cfg, (6,), seed)
        full = alone(m, p, 12)
        cut = next((i for i in range(2, 12) if full[i] not in full[:i]), None)
        if cut is not None:
            break
    assert cut is not None
    pool = make_pool(ctx, cfg, 2)

    # an EOS id ends the request with "stop" and is not emitted (scheduler.rs:203-206)
    sv = hip.Serve(m, pool, slots=2, eos=(full[cut], 0xFFFFFFFF))
    r = sv.submit(p, 12)
    toks, done, _ = split(sv.run())
    assert toks[r] == full[:cut] and done[r] == ("stop", 6, cut)
    sv.close()

    # the host's stop callback takes the place of the stop strings, at the same point of the round
    asked = []
    sv = hip.Serve(m, pool, slots=2, eos=NO_EOS, stop=lambda req, tok: asked.append((req, tok)) or tok == full[cut])
    r = sv.submit(p, 12)
    toks, done, _ = split(sv.run())
    assert toks[r] == full[:cut] and done[r] == ("stop", 6, cut)
    assert asked == [(r, t) for t in full[:cut + 1]]
    sv.close()
    sv = hip.Serve(m, pool, slots=2, eos=NO_EOS)

    # errors: an empty prompt at admission, a prompt beyond max_seq at its prefill; max_tokens 0 counts as 1
    r_empty, r_long, r_one = sv.submit([], 4), sv.submit([1] * (cfg["max_seq"] + 2), 4), sv.submit(p, 0)
    toks, done, errs = split(sv.run())
    assert errs[r_empty] == "empty prompt" and "max_seq exceeded" in errs[r_long]
    assert r_long not in done and toks[r_one] == full[:1] and done[r_one] == ("length", 6, 1)
    assert pool.active_batch() == []

    # a request that runs into max_seq ends with "length" (scheduler.rs:177-180)
    r = sv.submit(p, 1000)
    toks, done, _ = split(sv.run())
    if done[r][0] == "length":
        assert done[r] == ("length", 6, cfg["max_seq"] - 5) and len(toks[r]) == cfg["max_seq"] - 5
    else:
        # or it fell into a loop first: 24 equal tokens in a row end it, the 24th counted but not sent (scheduler.rs:219-222)
        assert done[r] == ("stop", 6, len(toks[r]) + 1) and len(set(toks[r][-23:])) == 1

    # cancellation: a running request finishes "cancelled" at its next token, a waiting one at once
    r1, r2, r3 = sv.submit(p, 12), sv.submit(p, 12), sv.submit(p, 12)
    ev = sv.tick() + sv.tick() + sv.tick()
    sv.cancel(r1)
    sv.cancel(r3)
    ev += sv.run()
    toks, done, _ = split(ev)
    assert done[r1][0] == "cancelled" and toks[r1] == full[:len(toks[r1])] and len(toks[r1]) < 12
    assert done[r3] == ("cancelled", 6, 0) and r3 not in toks
    assert toks[r2] == full and done[r2] == ("length", 6, 12)
    with pytest.raises(hip.KshError, match="not queued or running"):
        sv.cancel(r2)
    sv.close()
    m.bind_slot(None, 0)
    pool.close()


def test_sampled_requests_follow_the_host_sampler(ctx, model):
    """decode_token_sampled with temperature > 0: logits read back, sample_softcap_min_p with the request's
    generator state (seed | 1, advanced by 0x9E3779B9 before every token: scheduler.rs:151, 184)."""
    m, cfg = model
    (p,) = prompts_of(cfg, (7,), 703)
    temperature, min_p, seed, n_new = 0.9, 0.02, 1234, 10
    m.bind_slot(None, 0)
    m.reset()
    m.prefill_chunk(p[:-1])
    want, last, rng = [], p[-1], seed | 1
    for _ in range(n_new):
        rng = (rng + 0x9E3779B9) & 0xFFFFFFFF
        m.forward_token(last, want_logits=True, read_next=False)
        last = hip.sample_softcap_min_p(m.logits(), cfg["softcap"], temperature, min_p, rng)
        want.append(last)
    assert want != alone(m, p, n_new)        # the draw is not the argmax everywhere
    pool = make_pool(ctx, cfg, 1)
    sv = hip.Serve(m, pool, slots=1, eos=NO_EOS)
    r = sv.submit(p, n_new, temperature=temperature, min_p=min_p, seed=seed)
    toks, done, _ = split(sv.run())
    assert toks[r] == want and done[r] == ("length", 7, n_new)
    # the model's own entry point draws the same token
    m.bind_slot(None, 0)
    m.reset()
    m.prefill_chunk(p[:-1], use_graph=True)
    assert m.decode_token_sampled(p[-1], temperature, min_p, (seed | 1) + 0x9E3779B9) == want[0]
    sv.close()
    m.bind_slot(None, 0)
    pool.close()


def test_serve_create_errors(ctx, model):
    m, cfg = model
    owners = cfg["n_layers"] - cfg["shared_kv_layers"]
    bad = hip.KvPool(ctx, 1, cfg["max_seq"], owners + 1, 256, cfg["n_kv"])
    with pytest.raises(hip.KshError, match="kv layer mismatch"):
        hip.Serve(m, bad)
    bad.close()
    pool = make_pool(ctx, cfg, 1)
    with pytest.raises(hip.KshError, match="slots=0"):
        hip.Serve(m, pool, slots=0)
    # more slots asked for than the pool has: the request that finds no slot is told so (scheduler.rs:150-158)
    sv = hip.Serve(m, pool, slots=2, eos=NO_EOS)
    (p,) = prompts_of(cfg, (4,), 704)
    r1, r2 = sv.submit(p, 3), sv.submit(p, 3)
    toks, done, errs = split(sv.run())
    assert "admit failed: KvPool full" in errs[r2] and done[r1] == ("length", 4, 3)
    sv.close()
    m.bind_slot(None, 0)
    pool.close()


def test_a_token_repeated_24_times_ends_the_request(ctx):
    """scheduler.rs:219-222, 342-348: all-zero weights give all-zero logits, whose argmax is id 0 every time; the
    24th equal token in a row ends the request with "stop", counted in completion_tokens but not sent."""
    cfg = dict(synth.GEMMA4_TINY)
    w = synth.gemma4_weights(cfg, 611, oracle.quantize_q4k, oracle.quantize_q6k, ffn=FFN, swa_pattern=PATTERN, std=0.0)
    m = hip.Gemma4(ctx, cfg, w)
    pool = make_pool(ctx, cfg, 1)
    sv = hip.Serve(m, pool, slots=1, eos=NO_EOS)
    r = sv.submit([5, 6, 7], 40)
    toks, done, errs = split(sv.run())
    assert not errs and toks[r] == [0] * 23 and done[r] == ("stop", 3, 24)
    sv.close()
    pool.close()
    m.close()


def test_destroying_a_busy_scheduler_frees_its_slots(ctx, model):
    m, cfg = model
    pool = make_pool(ctx, cfg, 2)
    sv = hip.Serve(m, pool, slots=2, eos=NO_EOS)
    (p,) = prompts_of(cfg, (5,), 705)
    sv.submit(p, 30), sv.submit(p, 30), sv.submit(p, 30)
    sv.tick(), sv.tick()
    assert len(pool.active_batch()) == 2 and sv.pending() == (1, 2)
    sv.close()
    assert pool.active_batch() == []
    m.bind_slot(None, 0)
    pool.close()


@pytest.mark.parametrize("temperature,min_p", [(0.3, 0.05), (1.0, 0.5), (2.5, 0.001), (50.0, 0.9), (1.0, 1.5), (1.0, 0.0)])
def test_draws_from_the_narrowed_logits_are_the_host_samplers(ctx, model, temperature, min_p):
    """The device keeps only what can survive the min-p filter (few entries; more than a record holds; all of them; a
    filter above 1; no filter): the draw is the host sampler's on the whole row, for the single step and for a round."""
    m, cfg = model
    (p,) = prompts_of(cfg, (5,), 706)
    m.bind_slot(None, 0)
    m.reset()
    m.prefill_chunk(p[:-1])
    for seed in range(3, 60, 7):
        m.bind_slot(None, 4)
        got = m.decode_token_sampled(p[-1], temperature, min_p, seed)
        assert got == hip.sample_softcap_min_p(m.logits(), cfg["softcap"], temperature, min_p, seed)
    pool = make_pool(ctx, cfg, 4)
    slots = [pool.alloc() for _ in range(4)]
    temps, seeds = [temperature, 0.0, temperature, 2 * temperature], [11, 12, 13, 14]
    got = m.decode_round(pool, slots, p[:4], temps, [min_p] * 4, seeds)
    rows = m.round_logits(4)
    assert got == [hip.sample_softcap_min_p(rows[i], cfg["softcap"], temps[i], min_p, seeds[i]) for i in range(4)]
    pool.close()


def test_draws_of_rows_with_more_candidates_than_a_list_takes(ctx):
    """A vocabulary of 40960: lists of up to 5120 candidates are drawn from (dense ones among them), rows with more and rows
    without a filter are walked whole; all of them, and a greedy row, in one round."""
    cfg = dict(synth.GEMMA4_TINY, vocab=40960)
    dq4, dq6 = hip.device_quantizers(ctx, hip.Eng())
    w = synth.gemma4_weights(cfg, 612, dq4, lambda x: dq6([x]), ffn=FFN, swa_pattern=PATTERN, std=0.05)
    m = hip.Gemma4(ctx, cfg, w)
    (p,) = prompts_of(cfg, (6,), 708)
    pool = make_pool(ctx, cfg, 6)
    slots = [pool.alloc() for _ in range(6)]
    temps, min_p, seeds = [50.0, 0.0, 0.9, 1.0, 0.05, 0.0], [0.9, 0.5, 0.0, 0.05, 0.5, 0.0], [21, 22, 23, 24, 25, 26]
    m.decode_round(pool, slots, p)
    y = cfg["softcap"] * np.tanh(m.round_logits(6) / np.float32(cfg["softcap"]))
    far = np.sort(y[3])[::-1][3000] - y[3].max()      # a temperature at which some three thousand of row 3 pass
    temps[3] = float(far / np.log(min_p[3]))
    counts = [int((y[i] >= y[i].max() + t * np.log(q)).sum()) for i, (t, q) in enumerate(zip(temps, min_p)) if q]
    assert counts[0] > 5120 and 2500 < counts[2] < 3500 and counts[3] < 127, counts
    for _ in range(3):                                # (eager, captured, replayed)
        got = m.decode_round(pool, slots, p, temps, min_p, seeds)
        rows = m.round_logits(6)
        assert got == [hip.sample_softcap_min_p(rows[i], cfg["softcap"], temps[i], min_p[i], seeds[i]) for i in range(6)]
    # rows without a filter only, and greedy ones only
    got = m.decode_round(pool, slots, p, [0.9, 0.0] * 3, [0.0] * 6, seeds)
    assert got == [hip.sample_softcap_min_p(rows[i], cfg["softcap"], 0.9 if i % 2 == 0 else 0.0, 0.0, seeds[i]) for i in range(6)]
    assert m.decode_round(pool, slots, p) == [int(np.argmax(y[i])) for i in range(6)]
    pool.close()
    m.close()


@pytest.mark.parametrize("lens", [(90, 1, 130, 66, 2, 65), (225, 225), (9, 129)])
def test_prompts_prefilled_in_one_pass_fill_the_caches_of_passes_alone(ctx, lens):
    """The prefilling requests of a tick with more than 64 tokens share one pass over the weights (heads of 256 and 512; 65
    prompt tokens are 64 and the first decode input: a pass alone).  Every slot's K / V rows are the bytes of the prompt
    alone -- slots, positions, windows and the K slices of every GEMM are each prompt's own -- and nothing is written
    behind them."""
    cfg = dict(synth.GEMMA4_TINY, hd_swa=256, hd_full=512, max_seq=256, sliding_window=40)
    w = synth.gemma4_weights(cfg, 611, oracle.quantize_q4k, oracle.quantize_q6k, ffn=FFN, swa_pattern=PATTERN, std=0.05,
                             q6k_tensors=((1, "wdown"), (2, "wv")))
    m = hip.Gemma4(ctx, cfg, w)
    prompts = prompts_of(cfg, lens, 705)
    pool = make_pool(ctx, cfg, len(lens))
    sv = hip.Serve(m, pool, slots=len(lens), eos=NO_EOS)
    for p in prompts:
        sv.submit(p, 2)
    assert sv.tick() == []
    assert [pool.seq_len(i) for i in range(len(lens))] == [n - 1 for n in lens]
    owners = cfg["n_layers"] - cfg["shared_kv_layers"]
    for slot, p in enumerate(prompts):
        m.bind_slot(None, 0)
        m.reset()
        m.prefill_chunk(p[:-1])
        for layer in range(owners):
            row = cfg["n_kv"] * (cfg["hd_swa"] if PATTERN[layer] else cfg["hd_full"]) // 32 * 18
            for which, buf in ((0, pool.k_buf(slot, layer)), (1, pool.v_buf(slot, layer))):
                if len(p) > 1:
                    own = hip.Buffer(ctx, hip.lib().ksh_gemma4_kv(m.h, layer, which), owned=False)
                    assert np.array_equal(ctx.read_bytes(buf, row * (len(p) - 1)), ctx.read_bytes(own, row * (len(p) - 1))), (slot, layer, which)
                assert not np.any(ctx.read_bytes(buf, row, row * (len(p) - 1)))
    sv.close()
    m.bind_slot(None, 0)
    pool.close()
    m.close()


def test_joint_prompt_passes_do_not_depend_on_saved_plans(tmp_path, monkeypatch):
    """A plan that a search left for one of the pass lengths (whole rows where the library's rule cuts them into K slices)
    changes neither a pass alone nor a joint one: the two keep filling the caches with the same bytes."""
    monkeypatch.setenv("KSEARCH_BEAM_CACHE", str(tmp_path / "beam"))
    ctx = hip.Context()
    cfg = dict(synth.GEMMA4_TINY, hd_swa=256, hd_full=512, max_seq=256, sliding_window=40)
    h, whole = cfg["hidden"], hip.Sched(tg=512, nsg=8, nr0=128, k_split=1, lds_tile=64)
    for tp in (224, 512):                                  # a prompt of 225 alone; two of them in steps of 128 rows
        for hd in (256, 512):
            qd = cfg["n_q"] * hd
            for dims in ((h, qd, tp, 0, 0, 0, 1), (h, qd, tp), (qd, h, tp, hd, hd, 1), (qd, h, tp, 0, 0, 1), (qd, h, tp)):
                hip.plan_save("mul_mm_q4k", dims, ctx.device_name(), whole, 0.001)
        for f in (1024, 2048):
            for dims in ((h, f, tp), (h, f, tp, 0, 0, 3)):
                hip.plan_save("mul_mm_q4k", dims, ctx.device_name(), whole, 0.001)
    w = synth.gemma4_weights(cfg, 611, oracle.quantize_q4k, oracle.quantize_q6k, ffn=FFN, swa_pattern=PATTERN, std=0.05)
    m = hip.Gemma4(ctx, cfg, w)
    prompts = prompts_of(cfg, (225, 225), 707)
    pool = make_pool(ctx, cfg, 2)
    sv = hip.Serve(m, pool, slots=2, eos=NO_EOS)
    for p in prompts:
        sv.submit(p, 2)
    assert sv.tick() == []
    for slot, p in enumerate(prompts):
        m.bind_slot(None, 0)
        m.reset()
        m.prefill_chunk(p[:-1])
        for layer in range(cfg["n_layers"] - cfg["shared_kv_layers"]):
            n = cfg["n_kv"] * (cfg["hd_swa"] if PATTERN[layer] else cfg["hd_full"]) // 32 * 18 * (len(p) - 1)
            own = [hip.Buffer(ctx, hip.lib().ksh_gemma4_kv(m.h, layer, which), owned=False) for which in (0, 1)]
            for buf, mine in zip((pool.k_buf(slot, layer), pool.v_buf(slot, layer)), own):
                assert np.array_equal(ctx.read_bytes(buf, n), ctx.read_bytes(mine, n)), (slot, layer)
    sv.close()
    m.bind_slot(None, 0)
    pool.close()
    m.close()
    ctx.close()
