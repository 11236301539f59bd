"""Q4_K / Q6_K prefill GEMM on the matrix cores vs the CPU oracle (dequant,
bf16->f32 X, sequential f32 dot), 1e-3 relative; shapes and inputs of the
reference's check_mul_mm example plus the full benchmark configuration."""
import numpy as np
import pytest

import oracle
from ksearch_amd import hip, synth
from ksearch_amd.hip import DType
from tests.gpu_util import assert_close, rel_err
from tests.test_oracle_ops import check_mul_mm_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context()
    yield c
    c.close()


@pytest.fixture(scope="module")
def eng():
    return hip.Eng()


def run(ctx, eng, w, rows, cols, xf, xb, batch, q6=False):
    y = ctx.buffer_empty_f32(batch * rows)
    eng.matvec_batch(ctx, rows, cols, batch, DType.Q6K if q6 else DType.Q4K, ctx.buffer_bytes(w), ctx.buffer_bytes(xb), y)
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    want = oracle.matmul(oracle.Q6K if q6 else oracle.Q4K, w, rows, cols, xf, batch)
    return got, want


# crates/ksearch_kernels/examples/check_mul_mm.rs:296-304
@pytest.mark.parametrize("rows,cols,batch", [(64, 256, 16), (128, 256, 9), (2048, 1536, 256), (4096, 1536, 55)])
def test_mul_mm_check_mul_mm_shapes(ctx, eng, rows, cols, batch):
    w, x = check_mul_mm_inputs(rows, cols, batch)
    wq = oracle.quantize_q4k(w)
    xf, xb = synth.bf16_round(x)
    got, want = run(ctx, eng, wq, rows, cols, xf.reshape(batch, cols), xb.reshape(batch, cols), batch)
    assert_close(got, want, 1e-3, f"mul_mm {rows}x{cols} b{batch}")
    # mul_mm row t equals the GEMV on x[t] (the example's "mul_mm vs gemv" line)
    by = ctx.buffer_empty_f32(rows)
    bw = ctx.buffer_bytes(wq)
    for t in (0, batch - 1):
        eng.matvec_wd(ctx, rows, cols, DType.Q4K, bw, ctx.buffer_f32(xf.reshape(batch, cols)[t]), by)
        assert_close(got[t], ctx.read_f32(by, rows), 1e-3, f"mul_mm vs gemv t={t}")


@pytest.mark.parametrize("rows,cols,batch", [(1, 256, 1), (130, 512, 129), (257, 2048, 33)])
def test_mul_mm_random_blocks_ragged(ctx, eng, rows, cols, batch):
    w = synth.q4k_blocks(rows * cols // 256, seed=600 + rows)
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 601))
    got, want = run(ctx, eng, w, rows, cols, xf.reshape(batch, cols), xb.reshape(batch, cols), batch)
    assert_close(got, want, 1e-3, f"mul_mm {rows}x{cols} b{batch}")


def test_mul_mm_unit_columns_recover_weights(ctx, eng):
    # X = one-hot rows: Y[t] is column k_t of the dequantized matrix (pins the K order end to end)
    rows, cols = 64, 512
    w = synth.q4k_blocks(rows * cols // 256, seed=610)
    wd = oracle.dequant(oracle.Q4K, w, rows * cols).reshape(rows, cols)
    ks = [0, 1, 2, 3, 15, 16, 31, 32, 33, 63, 64, 127, 255, 256, 300, 511]
    x = np.zeros((len(ks), cols), dtype=np.float32)
    for t, k in enumerate(ks):
        x[t, k] = 1.0
    xf, xb = synth.bf16_round(x.reshape(-1))
    got, _ = run(ctx, eng, w, rows, cols, xf.reshape(len(ks), cols), xb.reshape(len(ks), cols), len(ks))
    for t, k in enumerate(ks):
        # the 1024-bias and the hi/lo split of the min term leave ~2^-22 of 1024*d
        assert np.allclose(got[t], wd[:, k], rtol=1e-5, atol=1e-5 * np.abs(wd).max()), k


def q6k_blocks_full_scales(n_blocks, seed):
    """Random Q6_K superblocks whose int8 scales span -128..127 (the synthetic set's stay within -32..31)."""
    blk = synth.q6k_blocks(n_blocks, seed).reshape(n_blocks, 210).copy()
    blk[:, 192:208] = np.random.default_rng(seed + 1).integers(-128, 128, size=(n_blocks, 16), dtype=np.int16).astype(np.int8).view(np.uint8)
    return blk.reshape(-1)


# Q6_K tensors in prefill: same shapes (1536 columns: rows of 1260 bytes, blocks at 2-byte alignment)
@pytest.mark.parametrize("rows,cols,batch", [(64, 256, 16), (128, 256, 9), (2048, 1536, 256), (4096, 1536, 55)])
def test_mul_mm_q6k_check_mul_mm_shapes(ctx, eng, rows, cols, batch):
    w, x = check_mul_mm_inputs(rows, cols, batch)
    wq = oracle.quantize_q6k(w)
    xf, xb = synth.bf16_round(x)
    got, want = run(ctx, eng, wq, rows, cols, xf.reshape(batch, cols), xb.reshape(batch, cols), batch, q6=True)
    assert_close(got, want, 1e-3, f"mul_mm q6k {rows}x{cols} b{batch}")
    by = ctx.buffer_empty_f32(rows)
    bw = ctx.buffer_bytes(wq)
    for t in (0, batch - 1):
        eng.matvec_wd(ctx, rows, cols, DType.Q6K, bw, ctx.buffer_f32(xf.reshape(batch, cols)[t]), by)
        assert_close(got[t], ctx.read_f32(by, rows), 1e-3, f"mul_mm q6k vs gemv t={t}")


@pytest.mark.parametrize("rows,cols,batch", [(1, 256, 1), (130, 512, 129), (257, 2048, 33), (300, 1280, 140)])
def test_mul_mm_q6k_random_blocks_ragged(ctx, eng, rows, cols, batch):
    # scales over the whole int8 range, so products beyond 2048 (rounded to even) occur
    w = q6k_blocks_full_scales(rows * cols // 256, seed=620 + rows)
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 621))
    got, want = run(ctx, eng, w, rows, cols, xf.reshape(batch, cols), xb.reshape(batch, cols), batch, q6=True)
    assert_close(got, want, 1e-3, f"mul_mm q6k {rows}x{cols} b{batch}")


@pytest.mark.parametrize("full_scales", [False, True])
def test_mul_mm_q6k_unit_columns_recover_weights(ctx, eng, full_scales):
    # one-hot rows of X return columns of the dequantized matrix: pins the ql / qh / scale indexing of every
    # position class.  Scales within -32..31: every scale * code is exact in f16 and the columns come back
    # bit-exact; over the whole int8 range a product beyond 2048 is rounded to an even integer (2^-11).
    rows, cols = 64, 512
    w = (q6k_blocks_full_scales if full_scales else synth.q6k_blocks)(rows * cols // 256, seed=630)
    wd = oracle.dequant(oracle.Q6K, w, rows * cols).reshape(rows, cols)
    ks = [0, 1, 2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 95, 96, 127, 128, 129, 191, 192, 255, 256, 300, 511]
    x = np.zeros((len(ks), cols), dtype=np.float32)
    for t, k in enumerate(ks):
        x[t, k] = 1.0
    xf, xb = synth.bf16_round(x.reshape(-1))
    got, _ = run(ctx, eng, w, rows, cols, xf.reshape(len(ks), cols), xb.reshape(len(ks), cols), len(ks), q6=True)
    for t, k in enumerate(ks):
        if full_scales:
            assert np.allclose(got[t], wd[:, k], rtol=2.0 ** -11, atol=0), k
        else:
            assert np.array_equal(got[t], wd[:, k]), k


def test_mul_mm_q6k_cfg2_shape(ctx, eng):
    tokens, rows, cols = 512, 8192, 2048
    w = q6k_blocks_full_scales(rows * cols // 256, seed=640)
    xf, xb = synth.bf16_round(synth.normal_f32(tokens * cols, 641))
    xf, xb = xf.reshape(tokens, cols), xb.reshape(tokens, cols)
    got, want = run(ctx, eng, w, rows, cols, xf, xb, tokens, q6=True)
    assert_close(got, want, 1e-3, "q6k 512x8192x2048")
    # linearity: twice the activations, twice the result, bit for bit.  128 tokens alone are 64 tiles, which the
    # library splits into K slices (another summation order: equal to f32 rounding); with the split switched off
    # (k_split = 1) the 128-token launch adds in the 512-token launch's order.
    xb2 = synth.bf16_round((2 * xf[:128]).reshape(-1))[1].reshape(128, cols)
    got2, _ = run(ctx, eng, w, rows, cols, 2 * xf[:128], xb2, 128, q6=True)
    assert_close(got2, 2 * got[:128], 2e-6, "K slices against the whole row")
    k1 = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, 128), (DType.Q6K, DType.BF16, DType.F32), (), dict(k_split=1)))
    assert "_kz" not in k1.name and k1.info.sched.k_split == 1
    y1 = ctx.buffer_empty_f32(128 * rows)
    ctx.encode_multi(k1, [ctx.buffer_bytes(w), ctx.buffer_bytes(xb2)], [y1])
    ctx.synchronize()
    assert np.array_equal(ctx.read_f32(y1, 128 * rows).reshape(128, rows), 2 * got[:128])


@pytest.mark.parametrize("wdt,xdt,batch,rows,cols,ks", [(DType.Q4K, DType.BF16, 200, 300, 1536, None), (DType.Q4K, DType.F32, 130, 256, 2048, 4),
                                                         (DType.Q6K, DType.F32, 70, 200, 1024, None), (DType.Q4K, DType.F32, 300, 2048, 512, None),
                                                         (DType.Q4K, DType.BF16, 256, 384, 8192, 8), (DType.Q4K, DType.F32, 65, 128, 256, None)])
def test_mul_mm_k_slices(ctx, wdt, xdt, batch, rows, cols, ks):
    """Few tiles: a row's superblocks go to K slices (rows of at least four superblocks), every slice stores its
    partial sums and a fold adds them in a fixed order.  Against the float64
    product at the accuracy of the whole-row launch (bf16 activations: 1e-3 against the oracle's f32 loop; f32
    activations: 2e-5), twice for bit-reproducibility, ragged tiles in both directions."""
    nb = rows * cols // 256
    w = synth.q4k_blocks(nb, 650) if wdt == DType.Q4K else synth.q6k_blocks(nb, 650)
    x = synth.normal_f32(batch * cols, 651).reshape(batch, cols)
    if xdt == DType.BF16:
        xf, xb = synth.bf16_round(x.reshape(-1))
        x, xin = xf.reshape(batch, cols), ctx.buffer_bytes(xb)
    else:
        xin = ctx.buffer_f32(x)
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, xdt, DType.F32), (), dict(k_split=ks) if ks else None))
    assert ("_kz" in k.name) == (k.info.sched.k_split > 1) == (cols >= 1024) and k.grid[2] == k.info.sched.k_split, (k.name, k.info.sched.k_split)
    assert (cols // 256) % k.info.sched.k_split == 0 and (ks is None or k.info.sched.k_split == ks)
    by, bw = ctx.buffer_empty_f32(batch * rows), ctx.buffer_bytes(w)
    runs = []
    for _ in range(2):
        ctx.encode_multi(k, [bw, xin], [by])
        ctx.synchronize()
        runs.append(ctx.read_f32(by, batch * rows).reshape(batch, rows))
    assert np.array_equal(runs[0], runs[1])
    odt = oracle.Q4K if wdt == DType.Q4K else oracle.Q6K
    worst = 0.0
    for t in range(0, batch, 7):
        worst = max(worst, float(rel_err(runs[0][t], oracle.matvec_f64(odt, w, rows, cols, x[t])).max()))
    assert worst <= 2e-5, worst


@pytest.mark.parametrize("xdt,batch,rows3,cols", [(DType.F32, 200, (384, 128, 128), 1024), (DType.BF16, 300, (2048, 256, 256), 512),
                                                  (DType.F32, 2048, (2048, 256, 256), 256), (DType.F32, 130, (200, 100, 0), 2048)])
def test_mul_mm_matrices_sharing_the_activations(ctx, xdt, batch, rows3, cols):
    """Up to three matrices over the same activations in one launch of the tile (q | k | v of a prompt chunk): every
    result against the float64 product and against the matrix's own launch, with K slices (few tiles) and as whole
    rows in two passes (2048 tokens), ragged row tiles, two matrices."""
    ws = [synth.q4k_blocks(r * cols // 256, 660 + i) for i, r in enumerate(rows3) if r]
    x = synth.normal_f32(batch * cols, 663).reshape(batch, cols)
    if xdt == DType.BF16:
        xf, xb = synth.bf16_round(x.reshape(-1))
        x, xin = xf.reshape(batch, cols), ctx.buffer_bytes(xb)
    else:
        xin = ctx.buffer_f32(x)
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows3[0], cols, batch, rows3[1], rows3[2]), (DType.Q4K, xdt, DType.F32)))
    assert k.name.endswith("_x%d" % len(ws)), k.name
    assert ("_kz" in k.name) == (cols >= 1024), k.name      # (rows of one or two superblocks: no slices)
    bws = [ctx.buffer_bytes(w) for w in ws]
    outs = [ctx.buffer_empty_f32(batch * r) for r in rows3 if r]
    ctx.encode_multi(k, [bws[0], xin] + bws[1:], outs)
    ctx.synchronize()
    for i, (w, r) in enumerate(zip(ws, [r for r in rows3 if r])):
        got = ctx.read_f32(outs[i], batch * r).reshape(batch, r)
        worst = max(float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, r, cols, x[t])).max()) for t in range(0, batch, 37))
        assert worst <= 2e-5, (i, worst)
        k1 = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (r, cols, batch), (DType.Q4K, xdt, DType.F32), (), dict(nr0=128)))
        y1 = ctx.buffer_empty_f32(batch * r)
        ctx.encode_multi(k1, [bws[i], xin], [y1])
        ctx.synchronize()
        assert_close(got, ctx.read_f32(y1, batch * r).reshape(batch, r), 2e-6, f"matrix {i} against its own launch")


@pytest.mark.parametrize("mode,batch,rows3,cols", [(1, 200, (384, 128, 128), 1536), (2, 96, (512, 512, 0), 2048), (3, 130, (256, 0, 0), 8192),
                                                   (1, 40, (300, 0, 0), 512), (2, 1056, (256, 0, 0), 512), (3, 70, (128, 0, 0), 12288)])
def test_mul_mm_with_the_rows_producer_inside(ctx, mode, batch, rows3, cols):
    """dims[5]: the producer of the rows runs inside the GEMM's preparation -- 1: rmsnorm(X, w); 2: x_new = res +
    rmsnorm(X, w_post) (stored, in place over res) and then rmsnorm(x_new, w_norm); 3: gelu(X) * up.  The rows the
    GEMM sees are the oracle's ops' results, the products against float64 at 2e-5; one to three
    matrices, K slices and whole rows, the small-batch form (40 tokens).  (x_new itself at 1e-5: its row sums are added
    in another order than the oracle's.)"""
    eps = 1e-6
    ws = [synth.q4k_blocks(r * cols // 256, 670 + i) for i, r in enumerate(rows3) if r]
    x = synth.normal_f32(batch * cols, 673).reshape(batch, cols)
    x[1] *= 40.0
    w0, w1 = 1.0 + 0.2 * synth.normal_f32(cols, 674), 1.0 + 0.2 * synth.normal_f32(cols, 675)
    res = synth.normal_f32(batch * cols, 676).reshape(batch, cols)
    up = synth.normal_f32(batch * cols, 677).reshape(batch, cols)
    bws = [ctx.buffer_bytes(w) for w in ws]
    ins, outs = [bws[0], ctx.buffer_f32(x)] + bws[1:], [ctx.buffer_empty_f32(batch * r) for r in rows3 if r]
    if mode == 1:
        ins.append(ctx.buffer_f32(w0))
        rows_in = np.stack([oracle.rmsnorm(x[t], w0, eps) for t in range(batch)])
    elif mode == 2:
        bres = ctx.buffer_f32(res)
        ins += [ctx.buffer_f32(w0), bres, ctx.buffer_f32(w1)]
        outs.append(bres)                                     # the new residual rows replace the old ones
        pairs = [oracle.rmsnorm_add_then_rmsnorm(x[t], w0, res[t], w1, eps) for t in range(batch)]
        x_new, rows_in = np.stack([p[0] for p in pairs]), np.stack([p[1] for p in pairs])
    else:
        ins.append(ctx.buffer_f32(up))
        rows_in = np.stack([oracle.gelu_mul(x[t], up[t]) for t in range(batch)])
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows3[0], cols, batch, rows3[1], rows3[2], mode), (DType.Q4K, DType.F32, DType.F32), (eps,)))
    ctx.encode_multi(k, ins, outs)
    ctx.synchronize()
    if mode == 2:
        assert_close(ctx.read_f32(bres, batch * cols).reshape(batch, cols), x_new, 1e-5, "new residual rows")
    for i, (w, r) in enumerate(zip(ws, [r for r in rows3 if r])):
        got = ctx.read_f32(outs[i], batch * r).reshape(batch, r)
        worst = max(float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, r, cols, rows_in[t])).max()) for t in range(0, batch, 13))
        assert worst <= 2e-5, (k.name, i, worst)


@pytest.mark.parametrize("batch", [96, 300])
def test_mul_mm_unfolded_results_feed_the_next_preparation(ctx, batch):
    """dims[6] = 1 leaves a GEMM's K slices as partial sums for a reader
    that adds them itself; dims[7] tells the next GEMM's prologue that its X is such a buffer.  The chain o-projection
    -> add-then-norm -> gate | up -> gelu * up -> down gives the very numbers of the same chain with every result
    folded by its own launch."""
    eps, hidden, ffn = 1e-6, 512, 1024
    wo, wg, wu, wd = (synth.q4k_blocks(r * c // 256, 680 + i) for i, (r, c) in enumerate(((hidden, hidden), (ffn, hidden), (ffn, hidden), (hidden, ffn))))
    bo, bg, bu, bd = (ctx.buffer_bytes(w) for w in (wo, wg, wu, wd))
    a = ctx.buffer_f32(synth.normal_f32(batch * hidden, 684))
    # (a small second norm weight keeps gelu(gate) * up of these synthetic weights inside the f16 range of the hi parts)
    w_post, w_norm = ctx.buffer_f32(1.0 + 0.2 * synth.normal_f32(hidden, 685)), ctx.buffer_f32(0.01 * (1.0 + 0.2 * synth.normal_f32(hidden, 686)))
    res0 = synth.normal_f32(batch * hidden, 687)
    f32 = (DType.Q4K, DType.F32, DType.F32)
    desc = lambda dims: hip.make_desc(hip.Kind.MATVEC_BATCH, dims, f32, (eps,))

    def run(kernel, ins, outs):
        ctx.encode_multi(kernel, ins, outs)
        ctx.synchronize()

    # folded: every GEMM finishes its own result
    y, g, u, out_a = (ctx.buffer_empty_f32(batch * n) for n in (hidden, ffn, ffn, hidden))
    res_a = ctx.buffer_f32(res0)
    run(ctx.compile(desc((hidden, hidden, batch))), [bo, a], [y])
    run(ctx.compile(desc((ffn, hidden, batch, ffn, 0, 2))), [bg, y, bu, w_post, res_a, w_norm], [g, u, res_a])
    run(ctx.compile(desc((hidden, ffn, batch, 0, 0, 3))), [bd, g, u], [out_a])
    # unfolded: the partial sums travel
    ko = ctx.compile(desc((hidden, hidden, batch, 0, 0, 0, 1)))
    zo = ko.grid[2]
    assert ko.name.endswith("_unfolded") and zo == ko.info.sched.k_split
    po = ctx.buffer_empty_f32(zo * batch * hidden)
    run(ko, [bo, a], [po])
    kg = ctx.compile(desc((ffn, hidden, batch, ffn, 0, 2, 1, zo)))
    zg = kg.grid[2]
    pg, res_b = ctx.buffer_empty_f32(zg * batch * 2 * ffn), ctx.buffer_f32(res0)
    run(kg, [bg, po, bu, w_post, res_b, w_norm], [pg, res_b])
    out_b = ctx.buffer_empty_f32(batch * hidden)
    run(ctx.compile(desc((hidden, ffn, batch, 0, 0, 3, 0, zg))), [bd, pg], [out_b])
    assert np.array_equal(ctx.read_f32(res_a, batch * hidden), ctx.read_f32(res_b, batch * hidden))
    assert np.array_equal(ctx.read_f32(out_a, batch * hidden), ctx.read_f32(out_b, batch * hidden))
    assert np.isfinite(ctx.read_f32(out_a, batch * hidden)).all() and np.abs(ctx.read_f32(out_a, batch * hidden)).max() > 0


@pytest.mark.parametrize("unfolded,k_split", [(0, 0), (1, 0), (0, 2), (1, 4)])
def test_mul_mm_f32_both_parts_in_one_workgroup(ctx, unfolded, k_split):
    """f32 activations on the tile: each row is scaled by its own power of two and split into two f16 parts at that
    scale, and every converted weight meets both parts in the same accumulator -- one launch, one result (or one set
    of partial sums; with K slices asked for, one per slice).  1024 tokens x 4096 rows x 1024 columns against
    float64; among the rows a small one, a large one, one far beyond the f16 range, one of zeros and one whose
    largest element is 10^7 times the others."""
    batch, rows, cols = 1024, 4096, 1024
    w = synth.q4k_blocks(rows * cols // 256, 690)
    x = synth.normal_f32(batch * cols, 691).reshape(batch, cols)
    x[3] *= 1e-3
    x[4] *= 300.0
    x[6] *= 1e12
    x[7] = 0.0
    x[8] *= 1e-3
    x[8, 5] = 1e4
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch, 0, 0, 0, unfolded), (DType.Q4K, DType.F32, DType.F32), (),
                                  dict(k_split=k_split) if k_split else None))
    nz = max(1, k_split)
    assert k.grid[2] == nz and ("_kz" in k.name) == bool(unfolded or k_split), (k.name, k.grid)
    y = ctx.buffer_empty_f32(nz * batch * rows if unfolded else batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), ctx.buffer_f32(x)], [y])
    ctx.synchronize()
    if unfolded:
        got = ctx.read_f32(y, nz * batch * rows).reshape(nz, batch, rows).astype(np.float64).sum(axis=0)
    else:
        got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    worst = max(float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, rows, cols, x[t])).max()) for t in (0, 3, 4, 5, 6, 8, 511, 1023))
    assert worst <= 2e-5, worst
    assert not got[7].any()


@pytest.mark.parametrize("rows,batch,cols,mode,shape", [
    (1, 65, 256, 0, "32x128"), (257, 33, 768, 0, "32x128"), (255, 96, 7936, 0, "32x128"), (300, 129, 1024, 2, "32x256"),
    (129, 65, 512, 3, "32x256"), (4095, 1000, 256, 0, "64x256"), (7937, 545, 512, 3, "64x256")])
def test_mul_mm_f32_rows_at_the_edges_of_its_tiles(ctx, rows, batch, cols, mode, shape):
    """Both shapes of the f32 rows' kernel where they can go wrong: one superblock and thirty-one, a row or a token past a
    tile or short of it, two matrices side by side (gelu(gate) * up), rows summed as in launches of their own.  Against
    float64 at the bar of the others (two f16 parts hold 22 bits of a row's largest, f32 sums: 2e-5); rows cut as in
    launches of their own against those launches, bit for bit."""
    ws = [ctx.buffer_bytes(synth.q4k_blocks(rows * cols // 256, 700 + i)) for i in range(2)]
    xs = synth.normal_f32(batch * cols, 702).reshape(batch, cols)
    x = ctx.buffer_f32(xs)

    def launch(dims, ins, sched=None):
        k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, dims, (DType.Q4K, DType.F32, DType.F32), (), sched))
        y = ctx.buffer_empty_f32(dims[2] * rows)
        ctx.encode_multi(k, ins, [y])
        ctx.synchronize()
        return k, ctx.read_f32(y, dims[2] * rows).reshape(dims[2], rows)

    if mode == 2:
        lens = [70, batch - 70] if batch - 70 <= 64 else [batch]     # (a prompt of up to 64 rows is summed as one of 65)
        as_ = np.concatenate([np.full(n, max(n, 65), np.float32) for n in lens])
        k, got = launch((rows, cols, batch, 0, 0, 0, 2), [ws[0], x, ctx.buffer_f32(as_)])
        for n, at in zip(lens, np.cumsum([0] + lens[:-1])):
            pad = np.zeros((max(n, 65), cols), np.float32)
            pad[:n] = xs[at:at + n]
            _, want = launch((rows, cols, len(pad)), [ws[0], ctx.buffer_f32(pad)], dict(nr0=128))
            assert np.array_equal(got[at:at + n], want[:n]), (n, at)
    else:
        dims = (rows, cols, batch, rows, 0, 0, 3) if mode == 3 else (rows, cols, batch)
        k, got = launch(dims, [ws[0], x, ws[1]] if mode == 3 else [ws[0], x], dict(k_split=1, nr0=128 if mode == 0 else 0))
        for t in sorted({0, 31, 32, batch // 2, batch - 1}):
            want = [oracle.matvec_f64(oracle.Q4K, synth.q4k_blocks(rows * cols // 256, 700 + i), rows, cols, xs[t]) for i in range(2)]
            if mode == 3:
                g = np.clip(want[0], -20.0, 20.0)     # (the kernels' gelu: tanh of a cubic, its argument held to +-20)
                want = 0.5 * g * (1.0 + np.tanh(0.7978845608 * (g + 0.044715 * g ** 3))) * want[1]
                # (either factor off by 2e-5 of its rms or value, the other up to four times its rms, gelu' <= 1.13, against a
                # product of at least 0.6 of the two rms: 2 * 4 * 1.13 / 0.6 * 2e-5)
                assert rel_err(got[t], want).max() <= 3e-4, t
            else:
                assert rel_err(got[t], want[0]).max() <= 2e-5, t
    assert shape in k.name, k.name


@pytest.mark.parametrize("rows,batch,cols,ks,shape", [
    (1, 2, 256, 1, "64x128"), (129, 65, 768, 1, "64x128"), (257, 63, 7936, 7, "64x128"), (127, 193, 2816, 11, "64x128"),
    (8193, 1025, 4096, 1, "128x128"), (4095, 1023, 1280, 5, "128x128")])
def test_mul_mm_bf16_rows_at_the_edges_of_its_tiles(ctx, rows, batch, cols, ks, shape):
    """Both shapes of the bf16 rows' kernel where they can go wrong: one superblock, a row or a token past a tile or short of
    it, slices of unequal length and of one superblock.  Against float64: bf16 values of normal size and codes times scales
    are exact in f16, the sums of x hold 22 bits, sums are f32 (2e-5, as for f32 rows)."""
    w = synth.q4k_blocks(rows * cols // 256, 730)
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 731))
    xs = xf.reshape(batch, cols)
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (DType.Q4K, DType.BF16, DType.F32), (),
                                  dict(nr0=128, tg=256, lds_tile=32, k_split=ks)))
    assert f"_{shape}x32" in k.name and k.info.sched.k_split == ks
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), ctx.buffer_bytes(xb)], [y])
    ctx.synchronize()
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    for t in sorted({0, 1, 31, 32, 62, 63, 64, 127, 128, batch - 2, batch - 1} & set(range(batch))):
        assert float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, rows, cols, xs[t])).max()) <= 2e-5, t


@pytest.mark.parametrize("xdt", [DType.F32, DType.BF16])
@pytest.mark.parametrize("rows,batch,cols", [(1, 2, 1024), (31, 32, 1280), (33, 33, 2048), (65, 64, 2304), (300, 3, 6400), (97, 50, 4096)])
def test_mul_mm_small_batch_edges(ctx, xdt, rows, batch, cols):
    """The small-batch form on both sides of its rule for the weights' way in (4 and 5, 8 and 9 superblocks; one and two parts; up to and
    past 32 tokens), waves without a superblock, with one and with several, a row past a tile or short of it.  Against float64:
    2e-5, as for the tiles."""
    w = synth.q4k_blocks(rows * cols // 256, 735)
    x = synth.normal_f32(batch * cols, 736)
    xb = ctx.buffer_f32(x)
    if xdt == DType.BF16:
        x, raw = synth.bf16_round(x)
        xb = ctx.buffer_bytes(raw)
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (DType.Q4K, xdt, DType.F32), (), dict(nr0=32)))
    assert "skinny" in k.name
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), xb], [y])
    ctx.synchronize()
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    for t in range(batch):
        assert float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, rows, cols, x.reshape(batch, cols)[t])).max()) <= 2e-5, t


@pytest.mark.parametrize("dims,xdt", [((512, 1024, 8), DType.F32), ((512, 1024, 1025), DType.BF16), ((512, 1024, 8, 512), DType.BF16)])
def test_mul_mm_few_tokens_refused(ctx, dims, xdt):
    """A schedule that names the form of one launch for what it does not take: an error, not another form."""
    with pytest.raises(RuntimeError):
        ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, dims, (DType.Q4K, xdt, DType.F32), (), dict(nr0=16)))


@pytest.mark.parametrize("wdt", [DType.Q4K, DType.Q6K])
@pytest.mark.parametrize("rows,batch,cols,rh", [(37, 5, 256, 1), (40, 16, 2304, 2), (70, 7, 1024, 4), (33, 29, 768, 1), (50, 75, 512, 1)])
def test_mul_mm_few_tokens_keep_their_infinities(ctx, wdt, rows, batch, cols, rh):
    """In the form of one launch a token with an infinity or no number is not finite, nor is a weight row with such a scale; every
    other result has the bits that it has without them."""
    size, at = (144, 0) if wdt == DType.Q4K else (210, 208)
    w = (synth.q4k_blocks if wdt == DType.Q4K else synth.q6k_blocks)(rows * cols // 256, 747)
    x, raw = synth.bf16_round(synth.normal_f32(batch * cols, 748))
    hurt, hurt_x = w.copy(), np.asarray(raw).view(np.uint16).copy().reshape(batch, cols)
    bad_rows, bad_tokens = {0: 0x7E00, 17: 0x7C00, rows - 1: 0xFC00}, {0: 0x7F80, batch // 2: 0x7FC0, batch - 1: 0xFF80}
    for r, bits in bad_rows.items():
        hurt.reshape(rows, cols // 256, size)[r, r % (cols // 256), at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
    for t, bits in bad_tokens.items():
        hurt_x[t, (37 * t + 5) % cols] = bits
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32), (), dict(nr0=16, unroll=rh)))
    assert "few" in k.name
    got = []
    for ww, xx in ((w, np.asarray(raw).view(np.uint16)), (hurt, hurt_x)):
        y = ctx.buffer_f32(np.zeros(batch * rows, np.float32))
        ctx.encode_multi(k, [ctx.buffer_bytes(ww), ctx.buffer_bytes(np.ascontiguousarray(xx).view(np.uint8))], [y])
        got.append(ctx.read_f32(y, batch * rows).reshape(batch, rows))
    touched = np.zeros((batch, rows), bool)
    touched[list(bad_tokens)] = True
    touched[:, list(bad_rows)] = True
    assert np.all(np.isfinite(got[0])) and not np.any(np.isfinite(got[1][touched]))
    assert np.array_equal(got[0][~touched].view(np.uint32), got[1][~touched].view(np.uint32))


@pytest.mark.parametrize("wdt,rows,cols,batch,few", [
    (DType.Q4K, 19, 24576, 5, False), (DType.Q6K, 64, 16384, 1000, False), (DType.Q4K, 300, 8448, 3, False), (DType.Q4K, 300, 8192, 3, True),
    (DType.Q6K, 128, 8192, 512, False), (DType.Q6K, 128, 8192, 256, True), (DType.Q6K, 128, 4096, 512, True), (DType.Q4K, 65536, 256, 1, False),
    (DType.Q4K, 14412, 256, 21, False), (DType.Q4K, 12300, 256, 9, True), (DType.Q6K, 10728, 256, 2, True)])
def test_mul_mm_few_tokens_left_open(ctx, wdt, rows, cols, batch, few):
    """Where an open call takes the form of one launch: not outside the sizes that its estimate holds for.  Either form against float64."""
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32)))
    assert ("few" in k.name) == few, k.name
    w = (synth.q4k_blocks if wdt == DType.Q4K else synth.q6k_blocks)(rows * cols // 256, 743)
    x, raw = synth.bf16_round(synth.normal_f32(batch * cols, 744))
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), ctx.buffer_bytes(raw)], [y])
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    for t in sorted({0, batch // 2, batch - 1}):
        want = oracle.matvec_f64(oracle.Q4K if wdt == DType.Q4K else oracle.Q6K, w, rows, cols, x.reshape(batch, cols)[t])
        assert np.abs(got[t] - want).max() <= (2e-5 if wdt == DType.Q4K or few else 1e-3) * max(np.abs(want).max(), np.abs(x.reshape(batch, cols)[t]).max()), t


@pytest.mark.parametrize("wdt,off", [(DType.Q4K, 0), (DType.Q6K, 0), (DType.Q6K, 14), (DType.Q6K, 6)])
@pytest.mark.parametrize("rows,batch,cols,rh", [(1, 1, 256, 1), (15, 2, 1792, 1), (17, 15, 2048, 2), (33, 16, 2304, 4), (65, 17, 4096, 1), (129, 31, 768, 1), (200, 32, 6400, 1),
                                                (63, 3, 8192, 4), (5000, 16, 512, 2), (12300, 9, 256, 4), (3000, 32, 2048, 0), (1000, 7, 2048, 0),
                                                (300, 33, 1024, 0), (250, 192, 768, 0), (250, 333, 768, 1), (70, 100, 2304, 1), (18, 1024, 256, 2)])
def test_mul_mm_few_tokens_edges(ctx, rows, batch, cols, rh, wdt, off):
    """The form of one launch: rows short of a tile and past one, odd numbers of tokens, waves without a superblock and with several, every
    number of row tiles, by schedule and left open; rows of activations of very different size, beyond f16's range too; Q6_K blocks at
    several two-byte addresses.  Against float64: 2e-5 of the largest result of the token, as for the tiles."""
    w = (synth.q4k_blocks if wdt == DType.Q4K else synth.q6k_blocks)(rows * cols // 256, 739)
    if wdt == DType.Q6K and rh == 4 and batch > 8:
        rh = 2             # (what a compute unit's LDS holds)
    x = synth.normal_f32(batch * cols, 740).reshape(batch, cols)
    x[batch // 2] *= 1e-9
    x[-1] *= 3e7
    x, raw = synth.bf16_round(x.ravel())
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32), (), dict(nr0=16, unroll=rh) if rh else None))
    assert "few" in k.name and (not rh or k.info.sched.unroll == rh)
    again = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32), (), k.info.sched))
    assert again.name == k.name
    y = ctx.buffer_f32(np.full(batch * rows + 64, 7.0, np.float32))
    ctx.encode_offsets_multi(k, [ctx.buffer_bytes(np.concatenate([np.full(off, 0xA5, np.uint8), w])), ctx.buffer_bytes(raw)], [off, 0], [y], [0])
    got = ctx.read_f32(y, batch * rows + 64)
    assert np.all(got[batch * rows:] == 7.0)
    for t in sorted({*range(min(batch, 40)), batch // 2, *range(max(0, batch - 35), batch)}):
        want = oracle.matvec_f64(oracle.Q4K if wdt == DType.Q4K else oracle.Q6K, w, rows, cols, x.reshape(batch, cols)[t])
        assert np.abs(got[t * rows:(t + 1) * rows] - want).max() <= 2e-5 * max(np.abs(want).max(), np.abs(x.reshape(batch, cols)[t]).max()), t


@pytest.mark.parametrize("xdt,cols,batch,pieces", [
    (DType.BF16, 256, 1, False), (DType.BF16, 1024, 32, False), (DType.BF16, 1280, 32, True), (DType.BF16, 1792, 33, False), (DType.BF16, 2048, 33, True), (DType.BF16, 2304, 32, True),
    (DType.F32, 1280, 32, False), (DType.F32, 2048, 5, True), (DType.F32, 2304, 31, False), (DType.F32, 2560, 3, False),
    (DType.F32, 3072, 32, False), (DType.F32, 3328, 32, True), (DType.F32, 2048, 33, False)])
def test_mul_mm_small_batch_way_in(ctx, xdt, cols, batch, pieces):
    """Which way the weights of the small-batch form come in, by pieces through LDS or a row a lane, on both sides of every line
    of its rule, and the result there against float64 (2e-5, as for the tiles)."""
    rows = 45
    w = synth.q4k_blocks(rows * cols // 256, 737)
    x = synth.normal_f32(batch * cols, 738)
    xb = ctx.buffer_f32(x)
    if xdt == DType.BF16:
        x, raw = synth.bf16_round(x)
        xb = ctx.buffer_bytes(raw)
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (DType.Q4K, xdt, DType.F32), (), dict(nr0=32)))
    wave = 64 * 16 * 4 if batch <= 32 else 2 * 64 * 16 * 4
    assert k.info.lds_bytes == 8 * (max(wave, 32 * 144) if pieces else wave)
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), xb], [y])
    ctx.synchronize()
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    for t in {0, batch // 2, batch - 1}:
        assert float(rel_err(got[t], oracle.matvec_f64(oracle.Q4K, w, rows, cols, x.reshape(batch, cols)[t])).max()) <= 2e-5, t


@pytest.mark.parametrize("rows,batch,cols,ks,at,shape", [
    (1, 1, 256, 1, 0, "32x128"), (33, 31, 768, 3, 2, "32x128"), (129, 33, 2816, 7, 14, "32x128"), (127, 32, 256, 1, 6, "32x128"),
    (4095, 65, 2816, 1, 10, "32x128"), (4097, 63, 6144, 8, 8, "64x128"), (4130, 64, 7936, 5, 4, "64x128"), (4223, 193, 768, 1, 12, "32x128")])
def test_mul_mm_q6k_few_bf16_rows(ctx, rows, batch, cols, ks, at, shape):
    """The Q6_K kernel of 32 or 64 tokens a workgroup where it can go wrong: a row or a token past a tile or short of it, slices
    of unequal length and of one superblock, blocks from any even address on (rows of 210 bytes begin at every one of eight).
    Against float64: these scales times codes stay below 2^11 and bf16 values are normal, both exact in f16; f32 sums (2e-5)."""
    w = synth.q6k_blocks(rows * cols // 256, 740)
    bw = ctx.buffer_bytes(bytes(at) + bytes(w))
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 741))
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (DType.Q6K, DType.BF16, DType.F32), (),
                                  dict(nr0=128, tg=256, lds_tile=64, k_split=ks)))
    assert f"_{shape}x64" in k.name and k.info.sched.k_split == ks, k.name
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_offsets_multi(k, [bw, ctx.buffer_bytes(xb)], [at, 0], [y], None)
    ctx.synchronize()
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    for t in sorted({0, 1, 30, 31, 32, 62, 63, 64, batch - 1} & set(range(batch))):
        want = oracle.matvec_f64(oracle.Q6K, w, rows, cols, xf.reshape(batch, cols)[t])
        assert rel_err(got[t], want).max() <= 2e-5, t


@pytest.mark.parametrize("rows,batch,prologue", [(31, 33, 0), (97, 64, 2), (200, 130, 0), (4130, 1000, 2)])
def test_mul_mm_f32_gate_up_pair(ctx, rows, batch, prologue):
    """dims[6] = 3: gelu(W x) * (W1 x) from one launch is the two matrices' products and KSH_GELU_MUL (64 rows of each
    matrix a tile; ragged in both directions)."""
    cols = 512 if prologue else 768
    ws = [ctx.buffer_bytes(synth.q4k_blocks(rows * cols // 256, 670 + i)) for i in range(2)]
    x, res, wv = (ctx.buffer_f32(synth.normal_f32(n, 672 + i)) for i, n in enumerate((batch * cols, batch * cols, cols)))
    pro = [wv, res, wv] if prologue else []
    outs = []
    for mode in (0, 3):
        k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch, rows, 0, prologue, mode), (DType.Q4K, DType.F32, DType.F32), (1e-6,),
                                      dict(k_split=1)))
        ys = [ctx.buffer_empty_f32(batch * rows) for _ in range(1 if mode else 2)]
        xn = [ctx.buffer_empty_f32(batch * cols)] if prologue else []
        ctx.encode_multi(k, [ws[0], x, ws[1]] + pro, ys + xn)
        if not mode:
            y = ctx.buffer_empty_f32(batch * rows)
            ctx.encode_multi(ctx.compile(hip.make_desc(hip.Kind.GELU_MUL, (batch * rows,))), ys, [y])
            ys = [y]
        ctx.synchronize()
        outs.append([ctx.read_f32(ys[0], batch * rows)] + [ctx.read_f32(b, batch * cols) for b in xn])
    assert_close(outs[1][0], outs[0][0], 1e-5, "gelu(gate) * up")
    if prologue:
        assert np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("wdt,batch,rows,cols", [(DType.Q6K, 77, 300, 7936), (DType.Q4K, 77, 300, 7936), (DType.Q4K, 64, 129, 7936),
                                                 (DType.Q6K, 1, 129, 2816), (DType.Q6K, 257, 10881, 1536), (DType.Q4K, 321, 7041, 768)])
def test_mul_mm_bf16_default_tile_and_slices(ctx, wdt, batch, rows, cols):
    """The launch bf16 rows get by themselves: slices of unequal length (31 and 11 superblocks), Q6_K products reading the
    rows of X as they are and behind a preparation (two rounds of tiles), tiles of 64 tokens two to a compute unit;
    ragged in both directions."""
    nb = rows * cols // 256
    w = synth.q4k_blocks(nb, 660) if wdt == DType.Q4K else synth.q6k_blocks(nb, 660)
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 661))
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32)))
    by = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), ctx.buffer_bytes(xb)], [by])
    ctx.synchronize()
    got = ctx.read_f32(by, batch * rows).reshape(batch, rows)
    odt = oracle.Q4K if wdt == DType.Q4K else oracle.Q6K
    for t in sorted({0, batch // 2, batch - 1}):
        assert_close(got[t], oracle.matvec_f64(odt, w, rows, cols, xf.reshape(batch, cols)[t]), 1e-4, f"{k.name} t={t}")


def test_mul_mm_k_slices_must_divide_the_row(ctx):
    with pytest.raises(hip.KshError, match="does not divide"):
        ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (256, 2048, 100), (DType.Q4K, DType.BF16, DType.F32), (), dict(k_split=3)))


@pytest.mark.parametrize("wdt,batch,rows,cols", [(DType.Q6K, 512, 300, 7936), (DType.Q4K, 512, 300, 7936), (DType.Q6K, 300, 1000, 2816),
                                                 (DType.Q4K, 40, 256, 2048)])
def test_mul_mm_reported_schedule_binds_again(ctx, wdt, batch, rows, cols, tmp_path, monkeypatch):
    """The schedule a bf16 launch reports (slice counts that divide 31 or 11 superblocks unevenly; the small-batch form) and
    the one a search saves are taken again, as an argument and from the plan file: the same launch, the same bits."""
    monkeypatch.setenv("KSEARCH_BEAM_CACHE", str(tmp_path / "beam"))
    nb = rows * cols // 256
    bw = ctx.buffer_bytes(synth.q4k_blocks(nb, 662) if wdt == DType.Q4K else synth.q6k_blocks(nb, 662))
    bx, by = ctx.buffer_bytes(synth.bf16_round(synth.normal_f32(batch * cols, 663))[1]), ctx.buffer_empty_f32(batch * rows)

    def desc(sched=None):
        return hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32), (), sched)

    def launch(k):
        ctx.encode_multi(k, [bw, bx], [by])
        ctx.synchronize()
        return k.name, tuple(k.grid), ctx.read_f32(by, batch * rows).tobytes()

    k = ctx.compile(desc())
    ks, nsb = k.info.sched.k_split, cols // 256
    assert nsb == 8 or nsb % ks, "the shape is here for a count that does not divide its superblocks"
    want = launch(k)
    assert launch(ctx.compile(desc(k.info.sched))) == want
    best, _, _ = ctx.beam_search(desc(), [bw, bx], [by], iters=3, force=True)
    ctx.compile(desc(best))
    # a plan file with that schedule, found by a context that has not bound the shape yet
    hip.plan_save(hip.plan_kind(desc()), (rows, cols, batch), ctx.device_name(), k.info.sched, 0.001)
    other = hip.Context()
    planned = other.compile(desc())
    assert (planned.name, tuple(planned.grid)) == want[:2]
    other.close()
    if nsb != 8:   # a bare count is held to divisors, as it was
        with pytest.raises(hip.KshError, match="does not divide"):
            ctx.compile(desc(dict(k_split=ks)))


def test_mul_mm_cfg2_full_size(ctx, eng):
    tokens, rows, cols = 512, 8192, 2048
    w, xf, xb = synth.cfg2_q4k_prefill()
    got, want = run(ctx, eng, w, rows, cols, xf, xb, tokens)
    assert_close(got, want, 1e-3, "cfg2")
    # linearity in X (size-independent property): W(2x) = 2 W(x) exactly in binary floating point
    # (on the first 128 tokens, none of whose values is small enough to lose bits as an f16 subnormal.  128 tokens alone
    # are 64 tiles, which the library would split into K slices -- the same sums in another order -- so the exact
    # check asks for whole rows, k_split = 1, and the default launch is held to f32 rounding.)
    xb2 = synth.bf16_round((2 * xf[:128]).reshape(-1))[1].reshape(128, cols)
    k1 = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, 128), (DType.Q4K, DType.BF16, DType.F32), (), dict(k_split=1)))
    assert "_kz" not in k1.name
    y1 = ctx.buffer_empty_f32(128 * rows)
    ctx.encode_multi(k1, [ctx.buffer_bytes(w), ctx.buffer_bytes(xb2)], [y1])
    ctx.synchronize()
    assert np.array_equal(ctx.read_f32(y1, 128 * rows).reshape(128, rows), 2 * got[:128])
    got3, _ = run(ctx, eng, w, rows, cols, xf[:128], xb[:128], 128)
    assert_close(got3, got[:128], 2e-6, "K slices against the whole row")


def test_mul_mm_errors(ctx):
    with pytest.raises(hip.KshError, match="not built"):
        ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (64, 256, 16), (DType.Q40, DType.BF16, DType.F32)))
    with pytest.raises(hip.KshError, match="multiple of 256"):
        ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (64, 100, 16), (DType.Q4K, DType.BF16, DType.F32)))


@pytest.mark.parametrize("wdt", [DType.Q4K, DType.Q6K])
@pytest.mark.parametrize("xdt", [DType.F32, DType.BF16])
@pytest.mark.parametrize("rows,cols,batch", [(2048, 2048, 256), (300, 7936, 40), (1536, 6144, 333), (8192, 2048, 512), (256, 512, 2)])
def test_mul_mm_candidates_are_what_their_handles_report(ctx, wdt, xdt, rows, cols, batch):
    """A schedule from the search's list binds, and the bound kernel reports the same tile and slices."""
    dims, dtypes = (rows, cols, batch), (wdt, xdt, DType.F32)
    for s in hip.beam_candidates(hip.make_desc(hip.Kind.MATVEC_BATCH, dims, dtypes)):
        got = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, dims, dtypes, (), s.as_dict())).info.sched
        assert all(getattr(got, f) == getattr(s, f) for f in ("tg", "nsg", "nr0", "lds_tile", "k_split")), (s.as_dict(), got.as_dict())


@pytest.mark.parametrize("wdt,rows,batch,cols,ks,shape", [
    (DType.Q6K, 4000, 1023, 4096, 1, "128x128"), (DType.Q6K, 3999, 1023, 4096, 1, "128x128"),
    (DType.Q4K, 297, 10, 7424, 29, "64x128"), (DType.Q4K, 2049, 100, 2048, 8, "64x128"), (DType.Q4K, 8193, 1025, 4096, 4, "128x128"),
    (DType.Q6K, 502, 31, 3584, 14, "32x128"), (DType.Q6K, 3371, 65, 2304, 9, "128x128"), (DType.Q6K, 2549, 733, 3072, 2, "128x128"),
    (DType.Q6K, 3000, 63, 2304, 8, "64x128")])
def test_mul_mm_bf16_partial_sums_kept_and_past(ctx, wdt, rows, batch, cols, ks, shape):
    """Partial sums of bf16 rows that stay in the L2s for the fold (small ones, and large results in few slices) and that go past them,
    of every shape of workgroup, and whole results of the tile of two roles in whole pieces of 64 bytes and not.  Against float64: 2e-5, as for the tiles."""
    w = (synth.q6k_blocks if wdt == DType.Q6K else synth.q4k_blocks)(rows * cols // 256, 745)
    xf, xb = synth.bf16_round(synth.normal_f32(batch * cols, 746))
    k = ctx.compile(hip.make_desc(hip.Kind.MATVEC_BATCH, (rows, cols, batch), (wdt, DType.BF16, DType.F32), (),
                                  dict(nr0=128, tg=256, lds_tile=64 if wdt == DType.Q6K else 32, k_split=ks)))
    assert f"_{shape}x" in k.name and k.info.sched.k_split == ks, k.name
    y = ctx.buffer_empty_f32(batch * rows)
    ctx.encode_multi(k, [ctx.buffer_bytes(w), ctx.buffer_bytes(xb)], [y])
    ctx.synchronize()
    got = ctx.read_f32(y, batch * rows).reshape(batch, rows)
    fmt = oracle.Q6K if wdt == DType.Q6K else oracle.Q4K
    for t in sorted({0, 1, batch // 2, batch - 1}):
        assert float(rel_err(got[t], oracle.matvec_f64(fmt, w, rows, cols, xf.reshape(batch, cols)[t])).max()) <= 2e-5, t
