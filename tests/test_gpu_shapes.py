"""Kernels at the sizes where their tilings can go wrong (partial tiles, remainders, the smallest and
largest of a dispatch's range), against the oracle under the reference's per-kernel tolerance."""
import numpy as np
import pytest

from modelspec_amd import api
from ops_lib import Prog, fast_values, within
from test_gpu_heldout import batches_of, load_logits
from test_gpu_ops import both

pytestmark = pytest.mark.gpu


def attention_case(ctx, oracle, B, L, S, H, heads):
    """Attention and its three gradients, random masked keys: results, oracle's, mask and bound."""
    q, G = (fast_values(s, B * L * H, 0.5).reshape(B * L, H) for s in (12, 15))
    k, v = (fast_values(s, B * S * H, 0.5).reshape(B * S, H) for s in (13, 14))
    mask = (np.random.default_rng(S).random((B, S)) < 0.7).astype(np.float32)
    mask[:, S // 2] = 1.0
    p = Prog()
    qi, ki, vi = p.input("q", (B * L, H)), p.input("k", (B * S, H)), p.input("v", (B * S, H))
    mi, Gi = p.input("mask", (B, S)), p.input("G", (B * L, H))
    attr = f"[heads = {heads}]"
    outs = [p.op("Attention", [qi, ki, vi, mi], (B * L, H), attr)]
    for op, rows in (("AttentionGradQ", B * L), ("AttentionGradK", B * S), ("AttentionGradV", B * S)):
        outs.append(p.op(op, [qi, ki, vi, mi, Gi], (rows, H), attr))
    got, want = both(ctx, oracle, p.out(*outs), {"q": q, "k": k, "v": v, "mask": mask, "G": G}, (0, 1, 2, 3))
    # r: sum over keys of |p| |v|-like terms, bounded by the largest row magnitudes.
    scale = np.abs(v).max() + np.abs(G).max() * (np.abs(q).max() + np.abs(k).max()) * np.sqrt(H // heads) * 2
    return got, want, mask, scale


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("B,L,S,H,heads", [
    (1, 1, 1, 16, 1), (2, 15, 15, 32, 2), (2, 17, 17, 64, 1), (3, 100, 100, 192, 3), (1, 150, 150, 64, 1),
    (2, 33, 33, 128, 1),     # head width 128: two-wave blocks, tiles of 32 rows
    (3, 300, 300, 32, 2),    # several streamed tiles, the last of 44 rows
    (43, 100, 100, 224, 14),  # over 4096 row tiles: four-wave blocks streaming 32-row tiles
    (2, 20, 48, 64, 2),      # fewer queries than keys, whole key tiles
    (2, 528, 528, 128, 2),   # long sequences: 64-row tiles forward, 32-row backward, partial last ones
    (1, 140, 144, 64, 1),    # the shortest of these, fewer queries than keys
])
def test_attention_over_partial_tiles(ctx, oracle, B, L, S, H, heads, mixed):
    """Partial tiles of rows, in f32 (also under mixed precision where a row count is no multiple of 16):
    rows past the end take no part and are not written, masked keys' gradients are +0."""
    if mixed and L % 16 == 0 and S % 16 == 0:
        pytest.skip("whole tiles under mixed precision are the f16 kernels', tested with them")
    ctx.set_precision(mixed)
    try:
        got, want, mask, scale = attention_case(ctx, oracle, B, L, S, H, heads)
    finally:
        ctx.set_precision(False)
    for idx, (g, w) in enumerate(zip(got, want)):
        ok, worst = within(g, w, np.abs(w) + scale)
        assert ok, (idx, worst)
    for g in (got[2], got[3]):
        assert np.all(g.reshape(B * S, H)[mask.reshape(-1) == 0] == 0)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("B,L,S,H,heads", [(2, 17, 17, 64, 1), (3, 100, 100, 192, 3), (1, 150, 150, 64, 1), (2, 20, 48, 64, 2),
                                           (2, 33, 33, 128, 1), (2, 90, 300, 32, 2), (43, 100, 100, 224, 14)])
def test_attention_over_partial_tiles_leaves_masked_keys_out(ctx, oracle, B, L, S, H, heads, mixed):
    """What a masked key and its value hold (NaN, infinities) reaches no result, and a run of live keys
    whose scores all overflow to -inf (those of a whole tile, before the first finite score) has
    probability 0: the oracle's values, which reads unmasked keys only."""
    rng = np.random.default_rng(S + H)
    q, G = (rng.uniform(0.1, 1.0, (B * L, H)).astype(np.float32) for _ in range(2))
    k, v = (rng.uniform(-1.0, 1.0, (B, S, H)).astype(np.float32) for _ in range(2))
    mask = (rng.random((B, S)) < 0.6).astype(np.float32)
    mask[:, S - 1] = 1.0
    k[:, :S * 2 // 3] = -3e38
    k[mask == 0], v[mask == 0] = np.nan, np.inf
    v[(mask == 0) & (np.arange(S) % 2 == 0)] = np.nan
    p = Prog()
    qi, ki, vi = p.input("q", (B * L, H)), p.input("k", (B * S, H)), p.input("v", (B * S, H))
    mi, Gi = p.input("mask", (B, S)), p.input("G", (B * L, H))
    attr = f"[heads = {heads}]"
    outs = [p.op("Attention", [qi, ki, vi, mi], (B * L, H), attr)]
    for op, rows in (("AttentionGradQ", B * L), ("AttentionGradK", B * S), ("AttentionGradV", B * S)):
        outs.append(p.op(op, [qi, ki, vi, mi, Gi], (rows, H), attr))
    inputs = {"q": q, "k": k.reshape(B * S, H), "v": v.reshape(B * S, H), "mask": mask, "G": G}
    ctx.set_precision(mixed)
    try:
        got, want = both(ctx, oracle, p.out(*outs), inputs, (0, 1, 2, 3))
    finally:
        ctx.set_precision(False)
    # |values| of at most 1: the bound of attention_case with unit magnitudes.
    for idx, (g, w) in enumerate(zip(got, want)):
        assert np.all(np.isfinite(w)), idx
        ok, worst = within(g, w, np.abs(w) + 1 + 4 * np.sqrt(H // heads))
        assert ok, (idx, worst)


def f16(x):
    return np.asarray(x, np.float32).astype(np.float16).astype(np.float64)


@pytest.fixture
def mixed(ctx):
    ctx.set_precision(True)
    yield ctx
    ctx.set_precision(False)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,k,n", [
    (8000, 72, 1496),   # 256 x 192 tiles (128 x 128 for both operands transposed), a K tail of 8
    (2000, 136, 2104),  # 128 x 128 tiles, partial ones at both edges, a K tail of 8
    (1000, 520, 1096),  # 64 x 64 tiles
    (1000, 24, 1096),   # one partial K tile
    (72, 1032, 88),     # 64 x 32 tiles, a K tail of 8
    (8, 256, 8),        # one partial tile
    (296, 9000, 200),   # split-K slices and their sum
    (520, 2052, 260),   # rows of 4 mod 8 halves: the other kernel's 128 x 128 tiles, K in slices
    (260, 1028, 516),   # the same, slices of 32 K and a K tail of 4
])
def test_mixed_gemm_tiles(mixed, m, k, n, ta, tb):
    """Every tile of the f16 GEMM at partial tiles and K tails, against the float64 product of the
    f16 operands (1e-5 of the sum of |terms|, f32 accumulation)."""
    rng = np.random.default_rng(m + k)
    a = rng.standard_normal((k, m) if ta else (m, k)).astype(np.float32)
    b = rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32)
    p = Prog()
    ai, bi = p.input("a", a.shape), p.input("b", b.shape)
    lhs = p.op("Transpose", [ai], (m, k)) if ta else ai
    rhs = p.op("Transpose", [bi], (k, n)) if tb else bi
    p.out(p.op("MatMul", [lhs, rhs], (m, n)))
    prog = mixed.program(p.text())
    prog.run({"a": a, "b": b})
    got = prog.output(0, m * n).reshape(m, n)
    A, Bm = f16(a.T if ta else a), f16(b.T if tb else b)
    bound = 1e-5 * (np.abs(A) @ np.abs(Bm)) + 1e-30
    worst = np.max(np.abs(got - A @ Bm) / bound)
    assert worst <= 1.0, worst


@pytest.mark.parametrize("rows,h,f", [(64, 64, 256), (2048, 256, 1024), (4096, 320, 1280), (304, 96, 392)])
def test_mixed_ffn_on_f16_values(mixed, rows, h, f):
    """gelu(x w1 + b1) w2 and its input gradient, the GELU's output and the pre-activation held as
    f16: each result within 2^-9 of the sum of |terms| of the float64 value, i.e. one f16 rounding
    (2^-11) of each factor of its last product and of the values behind it."""
    rng = np.random.default_rng(rows)
    x, dy = (rng.standard_normal((rows, h)).astype(np.float32) for _ in range(2))
    w1 = (rng.standard_normal((h, f)) / np.sqrt(h) * 2).astype(np.float32)
    w2 = (rng.standard_normal((f, h)) / np.sqrt(f)).astype(np.float32)
    b1 = rng.standard_normal(f).astype(np.float32)
    p = Prog()
    xi, gi, w1i, w2i = p.input("x", x.shape), p.input("dy", dy.shape), p.input("w1", w1.shape), p.input("w2", w2.shape)
    bi = p.input("b1", b1.shape)
    pre = p.op("AddRows", [p.op("MatMul", [xi, w1i], (rows, f)), bi], (rows, f))
    y = p.op("MatMul", [p.op("Gelu", [pre], (rows, f)), w2i], (rows, h))
    dg = p.op("MatMul", [gi, p.op("Transpose", [w2i], (h, f))], (rows, f))
    dx = p.op("MatMul", [p.op("GeluGrad", [pre, dg], (rows, f)), p.op("Transpose", [w1i], (f, h))], (rows, h))
    p.out(y, dx)
    prog = mixed.program(p.text())
    prog.run({"x": x, "dy": dy, "w1": w1, "w2": w2, "b1": b1})
    got_y, got_dx = (prog.output(k, rows * h).reshape(rows, h) for k in (0, 1))
    u = f16(x) @ f16(w1) + b1
    t = np.tanh(np.sqrt(2 / np.pi) * (u + 0.044715 * u ** 3))
    gelu = 0.5 * u * (1 + t)
    slope = 0.5 * (1 + t) + 0.5 * u * (1 - t * t) * np.sqrt(2 / np.pi) * (1 + 3 * 0.044715 * u * u)
    gated = (f16(dy) @ f16(w2).T) * slope
    for got, left, right in ((got_y, gelu, f16(w2)), (got_dx, gated, f16(w1).T)):
        bound = 2.0 ** -9 * ((np.abs(left) + 0.02) @ np.abs(right))
        worst = np.max(np.abs(got - left @ right) / bound)
        assert worst <= 1.0, worst


@pytest.mark.parametrize("rows,h", [(200, 64), (4096, 192), (16, 320), (1000, 96)])
def test_mixed_chains_of_products(mixed, rows, h):
    """x + a1 w1 + a2 w2 + a3 w3, each product read only by the next sum: one product over the
    concatenated K where h is a multiple of 64, separate ones (h = 96) otherwise."""
    rng = np.random.default_rng(h)
    x, a1, a2, a3 = (rng.standard_normal((rows, h)).astype(np.float32) for _ in range(4))
    w1, w2, w3 = (rng.standard_normal((h, h)).astype(np.float32) for _ in range(3))
    p = Prog()
    xi = p.input("x", (rows, h))
    total = xi
    for k in (1, 2, 3):
        ai, wi = p.input(f"a{k}", (rows, h)), p.input(f"w{k}", (h, h))
        total = p.op("Add", [total, p.op("MatMul", [ai, p.op("Transpose", [wi], (h, h))], (rows, h))], (rows, h))
    p.out(total)
    prog = mixed.program(p.text())
    prog.run({"x": x, "a1": a1, "a2": a2, "a3": a3, "w1": w1, "w2": w2, "w3": w3})
    got = prog.output(0, rows * h).reshape(rows, h)
    want, mag = x.astype(np.float64), np.abs(x).astype(np.float64)
    for a, w in ((a1, w1), (a2, w2), (a3, w3)):
        want, mag = want + f16(a) @ f16(w).T, mag + np.abs(f16(a)) @ np.abs(f16(w)).T
    assert np.max(np.abs(got - want) / mag) <= 1e-5


@pytest.mark.parametrize("rows,h", [(40, 512), (64, 1024), (16, 352), (2100, 512)])
def test_chains_of_products_over_a_deep_k(ctx, rows, h):
    """The same in f32 where the joined K would be split (1024 or more, few rows): the chain joins as
    far as its product stays unsplit, against float64 (1e-5 of the sum of |terms|)."""
    rng = np.random.default_rng(h + rows)
    inputs = {"x": rng.standard_normal((rows, h)).astype(np.float32)}
    p = Prog()
    total = p.input("x", (rows, h))
    want, mag = inputs["x"].astype(np.float64), np.abs(inputs["x"]).astype(np.float64)
    for k in (1, 2, 3):
        a, w = rng.standard_normal((rows, h)).astype(np.float32), rng.standard_normal((h, h)).astype(np.float32)
        inputs.update({f"a{k}": a, f"w{k}": w})
        ai, wi = p.input(f"a{k}", (rows, h)), p.input(f"w{k}", (h, h))
        total = p.op("Add", [total, p.op("MatMul", [ai, p.op("Transpose", [wi], (h, h))], (rows, h))], (rows, h))
        want = want + a.astype(np.float64) @ w.T
        mag = mag + np.abs(a.astype(np.float64)) @ np.abs(w.T)
    p.out(total)
    prog = ctx.program(p.text())
    prog.run(inputs)
    assert np.max(np.abs(prog.output(0, rows * h).reshape(rows, h) - want) / mag) <= 1e-5


@pytest.mark.parametrize("m,k,n,bias", [(70, 48, 30522, True), (4099, 32, 515, False), (37, 144, 60001, True), (2100, 16, 1001, False)])
def test_gemm_of_unaligned_output_rows(ctx, m, k, n, bias):
    """x wᵀ (+ b) into rows that are not 16-byte aligned, against float64 (1e-6 of the sum of |terms|
    and the bias: f32 accumulation of up to 144 terms)."""
    rng = np.random.default_rng(n)
    x, wt = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    p = Prog()
    y = p.op("MatMul", [p.input("x", x.shape), p.op("Transpose", [p.input("w", wt.shape)], (k, n))], (m, n))
    if bias:
        y = p.op("AddRows", [y, p.input("b", b.shape)], (m, n))
    p.out(y)
    prog = ctx.program(p.text())
    prog.run({"x": x, "w": wt, **({"b": b} if bias else {})})
    got = prog.output(0, m * n).reshape(m, n)
    X, W, bb = x.astype(np.float64), wt.astype(np.float64), b.astype(np.float64) * bias
    worst = np.max(np.abs(got - (X @ W.T + bb)) / (1e-6 * (np.abs(X) @ np.abs(W).T + np.abs(bb)) + 1e-30))
    assert worst <= 1.0, worst


@pytest.mark.parametrize("v", [8192, 8193, 16384, 16385, 32768, 32769])
def test_held_out_rows_of_many_classes(ctx, oracle, v):
    """The held-out reduction at the edges of its register-resident rows: ties across waves, a NaN, an
    infinity, -inf logits and a row of nothing else."""
    rows = 9
    rng = np.random.default_rng(v)
    x = (rng.standard_normal((1, rows, v)) * 4).astype(np.float32)
    labels = rng.integers(0, v, (1, rows)).astype(np.int32)
    weights = np.ones((1, rows), np.float32)
    x[0, 0, [5, 1029, v - 1]] = 40.0
    labels[0, 0] = 5
    x[0, 1, [v - 2, v - 1]] = 40.0
    labels[0, 1] = v - 2
    x[0, 2, 7:v - 3] = -np.inf
    labels[0, 2] = int(np.argmax(x[0, 2]))
    load_logits(ctx, rows, v)
    for case in ("finite", "nan", "inf", "all -inf"):
        if case == "nan":
            x[0, 3, v - 1] = np.nan
        elif case == "inf":
            x[0, 3, v - 1] = np.inf
        elif case == "all -inf":
            x[0, 4, :] = -np.inf
            labels[0, 4] = 0
        got = ctx.evaluate(batches_of(x, labels, weights), "labels", "weights")
        want = oracle.held_out_tally(x, labels, weights)
        assert got["correct"] == want["correct"] and got["selected"] == want["selected"], case
        if case == "finite":
            assert abs(got["loss"] - want["loss"]) <= 1e-5 * abs(want["loss"]) + 1e-6
        else:
            assert np.isnan(got["loss"]) == np.isnan(want["loss"]), case


def test_each_step_reads_its_own_inputs(ctx):
    """Eleven steps through the four staging slots, in one call, one by one, and one by one with a
    refused call before each (it uses no slot): the same losses, all different."""
    step, fwd = api.compile_config("mlp_micro")
    rng = np.random.default_rng(3)
    shapes = ((784, 256), (256,), (256, 10), (10,))
    values = [rng.standard_normal(s).astype(np.float32) * 0.05 for s in shapes]
    batches = [{"x": rng.random((8, 784), np.float32), "labels": rng.integers(0, 10, 8).astype(np.int32),
                "weights": np.ones(8, np.float32)} for _ in range(11)]
    ctx.load(step, fwd, 0, 1)
    got = []
    for how in ("one call", "one by one", "after refusals"):
        ctx.set_params(values)
        if how == "one call":
            got.append(ctx.run_steps(batches))
            continue
        losses = []
        for b in batches:
            if how == "after refusals":
                with pytest.raises(api.MsxError):
                    ctx.run_steps([{k: v for k, v in b.items() if k != "weights"}])
                with pytest.raises(api.MsxError):
                    ctx.run_steps([dict(b, labels=b["labels"] + 10)])
            losses.append(ctx.run_steps([b])[0])
        got.append(np.array(losses))
    assert len(set(got[0].tolist())) == 11
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("m,n", [(33, 40), (700, 36), (1030, 260)])  # tiles of 32 x 32, partial; of 32 x 64
@pytest.mark.parametrize("k", [4, 32, 36, 96, 128, 160, 224, 256, 292, 30])  # 1 to 10 K tiles, tails, unaligned
def test_gemm_of_few_and_many_k_tiles(ctx, m, n, k, ta, tb):
    """K tiles fewer and more than those in flight, against float64 (2e-6 of the sum of |terms|, 292 half
    units of 2^-24 growing as their root: f32 accumulation)."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((k, m) if ta else (m, k)).astype(np.float32)
    b = rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32)
    p = Prog()
    ai, bi = p.input("a", a.shape), p.input("b", b.shape)
    lhs = p.op("Transpose", [ai], (m, k)) if ta else ai
    rhs = p.op("Transpose", [bi], (k, n)) if tb else bi
    p.out(p.op("MatMul", [lhs, rhs], (m, n)))
    prog = ctx.program(p.text())
    prog.run({"a": a, "b": b})
    got = prog.output(0, m * n).reshape(m, n)
    A, B = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
    worst = np.max(np.abs(got - A @ B) / (2e-6 * (np.abs(A) @ np.abs(B)) + 1e-30))
    assert worst <= 1.0, worst


@pytest.mark.parametrize("rows,v", [(1, 4), (65, 256), (17, 1023), (33, 2048), (70, 2052), (40, 4096), (2500, 64), (8, 4100),
                                    (5, 8192), (9, 8196), (16, 2049)])
def test_cross_entropy_of_row_blocks(ctx, oracle, rows, v):
    """Loss and gradient at the edges of the row blocks' class counts, with more rows than blocks, odd
    class counts, zero weights and -inf logits, against the oracle."""
    rng = np.random.default_rng(v)
    x = (rng.standard_normal((rows, v)) * 3).astype(np.float32)
    x[0, 1:] = -np.inf
    labels = rng.integers(0, v, rows).astype(np.int32)
    labels[0] = 0
    weights = rng.choice(np.array([0.0, 1.0, 0.5], np.float32), rows)
    weights[0] = 1.0
    p = Prog()
    xi, li, wi = p.input("x", (rows, v)), p.input("labels", (rows,), "i32"), p.input("weights", (rows,))
    g = p.scalar(1.0)
    loss = p.op("CrossEntropy", [xi, li, wi], ())
    p.out(loss, p.op("CrossEntropyGrad", [xi, li, wi, g], (rows, v)))
    got, want = both(ctx, oracle, p, {"x": x, "labels": labels, "weights": weights}, (0, 1))
    for a, b in zip(got, want):
        ok, worst = within(a, b, np.abs(b) + 1e-6)
        assert ok, worst


@pytest.mark.parametrize("B,L,S,H,heads", [(1, 64, 64, 64, 1), (2, 48, 96, 128, 2), (3, 112, 112, 96, 3), (1, 64, 64, 768, 12),
                                           (2, 16, 16, 200, 1), (2, 32, 32, 1040, 1), (2, 33, 33, 64, 1)])
def test_mixed_products_of_attention_and_layer_norm(mixed, B, L, S, H, heads):
    """A product of each of attention's output, its gradients and a LayerNorm reads the f16 rounding of
    the f32 value beside it (1e-5 of the sum of |terms|), whether its producer writes the copy or not.
    Head widths without a kernel: the LayerNorm alone."""
    rng = np.random.default_rng(H)
    fits = H // heads in (16, 32, 64, 128)
    rows_s = {"q": B * L, "k": B * S, "v": B * S, "G": B * L}
    inputs = {n: rng.standard_normal((r, H)).astype(np.float32) * 0.5 for n, r in rows_s.items()}
    inputs["mask"] = np.ones((B, S), np.float32)
    inputs["w"] = rng.standard_normal((H, 24)).astype(np.float32)
    inputs["gamma"], inputs["beta"] = (rng.standard_normal(H).astype(np.float32) for _ in range(2))
    p = Prog()
    ids = {n: p.input(n, a.shape) for n, a in inputs.items()}
    values = [(p.op("LayerNorm", [ids["q"], ids["gamma"], ids["beta"]], (B * L, H)), B * L)]
    if fits:
        attr = f"[heads = {heads}]"
        operands = [ids[n] for n in ("q", "k", "v", "mask")]
        values.append((p.op("Attention", operands, (B * L, H), attr), B * L))
        for op, rows in (("AttentionGradQ", B * L), ("AttentionGradK", B * S), ("AttentionGradV", B * S)):
            values.append((p.op(op, operands + [ids["G"]], (rows, H), attr), rows))
    products = [p.op("MatMul", [v, ids["w"]], (rows, 24)) for v, rows in values]
    p.out(*[v for v, _ in values], *products)
    prog = mixed.program(p.text())
    prog.run(inputs)
    w = f16(inputs["w"])
    for e, (_, rows) in enumerate(values):
        value = f16(prog.output(e, rows * H).reshape(rows, H))
        got = prog.output(len(values) + e, rows * 24).reshape(rows, 24)
        worst = np.max(np.abs(got - value @ w) / (1e-5 * (np.abs(value) @ np.abs(w)) + 1e-30))
        assert worst <= 1.0, (e, worst)
