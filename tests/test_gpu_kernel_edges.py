"""Kernel variants at the sizes where they can go wrong: tile edges, remainders, the smallest and largest of the
range a dispatch rule gives them."""
import numpy as np
import pytest

import oracle
from helpers import mid_config, random_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from laya_amd.device import Context
    c = Context(0)
    yield c
    c.close()


def test_readout_option_counts(ctx):
    """The read-out keeps up to 256 options' exponentials in LDS and fetches the rest: one option, the last that
    fits, one past it, and more. Features of probabilities near 1/K: fp32 sums of K terms (K · 2^-24 ≈ 2e-5
    relative at most), held to 1e-5 absolute as the base-width read-out test does."""
    from laya_amd.batch import synthetic_batch
    from laya_amd.model import TrainableDecisionModel
    mc = mid_config(layers=1)
    o = oracle.OracleModel(mc, double=True)
    params = random_params(o.shapes, 5, std=0.05)
    batch = synthetic_batch(np.random.default_rng(6), [620, 520, 700, 12], [256, 257, 300, 1], [0, 1, 2, 0],
                            mc.encoder.vocab_size)
    o.set_params(params)
    o.forward(batch, training=False)
    probs_o, feats_o, _ = o.readout()
    m = TrainableDecisionModel(mc, ctx)
    m.set_params(params)
    m.forward(batch, training=False)
    _, probs, feats = m.readout()
    np.testing.assert_allclose(feats, feats_o, atol=1e-5)
    np.testing.assert_allclose(probs, probs_o, atol=1e-5)
    m.close()


def _bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7fff + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


def _rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rows,fan_in,fan_out", [
    (1, 32, 4), (5, 64, 64), (31, 96, 100), (33, 128, 132), (63, 256, 256), (65, 800, 96), (129, 768, 2304),
    (404, 1024, 544), (700, 768, 768), (512, 2048, 1024), (1100, 1024, 5248), (100, 100, 36), (97, 66, 30)])
def test_short_products(ctx, precision, rows, fan_in, fan_out):
    """Linear layers over few rows, forward (with bias and residual) and backward, at the edges of the 32- and 64-wide
    tiles and of the 32-deep stages, on both sides of the rules that choose among them, and shapes that they refuse (a K
    that is no multiple of 32, widths that are no multiple of 4); against fp64 on the same operands (rounded to bf16
    first for bf16 products). Operand rows spread over four decades and start from an unaligned size. fp32 accumulation
    rounds to about 2^-24 per addition: 1e-6 relative L2, as the other products' tests hold."""
    from laya_amd import ops
    from laya_amd.device import Context, DeviceArray
    c = ctx if precision == "fp32" else Context(0)
    c.set_matmul_precision(precision)
    r = np.random.default_rng(rows * 7 + fan_out)
    x = (r.standard_normal((rows, fan_in)) * 10.0 ** r.uniform(-2, 2, (rows, 1))).astype(np.float32)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    b = r.standard_normal(fan_out).astype(np.float32)
    res = r.standard_normal((rows, fan_out)).astype(np.float32)
    dy = (1e-4 * r.standard_normal((rows, fan_out))).astype(np.float32)
    dW0 = (1e-3 * r.standard_normal(W.shape)).astype(np.float32)
    low = (lambda a: _bf16(a).astype(np.float64)) if precision == "bf16" else (lambda a: a.astype(np.float64))
    Wp, bp = ops.Parameter(c, "W", W), ops.Parameter(c, "b", b)
    xd, yd = DeviceArray.from_numpy(c, x), DeviceArray(c, (rows, fan_out))
    ops.linear(Wp, bp, xd, rows, yd, residual=DeviceArray.from_numpy(c, res))
    assert _rel(yd.numpy(), low(x) @ low(W).T + b + res) < 1e-6
    Wp.gradient_buffer().upload(dW0)
    dxd = DeviceArray(c, (rows, fan_in))
    ops.linear_backward(Wp, bp, xd, DeviceArray.from_numpy(c, dy), rows, dxd)
    assert _rel(dxd.numpy(), low(dy) @ low(W)) < 1e-6
    assert _rel(Wp.gradient_buffer().numpy(), dW0 + low(dy).T @ low(x)) < 1e-6
    if c is not ctx:
        c.close()


def test_short_product_with_non_finite_operands(ctx):
    """A NaN or infinity stays in its own row: the scale comes from the finite values (the rows beside it are held to
    fp64 as above)."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    r = np.random.default_rng(3)
    x = r.standard_normal((96, 256)).astype(np.float32)
    W = (0.02 * r.standard_normal((128, 256))).astype(np.float32)
    x[40, 17], x[7, 200] = np.inf, np.nan
    yd = DeviceArray(ctx, (96, 128))
    ops.linear(ops.Parameter(ctx, "W", W), None, DeviceArray.from_numpy(ctx, x), 96, yd)
    y = yd.numpy()
    bad = np.isin(np.arange(96), (7, 40))
    assert not np.isfinite(y[bad]).any()
    assert _rel(y[~bad], x[~bad].astype(np.float64) @ W.astype(np.float64).T) < 1e-6


@pytest.mark.parametrize("p_drop", [0.0, 0.2])
@pytest.mark.parametrize("window", [-1, 64])
@pytest.mark.parametrize("lengths", [[1], [31, 33, 1], [128], [129, 32], [189], [300, 7], [640], [513, 512],
                                     [1000], [513, 300]])
def test_short_attention(ctx, lengths, window, p_drop):
    """Attention of grids small enough for 32 rows to a workgroup (up to 64 workgroups of 128 rows; 96 without a window
    on segments of 512 and more), where each wave takes a subtile of 32 keys or queries, and the next larger grids: row
    counts on both sides of a subtile, of a stage of four and of several stages, with RoPE where there is no dropout.
    Against the oracle in fp64; fp32 sums over up to 640 keys: 1e-5 relative L2, as the other attention tests hold."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    heads, hidden = 12, 768
    rows = sum(lengths)
    r = np.random.default_rng(rows + window)
    qkv = r.standard_normal((rows, 3 * hidden)).astype(np.float32)
    dctx = (1e-3 * r.standard_normal((rows, hidden))).astype(np.float32)
    theta = 10000.0 if p_drop == 0.0 else 0.0
    rotary = ops.Rotary(ctx, 64, theta, max(lengths)) if theta else None
    args = (np.asarray(lengths, np.int32), heads, ops.default_scale(64), window, theta, p_drop, 11)
    want_c = oracle.attention_forward(qkv, *args, double=True)
    want_d = oracle.attention_backward(qkv, dctx, *args, double=True)
    segs = ops.Segments(ctx, np.asarray(lengths, np.int32))
    shape = ops.AttentionShape(hidden, heads, ops.default_scale(64), window, rotary, p_drop, 11)
    q, c, l = DeviceArray.from_numpy(ctx, qkv), DeviceArray(ctx, (rows, hidden)), DeviceArray(ctx, (rows * heads,))
    d = DeviceArray(ctx, (rows, 3 * hidden))
    ops.attention_forward(q, segs, shape, c, l)
    ops.attention_backward(q, segs, shape, DeviceArray.from_numpy(ctx, dctx), d, c, l)
    assert _rel(c.numpy(), want_c) < 1e-5
    assert _rel(d.numpy(), want_d) < 1e-5


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rows,fan_in,fan_out,bf16_kernel", [
    (2500, 3072, 768, "gemm_bwd_pair_bf16w"), (6000, 768, 2304, "gemm_bwd_pair_bf16w"),
    (8003, 768, 2304, "gemm_bwd_pair_bf16w"), (5300, 768, 2304, ""), (6001, 768, 768, ""), (3232, 1152, 768, "gemm_nn_bf16"),
    (5500, 1024, 5248, "gemm_bwd_pair_bf16w")])
def test_backward_pair_of_few_input_gradient_tiles(ctx, precision, rows, fan_in, fan_out, bf16_kernel):
    """Pairs whose dX tile is more than a worker's share of the wide plan. In bf16 the workers with one more dX tile do no
    dW where that pays (the shapes that name the wide kernel: half of the workers busy, and either the balanced plan of
    128 x 128 tiles would be next or launches of their own are not faster); in fp32 only where exact splits would not be
    next and launches of their own are slower (the last shape). Against fp64 on the same operands, 1e-6 relative L2 widened by the square root of K over 768 for dW, whose sums run over the rows."""
    from laya_amd import ops
    from laya_amd.device import Context, DeviceArray
    c = ctx if precision == "fp32" else Context(0)
    c.set_matmul_precision(precision)
    r = np.random.default_rng(rows)
    x = r.standard_normal((rows, fan_in)).astype(np.float32)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    dy = (1e-4 * r.standard_normal((rows, fan_out))).astype(np.float32)
    low = (lambda a: _bf16(a).astype(np.float64)) if precision == "bf16" else (lambda a: a.astype(np.float64))
    Wp, dx = ops.Parameter(c, "W", W), DeviceArray(c, (rows, fan_in))
    c.profile_begin()
    ops.linear_backward(Wp, None, DeviceArray.from_numpy(c, x), DeviceArray.from_numpy(c, dy), rows, dx)
    ran = set(c.profile_end())
    assert ("gemm_bwd_pair_h2w" in ran) == (precision == "fp32" and fan_out == 5248), ran
    assert precision == "fp32" or not bf16_kernel or bf16_kernel in ran, ran
    assert _rel(dx.numpy(), low(dy) @ low(W)) < 1e-6
    assert _rel(Wp.gradient_buffer().numpy(), low(dy).T @ low(x)) < 1e-6 * np.sqrt(rows / 768)
    if c is not ctx:
        c.close()


def test_uneven_wide_pair_with_a_residual(ctx):
    """The first layer's QKV backward adds the residual gradient to dX in the wide pair's epilogue; with bf16 products
    over 8003 tokens some of its workers do no dW. Against the same step's fp32 products at bf16's bar, 2e-2 relative L2
    (without the residual the embedding gradient would be off by its own size)."""
    from laya_amd.batch import synthetic_batch
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    mc = mid_config(layers=1)
    params = random_params(oracle.OracleModel(mc).shapes, 7, std=0.02)
    lengths = [500] * 15 + [503]
    batch = synthetic_batch(np.random.default_rng(8), lengths, [4] * 16, [0] * 16, mc.encoder.vocab_size)
    d = np.random.default_rng(9).standard_normal(batch.n_markers).astype(np.float32)
    grads = []
    for policy in ("fp32", "bf16-backward"):
        c = Context(0)
        c.set_matmul_precision(policy)
        m = TrainableDecisionModel(mc, c)
        m.set_params(params)
        m.forward(batch, training=False)
        c.profile_begin()
        m.backward(d)
        ran = set(c.profile_end())
        assert policy == "fp32" or "gemm_bwd_pair_bf16w" in ran
        grads.append(m.grad("encoder.embeddings.tok_embeddings.weight"))
        m.close()
        c.close()
    assert _rel(grads[1], grads[0].astype(np.float64)) < 2e-2


@pytest.mark.parametrize("rows,fan_in,fan_out,kernel", [
    (12345, 768, 700, "x6"), (8003, 768, 2304, "x6w"), (7001, 1020, 1024, "x6w"), (5600, 768, 768, "x6"), (2500, 3072, 768, "h2s"),
    (1400, 3072, 768, "h2s"), (1403, 3076, 800, "h2s"), (1600, 2624, 1024, "h2s")])
def test_backward_pairs_keep_lines_far_below_the_largest(ctx, rows, fan_in, fan_out, kernel):
    """fp32 backward pairs on exact three-piece splits, or on two pieces scaled by row and column: rows and columns of dY,
    columns of W and of x 2^-26 below the rest, each of which a two-piece product under a scale of the others would keep
    to about 2^(26-39) = 1e-4, come out to fp32 precision, row by row and column by column (a sum of K terms rounded 2^-24
    each: 2e-6 holds dX's K of up to 2304, widened by the square root of the rows over 2304 for dW's)."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    r = np.random.default_rng(rows + fan_out)
    x = r.standard_normal((rows, fan_in)).astype(np.float32)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    dy = (1e-4 * r.standard_normal((rows, fan_out))).astype(np.float32)
    tiny = np.float32(2.0 ** -26)
    dy[7::50] *= tiny
    dy[:, 5::40] *= tiny
    W[:, 3::60] *= tiny
    x[:, 11::30] *= tiny
    Wp, dx = ops.Parameter(ctx, "W", W), DeviceArray(ctx, (rows, fan_in))
    ctx.profile_begin()
    ops.linear_backward(Wp, None, DeviceArray.from_numpy(ctx, x), DeviceArray.from_numpy(ctx, dy), rows, dx)
    assert "gemm_bwd_pair_" + kernel in ctx.profile_end()
    dy64, W64, x64 = (a.astype(np.float64) for a in (dy, W, x))
    bar = 2e-6 * max(1.0, np.sqrt(rows / 2304))
    for got, want, limit in ((dx.numpy(), dy64 @ W64, 2e-6), (Wp.gradient_buffer().numpy(), dy64.T @ x64, bar)):
        for axis in (0, 1):
            e = np.linalg.norm(got - want, axis=axis) / np.linalg.norm(want, axis=axis)
            print(rows, fan_in, fan_out, kernel, "worst line", e.max())
            assert e.max() < limit


def test_backward_pair_scaled_by_line_with_non_finite_operands(ctx):
    """A NaN or an infinity in dY stays in its own row of dX and its own row of dW; the scales of its lines come from
    their finite values. The other lines are held to fp64 as above. Rows of dY grow by 2^20 on the way down, so that the
    scales of dW's lines are lowered again and again."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    rows, fan_in, fan_out = 1403, 3076, 800
    r = np.random.default_rng(4)
    x = r.standard_normal((rows, fan_in)).astype(np.float32)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    dy = (r.standard_normal((rows, fan_out)) * 2.0 ** np.linspace(-30, -10, rows)[:, None]).astype(np.float32)
    clean = dy.copy()
    dy[700, 41], dy[90, 300], clean[700, 41], clean[90, 300] = np.inf, np.nan, 0.0, 0.0
    Wp, dxd = ops.Parameter(ctx, "W", W), DeviceArray(ctx, (rows, fan_in))
    ctx.profile_begin()
    ops.linear_backward(Wp, None, DeviceArray.from_numpy(ctx, x), DeviceArray.from_numpy(ctx, dy), rows, dxd)
    assert "gemm_bwd_pair_h2s" in ctx.profile_end()
    dx, dW = dxd.numpy(), Wp.gradient_buffer().numpy()
    for got, want, bad in ((dx, clean.astype(np.float64) @ W.astype(np.float64), (700, 90)),
                           (dW, clean.astype(np.float64).T @ x.astype(np.float64), (41, 300))):
        lines = np.isin(np.arange(len(got)), bad)
        assert not np.isfinite(got[lines]).any()
        e = np.linalg.norm(got[~lines] - want[~lines], axis=1) / np.linalg.norm(want[~lines], axis=1)
        assert e.max() < 2e-6


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rows,fan_in,fan_out,short", [
    (13824, 768, 64, "forward"), (32768, 64, 768, "dx"), (32768, 64, 64, "forward dx"), (8192, 256, 256, "forward dx"),
    (873, 3392, 640, "dx dw pair"), (404, 768, 768, "forward dx dw pair"), (512, 768, 2304, "forward dx dw pair")])
def test_short_products_only_where_they_fill_the_chip(ctx, precision, rows, fan_in, fan_out, short):
    """Narrow layers over many rows: a dW of a few tiles and a long K, a forward of many tiles and a short K, and a dX of
    the same leave the short kernels, whose K is dealt to one workgroup's waves only, for the tiles that split it over
    the chip, and so does a forward whose 32 x 64 tiles come in little more than one round; layers of ordinary width over
    few rows stay. The kernels that ran are read from the profile, the results
    held to fp64 as above (dW's sums run over the rows)."""
    from laya_amd import ops
    from laya_amd.device import Context, DeviceArray
    c = ctx if precision == "fp32" else Context(0)
    c.set_matmul_precision(precision)
    r = np.random.default_rng(rows + fan_in)
    x = r.standard_normal((rows, fan_in)).astype(np.float32)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    dy = (1e-4 * r.standard_normal((rows, fan_out))).astype(np.float32)
    low = (lambda a: _bf16(a).astype(np.float64)) if precision == "bf16" else (lambda a: a.astype(np.float64))
    Wp, frozen = ops.Parameter(c, "W", W), ops.Parameter(c, "F", W, False)
    xd, dyd = DeviceArray.from_numpy(c, x), DeviceArray.from_numpy(c, dy)
    y, dx = DeviceArray(c, (rows, fan_out)), DeviceArray(c, (rows, fan_in))
    want_dx, want_dW = low(dy) @ low(W), low(dy).T @ low(x)
    bar = 1e-6 * max(1.0, np.sqrt(rows / 768))

    got = []

    def run(kind, kernel, call):
        c.profile_begin()
        call()
        if any(k.startswith(kernel) and k.endswith(("_h2s", "_bf16s")) for k in c.profile_end()):
            got.append(kind)

    run("forward", "gemm_nt", lambda: ops.linear(Wp, None, xd, rows, y))
    assert _rel(y.numpy(), low(x) @ low(W).T) < 1e-6
    run("dx", "gemm_nn", lambda: ops.linear_backward(frozen, None, xd, dyd, rows, dx))
    assert _rel(dx.numpy(), want_dx) < 1e-6
    run("dw", "gemm_tn", lambda: ops.linear_backward(Wp, None, xd, dyd, rows, None))
    assert _rel(Wp.gradient_buffer().numpy(), want_dW) < bar
    Wp.zero_gradient()
    run("pair", "gemm_bwd_pair", lambda: ops.linear_backward(Wp, None, xd, dyd, rows, dx))
    assert _rel(dx.numpy(), want_dx) < 1e-6
    assert _rel(Wp.gradient_buffer().numpy(), want_dW) < bar
    assert got == short.split()
    if c is not ctx:
        c.close()


@pytest.mark.parametrize("rows,fan_in,fan_out,backward", [(3200, 1152, 768, False), (4500, 1152, 768, True)])
def test_fp32_products_of_even_estimates_run_short(ctx, rows, fan_in, fan_out, backward):
    """Where the estimates do not tell which tiles are faster, the short kernels take the product: each of a workgroup's
    waves sums its share of K in 32-bit accumulators of its own, a quarter of a sequential sum's terms or fewer. With
    independent rounding errors of at most 2^-24 of a partial sum, a sum of K / 16 matrix instructions over four waves
    stays below sqrt(K / 64) x 2^-24 of its norm (2.5e-7 for K = 1152, 2.1e-7 for 768), and the two pieces of an operand
    leave out less than 2^-22 of each value, independently: together below 5e-7."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    r = np.random.default_rng(rows)
    W = (0.02 * r.standard_normal((fan_out, fan_in))).astype(np.float32)
    a = r.standard_normal((rows, fan_out if backward else fan_in)).astype(np.float32)
    frozen, ad = ops.Parameter(ctx, "F", W, False), DeviceArray.from_numpy(ctx, a)
    out = DeviceArray(ctx, (rows, fan_in if backward else fan_out))
    ctx.profile_begin()
    if backward:
        x = DeviceArray.from_numpy(ctx, np.zeros((rows, fan_in), np.float32))
        ops.linear_backward(frozen, None, x, ad, rows, out)
    else:
        ops.linear(frozen, None, ad, rows, out)
    assert any(k.startswith("gemm_nn" if backward else "gemm_nt") and k.endswith("_h2s") for k in ctx.profile_end())
    W64 = W.astype(np.float64)
    assert _rel(out.numpy(), a.astype(np.float64) @ (W64 if backward else W64.T)) < 5e-7


@pytest.mark.parametrize("policy", ["fp32", "fp32-split3", "fp32-mfma"])
@pytest.mark.parametrize("head_dim,lengths,window", [(64, [300, 65], -1), (64, [700, 129], 64), (32, [200, 33], 8)])
def test_attention_backward_in_place(head_dim, lengths, window, policy):
    """dqkv may be qkv itself where RoPE is applied to a copy of q and k: v, read from the caller's array, is not
    overwritten before its last reader is done. The same bits as with an output of its own."""
    from laya_amd import ops
    from laya_amd.device import Context, DeviceArray
    c = Context(0)
    c.set_matmul_precision(policy)
    heads, rows = 4, sum(lengths)
    hidden = heads * head_dim
    r = np.random.default_rng(rows)
    qkv = r.standard_normal((rows, 3 * hidden)).astype(np.float32)
    dctx = DeviceArray.from_numpy(c, r.standard_normal((rows, hidden)).astype(np.float32))
    segs = ops.Segments(c, np.asarray(lengths, np.int32))
    shape = ops.AttentionShape(hidden, heads, ops.default_scale(head_dim), window,
                               ops.Rotary(c, head_dim, 10000.0, max(lengths)), 0.0, 0)
    q, ctxt, lse = DeviceArray.from_numpy(c, qkv), DeviceArray(c, (rows, hidden)), DeviceArray(c, (rows * heads,))
    ops.attention_forward(q, segs, shape, ctxt, lse)
    d = DeviceArray(c, (rows, 3 * hidden))
    ops.attention_backward(q, segs, shape, dctx, d, ctxt, lse)
    ops.attention_backward(q, segs, shape, dctx, q, ctxt, lse)
    np.testing.assert_array_equal(q.numpy(), d.numpy())
    c.close()


@pytest.mark.parametrize("words", [False, True])
@pytest.mark.parametrize("rows,fan_in,fan_out,measured", [(200, 768, 768, 0), (257, 768, 768, 0), (200, 784, 98, 1)])
def test_biased_backward_measures_only_what_it_reads(ctx, rows, fan_in, fan_out, measured, words):
    """The bias gradient of few rows is summed without a pass of its own over dY's magnitudes: the short pair reads none,
    and a pair that the short kernels refuse (a K that is no multiple of 32) measures dY with its other operands, in one
    launch for each product. The results as without a bias, to the bit."""
    from laya_amd import ops
    from laya_amd.device import DeviceArray
    r = np.random.default_rng(rows + fan_out)
    x, W = r.standard_normal((rows, fan_in)).astype(np.float32), r.standard_normal((fan_out, fan_in)).astype(np.float32)
    dy = r.standard_normal((rows, fan_out)).astype(np.float32)
    out = []
    for biased in (False, True):
        Wp = ops.Parameter(ctx, "W", W)
        b = ops.Parameter(ctx, "b", np.zeros(fan_out, np.float32)) if biased else None
        dx = DeviceArray(ctx, (rows, fan_in))
        dx_words = ops.magnitude_words(ctx) if words else None
        xd, dyd = DeviceArray.from_numpy(ctx, x), DeviceArray.from_numpy(ctx, dy)
        ctx.profile_begin()
        ops.linear_backward(Wp, b, xd, dyd, rows, dx, dx_words=dx_words)
        launches = ctx.profile_end().get("absmax", {}).get("launches", 0)
        if biased:
            assert launches == out[0][2]
            assert _rel(b.gradient_buffer().numpy(), dy.astype(np.float64).sum(0)) < 1e-6
        assert (launches > 0) == bool(measured)
        out.append((dx.numpy(), Wp.gradient_buffer().numpy(), launches))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("rows,fan_in,fan_out", [(1100, 768, 2304), (1618, 2624, 1024), (1618, 768, 3072),
                                                 (2200, 768, 2304), (2200, 1152, 768), (2700, 1024, 1024),
                                                 (3200, 1152, 768), (4800, 768, 768), (8192, 768, 32)])
def test_known_magnitudes_change_no_bits(ctx, rows, fan_in, fan_out):
    """Where the short products and the other tiles take about as long, the choice is the same whether the caller keeps
    the operands' magnitude words (and so spares their measuring) or not: the same bits."""
    from laya_amd import ops
    from laya_amd._native import check, lib
    from laya_amd.device import DeviceArray
    r = np.random.default_rng(rows)
    x, W, dy = (DeviceArray.from_numpy(ctx, r.standard_normal(s).astype(np.float32))
                for s in ((rows, fan_in), (fan_out, fan_in), (rows, fan_out)))
    xw, ww, dyw = (ops.magnitude_words(ctx) for _ in range(3))
    for a, w in ((x, xw), (W, ww), (dy, dyw)):
        ops.measure_words(ctx, a, w)
    runs = []
    for words in ((None, None, None), (xw.ptr, ww.ptr, dyw.ptr)):
        y, dx, dW = (DeviceArray(ctx, s) for s in ((rows, fan_out), (rows, fan_in), (fan_out, fan_in)))
        one_dx, one_dW = DeviceArray(ctx, (rows, fan_in)), DeviceArray(ctx, (fan_out, fan_in))
        size = (rows, fan_in, fan_out)
        check(lib().laya_linear_fwd_w(ctx.handle, x.ptr, *size[:2], W.ptr, fan_out, None, None, y.ptr, words[0], words[1],
                                      None))
        for d, g in ((dx, dW), (one_dx, None), (None, one_dW)):
            check(lib().laya_linear_bwd_w(ctx.handle, x.ptr, dy.ptr, *size, W.ptr, d and d.ptr, g and g.ptr, None,
                                          words[0], words[2], words[1], None))
        runs.append([a.numpy() for a in (y, dx, dW, one_dx, one_dW)])
    for a, b in zip(*runs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("lengths", [(33, 20), (64,), (129, 61), (404,)])
@pytest.mark.parametrize("inter", [1140, 1152])
def test_short_rope_and_geglu_epilogues(ctx, lengths, inter):
    """The QKV projection's RoPE and the MLP's GeGLU in the short products' epilogues: rows on both sides of a tile's edge
    and a GeGLU width that is no multiple of a tile's 32 columns, against the fp64 oracle (logits to 1e-5, as at the
    other widths); and their bf16 copies, which bf16 backward products read: the gradients with the copies are those
    without, to the bit."""
    from helpers import mixed_batch
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    mc = mid_config(layers=2, inter=inter)
    o = oracle.OracleModel(mc, double=True)
    params = random_params(o.shapes, 11, std=0.03)
    batch = mixed_batch(np.random.default_rng(12), list(lengths), mc.encoder.vocab_size)
    o.set_params(params)
    want = o.forward(batch, training=False)
    m = TrainableDecisionModel(mc, ctx)
    m.set_params(params)
    ctx.profile_begin()
    got = m.forward(batch, training=False)
    ran = set(ctx.profile_end())
    assert "gemm_nt_h2s" in ran and "geglu_fwd" not in ran
    assert _rel(got, want) < 1e-5
    m.close()
    d = np.random.default_rng(13).standard_normal(batch.n_markers).astype(np.float32)
    grads = []
    for copies in (True, False):
        c = Context(0)
        c.set_matmul_precision("bf16-backward")
        m = TrainableDecisionModel(mc, c)
        m.set_bf16_copies(copies)
        m.set_params(params)
        m.forward(batch, training=True, seed=5)
        m.backward(d)
        grads.append({n: m.grad(n) for n in m.names if m.has_grad(n)})
        m.close()
        c.close()
    for n, g in grads[0].items():
        np.testing.assert_array_equal(g, grads[1][n], err_msg=n)


def test_split_k_rope_projection(ctx):
    """A QKV projection past the short products' range whose 128 x 128 tiles still leave CUs idle (700 rows of 1536: 216
    tiles, K in two): its partials are summed, rotated and measured in one pass. Against the same model on exact splits,
    whose projection rotates in the product's epilogue: logits to 1e-5."""
    from laya_amd.batch import synthetic_batch
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    mc = mid_config(layers=1, hidden=1536, heads=24, inter=256, head_layers=1)
    lengths = [300, 400]
    batch = synthetic_batch(np.random.default_rng(14), lengths, [4, 4], [0, 1], mc.encoder.vocab_size)
    logits = []
    for policy in ("fp32", "fp32-split3"):
        c = Context(0)
        c.set_matmul_precision(policy)
        m = TrainableDecisionModel.synthetic(mc, 15, 0.03, c)
        c.profile_begin()
        logits.append(m.forward(batch, training=False))
        ran = set(c.profile_end())
        assert ({"gemm_nt_h2", "gemm_splitk_store"} <= ran) == (policy == "fp32"), ran
        m.close()
        c.close()
    assert _rel(logits[0], logits[1].astype(np.float64)) < 1e-5
