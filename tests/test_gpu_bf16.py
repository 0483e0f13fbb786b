"""The bf16 matrix-product path (bf16 operands on the bf16 matrix cores, fp32 accumulation, fp32 master
weights, gradients and statistics) against the oracle.

Two bars. Exactness: each product equals the fp64 product of the bf16-rounded operands up to fp32
accumulation order (relative L2 ≤ 2e-5) — this pins the rounding (nearest even), the fragment layouts and
the epilogues. Tolerance: against the exact fp32-input result, relative L2 ≤ 2e-2 per tensor, the bf16 bar.
"""
import numpy as np
import pytest

import oracle
from fixtures import rel_l2

pytestmark = pytest.mark.gpu

laya = pytest.importorskip("laya_amd.ops")


def bf16(a):
    """Round to bf16, nearest even (finite inputs)."""
    bits = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


@pytest.fixture(scope="module")
def ctx():
    from laya_amd.device import Context
    print("GPU bf16 tests: creating context on device 0", flush=True)
    c = Context(0)
    c.set_matmul_precision("bf16")
    yield c
    c.close()


def dev(ctx, a):
    from laya_amd.device import DeviceArray
    return DeviceArray.from_numpy(ctx, np.asarray(a))


@pytest.mark.parametrize("rows,inn,out", [(37, 96, 130), (333, 100, 260), (1000, 768, 2304), (2048, 1152, 768),
                                          (4100, 64, 96), (9000, 768, 2304),
                                          # the backward pair on 256 x 256 tiles (ragged columns, ragged last
                                          # dW unit; the model's shapes)
                                          (11000, 1148, 768), (13871, 768, 2304),
                                          # the balanced pair of 128 x 128 tiles: widths that the wide one refuses,
                                          # dY in float4s and not
                                          (9000, 768, 2300), (9000, 768, 2302)])
def test_bf16_linear_is_the_product_of_rounded_operands(ctx, rows, inn, out):
    """Forward with bias and residual (NT), dx (NN) and dW accumulated twice (TN, split-K at 4100 and 9000
    rows), in bf16."""
    print(f"bf16 linear rows={rows} in={inn} out={out}", flush=True)
    rng = np.random.default_rng(rows + 3 * inn + out)
    x = rng.standard_normal((rows, inn)).astype(np.float32)
    W = (0.05 * rng.standard_normal((out, inn))).astype(np.float32)
    b = rng.standard_normal(out).astype(np.float32)
    res = rng.standard_normal((rows, out)).astype(np.float32)
    dy = rng.standard_normal((rows, out)).astype(np.float32)
    w, bias = laya.Parameter(ctx, "w", W, True), laya.Parameter(ctx, "b", b, True)
    y = dev(ctx, np.zeros((rows, out), np.float32))
    dx = dev(ctx, np.zeros((rows, inn), np.float32))
    xd, dyd = dev(ctx, x), dev(ctx, dy)
    laya.linear(w, bias, xd, rows, y, residual=dev(ctx, res))
    laya.linear_backward(w, bias, xd, dyd, rows, dx)
    laya.linear_backward(w, bias, xd, dyd, rows, dx)
    xb, Wb, dyb = (bf16(a).astype(np.float64) for a in (x, W, dy))
    y_exact = xb @ Wb.T + b + res
    dx_exact = dyb @ Wb
    dW_exact = 2 * dyb.T @ xb
    assert rel_l2(y_exact, y.numpy()) < 2e-5
    assert rel_l2(dx_exact, dx.numpy()) < 2e-5
    assert rel_l2(dW_exact, w.gradient.numpy()) < 2e-5
    assert rel_l2(2 * dy.sum(0, dtype=np.float64), bias.gradient.numpy()) < 1e-6  # the bias sum stays fp32
    x64, W64, dy64 = (a.astype(np.float64) for a in (x, W, dy))
    assert rel_l2(x64 @ W64.T + b + res, y.numpy()) < 2e-2
    assert rel_l2(dy64 @ W64, dx.numpy()) < 2e-2
    assert rel_l2(2 * dy64.T @ x64, w.gradient.numpy()) < 2e-2


def test_bf16_precision_switch_is_per_context():
    """fp32 stays the default: a second context multiplies in fp32 while another is in bf16."""
    from laya_amd.device import Context
    a, b = Context(0), Context(0)
    try:
        b.set_matmul_precision("bf16")
        rng = np.random.default_rng(0)
        x = rng.standard_normal((300, 256)).astype(np.float32)
        W = (0.05 * rng.standard_normal((128, 256))).astype(np.float32)
        outs = []
        for c in (a, b):
            w = laya.Parameter(c, "w", W, False)
            y = dev(c, np.zeros((300, 128), np.float32))
            laya.linear(w, None, dev(c, x), 300, y)
            outs.append(y.numpy())
        exact = x.astype(np.float64) @ W.astype(np.float64).T
        rounded = bf16(x).astype(np.float64) @ bf16(W).astype(np.float64).T
        assert rel_l2(exact, outs[0]) < 1e-6
        assert rel_l2(rounded, outs[1]) < 2e-5 and rel_l2(exact, outs[1]) > 1e-4
        with pytest.raises(ValueError):
            a.set_matmul_precision("fp16")
    finally:
        a.close()
        b.close()


def _heads(n):
    """choice K = 8, score K = 4, noul K = 2, cycling."""
    return [(8, 4, 2)[i % 3] for i in range(n)], [i % 3 for i in range(n)]


def _grads_match(names, want, got, bar, skip=("scorer.3.bias",)):
    """Per-tensor relative L2 against the fp32 result; the output bias's gradient is Σ of a softmax-CE
    gradient, zero up to rounding in any implementation, so it has no relative error to measure."""
    errors = {n: rel_l2(want[n], got[n]) for n in names if n not in skip and n in want}
    top = sorted(errors.items(), key=lambda kv: -kv[1])[:8]
    print("largest gradient rel-L2: " + ", ".join(f"{n} {e:.2e}" for n, e in top), flush=True)
    bad = {n: e for n, e in errors.items() if e >= bar}
    assert not bad, bad
    return max(errors.values())


def _bf16_vs_oracle(ctx, batch, seed):
    """The backward products in bf16 (forward in fp32) against the fp32 oracle."""
    from laya_amd.config import modernbert_base
    from laya_amd.model import TrainableDecisionModel
    import helpers
    mc = modernbert_base()
    o = oracle.OracleModel(mc)
    params = helpers.random_params(o.shapes, seed, std=0.02)
    rng = np.random.default_rng(seed + 1)
    targets = np.concatenate([np.eye(k, dtype=np.float32)[rng.integers(k)] for k in batch.n_options])
    o.set_params(params)
    o.set_head_dropout(0.1)
    logits_o = o.forward(batch, training=True, keep_tape=True, seed=seed).astype(np.float32)
    _, g = oracle.cross_entropy(batch.n_options, logits_o, targets, 1.0, float(batch.n_items))
    o.backward(g)
    ctx.set_matmul_precision("bf16-backward")
    try:
        m = TrainableDecisionModel(mc, ctx)
        m.set_params(params)
        m.head_dropout = 0.1
        logits_m = m.forward(batch, training=True, seed=seed)
        m.backward(g)
    finally:
        ctx.set_matmul_precision("bf16")
    assert rel_l2(logits_o, logits_m) < 1e-4  # the forward is fp32
    names = [n for n in m.names if m.has_grad(n)]
    worst = _grads_match(names, {n: o.grad(n) for n in names}, {n: m.grad(n) for n in names}, 2e-2)
    print(f"bf16 backward vs fp32 oracle: worst gradient rel-L2 {worst:.2e} over {len(names)} tensors", flush=True)
    m.close()


def test_bf16_modernbert_base_gradients_match_the_fp32_oracle(ctx):
    """Batch 32 × 1024 in bf16 at reduced size: ModernBERT-base (22 layers, 164M parameters), 4 × 256 tokens
    without padding, heads choice 8 / score 4 / noul 2, summed CE, head dropout 0.1: every gradient of the
    bf16 backward products within the bf16 bar of the fp32 oracle."""
    from laya_amd.batch import synthetic_batch
    print("bf16 model: ModernBERT-base 22 layers, 4 x 256", flush=True)
    rng = np.random.default_rng(31)
    opts, qt = _heads(4)
    _bf16_vs_oracle(ctx, synthetic_batch(rng, [256] * 4, opts, qt, 50368), 31)


def test_bf16_packed_zipf_batch_gradients_match_the_fp32_oracle(ctx):
    """The variable-length packed batch in bf16 at reduced size: 6 sequences of lengths U[16, 400]
    concatenated with per-sequence RoPE positions, ids Zipf(1.1) over the 50368 vocabulary (repeated ids
    in the embedding-gradient scatter)."""
    from laya_amd.batch import synthetic_batch
    print("bf16 model: ModernBERT-base 22 layers, 6 packed sequences, Zipf ids", flush=True)
    rng = np.random.default_rng(41)
    lengths = rng.integers(16, 401, 6)
    opts, qt = _heads(6)
    _bf16_vs_oracle(ctx, synthetic_batch(rng, lengths, opts, qt, 50368, zipf=1.1), 41)


def _grads(m, c, batch, targets, seed, forward_policy, backward_policy):
    c.set_matmul_precision(forward_policy)
    m.zero_gradients()
    logits = m.forward(batch, training=True, seed=seed)
    _, g = oracle.cross_entropy(batch.n_options, logits, targets, 1.0, float(batch.n_items))
    c.set_matmul_precision(backward_policy)
    m.backward(g)
    return logits, {n: m.grad(n) for n in m.names if m.has_grad(n)}


def _bf16_at_full_size(batch, seed):
    """At full size, on the GPU (the fp32 path is held to the oracle at 1e-4 on smaller inputs):
    - the bf16 backward products on an fp32 forward against the fp32 backward: every gradient within 2e-2;
    - with the forward in bf16 too (every product in bf16), the bf16 backward against an fp32 backward of
      the same bf16 forward: every gradient within 2e-2, and the bf16 forward's logits within 2e-2 of fp32.
    (A bf16 forward evaluates a slightly different function — activations move by ~1e-2 and near-zero
    ReLU inputs flip — so its gradients are compared with the backward of that same forward.)"""
    from laya_amd.config import modernbert_base
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    c = Context(0)
    try:
        m = TrainableDecisionModel.synthetic(modernbert_base(), seed=seed, std=0.02, ctx=c)
        m.head_dropout = 0.1
        rng = np.random.default_rng(seed)
        targets = np.concatenate([np.eye(k, dtype=np.float32)[rng.integers(k)] for k in batch.n_options])
        l32, g32 = _grads(m, c, batch, targets, seed, "fp32", "fp32")
        _, gbwd = _grads(m, c, batch, targets, seed, "fp32", "bf16-backward")
        worst = _grads_match(g32.keys(), g32, gbwd, 2e-2)
        print(f"bf16 backward products vs fp32: worst gradient rel-L2 {worst:.2e}", flush=True)
        l16, gf = _grads(m, c, batch, targets, seed, "bf16-forward", "bf16-forward")  # bf16 forward, fp32 backward
        _, gall = _grads(m, c, batch, targets, seed, "bf16", "bf16")
        assert rel_l2(l32, l16) < 2e-2
        worst = _grads_match(gf.keys(), gf, gall, 2e-2)
        print(f"every product in bf16: logits rel-L2 {rel_l2(l32, l16):.2e}; bf16 vs fp32 backward of the bf16 "
              f"forward: worst gradient rel-L2 {worst:.2e}", flush=True)
        m.close()
    finally:
        c.close()


def test_bf16_at_batch_32x1024(ctx):
    """Batch 32 × 1024, no padding, bf16 products (32,768 tokens)."""
    from laya_amd.batch import synthetic_batch
    print("bf16 model: 32 x 1024 full size", flush=True)
    rng = np.random.default_rng(51)
    opts, qt = _heads(32)
    _bf16_at_full_size(synthetic_batch(rng, [1024] * 32, opts, qt, 50368), 51)


def test_bf16_at_64_packed_zipf_sequences(ctx):
    """64 sequences of lengths U[16, 2048] packed without padding, Zipf(1.1) ids, bf16 products."""
    from laya_amd.batch import synthetic_batch
    print("bf16 model: 64 packed sequences U[16, 2048], Zipf ids, full size", flush=True)
    rng = np.random.default_rng(61)
    lengths = rng.integers(16, 2049, 64)
    opts, qt = _heads(64)
    _bf16_at_full_size(synthetic_batch(rng, lengths, opts, qt, 50368, zipf=1.1), 61)


@pytest.mark.parametrize("shape", ["32x1024", "64 packed zipf"])
def test_bf16_weights_one_piece_products_equal_two_piece_ones(shape):
    """With bf16 weights the forward's two-piece products take each weight as one fp16 piece and skip the
    products of the low piece: a bf16 value scaled into fp16's range is exact there, so that piece is zero and
    its products add nothing. At the bf16 workloads' full sizes (the 256 x 256, 192 x 256 and 128 x 128
    kernels), under their policy (fp32-accurate forward, bf16 backward products), the step with bf16 weights
    on equals bit for bit the step of the same model with bf16 weights off, its fp32 weights already holding
    the bf16 values (products carrying both pieces)."""
    from laya_amd.batch import synthetic_batch
    from laya_amd.config import modernbert_base
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel, synthetic_params
    print(f"bf16 weights, one-piece vs two-piece forward products: {shape}", flush=True)
    rng = np.random.default_rng(101)
    if shape == "32x1024":
        lengths = [1024] * 32
        batch = synthetic_batch(rng, lengths, *_heads(32), 50368)
    else:
        lengths = rng.integers(16, 2049, 64)
        batch = synthetic_batch(rng, lengths, *_heads(64), 50368, zipf=1.1)
    targets = np.concatenate([np.eye(k, dtype=np.float32)[rng.integers(k)] for k in batch.n_options])
    c = Context(0)
    try:
        c.set_matmul_precision("bf16-backward")
        m = TrainableDecisionModel(modernbert_base(), c)
        params = synthetic_params(m.shapes, 101)
        pw = _product_weights(m.shapes)
        m.set_params({n: (bf16(v) if n in pw else v) for n, v in params.items()})
        m.head_dropout = 0.1
        steps, ran = [], []
        for on in (True, False):
            m.set_bf16_weights(on)
            m.zero_gradients()
            c.profile_begin()
            logits = m.forward(batch, training=True, seed=7)
            ran.append(sorted(n for n in c.profile_end() if n.startswith("gemm_nt_h2")))
            _, g = oracle.cross_entropy(batch.n_options, logits, targets, 1.0, float(batch.n_items))
            m.backward(g)
            steps.append((logits, {n: m.grad(n) for n in m.names if m.has_grad(n)}))
        print(f"forward products: {ran[0]} against {ran[1]}", flush=True)
        assert "gemm_nt_h2b1w" in ran[0] and not any("b1" in n for n in ran[1]), ran
        (l1, g1), (l2, g2) = steps
        np.testing.assert_array_equal(l1, l2)
        for n in g1:
            np.testing.assert_array_equal(g1[n], g2[n], err_msg=n)
        print(f"{shape}: logits and {len(g1)} gradients equal bit for bit", flush=True)
        m.close()
    finally:
        c.close()


def _copies_step(m, batch, d, seed=5):
    m.zero_gradients()
    logits = m.forward(batch, training=True, seed=seed)
    m.backward(d)
    return logits, {n: m.grad(n) for n in m.names if m.has_grad(n)}


@pytest.mark.parametrize("policy", ["bf16-backward", "bf16"])
def test_bf16_copies_give_bitwise_the_same_step(policy):
    """The bf16 copies (weights, and the saved activations the products read) hold exactly the values the
    products would round their fp32 operands to (nearest even), so a step reading them equals a step
    rounding in-kernel bit for bit — with head dropout, and with the encoder layers recomputed."""
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    import helpers
    print(f"bf16 copies: on vs off, policy {policy}", flush=True)
    c = Context(0)
    try:
        c.set_matmul_precision(policy)
        cfg = helpers.mid_config(layers=4)
        m = TrainableDecisionModel(cfg, c)
        m.set_params(helpers.random_params(m.shapes, 71, std=0.03))
        m.head_dropout = 0.1
        batch = helpers.mixed_batch(np.random.default_rng(72), [300, 129, 64, 17, 211, 1200], cfg.encoder.vocab_size)
        d = np.random.default_rng(73).standard_normal(batch.n_markers).astype(np.float32)
        m.set_bf16_copies(False)
        l0, g0 = _copies_step(m, batch, d)
        with pytest.raises(Exception):
            m.param_bf16("encoder.layers.1.attn.Wqkv.weight")  # no copy is kept with the option off
        m.set_bf16_copies(True)
        l1, g1 = _copies_step(m, batch, d)
        np.testing.assert_array_equal(l0, l1)
        for n in g0:
            np.testing.assert_array_equal(g0[n], g1[n], err_msg=n)
        m.layer_checkpointing = m.CHECKPOINT_RECOMPUTE
        l2, g2 = _copies_step(m, batch, d)
        assert m.recomputing
        np.testing.assert_array_equal(l0, l2)
        for n in g0:
            np.testing.assert_array_equal(g0[n], g2[n], err_msg=n)
        m.close()
    finally:
        c.close()


def test_adamw_keeps_the_bf16_weight_copy_current():
    """Through optimizer steps the weights' bf16 copy is bf16(master) to the bit: refreshed from the masters
    after host writes, and written by the AdamW kernel with each update."""
    from laya_amd.device import Context
    from laya_amd.model import TrainableDecisionModel
    import helpers
    print("bf16 copies: the weight copy through AdamW steps", flush=True)
    c = Context(0)
    try:
        c.set_matmul_precision("bf16-backward")
        cfg = helpers.mid_config(layers=2)
        m = TrainableDecisionModel(cfg, c)
        m.set_params(helpers.random_params(m.shapes, 81, std=0.03))
        rng = np.random.default_rng(82)
        batch = helpers.mixed_batch(rng, [200, 90, 33], cfg.encoder.vocab_size)
        targets = np.concatenate([np.eye(k, dtype=np.float32)[rng.integers(k)] for k in batch.n_options])
        m.set_trainable_encoder_layers(1)  # frozen layers keep their copy as refreshed
        for step in range(3):
            m.train_step(batch, targets, seed=step, ce_weight=1.0, loss_scale=1.0, max_norm=1.0, lr_encoder=1e-3,
                         lr_head=1e-3, weight_decay=0.01)
            if step == 1:
                m.set_param("scorer.0.weight", np.full(m.shapes["scorer.0.weight"], 1.0 + 2 ** -9, np.float32))
        m.forward(batch)  # refreshes the copy after the host write
        for n in m.names:
            np.testing.assert_array_equal(m.param_bf16(n), bf16(m.param(n)), err_msg=n)
        m.close()
    finally:
        c.close()


def _forward_backward(ctx, mc, params, batch, targets, seed, policy, bf16_weights=False):
    from laya_amd.model import TrainableDecisionModel
    ctx.set_matmul_precision(policy)
    try:
        m = TrainableDecisionModel(mc, ctx)
        m.set_params(params)
        m.head_dropout = 0.1
        if bf16_weights:
            m.set_bf16_weights(True)
        logits = m.forward(batch, training=True, seed=seed)
        _, g = oracle.cross_entropy(batch.n_options, logits, targets, 1.0, float(batch.n_items))
        m.backward(g)
        grads = {n: m.grad(n) for n in m.names if m.has_grad(n)}
        m.close()
    finally:
        ctx.set_matmul_precision("bf16")
    return logits, g, grads


def _product_weights(names):
    """The weights the matrix products read (the linears of the encoder, head and scorer)."""
    return [n for n in names if n.endswith(("Wqkv.weight", "Wo.weight", "Wi.weight", "in_proj_weight",
                                            "out_proj.weight", "linear1.weight", "linear2.weight",
                                            "scorer.1.weight", "scorer.3.weight"))]


def _modernbert_base_case(seed, n=4, length=256):
    from laya_amd.batch import synthetic_batch
    from laya_amd.config import modernbert_base
    import helpers
    mc = modernbert_base()
    shapes = oracle.OracleModel(mc).shapes
    rng = np.random.default_rng(seed)
    opts, qt = _heads(n)
    batch = synthetic_batch(rng, [length] * n, opts, qt, 50368)
    targets = np.concatenate([np.eye(k, dtype=np.float32)[rng.integers(k)] for k in batch.n_options])
    # Head linear1 biases away from the ReLU's kink (tests/helpers.fixture_params): no ReLU input lies within
    # rounding of zero, so the comparison sees the products' rounding and nothing else.
    return mc, shapes, helpers.fixture_params(shapes, seed), batch, targets


def test_bf16_weights_match_the_oracle_fed_the_rounded_weights(ctx):
    """bf16 weights as the reference's PackedMatrixBf16 keeps them (a bf16 weight widened exactly to fp32 inside
    an fp32 product, PackedMatrixBf16.cs:7-21): ModernBERT-base, 22 layers, 4 × 256 tokens, every product
    fp32-accurate (the default two-piece products) on fp32 activations, the products reading each weight
    rounded to bf16. Against the oracle (fp32 and fp64) fed the same bf16-rounded weights: logits to 1e-5 and
    every gradient within max(1e-4, 4 × the fp32 oracle's error) of fp64 — the fp32 bar. Then AdamW updates the
    fp32 masters and the products follow the rounding of the updated weights."""
    from laya_amd.config import modernbert_base  # noqa: F401
    from laya_amd.model import TrainableDecisionModel
    print("bf16 weights: ModernBERT-base 22 layers, 4 x 256, vs the oracle with bf16-rounded weights", flush=True)
    mc, shapes, params, batch, targets = _modernbert_base_case(71)
    rounded = dict(params)
    pw = _product_weights(shapes)
    assert len(pw) == 4 * 22 + 4 * 2 + 2
    for n in pw:
        rounded[n] = bf16(params[n])
    seed = 71
    logits, g, grads = _forward_backward(ctx, mc, params, batch, targets, seed, "fp32", bf16_weights=True)
    o, o64 = oracle.OracleModel(mc), oracle.OracleModel(mc, double=True)
    for r in (o, o64):
        r.set_params(rounded)
        r.set_head_dropout(0.1)
        r.forward(batch, training=True, keep_tape=True, seed=seed)
        r.backward(g)
    lo = o64.forward(batch, training=True, keep_tape=False, seed=seed)
    assert np.abs(logits - lo).max() < 1e-5
    worst = (0.0, "")
    for n in grads:
        exact = o64.grad(n)
        bar = max(1e-4, 4 * rel_l2(exact, o.grad(n)))
        r = rel_l2(exact, grads[n])
        assert r < bar, (n, r, bar)
        if bar == 1e-4:
            worst = max(worst, (r, n))
    print(f"bf16 weights vs the oracle fed bf16-rounded weights: worst gradient rel-L2 {worst[0]:.2e} ({worst[1]})",
          flush=True)
    # The unrounded weights move the logits by the weights' rounding, not more.
    lf = oracle.OracleModel(mc, double=True)
    lf.set_params(params)
    lf.set_head_dropout(0.1)
    print(f"logits vs unrounded weights: rel-L2 {rel_l2(lf.forward(batch, True, False, seed), logits):.2e}",
          flush=True)
    # After an AdamW step the products read the rounding of the updated masters.
    ctx.set_matmul_precision("fp32")
    try:
        m = TrainableDecisionModel(mc, ctx)
        m.set_params(params)
        m.set_bf16_weights(True)
        m.forward(batch, training=True, seed=seed)
        m.backward(g)
        m.adamw_step(1e-3, 1e-3)
        masters = {n: m.param(n) for n in shapes}
        lg = m.forward(batch, training=False)
        ref = oracle.OracleModel(mc, double=True)
        ref.set_params({n: (bf16(v) if n in pw else v) for n, v in masters.items()})
        assert np.abs(lg - ref.forward(batch, training=False, keep_tape=False)).max() < 1e-5
        m.close()
    finally:
        ctx.set_matmul_precision("bf16")


@pytest.mark.parametrize("weights", ["relu-clear", "generic"])
def test_every_product_in_bf16_against_the_fp32_oracle(ctx, weights):
    """Every product on bf16 operands (forward and backward, weights and activations rounded to bf16, fp32
    accumulation, statistics and masters) against the fp32 oracle with the unrounded weights, at ModernBERT-base
    (22 layers, 4 × 256). With head linear1 biases away from the ReLU's kink ("relu-clear") the difference is
    the products' rounding alone and every gradient is held to the bf16 bar, 2e-2. With the benchmark's kind of
    initialisation ("generic": zero biases, unit γ) ~10³ of the head's 6.3M ReLU inputs lie within bf16
    rounding of zero and are decided the other way; that is measured and printed, held only to 1e-1."""
    from laya_amd.model import synthetic_params
    print(f"every product in bf16 vs the fp32 oracle, {weights} weights", flush=True)
    mc, shapes, params, batch, targets = _modernbert_base_case(81)
    if weights == "generic":
        params = synthetic_params(shapes, 81)
    seed = 81
    logits, g, grads = _forward_backward(ctx, mc, params, batch, targets, seed, "bf16")
    o = oracle.OracleModel(mc)
    o.set_params(params)
    o.set_head_dropout(0.1)
    lo = o.forward(batch, training=True, keep_tape=True, seed=seed)
    o.backward(g)
    print(f"logits rel-L2 vs fp32: {rel_l2(lo, logits):.2e}", flush=True)
    worst = _grads_match(list(grads), {n: o.grad(n) for n in grads}, grads, 2e-2 if weights == "relu-clear" else 1e-1)
    print(f"every product in bf16 ({weights}): worst gradient rel-L2 vs the fp32 oracle {worst:.2e}", flush=True)


def test_bf16_weights_with_bf16_backward_products_against_the_oracle(ctx):
    """The policy the bf16 benchmark workloads run: bf16 weights (each product reads the weight rounded to bf16,
    PackedMatrixBf16.cs:7-21) with a forward of fp32-accurate products on fp32 activations, and the backward
    products on bf16 operands (weights, output gradients and saved activations rounded to bf16, fp32
    accumulation). ModernBERT-base, 22 layers, 4 × 256, the benchmark's kind of initialisation (zero biases,
    unit γ), against the oracle fed the same bf16-rounded weights: logits to 1e-5 (the forward is the oracle's
    function) and every gradient within the bf16 bar, 2e-2."""
    from laya_amd.model import synthetic_params
    print("bf16 weights + bf16 backward products vs the oracle with bf16-rounded weights", flush=True)
    mc, shapes, _, batch, targets = _modernbert_base_case(91)
    params = synthetic_params(shapes, 91)
    rounded = {n: (bf16(v) if n in _product_weights(shapes) else v) for n, v in params.items()}
    seed = 91
    logits, g, grads = _forward_backward(ctx, mc, params, batch, targets, seed, "bf16-backward", bf16_weights=True)
    o = oracle.OracleModel(mc)
    o.set_params(rounded)
    o.set_head_dropout(0.1)
    lo = o.forward(batch, training=True, keep_tape=True, seed=seed)
    assert np.abs(logits - lo).max() < 1e-5
    o.backward(g)
    worst = _grads_match(list(grads), {n: o.grad(n) for n in grads}, grads, 2e-2)
    print(f"bf16 weights + bf16 backward products: worst gradient rel-L2 vs the oracle {worst:.2e}", flush=True)
