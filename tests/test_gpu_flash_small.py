"""The flash attention kernel for few tokens (one workgroup per head and 16 or
32 queries, its waves splitting the keys in groups of 32) against the oracle:
one token, tokens that end inside a query block, a key group and a round of
eight groups, exactly on them, and three rounds; a kernel of several parts;
and a block whose attention reads the operands its QKV projection wrote; and
infinities, in scores and values (not in bf16x3, where an infinity has no hi
and lo parts).

Tolerance for f32 storage: |got - want| <= 1e-4 + 1e-4 |want|
(reference.rs:22-24); for f16 storage, max abs error <= 2e-2 against the
oracle on the same f16-rounded inputs.
"""

import numpy as np
import pytest

import oracle
from beatlm_amd import hip, ir
from tests.blockdata import block_graph, block_values, block_weights, max_abs_err
from tests.test_gpu_sweep import attention_graph

pytestmark = pytest.mark.gpu

X, Y = 0, 20
F16_TOL = 2e-2
MATHS = ["bf16x3", "f32", "f16"]


def compare(got, want, math, what):
    if math == "f16":
        err = max_abs_err(got, want)
        assert err <= F16_TOL, f"{what}: max abs error {err:.3e}"
    else:
        bad = oracle.first_mismatch(got, want)
        assert bad is None, f"{what}: element {bad[0]} is {bad[1]}, the oracle says {bad[2]}"


@pytest.fixture
def math(ctx, request):
    if request.param == "f32":
        ctx.set_f32_math(hip.F32_MATH_MFMA_F32)
    yield request.param
    ctx.set_f32_math(hip.F32_MATH_SPLIT_BF16)


@pytest.mark.parametrize("t,h,parts", [(1, 1, 1), (15, 2, 1), (32, 1, 1), (33, 3, 1), (64, 2, 1), (256, 1, 1), (257, 6, 1),
                                       (290, 2, 3), (700, 2, 1)])
@pytest.mark.parametrize("math", MATHS, indirect=True)
@pytest.mark.parametrize("blocks", ["1", "2"])
def test_attention_of_few_tokens_matches_the_oracle(ctx, monkeypatch, t, h, parts, math, blocks):
    monkeypatch.setenv("BL_FLASH_SMALL", blocks)
    # Scores of up to +-40, so that the running maximum moves and most
    # probabilities are small.
    qkv = oracle.uniform(t + 100 * h, t * 3 * h * 64, -3.0, 3.0)
    if math == "f16":
        qkv = qkv.astype(np.float16)
    want = oracle.attention(qkv.astype(np.float32), t, h, 64, 0.125)
    prep = ir.prepare(ctx, attention_graph(t, h, 64), parts=parts, dtype=hip.F16 if math == "f16" else hip.F32)
    try:
        assert all("keys over waves" in prep.kernels.label(k) for k in range(len(prep.kernels)))
        prep.write(X, qkv)
        prep.run()
        ctx.synchronize()
        compare(prep.read(Y).astype(np.float32), want, math, f"t={t} h={h} parts={parts}")
    finally:
        prep.close()


@pytest.mark.parametrize("t", [50, 257])
@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_a_small_blocks_attention_reads_its_projections_operands(ctx, t, math):
    """The planner's own choice in an encoder block, run twice (the second pass
    finds the first one's operands and statistics)."""
    d, h, mlp = 128, 2, 512
    x, w = oracle.uniform(21, t * d, -2.0, 2.0), block_weights(d, mlp, 100, "reference")
    g, ids = block_graph(t, d, h, mlp, 1e-6)
    prep = ir.prepare(ctx, g, dtype=hip.F16 if math == "f16" else hip.F32)
    try:
        labels = [prep.kernels.label(k) for k in range(len(prep.kernels))]
        assert any("keys over waves" in lab for lab in labels), labels
        vals = block_values(ids, x, w)
        if math == "f16":
            vals = {k: v.astype(np.float16) for k, v in vals.items()}
        for tid, v in vals.items():
            prep.write(tid, v)
        for _ in range(2):
            prep.run()
        ctx.synchronize()
        got = prep.read(ids.output).astype(np.float32)
    finally:
        prep.close()
    if math == "f16":
        x, w = (x.astype(np.float16).astype(np.float32), {k: v.astype(np.float16).astype(np.float32) for k, v in w.items()})
    compare(got, oracle.vit_block(x, w, t, h, d // h, mlp, 1e-6), math, f"block of {t} tokens")


@pytest.mark.parametrize("t,first,count", [(70, 32, 32), (290, 0, 64), (300, 128, 100)])
@pytest.mark.parametrize("math", ["f32", "f16"], indirect=True)
@pytest.mark.parametrize("blocks", ["1", "2"])
def test_keys_with_scores_of_minus_infinity_take_no_part(ctx, monkeypatch, t, first, count, math, blocks):
    """Keys first .. first + count - 1 score -inf against every query (whole
    groups of 32 of them): their probabilities are zero, as a softmax over
    the row has them."""
    monkeypatch.setenv("BL_FLASH_SMALL", blocks)
    qkv = oracle.uniform(t, t * 192, -3.0, 3.0)
    if math == "f16":
        qkv = qkv.astype(np.float16)
    v = qkv.reshape(t, 3, 64)
    v[:, 0, 5] = 1.0
    v[first : first + count, 1, 5] = -np.inf
    kept = np.delete(v, np.s_[first : first + count], 0)
    s = v[:, 0].astype(np.float64) @ kept[:, 1].astype(np.float64).T * 0.125
    p = np.exp(s - s.max(1, keepdims=True))
    want = (p / p.sum(1, keepdims=True)) @ kept[:, 2].astype(np.float64)
    prep = ir.prepare(ctx, attention_graph(t, 1, 64), dtype=hip.F16 if math == "f16" else hip.F32)
    try:
        assert "keys over waves" in prep.kernels.label(0)
        prep.write(X, qkv)
        prep.run()
        ctx.synchronize()
        compare(prep.read(Y).astype(np.float32), want.reshape(-1).astype(np.float32), math, f"t={t}")
    finally:
        prep.close()


@pytest.mark.parametrize("t", [33, 257, 290])
@pytest.mark.parametrize("math", ["f32", "f16"], indirect=True)
@pytest.mark.parametrize("blocks", ["1", "2"])
def test_an_infinite_value_of_the_last_token_stays_infinite(ctx, monkeypatch, t, math, blocks):
    """One column of the last token's value is +inf: that column of every
    query's output is, and no other column is touched."""
    monkeypatch.setenv("BL_FLASH_SMALL", blocks)
    qkv = oracle.uniform(t + 1, t * 192, -1.0, 1.0)
    if math == "f16":
        qkv = qkv.astype(np.float16)
    qkv.reshape(t, 3, 64)[-1, 2, 9] = np.inf
    want = oracle.attention(np.where(np.isinf(qkv), 0, qkv).astype(np.float32), t, 1, 64, 0.125).reshape(t, 64)
    prep = ir.prepare(ctx, attention_graph(t, 1, 64), dtype=hip.F16 if math == "f16" else hip.F32)
    try:
        prep.write(X, qkv)
        prep.run()
        ctx.synchronize()
        got = prep.read(Y).astype(np.float32).reshape(t, 64)
        assert np.all(np.isposinf(got[:, 9])), got[:4, 9]
        rest = np.arange(64) != 9
        compare(got[:, rest].reshape(-1), want[:, rest].reshape(-1), math, f"t={t}")
    finally:
        prep.close()


@pytest.mark.parametrize("math,t,h,parts,few", [
    ("f16", 1200, 6, 1, True), ("f16", 1370, 6, 4, True), ("f16", 2501, 6, 4, False), ("f16", 5477, 6, 4, False), ("f16", 8192, 1, 1, False),
    ("f32", 1370, 6, 4, True), ("f32", 5477, 6, 2, False), ("f32", 8192, 1, 4, False),
    ("bf16x3", 626, 6, 1, True), ("bf16x3", 626, 6, 4, False), ("bf16x3", 362, 6, 4, True), ("bf16x3", 700, 6, 1, False)], indirect=["math"])
def test_parts_of_a_long_sequence_keep_the_kernel_that_shares_out_its_keys(ctx, math, t, h, parts, few):
    """The few-token kernel's time grows with the tokens however few a part's
    rows: every part of one kernel is planned by both (a projection before it,
    so that the choice is the planner's in f16 and bf16x3 too)."""
    d, g = 64 * h, ir.Graph()
    for tid, n in ((0, t * d), (1, 3 * d * d), (2, 3 * d)):
        g.tensor(tid, ir.WEIGHT if tid else ir.INPUT, n)
    ops = [ir.op(ir.OP_MATMUL, [0, 1, 2], [t, d, 3 * d]), ir.op(ir.OP_ATTENTION_SCORES, [10], [t, h, 64]),
           ir.op(ir.OP_SCALE, [11], [t * h * t], 0.125), ir.op(ir.OP_SOFTMAX, [12], [t * h, t]), ir.op(ir.OP_ATTENTION_VALUES, [13, 10], [t, h, 64])]
    for i, o in enumerate(ops):
        g.tensor(10 + i, ir.OUTPUT if i == 4 else ir.ACTIVATION, ir.output_elements(o))
        g.push(o, 10 + i)
    prep = ir.realise(ctx, g.lower().fuse_attention().split([1, parts]), hip.F16 if math == "f16" else hip.F32)
    try:
        labels = [prep.kernels.label(k) for k in range(1, len(prep.kernels))]
        assert all(("keys over waves" in lab) == few for lab in labels), labels
    finally:
        prep.close()
