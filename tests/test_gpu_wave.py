"""The wave-split product (eight waves of a workgroup splitting the k-steps of
one small tile) against the oracle at the edges of its tiles and k-steps: one
row, a row more or less than a tile, columns that end inside a tile, fewer
k-steps than waves, exactly as many, and one more than two or four rounds of
them; the 3x3 convolution's windows where a k-step lies inside a tap (64 or 32
channels a step) and where it straddles two; the patch gather with even and
odd patch rows; residual units whose image passes between convolutions as bf16
planes.

Tolerance for f32 storage: |got - want| <= 1e-4 + 1e-4 |want|
(reference.rs:22-24); for f16 storage, max abs error <= 2e-2 against the
oracle on the same f16-rounded inputs.
"""

import numpy as np
import pytest

import oracle
from beatlm_amd import hip, ir
from tests.blockdata import CHAIN as H_, CHAIN_OUT as Y, block_values, block_weights, chain, max_abs_err

pytestmark = pytest.mark.gpu

F16_TOL = 2e-2
MATHS = ["bf16x3", "f32", "f16"]
TILES = {"1": "wave 16x32", "2": "wave 32x32", "3": "wave 32x64"}


def check(ctx, monkeypatch, vals, ops, want, math, tile, waves):
    """Runs the chain with the wave-split tile forced and compares its output;
    `waves`: the kernels that must take it."""
    monkeypatch.setenv("BL_GEMM_WAVE", tile)
    if math == "f32":
        ctx.set_f32_math(hip.F32_MATH_MFMA_F32)
    try:
        prep = ir.prepare(ctx, chain(vals, ops), dtype=hip.F16 if math == "f16" else hip.F32)
        try:
            labels = [prep.kernels.label(k) for k in range(len(prep.kernels))]
            assert sum(TILES[tile] in lab for lab in labels) == waves, labels
            for tid, v in vals.items():
                prep.write(tid, v)
            prep.run()
            ctx.synchronize()
            got = prep.read(Y).astype(np.float32)
        finally:
            prep.close()
    finally:
        ctx.set_f32_math(hip.F32_MATH_SPLIT_BF16)
    if math == "f16":
        err = max_abs_err(got, want)
        assert err <= F16_TOL, f"{labels}: max abs error {err:.3e}"
    else:
        bad = oracle.first_mismatch(got, want)
        assert bad is None, f"{labels}: element {bad[0]} is {bad[1]}, the oracle says {bad[2]}"


def stored(math, *arrays):
    """The values as stored, and as the oracle reads them."""
    kept = [a.astype(np.float16) if math == "f16" else a for a in arrays]
    return kept, [a.astype(np.float32) for a in kept]


@pytest.mark.parametrize("m,k,n", [(1, 64, 8), (15, 512, 40), (17, 576, 32), (33, 1088, 72), (64, 2112, 136), (257, 1536, 384),
                                   (31, 4160, 64)])
@pytest.mark.parametrize("math", MATHS)
@pytest.mark.parametrize("tile", TILES)
def test_a_wave_split_product_matches_the_oracle(ctx, monkeypatch, m, k, n, math, tile):
    (a, b, bias), (af, bf, biasf) = stored(math, oracle.uniform(3 + k, m * k, -2.0, 2.0), oracle.fan_in_weights(4 + n, k * n, k),
                                           oracle.uniform(5 + n, n, -0.1, 0.1))
    check(ctx, monkeypatch, {0: a, 1: b, 2: bias}, [ir.op(ir.OP_MATMUL, [0, 1, 2], [m, k, n])],
          oracle.matmul(af, bf, biasf, m, k, n), math, tile, 1)


@pytest.mark.parametrize("h,w,cin,cout,stride", [(5, 7, 64, 64, 1), (9, 13, 96, 40, 1), (6, 5, 48, 24, 2), (10, 9, 384, 64, 2),
                                                 (3, 3, 32, 8, 1), (1, 1, 128, 32, 1)])
@pytest.mark.parametrize("math", MATHS)
@pytest.mark.parametrize("tile", TILES)
def test_a_wave_split_convolution_matches_the_oracle(ctx, monkeypatch, h, w, cin, cout, stride, math, tile):
    (x, wt, b), (xf, wf, bf) = stored(math, oracle.uniform(6 + cin, h * w * cin, -2.0, 2.0),
                                      oracle.fan_in_weights(7 + cout, 9 * cin * cout, 9 * cin), oracle.uniform(8, cout, -0.1, 0.1))
    check(ctx, monkeypatch, {0: x, 1: wt, 2: b}, [ir.op(ir.OP_CONV3X3, [0, 1, 2], [h, w, cin, cout, stride])],
          oracle.conv3x3(xf, wf, bf, h, w, cin, cout, stride), math, tile, 1)


@pytest.mark.parametrize("channels", [32, 64])
@pytest.mark.parametrize("math", MATHS)
@pytest.mark.parametrize("tile", TILES)
def test_a_wave_split_residual_unit_matches_the_oracle(ctx, monkeypatch, channels, math, tile):
    """relu -> conv -> relu -> conv -> + x: the ReLU prologues, the first
    convolution's output kept as bf16 planes, and the skip in the epilogue."""
    side, c = 11, channels
    px = side * side * c
    (x, w1, b1, w2, b2), f = stored(math, oracle.uniform(31, px, -2.0, 2.0), oracle.fan_in_weights(32, 9 * c * c, 9 * c),
                                    oracle.uniform(33, c, -0.1, 0.1), oracle.fan_in_weights(34, 9 * c * c, 9 * c),
                                    oracle.uniform(35, c, -0.1, 0.1))
    ops = [ir.op(ir.OP_RELU, [0], [px]), ir.op(ir.OP_CONV3X3, [H_, 1, 2], [side, side, c, c, 1]), ir.op(ir.OP_RELU, [H_ + 1], [px]),
           ir.op(ir.OP_CONV3X3, [H_ + 2, 3, 4], [side, side, c, c, 1]), ir.op(ir.OP_ADD, [H_ + 3, 0], [px])]
    h = np.maximum(oracle.conv3x3(np.maximum(f[0], 0), f[1], f[2], side, side, c, c, 1), 0)
    want = oracle.conv3x3(h, f[3], f[4], side, side, c, c, 1) + f[0]
    check(ctx, monkeypatch, dict(enumerate([x, w1, b1, w2, b2])), ops, want, math, tile, 2)


@pytest.mark.parametrize("gh,gw,p,cin", [(3, 5, 14, 3), (1, 1, 7, 3), (4, 9, 5, 5), (6, 3, 16, 4)])
@pytest.mark.parametrize("math", MATHS)
@pytest.mark.parametrize("tile", TILES)
def test_a_wave_split_patch_embedding_matches_the_oracle(ctx, monkeypatch, gh, gw, p, cin, math, tile):
    cout, k = 40, p * p * cin
    (x, w, b), (xf, wf, bf) = stored(math, oracle.uniform(41, gh * p * gw * p * cin, -2.0, 2.0), oracle.fan_in_weights(42, k * cout, k),
                                     oracle.uniform(43, cout, -0.1, 0.1))
    check(ctx, monkeypatch, {0: x, 1: w, 2: b}, [ir.op(ir.OP_PATCH_EMBED, [0, 1, 2], [gh, gw, p, cin, cout])],
          oracle.patch_embed(xf, wf, bf, gh, gw, p, cin, cout), math, tile, 1)


@pytest.mark.parametrize("t", [17, 64, 65, 257])
@pytest.mark.parametrize("math", MATHS)
@pytest.mark.parametrize("tile", TILES)
def test_wave_split_products_of_a_block_match_the_oracle(ctx, monkeypatch, t, math, tile):
    """Two encoder blocks with every product wave-split: the QKV projections
    write the attention's operands (tokens that end inside a 16-token run) and,
    with fc1, apply folded LayerNorms whose rows' common offset is ten times
    their spread; the out-projections and fc2 leave row statistics."""
    d, h, mlp, eps = 192, 3, 768, 1e-6
    monkeypatch.setenv("BL_GEMM_WAVE", tile)
    x = oracle.uniform(61, t * d, -2.0, 2.0) + np.float32(0.0 if math == "f16" else 20.0)
    ws = [block_weights(d, mlp, seed, "reference") for seed in (100, 200)]
    g = ir.Graph()
    g.tensor(0, ir.INPUT, t * d)
    a = g.vit_block(ir.VitDims(t, d, h, mlp, eps), 0, 100, ir.ACTIVATION)
    b = g.vit_block(ir.VitDims(t, d, h, mlp, eps), a.output, a.next_id, ir.OUTPUT)
    vals = block_values(a, x, ws[0]) | block_values(b, x, ws[1])
    if math == "f16":
        vals = {k: v.astype(np.float16) for k, v in vals.items()}
    if math == "f32":
        ctx.set_f32_math(hip.F32_MATH_MFMA_F32)
    try:
        prep = ir.prepare(ctx, g, dtype=hip.F16 if math == "f16" else hip.F32)
        try:
            labels = [prep.kernels.label(k) for k in range(len(prep.kernels))]
            assert sum(TILES[tile] in lab for lab in labels) == 8 and sum("folded into" in lab for lab in labels) == 3, labels
            for tid, v in vals.items():
                prep.write(tid, v)
            prep.run()
            ctx.synchronize()
            got = prep.read(b.output).astype(np.float32)
        finally:
            prep.close()
    finally:
        ctx.set_f32_math(hip.F32_MATH_SPLIT_BF16)
    if math == "f16":
        x, ws = x.astype(np.float16).astype(np.float32), [{k: v.astype(np.float16).astype(np.float32) for k, v in w.items()} for w in ws]
    want = oracle.vit_block(oracle.vit_block(x, ws[0], t, h, 64, mlp, eps), ws[1], t, h, 64, mlp, eps)
    if math == "f16":
        err = max_abs_err(got, want)
        assert err <= F16_TOL, f"{labels}: max abs error {err:.3e}"
    else:
        bad = oracle.first_mismatch(got, want)
        assert bad is None, f"{labels}: element {bad[0]} is {bad[1]}, the oracle says {bad[2]}"
