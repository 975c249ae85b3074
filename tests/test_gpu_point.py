"""Launches that took two kernels' place, against the oracle: the transposed
convolution as a product over input pixels (channels that end inside a 32-wide
slice, columns that end inside a 64-wide block, rows that end inside a
16-pixel tile), the 1x1 convolution that blends its resampled input's corners
as it loads them, the direct convolution that adds up its channels for a
one-column product, and the taps' LayerNorm that writes the feature map; each
run twice over the same inputs.

Tolerance for f32 storage: |got - want| <= 1e-4 + 1e-4 |want|
(reference.rs:22-24); for f16 storage, max abs error <= 2e-2 against the
oracle on the same f16-rounded inputs.
"""

import numpy as np
import pytest

import oracle
from beatlm_amd import hip, ir
from tests.blockdata import CHAIN as H_, CHAIN_OUT as Y, chain, max_abs_err

pytestmark = pytest.mark.gpu

F16_TOL = 2e-2
MATHS = ["bf16x3", "f32", "f16"]


def check(ctx, arrays, ops, oracle_of, math, marks):
    """`arrays` in storage type are tensors 0 ..; oracle_of takes them as f32;
    `marks`: texts that some label must hold."""
    kept = [a.astype(np.float16) if math == "f16" else a for a in arrays]
    want = oracle_of(*[a.astype(np.float32) for a in kept])
    vals = dict(enumerate(kept))
    if math == "f32":
        ctx.set_f32_math(hip.F32_MATH_MFMA_F32)
    try:
        prep = ir.prepare(ctx, chain(vals, ops), dtype=hip.F16 if math == "f16" else hip.F32)
        try:
            labels = [prep.kernels.label(k) for k in range(len(prep.kernels))]
            for mark in marks:
                assert any(mark in lab for lab in labels), (mark, labels)
            for tid, v in vals.items():
                prep.write(tid, v)
            for _ in range(2):
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


@pytest.mark.parametrize("h,w,cin,cout,f", [(1, 1, 8, 8, 2), (3, 5, 48, 48, 4), (4, 4, 96, 24, 2), (7, 9, 40, 16, 3), (37, 37, 32, 8, 1)])
@pytest.mark.parametrize("math", MATHS)
def test_a_transposed_convolution_as_a_product_matches_the_oracle(ctx, h, w, cin, cout, f, math):
    arrays = [oracle.uniform(1 + cin, h * w * cin, -2.0, 2.0), oracle.fan_in_weights(2 + cout, f * f * cin * cout, cin),
              oracle.uniform(3, cout, -0.1, 0.1)]
    check(ctx, arrays, [ir.op(ir.OP_CONV_TRANSPOSE, [0, 1, 2], [h, w, cin, cout, f])],
          lambda x, wt, b: oracle.conv_transpose(x, wt, b, h, w, cin, cout, f), math, ["rows"])


@pytest.mark.parametrize("ih,iw,oh,ow,c,n", [(1, 1, 3, 2, 8, 8), (5, 7, 10, 14, 64, 64), (6, 4, 11, 9, 96, 72), (9, 9, 5, 4, 32, 136),
                                             (3, 8, 1, 1, 40, 16)])
@pytest.mark.parametrize("math", MATHS)
def test_a_resampling_blended_into_its_product_matches_the_oracle(ctx, ih, iw, oh, ow, c, n, math):
    """conv -> resize -> 1x1 -> relu, the product writing the program's output
    (one that lies over the convolution's: test_gpu_plans.py)."""
    arrays = [oracle.uniform(11 + c, ih * iw * c, -2.0, 2.0), oracle.fan_in_weights(12, 9 * c * c, 9 * c), oracle.fan_in_weights(13 + n, c * n, c),
              oracle.uniform(14, n, -0.1, 0.1)]
    ops = [ir.op(ir.OP_CONV3X3, [0, 1, ir.NONE], [ih, iw, c, c, 1]), ir.op(ir.OP_RESIZE_BILINEAR, [H_], [ih, iw, oh, ow, c]),
           ir.op(ir.OP_MATMUL, [H_ + 1, 2, 3], [oh * ow, c, n]), ir.op(ir.OP_RELU, [H_ + 2], [oh * ow * n])]

    def want(x, wc, w, b):
        y = oracle.resize_bilinear(oracle.conv3x3(x, wc, None, ih, iw, c, c, 1), ih, iw, oh, ow, c)
        return np.maximum(oracle.matmul(y, w, b, oh * ow, c, n), 0)

    check(ctx, arrays, ops, want, math, ["rows < resize 1", "fused into 2"])


@pytest.mark.parametrize("h,w,cin", [(130, 255, 32), (67, 513, 40)])
@pytest.mark.parametrize("math", ["bf16x3", "f16"])
def test_a_convolution_that_adds_up_its_channels_matches_the_oracle(ctx, h, w, cin, math):
    """conv (direct) -> relu -> 1x1 to one channel -> relu."""
    arrays = [oracle.uniform(21, h * w * cin, -2.0, 2.0), oracle.fan_in_weights(22, 9 * cin * 32, 9 * cin), oracle.uniform(23, 32, -0.1, 0.1),
              oracle.fan_in_weights(24, 32, 32), oracle.uniform(25, 1, -0.1, 0.1)]
    ops = [ir.op(ir.OP_CONV3X3, [0, 1, 2], [h, w, cin, 32, 1]), ir.op(ir.OP_RELU, [H_], [h * w * 32]),
           ir.op(ir.OP_MATMUL, [H_ + 1, 3, 4], [h * w, 32, 1]), ir.op(ir.OP_RELU, [H_ + 2], [h * w])]
    check(ctx, arrays, ops, lambda x, wc, bc, w1, b1: np.maximum(
        oracle.matmul(np.maximum(oracle.conv3x3(x, wc, bc, h, w, cin, 32, 1), 0), w1, b1, h * w, 32, 1), 0),
        math, ["direct", "< product 1"])


@pytest.mark.parametrize("grid,d", [(1, 64), (5, 384), (6, 48)])
@pytest.mark.parametrize("math", MATHS)
def test_a_layernorm_that_writes_the_map_matches_the_oracle(ctx, grid, d, math):
    t = grid * grid + 1
    arrays = [oracle.uniform(31, t * d, -2.0, 2.0), oracle.uniform(32, d, 0.5, 1.5), oracle.uniform(33, d, -0.5, 0.5)]
    ops = [ir.op(ir.OP_LAYER_NORM, [0, 1, 2], [t, d], 1e-6), ir.op(ir.OP_TOKENS_TO_MAP, [H_], [grid, grid, d])]
    check(ctx, arrays, ops, lambda x, g, b: oracle.layernorm(x, g, b, t, d, 1e-6).reshape(t, d)[1:].reshape(-1), math,
          ["> map 1", "fused into 0"])
