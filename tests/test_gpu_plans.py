"""Plans of several kernels composed: launches that take two kernels' place
next to other plans that read or write the same tensors, programs of several
binding sets whose kernels interleave, parts that do not cover their tensor,
and outputs the memory plan lays over what an earlier kernel still reads.

Tolerance for f32 storage: |got - want| <= 1e-4 + 1e-4 |want|
(reference.rs:22-24); for f16 storage, max abs error <= 2e-2 against the
oracle on the same f16-rounded inputs.
"""

import numpy as np
import pytest

import oracle
from beatlm_amd import hip, ir
from tests.blockdata import max_abs_err

pytestmark = pytest.mark.gpu

EPS = 1e-6
F16_TOL = 2e-2
MATHS = ["bf16x3", "f32", "f16"]
STAND_IN = 1 << 18


@pytest.fixture
def math(ctx, request):
    if request.param == "f32":
        ctx.set_f32_math(hip.F32_MATH_MFMA_F32)
    yield request.param
    ctx.set_f32_math(hip.F32_MATH_SPLIT_BF16)


def compare(got, want, math, what):
    if math == "f16":
        err = max_abs_err(got, want)
        assert err <= F16_TOL, f"{what}: max abs error {err:.3e}"
    else:
        bad = oracle.first_mismatch(got, want)
        assert bad is None, f"{what}: element {bad[0]} is {bad[1]}, the oracle says {bad[2]}"


class Net:
    """A graph from (operation, output role) pairs: tensor i of `inputs`
    ((role, elements) each) is i, operation i writes 100 + i. Planned and
    prepared through the C ABI; `change(specs)` may edit the specs, and every
    tensor that is no weight gets stand-ins of its own in each set past the first."""

    def __init__(self, ctx, inputs, ops, math, sets=1, change=None):
        g = ir.Graph()
        for i, (role, n) in enumerate(inputs):
            g.tensor(i, role, n)
        for i, (o, role) in enumerate(ops):
            g.tensor(100 + i, role, ir.output_elements(o))
            g.push(o, 100 + i)
        self.program = g.lower().fuse_attention()
        self.f16 = math == "f16"
        self.program.set_dtype(hip.F16 if self.f16 else hip.F32)
        tensors = self.program.tensors()
        descs, own, last = list(tensors), [{t.id: t.id for t in tensors}], len(self.program) - 1
        for s in range(1, sets):
            own.append({})
            for t in tensors:
                if self.program.role(t.id) != ir.WEIGHT:
                    own[s][t.id] = s * STAND_IN + t.id
                    descs.append(ir.tensor_desc(own[s][t.id], t.dtype, t.elements, 0, last))
        self.plan = ir.Plan(descs, ir.profile("mi355x"))
        self.own, self.elements = own, {t.id: t.elements for t in tensors}
        self.arenas = hip.Arenas(ctx, self.plan.arenas())
        specs = self.program.specs(self.plan)
        if change:
            change(specs)
        subs = None
        if sets > 1:
            subs = []
            for mine in own:
                at = {t: self.plan.placement(s) for t, s in mine.items() if t != s}
                subs.append([hip.Substitution(t, mine[t], p.arena, 0, p.offset, p.size) for t, p in at.items()])
        internal = [t.id for t in tensors if self.program.role(t.id) == ir.ACTIVATION]
        self.kernels = hip.Kernels(ctx, self.arenas, specs, sets=subs, internal=internal)
        self.labels = [self.kernels.label(k) for k in range(len(self.kernels))]
        self.ctx = ctx

    def __enter__(self):
        return self

    def __exit__(self, *_):
        self.kernels.close()
        self.arenas.close()

    def at(self, tid, s=0):
        return self.plan.placement(self.own[s].get(tid, tid))

    def write(self, tid, v, s=0):
        p = self.at(tid, s)
        self.arenas.write(p.arena, p.offset, np.ascontiguousarray(v, np.float16 if self.f16 else np.float32))

    def read(self, tid, s=0):
        p = self.at(tid, s)
        return self.arenas.read(p.arena, p.offset, self.elements[tid], np.float16 if self.f16 else np.float32).astype(np.float32)

    def overlap(self, a, b):
        """Whether the plan lays tensors a and b over each other in set 0."""
        p, q = self.at(a), self.at(b)
        return p.arena == q.arena and p.offset < q.offset + q.size and q.offset < p.offset + p.size


def stored(math, a):
    """The values as stored, as the oracle reads them."""
    return a.astype(np.float16).astype(np.float32) if math == "f16" else a


@pytest.mark.parametrize("h,w,oh,ow,heads", [(4, 4, 8, 8, 1), (3, 5, 9, 7, 2)])
@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_attention_over_a_projection_of_a_resampling(ctx, h, w, oh, ow, heads, math):
    """resize -> QKV projection -> attention: the attention's keys and values
    are the projection's, whoever writes them."""
    t, n = oh * ow, 3 * heads * 64
    wq, bq = (stored(math, a) for a in (oracle.fan_in_weights(41, 64 * n, 64), oracle.uniform(42, n, -0.1, 0.1)))
    ops = [(ir.op(ir.OP_RESIZE_BILINEAR, [0], [h, w, oh, ow, 64]), ir.ACTIVATION), (ir.op(ir.OP_MATMUL, [100, 1, 2], [t, 64, n]), ir.ACTIVATION),
           (ir.op(ir.OP_ATTENTION_SCORES, [101], [t, heads, 64]), ir.ACTIVATION),
           (ir.op(ir.OP_SCALE, [102], [t * heads * t], 0.125), ir.ACTIVATION), (ir.op(ir.OP_SOFTMAX, [103], [t * heads, t]), ir.ACTIVATION),
           (ir.op(ir.OP_ATTENTION_VALUES, [104, 101], [t, heads, 64]), ir.OUTPUT)]
    with Net(ctx, [(ir.INPUT, h * w * 64), (ir.WEIGHT, 64 * n), (ir.WEIGHT, n)], ops, math) as net:
        assert "flash_attention" in net.labels[-1], net.labels
        net.write(1, wq)
        net.write(2, bq)
        for seed in (43, 44):
            x = stored(math, oracle.uniform(seed, h * w * 64, -2.0, 2.0))
            net.write(0, x)
            net.kernels.encode_all()
            ctx.synchronize()
            qkv = oracle.matmul(oracle.resize_bilinear(x, h, w, oh, ow, 64), wq, bq, t, 64, n)
            compare(net.read(105), oracle.attention(qkv, t, heads, 64, 0.125), math, f"{net.labels}, input {seed}")


def fused_stage(ctx, math, sets):
    """conv 256 -> 64, conv 64 -> 64 = x, resampled, 1x1 = y, relu: x moves to
    the workspace, since the plan lays y over it."""
    h, w, oh, ow = 8, 8, 16, 16
    arrays = [stored(math, a) for a in (oracle.fan_in_weights(51, 9 * 256 * 64, 9 * 256), oracle.fan_in_weights(52, 9 * 64 * 64, 9 * 64),
                                        oracle.fan_in_weights(53, 64 * 64, 64), oracle.uniform(54, 64, -0.1, 0.1))]
    ops = [(ir.op(ir.OP_CONV3X3, [0, 1, ir.NONE], [h, w, 256, 64, 1]), ir.ACTIVATION),
           (ir.op(ir.OP_CONV3X3, [100, 2, ir.NONE], [h, w, 64, 64, 1]), ir.ACTIVATION),
           (ir.op(ir.OP_RESIZE_BILINEAR, [101], [h, w, oh, ow, 64]), ir.ACTIVATION),
           (ir.op(ir.OP_MATMUL, [102, 3, 4], [oh * ow, 64, 64]), ir.ACTIVATION),
           (ir.op(ir.OP_RESIZE_BILINEAR, [103], [oh, ow, 5, 7, 64]), ir.OUTPUT)]
    net = Net(ctx, [(ir.INPUT, h * w * 256)] + [(ir.WEIGHT, a.size) for a in arrays], ops, math, sets)
    assert net.overlap(101, 103) and "> workspace" in net.labels[1] and "< resize 2" in net.labels[3], net.labels
    for i, a in enumerate(arrays):
        net.write(1 + i, a)

    def want(x):
        y = oracle.conv3x3(x, arrays[0], None, h, w, 256, 64, 1)
        y = oracle.resize_bilinear(oracle.conv3x3(y, arrays[1], None, h, w, 64, 64, 1), h, w, oh, ow, 64)
        return oracle.resize_bilinear(oracle.matmul(y, arrays[2], arrays[3], oh * ow, 64, 64), oh, ow, 5, 7, 64)

    return net, want, [stored(math, oracle.uniform(55 + s, h * w * 256, -2.0, 2.0)) for s in range(3)]


@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_a_moved_tensor_follows_each_new_input(ctx, math):
    net, want, xs = fused_stage(ctx, math, 1)
    with net:
        for x in xs:
            net.write(0, x)
            net.kernels.encode_all()
            ctx.synchronize()
            compare(net.read(104), want(x), math, f"{net.labels}")


@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_a_moved_tensor_outlives_another_sets_kernels(ctx, math):
    """Every kernel of set 1 between the moved tensor's writer and its reader
    of set 0 (on the f32 matrix cores the first convolution splits k: its
    partial sums lie in the workspace too)."""
    net, want, xs = fused_stage(ctx, math, 2)
    with net:
        assert math != "f32" or "splitk" in net.labels[0], net.labels
        for s in (0, 1):
            net.write(0, xs[s], s)
        for k in (0, 1):
            net.kernels.encode(k, 0)
        for k in range(5):
            net.kernels.encode(k, 1)
        for k in (2, 3, 4):
            net.kernels.encode(k, 0)
        ctx.synchronize()
        for s in (0, 1):
            compare(net.read(104, s), want(xs[s]), math, f"set {s}, {net.labels}")


@pytest.mark.parametrize("operand", ["bias", "channel scale"])
@pytest.mark.parametrize("math", ["bf16x3", "f16"], indirect=True)
def test_a_one_column_product_over_what_its_convolution_reads(ctx, operand, math):
    """The plan lays the product's output over the convolution's bias (its
    channel scale): the convolution's workgroups all read those, so the
    product keeps a launch of its own."""
    h, w = 130, 255
    wc, ch, w1, b1 = (stored(math, a) for a in (oracle.fan_in_weights(62, 9 * 32 * 32, 9 * 32), oracle.uniform(63, 32, 0.5, 1.5),
                                                oracle.fan_in_weights(64, 32, 32), oracle.uniform(65, 1, -0.1, 0.1)))
    x = stored(math, oracle.uniform(61, h * w * 32, -2.0, 2.0))
    ops = [(ir.op(ir.OP_RELU, [2], [32]), ir.ACTIVATION)]
    if operand == "bias":
        ops += [(ir.op(ir.OP_CONV3X3, [0, 1, 100], [h, w, 32, 32, 1]), ir.ACTIVATION)]
    else:
        ops += [(ir.op(ir.OP_CONV3X3, [0, 1, ir.NONE], [h, w, 32, 32, 1]), ir.ACTIVATION),
                (ir.op(ir.OP_CHANNEL_SCALE, [101, 100], [h * w, 32]), ir.ACTIVATION)]
    c = 100 + len(ops) - 1
    ops += [(ir.op(ir.OP_MATMUL, [c, 3, 4], [h * w, 32, 1]), ir.ACTIVATION), (ir.op(ir.OP_RESIZE_BILINEAR, [c + 1], [h, w, 20, 30, 1]), ir.OUTPUT)]
    with Net(ctx, [(ir.INPUT, x.size), (ir.WEIGHT, wc.size), (ir.WEIGHT, 32), (ir.WEIGHT, 32), (ir.WEIGHT, 1)], ops, math) as net:
        assert net.overlap(100, c + 1) and "direct" in net.labels[1], net.labels
        assert "product" not in net.labels[1], net.labels
        for i, a in enumerate((x, wc, ch, w1, b1)):
            net.write(i, a)
        net.kernels.encode_all()
        ctx.synchronize()
        y = oracle.conv3x3(x, wc, ch if operand == "bias" else None, h, w, 32, 32, 1)
        if operand != "bias":
            y = oracle.channel_scale(y, ch)
        want = oracle.resize_bilinear(oracle.matmul(y, w1, b1, h * w, 32, 1), h, w, 20, 30, 1)
        compare(net.read(c + 2), want, math, f"{net.labels}")


def part(specs, k, start, end):
    specs[k].part = hip.Part(0, 1, start, end)


@pytest.mark.parametrize("which", ["map", "layernorm", "resampled product", "resampling", "one column", "transposed"])
@pytest.mark.parametrize("math", ["bf16x3", "f16"], indirect=True)
def test_a_lone_part_that_does_not_cover_its_tensor_writes_its_own_range(ctx, which, math):
    """Part 1 of 1 may cover less than its tensor: the rest of the output stays
    as the host left it (outputs here start at 7)."""
    u = lambda seed, n: stored(math, oracle.uniform(seed, n, -1.0, 1.0))
    if which in ("map", "layernorm"):
        t, d = 26, 64
        arrays = [u(71, t * d), u(72, d), u(73, d)]
        ops = [(ir.op(ir.OP_LAYER_NORM, [0, 1, 2], [t, d], EPS), ir.ACTIVATION), (ir.op(ir.OP_TOKENS_TO_MAP, [100], [5, 5, d]), ir.OUTPUT)]
        full = oracle.layernorm(*arrays, t, d, EPS).reshape(t, d)[1:].reshape(-1)
        if which == "map":
            change, lo, hi = (lambda s: part(s, 1, 3 * d, 17 * d)), 3 * d, 17 * d
        else:
            # Rows 1 .. 9 alone are the LayerNorm's: map rows 0 .. 8 are checked.
            change, lo, hi = (lambda s: part(s, 0, 0, 10)), 0, 9 * d
    elif which in ("resampled product", "resampling"):
        arrays = [u(74, 64 * 64), u(75, 64 * 64), u(76, 64)]
        ops = [(ir.op(ir.OP_RESIZE_BILINEAR, [0], [8, 8, 16, 16, 64]), ir.ACTIVATION), (ir.op(ir.OP_MATMUL, [100, 1, 2], [256, 64, 64]), ir.OUTPUT)]
        full = oracle.matmul(oracle.resize_bilinear(arrays[0], 8, 8, 16, 16, 64), arrays[1], arrays[2], 256, 64, 64)
        if which == "resampled product":
            change, lo, hi = (lambda s: part(s, 1, 64, 128)), 64 * 64, 128 * 64
        else:
            change, lo, hi = (lambda s: part(s, 0, 0, 100)), 0, 100 * 64
    elif which == "one column":
        h, w = 130, 255
        arrays = [u(77, h * w * 32), stored(math, oracle.fan_in_weights(78, 9 * 32 * 32, 9 * 32)), u(79, 32), u(80, 1)]
        ops = [(ir.op(ir.OP_CONV3X3, [0, 1, ir.NONE], [h, w, 32, 32, 1]), ir.ACTIVATION), (ir.op(ir.OP_MATMUL, [100, 2, 3], [h * w, 32, 1]), ir.OUTPUT)]
        full = oracle.matmul(oracle.conv3x3(arrays[0], arrays[1], None, h, w, 32, 32, 1), arrays[2], arrays[3], h * w, 32, 1)
        change, lo, hi = (lambda s: part(s, 0, 0, 33088)), 0, 33088
    else:
        arrays = [u(81, 9 * 9 * 48), u(82, 4 * 48 * 48), u(83, 48)]
        ops = [(ir.op(ir.OP_CONV_TRANSPOSE, [0, 1, 2], [9, 9, 48, 48, 2]), ir.OUTPUT)]
        full = oracle.conv_transpose(arrays[0], arrays[1], arrays[2], 9, 9, 48, 48, 2)
        change, lo, hi = (lambda s: part(s, 0, 50, 201)), 50 * 48, 201 * 48
    whole = which in ("layernorm", "resampling", "one column")  # the last kernel writes all: the rest of its input is arbitrary
    out = 100 + len(ops) - 1
    with Net(ctx, [(ir.INPUT, arrays[0].size)] + [(ir.WEIGHT, a.size) for a in arrays[1:]], ops, math, change=change) as net:
        for i, a in enumerate(arrays):
            net.write(i, a)
        net.write(out, np.full(full.size, 7.0))
        net.kernels.encode_all()
        ctx.synchronize()
        got = net.read(out)
        compare(got[lo:hi], full[lo:hi], math, f"{net.labels}")
        assert whole or (np.all(got[:lo] == 7.0) and np.all(got[hi:] == 7.0)), net.labels
        assert not any("fused" in lab for lab in net.labels), net.labels


@pytest.mark.parametrize("product", ["transposed convolution", "matmul"])
@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_weights_that_a_kernel_writes_are_packed_again_in_every_set(ctx, product, math):
    """The weights are a kernel's output, at a place of its own in each set."""
    if product == "matmul":
        x, n = stored(math, oracle.uniform(91, 40 * 64, -1.0, 1.0)), 64 * 64
        o = ir.op(ir.OP_MATMUL, [0, 100, ir.NONE], [40, 64, 64])
        want = lambda w: oracle.matmul(x, w, None, 40, 64, 64)
    else:
        x, n = stored(math, oracle.uniform(92, 9 * 9 * 48, -1.0, 1.0)), 4 * 48 * 48
        o = ir.op(ir.OP_CONV_TRANSPOSE, [0, 100, ir.NONE], [9, 9, 48, 48, 2])
        want = lambda w: oracle.conv_transpose(x, w, None, 9, 9, 48, 48, 2)
    with Net(ctx, [(ir.INPUT, x.size), (ir.INPUT, n)], [(ir.op(ir.OP_RELU, [1], [n]), ir.ACTIVATION), (o, ir.OUTPUT)], math, 2) as net:
        for seed in (93, 94):
            for s in (0, 1):
                w = stored(math, oracle.uniform(seed + 10 * s, n, -0.2, 0.2))
                net.write(0, x, s)
                net.write(1, w, s)
                net.kernels.encode_all(s)
                ctx.synchronize()
                compare(net.read(101, s), want(np.maximum(w, 0)), math, f"set {s}, weights {seed}: {net.labels}")


@pytest.mark.parametrize("math", MATHS, indirect=True)
def test_tokens_over_the_image_their_patches_come_from(ctx, math):
    """The plan lays the tokens over an image whose last reader is the patch
    embedding: the class-token prepend keeps a launch of its own."""
    grid, p, c, d = 5, 14, 3, 64
    image, rows = (grid * p) ** 2 * c, grid * grid
    arrays = [stored(math, a) for a in (oracle.uniform(111, image, 0.0, 1.0), oracle.fan_in_weights(112, p * p * c * d, p * p * c),
                                        oracle.uniform(113, d, -0.1, 0.1), oracle.uniform(114, d, -1.0, 1.0))]
    ops = [(ir.op(ir.OP_RELU, [0], [image]), ir.ACTIVATION), (ir.op(ir.OP_PATCH_EMBED, [100, 1, 2], [grid, grid, p, c, d]), ir.ACTIVATION),
           (ir.op(ir.OP_PREPEND_TOKEN, [3, 101], [rows, d]), ir.ACTIVATION), (ir.op(ir.OP_TOKENS_TO_MAP, [102], [grid, grid, d]), ir.OUTPUT)]
    with Net(ctx, [(ir.INPUT, image)] + [(ir.WEIGHT, a.size) for a in arrays[1:]], ops, math) as net:
        assert net.overlap(100, 102), net.labels
        assert not any("prepend" in lab and "fused" in lab or "< prepend" in lab for lab in net.labels), net.labels
        for i, a in enumerate(arrays):
            net.write(i, a)
        net.kernels.encode_all()
        ctx.synchronize()
        compare(net.read(103), oracle.patch_embed(arrays[0], arrays[1], arrays[2], grid, grid, p, c, d), math, f"{net.labels}")


@pytest.mark.parametrize("t,m", [(40, 192), (700, 384)])
def test_a_product_over_the_input_of_its_folded_layernorm(ctx, t, m):
    """x -> LayerNorm -> product, x used no further: the plan lays the product
    over x, which an f16 product with the LayerNorm folded in would still read."""
    d = 128
    arrays = [stored("f16", a) for a in (oracle.uniform(121, t * d, -1.0, 1.0), oracle.fan_in_weights(122, d * d, d), oracle.uniform(123, d, 0.8, 1.2),
                                         oracle.uniform(124, d, -0.1, 0.1), oracle.fan_in_weights(125, d * m, d))]
    ops = [(ir.op(ir.OP_MATMUL, [0, 1, ir.NONE], [t, d, d]), ir.ACTIVATION), (ir.op(ir.OP_LAYER_NORM, [100, 2, 3], [t, d], EPS), ir.ACTIVATION),
           (ir.op(ir.OP_MATMUL, [101, 4, ir.NONE], [t, d, m]), ir.ACTIVATION), (ir.op(ir.OP_RESIZE_BILINEAR, [102], [1, t, 1, t, m]), ir.OUTPUT)]
    with Net(ctx, [(ir.INPUT, t * d)] + [(ir.WEIGHT, a.size) for a in arrays[1:]], ops, "f16") as net:
        assert net.overlap(100, 102), net.labels
        assert not any("layernorm 1" in lab for lab in net.labels), net.labels
        for i, a in enumerate(arrays):
            net.write(i, a)
        net.kernels.encode_all()
        ctx.synchronize()
        n = oracle.layernorm(oracle.matmul(arrays[0], arrays[1], None, t, d, d), arrays[2], arrays[3], t, d, EPS)
        compare(net.read(103), oracle.matmul(n, arrays[4], None, t, d, m), "f16", f"{net.labels}")


@pytest.mark.parametrize("t1,t2", [(300, 705), (257, 641), (900, 1985)])
@pytest.mark.parametrize("math", ["bf16x3", "f16"], indirect=True)
def test_attentions_of_two_sizes_share_their_scratch(ctx, monkeypatch, t1, t2, math):
    """The larger attention's keys past its last token lie where the smaller
    one's partial results would: they must stay finite, whatever ran before."""
    monkeypatch.setenv("BL_FLASH_SMALL", "0")
    heads, d = 2, 128
    arrays, ops = [], []
    for i, t in enumerate((t1, t2)):
        arrays += [stored(math, a) for a in (oracle.uniform(131 + i, t * d, -1.0, 1.0), oracle.fan_in_weights(133 + i, 3 * d * d, d),
                                             oracle.uniform(135 + i, 3 * d, -0.1, 0.1))]
        b = 100 + 5 * i
        # The first qkv is an output: the two lie at places of their own.
        ops += [(ir.op(ir.OP_MATMUL, [3 * i, 3 * i + 1, 3 * i + 2], [t, d, 3 * d]), ir.ACTIVATION if i else ir.OUTPUT),
                (ir.op(ir.OP_ATTENTION_SCORES, [b], [t, heads, 64]), ir.ACTIVATION), (ir.op(ir.OP_SCALE, [b + 1], [t * heads * t], 0.125), ir.ACTIVATION),
                (ir.op(ir.OP_SOFTMAX, [b + 2], [t * heads, t]), ir.ACTIVATION),
                (ir.op(ir.OP_ATTENTION_VALUES, [b + 3, b], [t, heads, 64]), ir.OUTPUT)]
    with Net(ctx, [(ir.WEIGHT if i % 3 else ir.INPUT, a.size) for i, a in enumerate(arrays)], ops, math) as net:
        for i, a in enumerate(arrays):
            net.write(i, a)
        for _ in range(3):
            net.kernels.encode_all()
        ctx.synchronize()
        for i, t in enumerate((t1, t2)):
            qkv = stored(math, oracle.matmul(arrays[3 * i], arrays[3 * i + 1], arrays[3 * i + 2], t, d, 3 * d))
            compare(net.read(104 + 5 * i), oracle.attention(qkv, t, heads, 64, 0.125), math, f"{t} tokens, {net.labels}")
