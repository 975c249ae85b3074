"""The workloads this framework's speed is measured on: encoder blocks, the
encoder with its embeddings and taps, the DPT decoder, the whole depth model
and a block run as frame-budget slices, each through the public entry points
(`ir.Graph` -> `ir.prepare` -> `Prepared.run`, `Kernels.encode` with a
`hip.Timer`).

A case is a dict of plain values:

  kind     "block"    `blocks` chained pre-LN encoder blocks of `tokens` tokens,
                      run once per job slot (`slots`)
           "encoder"  patch embedding, class token and positions, `blocks`
                      blocks, the last two tapped through the final LayerNorm
           "decoder"  the DPT decoder over four [grid][grid][384] feature maps
           "model"    the whole Depth Anything V2 Small (12 blocks, decoder)
           "slices"   `blocks` blocks, every kernel split into `parts`, each
                      slice encoded alone with the slice timer, as a frame loop
                      does
  width    384, 768 or 1024 (ViT-S, ViT-B, ViT-L; heads of 64, MLP 4 x width)
  dtype    "f32" or "f16" storage; `math` "split" (bf16x3, the default) or
           "mfma" (the f32 matrix cores) for f32
"""

import math

import numpy as np
import torch

from beatlm_amd import hip, ir

EPS = 1e-6
PATCH = 14
WIDTHS = {"s": 384, "b": 768, "l": 1024}
_context = None


def listed():
    return [
        # One ViT-S block of a 224-pixel frame: the smallest call, and the
        # repository's first benchmark configuration.
        {"name": "block_s_257_f32", "kind": "block", "width": 384, "tokens": 257, "blocks": 1, "slots": 1, "dtype": "f32", "math": "split"},
        # Two blocks of the headline encoder (518 pixels): LayerNorms folded
        # across the boundary as in the 12-block model.
        {"name": "blocks_s_1370_f32", "kind": "block", "width": 384, "tokens": 1370, "blocks": 2, "slots": 1, "dtype": "f32", "math": "split"},
        # The same at 350 pixels on the f32 matrix cores, the option a user
        # takes who wants plain f32 products.
        {"name": "blocks_s_626_f32_mfma", "kind": "block", "width": 384, "tokens": 626, "blocks": 2, "slots": 1, "dtype": "f32", "math": "mfma"},
        # ViT-B at 518 pixels in f16 storage.
        {"name": "blocks_b_1370_f16", "kind": "block", "width": 768, "tokens": 1370, "blocks": 2, "slots": 1, "dtype": "f16", "math": "split"},
        # ViT-L at 518 pixels, four frames in four job slots.
        {"name": "block_l_1370x4_f16", "kind": "block", "width": 1024, "tokens": 1370, "blocks": 1, "slots": 4, "dtype": "f16", "math": "split"},
        # ViT-S at 1036 pixels: the long sequence.
        {"name": "blocks_s_5477_f16", "kind": "block", "width": 384, "tokens": 5477, "blocks": 2, "slots": 1, "dtype": "f16", "math": "split"},
        # Image to feature maps at 266 pixels: patch embedding, class token,
        # positions, taps.
        {"name": "encoder_s_266_f32", "kind": "encoder", "width": 384, "grid": 19, "blocks": 2, "dtype": "f32", "math": "split"},
        # The decoder alone, at a small image in f16 and at 518 pixels in f32.
        {"name": "decoder_266_f16", "kind": "decoder", "grid": 19, "dtype": "f16", "math": "split"},
        {"name": "decoder_518_f32", "kind": "decoder", "grid": 37, "dtype": "f32", "math": "split"},
        # The whole depth model on its smallest and its native image side.
        {"name": "model_182_f32", "kind": "model", "grid": 13, "dtype": "f32", "math": "split"},
        {"name": "model_518_f32", "kind": "model", "grid": 37, "dtype": "f32", "math": "split"},
        # A block as frame-budget slices: kernels split in two, each slice
        # encoded and timed alone.
        {"name": "slices_s_1370_f32", "kind": "slices", "width": 384, "tokens": 1370, "blocks": 1, "parts": 2, "dtype": "f32", "math": "split"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["block", "encoder", "decoder", "model", "slices"], [5, 1, 2, 2, 1])[0]
    dtype = rng.choice(["f32", "f16"])
    math_ = "mfma" if dtype == "f32" and rng.random() < 0.2 else "split"
    if kind in ("block", "slices"):
        # The f32 matrix cores run a product several times longer: ViT-S alone.
        width = WIDTHS[rng.choice(["s", "s", "b", "l"]) if math_ == "split" else "s"]
        # Any token count (register tokens, other patch sizes), up to 1036
        # pixels for ViT-S and 700 for the wider ones.
        tokens = _log_int(rng, 65, 5477 if width == 384 and dtype == "f16" else 2501 if width == 384 else 1370)
        if kind == "slices":
            return {"kind": kind, "width": width, "tokens": tokens, "blocks": 1, "parts": rng.randint(1, 4), "dtype": dtype, "math": math_}
        slots = rng.choice([1, 1, 2, 4]) if tokens <= 1370 else 1
        return {"kind": kind, "width": width, "tokens": tokens, "blocks": rng.choice([1, 2]) if slots == 1 else 1, "slots": slots,
                "dtype": dtype, "math": math_}
    grid = _log_int(rng, 7, 37)
    if kind == "encoder":
        return {"kind": kind, "width": WIDTHS[rng.choice(["s", "b", "l"])], "grid": grid, "blocks": 2, "dtype": dtype, "math": math_}
    return {"kind": kind, "grid": min(grid, 25) if math_ == "mfma" else grid, "dtype": dtype, "math": math_}


# ---- graphs ----


class _Built:
    """A case's graph: its tensors by name, inputs, and outputs."""

    def __init__(self):
        self.graph = ir.Graph()
        self.inputs = {}  # name -> (tensor id, elements)
        self.weights = {}  # name -> (tensor id, elements)
        self.outputs = []  # (tensor id, shape)


def _block_names(b, ids, d):
    sizes = {"norm1_g": d, "norm1_b": d, "qkv_w": 3 * d * d, "qkv_b": 3 * d, "proj_w": d * d, "proj_b": d, "ls1": d,
             "norm2_g": d, "norm2_b": d, "fc1_w": 4 * d * d, "fc1_b": 4 * d, "fc2_w": 4 * d * d, "fc2_b": d, "ls2": d}
    return {f"block{b}.{n}": (getattr(ids, n), sizes[n]) for n in ir.BLOCK_WEIGHTS}


def _encoder(u, grid, width, layers, taps, role):
    enc = ir.vit_encoder(u.graph, grid, PATCH, 3, width, width // 64, 4 * width, EPS, taps, 0, role)
    e, tokens = enc.embed, grid * grid + 1
    u.inputs["image"] = (e.image, (grid * PATCH) ** 2 * 3)
    u.weights.update({"patch_w": (e.patch_w, PATCH * PATCH * 3 * width), "patch_b": (e.patch_b, width),
                      "cls": (e.cls, width), "pos": (e.pos, tokens * width),
                      "final_g": (enc.final_g, width), "final_b": (enc.final_b, width)})
    for b in range(layers):
        u.weights.update(_block_names(b, enc.blocks[b], width))
    return enc


def _build(case):
    u = _Built()
    kind = case["kind"]
    cfg = ir.DepthConfig.small()
    if kind in ("block", "slices"):
        t, d = case["tokens"], case["width"]
        u.graph.tensor(0, ir.INPUT, t * d)
        u.inputs["x"] = (0, t * d)
        x, nid = 0, 100
        for b in range(case["blocks"]):
            last = b + 1 == case["blocks"]
            ids = u.graph.vit_block(ir.VitDims(t, d, d // 64, 4 * d, EPS), x, nid, ir.OUTPUT if last else ir.ACTIVATION)
            u.weights.update(_block_names(b, ids, d))
            x, nid = ids.output, ids.next_id
        u.outputs = [(x, (t, d))]
    elif kind == "encoder":
        grid, d, n = case["grid"], case["width"], case["blocks"]
        enc = _encoder(u, grid, d, n, tuple(range(max(1, n - 1), n + 1)), ir.OUTPUT)
        u.outputs = [(f, (grid, grid, d)) for f in enc.features]
    elif kind == "decoder":
        grid = case["grid"]
        n = grid * grid * cfg.hidden_size
        for i in range(4):
            u.graph.tensor(i, ir.INPUT, n)
            u.inputs[f"feature{i}"] = (i, n)
        depth, weights, _ = ir.depth_decoder(u.graph, cfg, grid * PATCH, [0, 1, 2, 3], 10)
        u.weights.update({name: (tid, size) for tid, name, size in weights})
        u.outputs = [(depth, (grid * PATCH, grid * PATCH))]
    else:
        grid = case["grid"]
        enc = _encoder(u, grid, cfg.hidden_size, cfg.num_layers, cfg.out_indices, ir.ACTIVATION)
        depth, weights, _ = ir.depth_decoder(u.graph, cfg, grid * PATCH, enc.features, enc.next_id)
        u.weights.update({name: (tid, size) for tid, name, size in weights})
        u.outputs = [(depth, (grid * PATCH, grid * PATCH))]
    return u


# ---- values ----


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _values(case, u, seed):
    """Every input and weight, drawn as the benchmark draws them: images U[0, 1]
    normalised with the checkpoint's mean and deviation, Xavier weights, LN
    gamma 1 + 0.1 N, beta 0.1 N, biases U(-0.1, 0.1), LayerScale U(0.1, 1),
    decoder weights U(+-sqrt(6/fan-in)); in the storage type."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    cfg = ir.DepthConfig.small()
    dtype = torch.float16 if case["dtype"] == "f16" else torch.float32

    def uniform(n, lo, hi):
        return torch.rand(n, generator=gen, device=dev, dtype=torch.float32) * (hi - lo) + lo

    def normal(n, mean=0.0, sd=1.0):
        return torch.randn(n, generator=gen, device=dev, dtype=torch.float32) * sd + mean

    d = case.get("width", cfg.hidden_size)
    fans = {"qkv_w": (d, 3 * d), "proj_w": (d, d), "fc1_w": (d, 4 * d), "fc2_w": (4 * d, d), "patch_w": (3 * PATCH * PATCH, d)}
    vals = {}
    slots = case.get("slots", 1)
    for name, (_, n) in u.inputs.items():
        for slot in range(slots):
            if name == "image":
                mean = torch.tensor([0.485, 0.456, 0.406], device=dev)
                sd = torch.tensor([0.229, 0.224, 0.225], device=dev)
                v = ((uniform(n, 0.0, 1.0).view(-1, 3) - mean) / sd).reshape(-1)
            else:
                v = normal(n)
            vals[name, slot] = v.to(dtype)
    for name, (_, n) in u.weights.items():
        last = name.split(".")[-1]
        if last in fans:
            a = math.sqrt(6.0 / sum(fans[last]))
            v = uniform(n, -a, a)
        elif last in ("norm1_g", "norm2_g", "final_g"):
            v = normal(n, 1.0, 0.1)
        elif last in ("norm1_b", "norm2_b", "final_b"):
            v = normal(n, 0.0, 0.1)
        elif last in ("ls1", "ls2"):
            v = uniform(n, 0.1, 1.0)
        elif last == "cls":
            v = normal(n)
        elif last == "pos":
            v = normal(n, 0.0, 0.02)
        elif last == "weight":
            a = math.sqrt(6.0 / cfg.fan_in(name))  # keeps the spread through a convolution and its ReLU
            # The head's last product mostly adds: depths mostly above its ReLU's zero.
            v = uniform(n, -0.5 * a if name.startswith("head.conv3") else -a, a)
        else:  # biases
            v = uniform(n, -0.1, 0.1)
        vals[name] = v.to(dtype)
    return vals


# ---- running ----


def _ctx():
    global _context
    if _context is None:
        _context = hip.Context(0)
    return _context


class _DeviceArray:
    """Device bytes of a prepared program as torch sees them; it holds the
    program, so that the memory outlives a tensor over it."""

    def __init__(self, prep, ptr, shape, f16):
        self.prep = prep
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f2" if f16 else "<f4", "data": (ptr, False), "version": 2}


def _view(prep, tid, shape, slot=0):
    p = prep.plan.placement(prep.slot_tensor(tid, slot))
    ptr = prep.arenas.device_ptr(p.arena, p.offset)
    return torch.as_tensor(_DeviceArray(prep, ptr, shape, prep.dtype == hip.F16), device="cuda"), p


class _State:
    pass


def prepare(case, seed):
    """The program built once, its weights and inputs in device memory."""
    ctx = _ctx()
    u = _build(case)
    dtype = hip.F16 if case["dtype"] == "f16" else hip.F32
    ctx.set_f32_math(hip.F32_MATH_MFMA_F32 if case["math"] == "mfma" else hip.F32_MATH_SPLIT_BF16)
    slots = case.get("slots", 1)
    prep = ir.prepare(ctx, u.graph, parts=case.get("parts", 1), dtype=dtype, slots=slots)
    ctx.set_f32_math(hip.F32_MATH_SPLIT_BF16)
    for key, v in _values(case, u, seed).items():
        name, slot = key if isinstance(key, tuple) else (key, 0)
        tid, n = u.inputs.get(name) or u.weights[name]
        view, p = _view(prep, tid, (n,), slot)
        view.copy_(v)
        prep.arenas.invalidate(p.arena, p.offset, n * view.element_size())
    torch.cuda.synchronize()
    s = _State()
    s.prep, s.slots = prep, slots
    s.outputs = [_view(prep, tid, shape, slot)[0] for slot in range(slots) for tid, shape in u.outputs]
    s.timer = None
    if case["kind"] == "slices":
        s.timer = hip.Timer(ctx, len(prep.kernels))
        s.frame = 0
    return s


def run(state):
    """One frame: every kernel of the program, for every job slot; or, for
    slices, every slice encoded alone between the timer's events."""
    prep = state.prep
    if state.timer is None:
        for slot in range(state.slots):
            prep.run(slot)
        return state.outputs
    timer = state.timer
    state.frame += 1
    timer.begin_frame(state.frame)
    for k in range(len(prep.kernels)):
        prep.kernels.encode(k, 0, timer, k)
    timer.submitted(timer.resolve())
    timer.collect()
    return state.outputs


# ---- work and tolerance ----


def _conv_shapes(grid):
    """(output pixels, k, cout, input elements) of every decoder product."""
    cfg = ir.DepthConfig.small()
    f = cfg.fusion_hidden_size
    out, sizes = [], []
    for ch, kind in zip(cfg.neck_hidden_sizes, cfg.reassemble):
        out.append((grid * grid, cfg.hidden_size, ch))
        if kind[0] == "up":
            side = grid * kind[1]
            out.append((side * side, ch, ch))
        elif kind[0] == "down":
            side = (grid - 1) // kind[1] + 1
            out.append((side * side, 9 * ch, ch))
        else:
            side = grid
        out.append((side * side, 9 * ch, f))
        sizes.append(side)
    sizes = sizes[::-1]
    for i, side in enumerate(sizes):
        to = sizes[i + 1] if i + 1 < len(sizes) else 2 * side
        out += [(side * side, 9 * f, f)] * (4 if i else 2)
        out.append((to * to, f, f))
    full = grid * PATCH
    side = 2 * sizes[-1]
    out += [(side * side, 9 * f, f // 2), (full * full, 9 * (f // 2), cfg.head_hidden_size), (full * full, cfg.head_hidden_size, 1)]
    return out


def work(case):
    """Products (2 per multiply-add), and each input, weight and output once."""
    u = _build(case)
    elt = 2 if case["dtype"] == "f16" else 4
    slots = case.get("slots", 1)
    n = slots * (sum(x[1] for x in u.inputs.values()) + sum(math.prod(s) for _, s in u.outputs)) + sum(x[1] for x in u.weights.values())
    flops = 0
    if case["kind"] != "decoder":
        d = case.get("width", 384)
        t = case.get("tokens") or case["grid"] ** 2 + 1
        blocks = case.get("blocks", 12)
        flops += slots * blocks * (24 * t * d * d + 4 * t * t * d)
        if "grid" in case:
            flops += 2 * (t - 1) * 3 * PATCH * PATCH * d
    if case["kind"] in ("decoder", "model"):
        flops += sum(2 * px * k * co for px, k, co in _conv_shapes(case["grid"]))
    return {"bytes": n * elt, "flops": flops}


def tolerance(case):
    """About four times what each kind was measured to be off the 64-bit result
    (exact): blocks 2.5e-6 in f32 (products of operands split into two bf16
    parts; 2.3e-7 on the f32 matrix cores) and 4.3e-4 in f16 storage, which
    rounds every activation; taps through the final LayerNorm 5.0e-6 and
    5.2e-4; the decoder up to 1.3e-5 and 7.4e-4, and the model about as much."""
    f32, f16 = {"block": (1e-5, 2e-3), "slices": (1e-5, 2e-3), "encoder": (2e-5, 2e-3), "decoder": (4e-5, 3e-3),
                "model": (4e-5, 4e-3)}[case["kind"]]
    return {"rel": f16 if case["dtype"] == "f16" else f32}


# ---- the same in 64 bits ----


def _ln(x, g, b):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + EPS) * g + b


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _blocks64(x, w, d, blocks, taps=()):
    t, h = x.shape[0], d // 64
    taken = []
    for b in range(blocks):
        p = {n: w[f"block{b}.{n}"] for n in ir.BLOCK_WEIGHTS}
        y = _ln(x, p["norm1_g"], p["norm1_b"])
        qkv = (y @ p["qkv_w"].view(d, 3 * d) + p["qkv_b"]).view(t, 3, h, 64)
        o = torch.empty(t, h, 64, dtype=x.dtype, device=x.device)
        for head in range(h):
            q, k, v = (qkv[:, i, head].contiguous() for i in range(3))
            o[:, head] = torch.softmax(q @ k.t().contiguous() * 0.125, -1) @ v
        x = x + (o.view(t, d) @ p["proj_w"].view(d, d) + p["proj_b"]) * p["ls1"]
        y = _ln(x, p["norm2_g"], p["norm2_b"])
        y = _gelu(y @ p["fc1_w"].view(d, 4 * d) + p["fc1_b"])
        x = x + (y @ p["fc2_w"].view(4 * d, d) + p["fc2_b"]) * p["ls2"]
        if b + 1 in taps:
            taken.append(x)
    return x, taken


def _encoder64(case, w, grid, d, blocks, taps):
    side = grid * PATCH
    img = w["image", 0].view(grid, PATCH, grid, PATCH, 3).permute(0, 2, 1, 3, 4).reshape(grid * grid, -1)
    x = img @ w["patch_w"].view(-1, d) + w["patch_b"]
    assert side * side * 3 == w["image", 0].numel()
    x = torch.cat([w["cls"].view(1, d), x]) + w["pos"].view(-1, d)
    _, taken = _blocks64(x, w, d, blocks, taps)
    return [_ln(x, w["final_g"], w["final_b"])[1:].view(grid, grid, d) for x in taken]


def _conv3_64(x, w, b, cout, stride=1):
    """NHWC x, HWIO w, padding 1, as a sum over the nine taps."""
    h, wd, cin = x.shape
    oh, ow = (h - 1) // stride + 1, (wd - 1) // stride + 1
    pad = torch.zeros(h + 2, wd + 2, cin, dtype=x.dtype, device=x.device)
    pad[1:-1, 1:-1] = x
    w = w.view(3, 3, cin, cout)
    out = torch.zeros(oh * ow, cout, dtype=x.dtype, device=x.device)
    for ky in range(3):
        for kx in range(3):
            tap = pad[ky : ky + (oh - 1) * stride + 1 : stride, kx : kx + (ow - 1) * stride + 1 : stride]
            out += tap.reshape(oh * ow, cin) @ w[ky, kx]
    return (out if b is None else out + b).view(oh, ow, cout)


def _resize64(x, oh, ow):
    """Bilinear, corners aligned."""

    def axis(n, to):
        pos = torch.arange(to, dtype=torch.float64, device=x.device) * ((n - 1) / (to - 1) if to > 1 else 0.0)
        lo = pos.floor().clamp(max=n - 1)
        i = lo.long()
        return i, (i + 1).clamp(max=n - 1), pos - lo

    y0, y1, ly = axis(x.shape[0], oh)
    x0, x1, lx = axis(x.shape[1], ow)
    rows = x[y0] * (1 - ly).view(-1, 1, 1) + x[y1] * ly.view(-1, 1, 1)
    return rows[:, x0] * (1 - lx).view(1, -1, 1) + rows[:, x1] * lx.view(1, -1, 1)


def _decoder64(features, w, grid):
    cfg = ir.DepthConfig.small()
    fw = cfg.fusion_hidden_size

    def conv(x, name, cout, stride=1, bias=True):
        return _conv3_64(x, w[name + ".weight"], w[name + ".bias"] if bias else None, cout, stride)

    def one(x, name, cout):
        return x @ w[name + ".weight"].view(x.shape[-1], cout) + w[name + ".bias"]

    def unit(x, name):
        y = conv(torch.relu(x), name + ".convolution1", fw)
        return conv(torch.relu(y), name + ".convolution2", fw) + x

    stages = []
    for i, x in enumerate(features):
        ch, kind = cfg.neck_hidden_sizes[i], cfg.reassemble[i]
        pre = f"neck.reassemble_stage.layers.{i}"
        m = one(x, pre + ".projection", ch)
        if kind[0] == "up":
            f = kind[1]
            taps = w[pre + ".resize.weight"].view(f, f, ch, ch)
            up = torch.empty(grid, f, grid, f, ch, dtype=m.dtype, device=m.device)
            for ky in range(f):
                for kx in range(f):
                    up[:, ky, :, kx] = m @ taps[ky, kx]
            m = up.view(grid * f, grid * f, ch) + w[pre + ".resize.bias"]
        elif kind[0] == "down":
            m = conv(m, pre + ".resize", ch, kind[1])
        stages.append(conv(m, f"neck.convs.{i}", fw, 1, False))
    fused = None
    for layer in range(len(stages)):
        x = stages[len(stages) - 1 - layer]
        name = f"neck.fusion_stage.layers.{layer}"
        if fused is not None:
            x = unit(x, name + ".residual_layer1") + fused
        x = unit(x, name + ".residual_layer2")
        nxt = len(stages) - 2 - layer
        to = stages[nxt].shape[:2] if nxt >= 0 else (2 * x.shape[0], 2 * x.shape[1])
        fused = one(_resize64(x, *to), name + ".projection", fw)
    full = grid * PATCH
    x = _resize64(conv(fused, "head.conv1", fw // 2), full, full)
    x = torch.relu(conv(x, "head.conv2", cfg.head_hidden_size))
    return torch.relu(one(x, "head.conv3", 1)).view(full, full)


def exact(case, seed):
    u = _build(case)
    w = {k: v.to(torch.float64) for k, v in _values(case, u, seed).items()}
    kind = case["kind"]
    if kind in ("block", "slices"):
        d = case["width"]
        outs = [_blocks64(w["x", slot].view(-1, d), w, d, case["blocks"])[0] for slot in range(case.get("slots", 1))]
    elif kind == "encoder":
        n = case["blocks"]
        outs = _encoder64(case, w, case["grid"], case["width"], n, tuple(range(max(1, n - 1), n + 1)))
    elif kind == "decoder":
        grid = case["grid"]
        outs = [_decoder64([w[f"feature{i}", 0].view(grid, grid, -1) for i in range(4)], w, grid)]
    else:
        cfg = ir.DepthConfig.small()
        feats = _encoder64(case, w, case["grid"], cfg.hidden_size, cfg.num_layers, cfg.out_indices)
        outs = [_decoder64(feats, w, case["grid"])]
    return [np.asarray(o.cpu()) for o in outs]
