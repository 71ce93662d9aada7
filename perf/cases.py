"""What a program does with this framework, as measurable cases: the calls of
one layer of a quantised mixture-of-experts model, in decode and in prefill,
through the Python binding's public entry points.

The shapes are those of the benchmark and the tests: hidden 2048, 64 experts of
width 1536, the latent-attention projections (768 / 3840 / 576 / 2048 outputs),
a vocabulary of 154,880, cached positions of 576 values, and batches of up to
256 tokens (the most a MoE layer call takes).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mobile-moe.zig_amd", "python"))
import mmhip as mm  # noqa: E402

Q8, IQ2, F32, F16 = "q8_0", "iq2_xxs", "f32", "f16"
TYPE = {Q8: mm.Q8_0, IQ2: mm.IQ2_XXS, F32: mm.F32, F16: mm.F16}

_MLA = dict(hidden=2048, q_lora=768, q_out=3840, kv=576, o_in=2560)
_MOE = dict(hidden=2048, inter=1536, experts=64, shared=1536, router=F32)


def listed():
    return [
        # One decode step's four latent-attention projections of a layer, one
        # token: the smallest calls there are, four launches.
        dict(name="proj_decode_q8", kind="proj", fmt=Q8, tokens=1, **_MLA),
        # The engine's seam: one matrix times one vector, both on the host,
        # the weight resident (what a host program calls for each projection).
        dict(name="seam_gemv_iq2", kind="seam", fmt=IQ2, rows=1536, cols=2048, batch=1),
        # The products of 64 experts with one step's activations, one launch
        # (the headline of the benchmark).
        dict(name="experts_step_iq2", kind="experts", fmt=IQ2, experts=64, hidden=2048, inter=1536),
        # The output projection over the whole vocabulary and the greedy token.
        dict(name="logits_q8", kind="logits", fmt=Q8, vocab=154880, hidden=2048),
        # The MoE layer for one token (decode), in both expert formats.
        dict(name="moe_decode_iq2", kind="moe", fmt=IQ2, tokens=1, **_MOE),
        dict(name="moe_decode_q8", kind="moe", fmt=Q8, tokens=1, **_MOE),
        # The MoE layer for a prompt chunk: 64 tokens, and the largest call.
        dict(name="moe_prefill_iq2_64", kind="moe", fmt=IQ2, tokens=64, **_MOE),
        dict(name="moe_prefill_q8_256", kind="moe", fmt=Q8, tokens=256, **_MOE),
        # The same projections for a prompt: a ragged chunk, and the largest.
        dict(name="proj_prefill_iq2_77", kind="proj", fmt=IQ2, tokens=77, **_MLA),
        dict(name="proj_prefill_q8_256", kind="proj", fmt=Q8, tokens=256, **_MLA),
        # Latent vectors of 300 cached positions expanded to keys with the
        # f32 matrix k_b.
        dict(name="kv_expand_f32_300", kind="expand", fmt=F32, rows=2560, cols=512, batch=300),
        # A long context's cache rows written as Q8_0 blocks and read back.
        dict(name="kv_codec_q8", kind="codec", positions=131072, row=576),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, step, lo, hi):
    return step * rng.randint((lo + step - 1) // step, hi // step)


def draw(rng):
    kind = rng.choice(["proj", "proj", "moe", "moe", "moe", "seam", "experts", "logits", "expand", "codec"])
    fmt = rng.choice([Q8, IQ2])
    step = 32 if fmt == Q8 else 256  # columns come in whole blocks
    if kind == "proj":
        return dict(kind=kind, fmt=fmt, tokens=rng.choice([1, _log(rng, 2, 256), rng.randint(2, 256)]),
                    hidden=_mult(rng, step, 768, 2048), q_lora=_mult(rng, step, 512, 1024),
                    q_out=rng.randint(1024, 3840), kv=rng.randint(300, 700), o_in=_mult(rng, step, 1024, 2560))
    if kind == "moe":
        inter = _mult(rng, step, 512, 1536)
        return dict(kind=kind, fmt=fmt, tokens=rng.choice([1, _log(rng, 2, 256), rng.randint(2, 256)]),
                    hidden=_mult(rng, step, 768, 2048), inter=inter, experts=rng.randint(8, 64),
                    shared=rng.choice([0, inter, inter, _mult(rng, step, 512, 1536)]), router=rng.choice([F32, F16]))
    if kind == "seam":
        return dict(kind=kind, fmt=rng.choice([Q8, IQ2, F32]), rows=_log(rng, 200, 8192),
                    cols=_mult(rng, 256, 512, 4096), batch=rng.choice([1, 1, rng.randint(2, 64)]))
    if kind == "experts":
        return dict(kind=kind, fmt=fmt, experts=rng.randint(4, 64), hidden=_mult(rng, step, 768, 2048),
                    inter=_mult(rng, step, 512, 1536))
    if kind == "logits":
        return dict(kind=kind, fmt=fmt, vocab=rng.randint(32000, 154880), hidden=_mult(rng, step, 768, 2048))
    if kind == "expand":
        return dict(kind=kind, fmt=rng.choice([F32, F16]), rows=rng.randint(1024, 2560), cols=rng.randint(256, 512),
                    batch=_log(rng, 2, 300))
    return dict(kind=kind, positions=_log(rng, 256, 131072), row=rng.choice([576, 512, 64, rng.randint(64, 640)]))


# ---- weights and inputs -------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _raw(g, fmt, rows, cols, count=1):
    """Raw weight bytes on the device, as a model file holds them: block codes
    uniform, block scales half-normal, plain weights normal."""
    n = count * rows * cols
    if fmt in (F32, F16):
        w = torch.randn(n, generator=g, device="cuda") * 0.02
        return (w if fmt == F32 else w.half()).view(torch.uint8)
    size, nbytes, sigma = (32, 34, 0.02 / 127) if fmt == Q8 else (256, 66, 4e-4)
    blocks = torch.empty(n // size, nbytes, dtype=torch.uint8, device="cuda")
    d = (torch.randn(n // size, generator=g, device="cuda").abs() * sigma).half()
    blocks[:, :2] = d.view(torch.uint8).view(-1, 2)
    if fmt == Q8:
        codes = torch.randint(-127, 128, (n // size, 32), generator=g, device="cuda", dtype=torch.int8)
        blocks[:, 2:] = codes.view(torch.uint8)
    else:
        blocks[:, 2:] = torch.randint(0, 256, (n // size, 64), generator=g, device="cuda", dtype=torch.uint8)
    return blocks.view(-1)


def _x(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _mla_shapes(c):
    return dict(q_a=(c["q_lora"], c["hidden"]), q_b=(c["q_out"], c["q_lora"]), kv_a=(c["kv"], c["hidden"]),
                o_proj=(c["hidden"], c["o_in"]))


def _inputs(case, seed):
    """Every raw weight and input of a case, on the device, from the seed alone."""
    c, g, kind = case, _gen(seed), case["kind"]
    if kind == "proj":
        shapes = _mla_shapes(c)
        return dict(w={n: _raw(g, c["fmt"], r, k) for n, (r, k) in shapes.items()},
                    x={n: _x(g, c["tokens"], k) for n, (r, k) in shapes.items()})
    if kind in ("seam", "expand"):
        return dict(w=_raw(g, c["fmt"], c["rows"], c["cols"]), x=_x(g, c["batch"], c["cols"]))
    if kind == "experts":
        return dict(gate=_raw(g, c["fmt"], c["inter"], c["hidden"], c["experts"]),
                    down=_raw(g, c["fmt"], c["hidden"], c["inter"], c["experts"]),
                    xg=_x(g, c["hidden"]), xd=_x(g, c["experts"], c["inter"]))
    if kind == "logits":
        return dict(w=_raw(g, c["fmt"], c["vocab"], c["hidden"]), x=_x(g, c["hidden"]))
    if kind == "codec":
        return dict(x=_x(g, c["positions"], c["row"]))
    # MoE: router logits N(0, 0.02 sqrt(hidden)) plus the log of a popularity
    # of 1 / rank, carried by one hidden coordinate that is about constant:
    # a few experts take many tokens and most take few, as in a trained model.
    H, I, E, S = c["hidden"], c["inter"], c["experts"], c["shared"]
    x = _x(g, c["tokens"], H)
    x[:, 0] = 4.0
    router = torch.randn(E, H, generator=g, device="cuda") * 0.02
    rank = torch.randperm(E, generator=g, device="cuda").float() + 1
    router[:, 0] = -torch.log(rank) / 4.0
    if c["router"] == F16:
        router = router.half()
    w = dict(gate=_raw(g, c["fmt"], I, H, E), up=_raw(g, c["fmt"], I, H, E), down=_raw(g, c["fmt"], H, I, E))
    if S:
        w.update(sg=_raw(g, c["fmt"], S, H), su=_raw(g, c["fmt"], S, H), sd=_raw(g, c["fmt"], H, S))
    return dict(x=x, router=router, **w)


class _Ptr:
    """A device tensor as the binding takes device buffers (an address)."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


class _State:
    """What a program keeps between calls; frees the library's handles with it."""

    def __init__(self, case):
        self.case, self.handles, self.hosts = case, [], []

    def weight(self, raw, rows, cols, count=1):
        w = context().weight_from_device(_Ptr(raw), TYPE[self.case["fmt"]], rows, cols, count)
        self.handles.append(w)
        return w

    def out(self, *shape, dtype=torch.float32):
        return torch.zeros(*shape, dtype=dtype, device="cuda")

    def __del__(self):
        for h in self.handles:
            h.free()
        for a in self.hosts:
            context().forget(a)


_ctx = None


def context():
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = mm.Context(0)
    return _ctx


def prepare(case, seed):
    c, s, d = case, _State(case), _inputs(case, seed)
    torch.cuda.synchronize()  # the library uploads on a stream of its own
    kind = c["kind"]
    if kind == "proj":
        s.calls = []
        for n, (r, k) in _mla_shapes(c).items():
            s.calls.append((s.weight(d["w"][n], r, k), _Ptr(d["x"][n]), _Ptr(s.out(c["tokens"], r))))
        s.y = [y.t for _, _, y in s.calls]
    elif kind == "seam":
        s.w, s.x = d["w"].cpu().numpy(), d["x"].cpu().numpy()
        s.hosts.append(s.w)
    elif kind == "expand":
        s.w, s.x, s.y = s.weight(d["w"], c["rows"], c["cols"]), _Ptr(d["x"]), s.out(c["batch"], c["rows"])
        s.yp = _Ptr(s.y)
    elif kind == "experts":
        E, H, I = c["experts"], c["hidden"], c["inter"]
        wg, wd = s.weight(d["gate"], I, H, E), s.weight(d["down"], H, I, E)
        s.x, s.y = [_Ptr(d["xg"]), _Ptr(d["xd"])], [s.out(E, I), s.out(E, H)]
        s.groups = context().gemv_groups([(wg, 0, E, s.x[0], 0, _Ptr(s.y[0]), I), (wd, 0, E, s.x[1], I, _Ptr(s.y[1]), H)])
    elif kind == "logits":
        s.w, s.x = s.weight(d["w"], c["vocab"], c["hidden"]), _Ptr(d["x"])
        s.y, s.token = s.out(c["vocab"]), s.out(1, dtype=torch.int32)
        s.yp, s.tp = _Ptr(s.y), _Ptr(s.token)
    elif kind == "codec":
        n, row = c["positions"], c["row"]
        s.x, s.blocks, s.y = _Ptr(d["x"]), s.out(n, (row + 31) // 32 * 34, dtype=torch.uint8), s.out(n, row)
        s.bp, s.yp = _Ptr(s.blocks), _Ptr(s.y)
    else:
        h = {k: v.view(torch.uint8).view(-1).cpu().numpy() for k, v in d.items() if k != "x"}
        s.layer = mm.MoeLayer(context(), hidden=c["hidden"], inter=c["inter"], n_experts=c["experts"],
                              expert_type=TYPE[c["fmt"]], router=h["router"], gate=h["gate"], up=h["up"], down=h["down"],
                              shared=(h["sg"], h["su"], h["sd"]) if c["shared"] else None,
                              shared_inter=c["shared"] or None, router_type=TYPE[c["router"]])
        s.layer._keep = []  # the weights are on the device now
        s.handles.append(s.layer)
        s.x, s.y = _Ptr(d["x"]), s.out(c["tokens"], c["hidden"])
        s.yp = _Ptr(s.y)
    torch.cuda.synchronize()
    return s


def run(s):
    c, ctx = s.case, context()
    kind = c["kind"]
    if kind == "proj":
        for w, x, y in s.calls:
            if c["tokens"] == 1:
                ctx.gemv_batched_dev(w, 0, 1, x, 0, y, 0)
            else:
                ctx.qmm_dev(w, 0, x, y, c["tokens"])
        return s.y
    if kind == "seam":
        if c["batch"] == 1:
            return ctx.mat_vec_mul(s.w, TYPE[c["fmt"]], s.x, c["rows"], c["cols"], resident=True)
        return ctx.batch_mat_mul(s.w, TYPE[c["fmt"]], s.x, c["rows"], c["batch"], c["cols"], resident=True)
    if kind == "expand":
        ctx.qmm_dev(s.w, 0, s.x, s.yp, c["batch"])
        return s.y
    if kind == "experts":
        ctx.gemv_grouped_dev(s.groups)
        return s.y
    if kind == "logits":
        ctx.gemv_batched_dev(s.w, 0, 1, s.x, 0, s.yp, 0)
        ctx.argmax_dev(s.tp, s.yp, c["vocab"])
        return [s.y, s.token]
    if kind == "codec":
        ctx.quantize_q8_0_rows_dev(s.bp, s.x, c["row"], c["positions"], c["row"])
        ctx.dequantize_q8_0_rows_dev(s.yp, c["row"], s.bp, c["positions"], c["row"])
        return [s.blocks, s.y]
    s.layer.ffn_dev(s.x, s.yp, c["tokens"])
    return s.y


# ---- what a pass cannot do without --------------------------------------

def _wbytes(fmt, rows, cols):
    return rows * cols * {Q8: 34 / 32, IQ2: 66 / 256, F32: 4, F16: 2}[fmt]


def _touched(case):
    """Routed experts that the tokens of a call are expected to reach."""
    p = 1.0 / np.arange(1, case["experts"] + 1)
    p /= p.sum()
    k = min(4, case["experts"])
    return min(float(case["experts"]), max(float(k), float(np.sum(1 - (1 - p) ** (k * case["tokens"])))))


def work(case):
    c, kind = case, case["kind"]
    if kind == "proj":
        t, shapes = c["tokens"], _mla_shapes(c).values()
        return dict(bytes=sum(_wbytes(c["fmt"], r, k) + 4 * t * (r + k) for r, k in shapes),
                    flops=sum(2 * t * r * k for r, k in shapes))
    if kind in ("seam", "expand"):
        r, k, b = c["rows"], c["cols"], c["batch"]
        return dict(bytes=_wbytes(c["fmt"], r, k) + 4 * b * (r + k), flops=2 * b * r * k)
    if kind == "experts":
        E, H, I = c["experts"], c["hidden"], c["inter"]
        return dict(bytes=2 * E * _wbytes(c["fmt"], I, H) + 4 * (H + 2 * E * I + E * H), flops=4 * E * H * I)
    if kind == "logits":
        return dict(bytes=_wbytes(c["fmt"], c["vocab"], c["hidden"]) + 4 * (c["vocab"] + c["hidden"]) + 4,
                    flops=2 * c["vocab"] * c["hidden"])
    if kind == "codec":
        n = c["positions"]
        return dict(bytes=2 * n * (4 * c["row"] + (c["row"] + 31) // 32 * 34), flops=4 * n * c["row"])
    t, H, I, E, S = c["tokens"], c["hidden"], c["inter"], c["experts"], c["shared"]
    return dict(bytes=3 * _touched(c) * _wbytes(c["fmt"], I, H) + (3 * _wbytes(c["fmt"], S, H) if S else 0) +
                _wbytes(c["router"], E, H) + 8 * t * H, flops=2 * t * (E * H + 3 * H * (min(4, E) * I + S)))


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"
    if case["fmt"] in (F32, F16):
        return {"rel": 2e-6}
    # Activations enter the products as 16-bit block fixed point.
    return {"rel": 3e-4 if kind == "moe" else 1e-4}


# ---- the same results in 64 bits ----------------------------------------

# The IQ2_XXS codebook (public GGUF format data): eight magnitudes of
# 8, 25 and 43 per entry, as the base-3 digits of a number, the first lowest.
_GRID = [
    0, 2, 4, 6, 8, 10, 12, 18, 20, 24, 26, 28, 30, 36, 42, 46, 48, 54, 56, 62,
    74, 82, 84, 90, 94, 108, 138, 150, 162, 164, 182, 218, 244, 246, 252, 262, 264, 270, 272, 276,
    288, 298, 300, 306, 318, 324, 326, 330, 342, 356, 376, 378, 388, 412, 414, 432, 462, 480, 486, 490,
    492, 498, 510, 514, 516, 522, 524, 546, 570, 594, 650, 660, 730, 732, 738, 748, 756, 774, 786, 792,
    796, 810, 816, 828, 846, 854, 864, 912, 922, 972, 978, 990, 994, 1006, 1026, 1068, 1100, 1134, 1148, 1216,
    1218, 1224, 1242, 1270, 1296, 1300, 1368, 1414, 1458, 1460, 1466, 1488, 1504, 1512, 1514, 1564, 1572, 1620, 1622, 1702,
    1704, 1710, 1728, 1742, 1782, 1810, 1830, 1926, 1950, 1962, 2010, 2136, 2188, 2190, 2196, 2202, 2206, 2208, 2214, 2220,
    2228, 2232, 2242, 2244, 2250, 2268, 2286, 2314, 2322, 2326, 2350, 2358, 2382, 2390, 2400, 2430, 2436, 2448, 2484, 2500,
    2522, 2532, 2592, 2674, 2676, 2682, 2700, 2704, 2754, 2796, 2800, 2810, 2866, 2898, 2916, 2922, 2926, 2932, 2934, 2970,
    2976, 3000, 3026, 3072, 3142, 3222, 3224, 3248, 3322, 3360, 3402, 3412, 3418, 3450, 3510, 3570, 3648, 3654, 3672, 3696,
    3726, 3766, 3822, 3852, 3888, 3892, 3978, 3980, 4026, 4160, 4374, 4376, 4382, 4402, 4430, 4458, 4470, 4482, 4546, 4618,
    4620, 4626, 4630, 4644, 4662, 4698, 4730, 4764, 4786, 4806, 4824, 4862, 4944, 5032, 5106, 5112, 5124, 5130, 5176, 5198,
    5238, 5296, 5346, 5366, 5376, 5464, 5644, 5688, 5834, 5868, 5890, 5920, 5994, 6090, 6354, 6402,
]


def _weights64(raw, fmt, rows, cols):
    """Raw bytes of one matrix as float64 [rows, cols]."""
    if fmt == F32:
        return raw.view(torch.float32).double().view(rows, cols)
    if fmt == F16:
        return raw.view(torch.float16).double().view(rows, cols)
    size, nbytes = (32, 34) if fmt == Q8 else (256, 66)
    b = raw.view(-1, nbytes)
    d = b[:, :2].contiguous().view(torch.float16).double()
    if fmt == Q8:
        return (b[:, 2:].contiguous().view(torch.int8).double() * d).view(rows, cols)
    n = torch.tensor(_GRID, device=raw.device).view(256, 1)
    digits = torch.div(n, 3 ** torch.arange(8, device=raw.device), rounding_mode="floor") % 3
    grid = torch.tensor([8.0, 25.0, 43.0], dtype=torch.float64, device=raw.device)[digits]
    words = b[:, 2:].contiguous().view(torch.int32).view(-1, 8, 2).long() & 0xFFFFFFFF
    group = torch.arange(4, device=raw.device)
    idx = (words[..., :1] >> (8 * group)) & 255
    code = (words[..., 1:] >> (7 * group)) & 127
    bits = (code[..., None] >> torch.arange(7, device=raw.device)) & 1
    bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)
    scale = d.view(-1, 1) * (0.5 + (words[..., 1] >> 28).double()) / 4
    return (grid[idx] * (1.0 - 2.0 * bits) * scale[..., None, None]).view(rows, cols)


def _product64(raw, fmt, rows, cols, x):
    """x . W^T in float64, a few thousand rows of the matrix at a time."""
    step = 16384
    raw = raw.view(rows, -1)
    return torch.cat([x.double() @ _weights64(raw[r:r + step].reshape(-1), fmt, min(step, rows - r), cols).t().contiguous()
                      for r in range(0, rows, step)], -1)


def exact(case, seed):
    c, d, kind = case, _inputs(case, seed), case["kind"]
    if kind == "proj":
        return [_product64(d["w"][n], c["fmt"], r, k, d["x"][n]) for n, (r, k) in _mla_shapes(c).items()]
    if kind == "seam":
        y = _product64(d["w"], c["fmt"], c["rows"], c["cols"], d["x"])
        return (y[0] if c["batch"] == 1 else y).cpu().numpy()
    if kind == "expand":
        return _product64(d["w"], c["fmt"], c["rows"], c["cols"], d["x"])
    if kind == "experts":
        E, H, I = c["experts"], c["hidden"], c["inter"]
        gate, down = d["gate"].view(E, -1), d["down"].view(E, -1)
        return [torch.stack([_product64(gate[e], c["fmt"], I, H, d["xg"].view(1, -1))[0] for e in range(E)]),
                torch.stack([_product64(down[e], c["fmt"], H, I, d["xd"][e].view(1, -1))[0] for e in range(E)])]
    if kind == "logits":
        return [_product64(d["w"], c["fmt"], c["vocab"], c["hidden"], d["x"].view(1, -1))[0], None]
    if kind == "codec":
        n, row = c["positions"], c["row"]
        nb = (row + 31) // 32
        x = torch.nn.functional.pad(d["x"], (0, nb * 32 - row)).view(n, nb, 32)
        scale = x.abs().amax(-1) / 127.0  # in 32 bits: the format's own rounding
        q = x / scale[..., None]
        q = torch.where(scale[..., None] > 0, torch.sign(q) * torch.floor(q.abs() + 0.5), torch.zeros_like(q))
        return [None, (q.double() * scale.half().double()[..., None]).view(n, nb * 32)[:, :row]]
    T, H, I, E, S, f = c["tokens"], c["hidden"], c["inter"], c["experts"], c["shared"], c["fmt"]
    x = d["x"].double()
    top, ids = torch.topk(x @ d["router"].double().t().contiguous(), min(4, E), dim=-1)
    share = torch.softmax(top, -1)
    y = torch.zeros(T, H, dtype=torch.float64, device="cuda")

    def expert(gate, up, down, width, v):
        g = _product64(gate, f, width, H, v)
        return _product64(down, f, H, width, g / (1 + torch.exp(-g)) * _product64(up, f, width, H, v))

    gate, up, down = (d[k].view(E, -1) for k in ("gate", "up", "down"))
    for e in range(E):
        t, k = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            y[t] += share[t, k, None] * expert(gate[e], up[e], down[e], I, x[t])
    if S:
        y += expert(d["sg"], d["su"], d["sd"], S, x)
    return y
