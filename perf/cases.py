"""The attention section of the Klein DiT blocks as programs call it, over the sizes it meets.

A Klein 4B denoising step runs 5 double and 20 single blocks (24 heads of 128, hidden width
3072).  One image of H x W pixels is a sequence of 512 text tokens and (H/16) x (W/16) image
tokens; generation runs from previews of 256 pixels to 2048, in several aspect ratios, at
batch 1 to 4, and one GPU of a head-parallel group holds 24 / n heads.  Per block a program
calls either the bfloat16 path (``modules.double_attention`` / ``single_attention``, or their
parts ``kernels.qk_prep`` and ``kernels.attend_merged``) or the int8 path
(``modules.double_attention_int8``, ``w8a8.qk_prep``, ``w8a8.linear``); at load time it
calibrates and quantises each projection (``w8a8.absmax_cols``, ``w8a8.quantize_linear``).

A case is one such call:

  kind        batch  text  rows  cols  heads   and
  double      B      T     h     w     24      bf16 QKV of both streams -> both attention outputs
  single      B      T     h     w     24      bf16 linear1 output (QKV + MLP columns) -> attention
  attend      B      T     h     w     H       q, k, v -> merged attention output
  qk_prep     B      T     h     w     24      rope: "tables" (cos / sin lanes), "ids", or "pe" (plain branch)
  linear8     B      T     h     w     24      bf16 activation -> int8 projection -> bf16 QKV
  qkv8        B      T     h     w     24      block input, modulation -> int8 projection -> q, k, v
  double8     B      T     h     w     24      both block inputs -> both attention outputs, int8 projections
  calibrate   B      T     h     w     24      one calibration batch and a weight -> the int8 projection

Sequence lengths are T + h * w; h = 0 is a text stream alone.
"""

from __future__ import annotations

import math

import torch

from flicker_amd import kernels, modules, rope, w8a8

HEADS, DIM, HIDDEN, MLP = 24, 128, 3072, 18432   # MLP: the two gated halves of linear1
WIDTH = 3 * HEADS * DIM
GAIN = 1.0 / math.sqrt(DIM)


def _case(name, kind, batch, text, rows, cols, heads=HEADS, **more):
    case = {"kind": kind, "batch": batch, "text": text, "rows": rows, "cols": cols, "heads": heads, **more}
    return {"name": name, **case} if name else case


def listed():
    return [
        # The smallest call of a block: a text stream's qk_prep, where launches and latency count.
        _case("qk_prep_text", "qk_prep", 1, 512, 0, 0, rope="tables"),
        # A 256-pixel preview through a double block's attention section.
        _case("double_256px", "double", 1, 512, 16, 16),
        # A 512-pixel image through a single block, QKV read in place from linear1's wide output.
        _case("single_512px", "single", 1, 512, 32, 32),
        # One of eight GPUs' three heads of a 1024-pixel image.
        _case("attend_3_heads", "attend", 1, 512, 64, 64, heads=3),
        # The ordinary 1024-pixel image, and the largest one of 2048.
        _case("attend_1024px", "attend", 1, 512, 64, 64),
        _case("attend_2048px", "attend", 1, 512, 128, 128),
        # Four images at a time, and a 1536 x 640 banner whose lanes come from the position ids.
        _case("qk_prep_1024px_b4", "qk_prep", 4, 512, 64, 64, rope="tables"),
        _case("qk_prep_ids_banner", "qk_prep", 1, 512, 96, 40, rope="ids"),
        # The int8 projection of the text stream alone.
        _case("linear8_text", "linear8", 1, 512, 0, 0),
        # A single block's int8 projection at 1008 x 752 pixels: no tile divides its 3473 tokens.
        _case("qkv8_ragged", "qkv8", 1, 512, 63, 47),
        # A double block's whole attention section on the int8 path.
        _case("double8_1024px", "double8", 1, 512, 64, 64),
        # Load time: one 1024-pixel calibration batch and the weight it scales.
        _case("calibrate_1024px", "calibrate", 1, 512, 64, 64),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("double", "single", "attend", "qk_prep", "linear8", "qkv8", "double8", "calibrate"))
    batch = rng.choice((1, 1, 1, 2, 4))
    side = _log_int(rng, 8, 96 if batch == 1 else 64)      # image tokens along one side
    ratio = rng.uniform(0.5, 2.0)
    rows, cols = max(4, round(side * math.sqrt(ratio))), max(4, round(side / math.sqrt(ratio)))
    text = rng.choice((512, 512, 512, 256, 128))
    heads, more = HEADS, {}
    if kind == "qk_prep":
        more["rope"] = rng.choice(("tables", "ids", "pe"))
    if kind == "attend":
        heads = rng.choice((24, 24, 12, 6, 3))
    if kind in ("double", "single") or more.get("rope") in ("tables", "ids"):
        # the bounded path's gate: each stream's length is a multiple of 64
        rows, cols = max(8, rows // 8 * 8), max(8, cols // 8 * 8)
    if kind in ("linear8", "qk_prep") and rng.random() < 0.25:
        rows, cols = 0, 0                                  # a shorter text stream alone
        gated = more.get("rope") in ("tables", "ids")
        text = 64 * rng.randrange(1, 8) if gated else rng.randrange(17, 512)
    return _case(None, kind, batch, text, rows, cols, heads, **more)


def _length(case):
    return case["text"] + case["rows"] * case["cols"]


def work(case):
    batch, length, heads = case["batch"], _length(case), case["heads"]
    tokens = batch * length
    qkv, out = 2 * tokens * 3 * heads * DIM, 2 * tokens * heads * DIM
    lanes = 16 * length if case.get("rope") == "ids" else 2 * 4 * length * DIM
    attention = 4 * batch * heads * length * length * DIM
    projection = 2 * tokens * HIDDEN * WIDTH
    x, w8 = 2 * tokens * HIDDEN, HIDDEN * WIDTH
    kind = case["kind"]
    if kind in ("double", "single"):
        return {"bytes": qkv + lanes + out, "flops": attention}
    if kind == "attend":
        return {"bytes": qkv + out, "flops": attention}
    if kind == "qk_prep":
        return {"bytes": 2 * qkv + lanes, "flops": 0}
    if kind == "linear8":
        return {"bytes": x + w8 + qkv, "flops": projection}
    if kind == "qkv8":
        return {"bytes": x + w8 + lanes + qkv, "flops": projection}
    if kind == "double8":
        return {"bytes": x + 2 * w8 + lanes + out, "flops": projection + attention}
    return {"bytes": x + 3 * w8, "flops": 0}               # calibrate: X and W read, WqT written


def tolerance(case):
    # Calibration is maxima, single float32 operations and the codes they fix.  The others end
    # in bfloat16: against 64 bits they measure 1.7e-3 off from the last rounding alone, 2.3e-3
    # to 2.9e-3 with those of P or of the normed rows on the way, 4.6e-3 through a bf16 section.
    return "exact" if case["kind"] == "calibrate" else {"rel": 1e-2}


# ---------------------------------------------------------------- inputs ----------------


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _scales(gen):
    return tuple((1 + 0.05 * _normal(gen, DIM)).to(torch.bfloat16) for _ in range(2))


def _ids(case):
    return rope.sequence_ids(case["text"], case["rows"], case["cols"])


def _activation(gen, batch, length):
    """A block input with 1% of its channels 20 times the others, as DiT activations have."""
    x = _normal(gen, batch, length, HIDDEN)
    x[..., torch.randperm(HIDDEN, generator=gen, device="cuda")[:HIDDEN // 100]] *= 20.0
    return x.to(torch.bfloat16)


def _weight(gen):
    return (0.02 * _normal(gen, HIDDEN, WIDTH)).to(torch.bfloat16)


def _modulation(gen, batch):
    return tuple((0.2 * _normal(gen, batch, HIDDEN)).to(torch.bfloat16) for _ in range(2))


def _absmax(x):
    return x.reshape(-1, HIDDEN).abs().amax(0).float()


def _inputs(case, seed):
    """The case's tensors, from plain torch alone."""
    gen = torch.Generator("cuda").manual_seed(seed)
    kind, batch, length, heads = case["kind"], case["batch"], _length(case), case["heads"]
    text = case["text"]
    if kind == "double":
        return {"txt": _normal(gen, batch, text, WIDTH).to(torch.bfloat16),
                "img": _normal(gen, batch, length - text, WIDTH).to(torch.bfloat16),
                "txt_scales": _scales(gen), "img_scales": _scales(gen)}
    if kind == "single":
        return {"linear1": _normal(gen, batch, length, WIDTH + MLP).to(torch.bfloat16), "scales": _scales(gen)}
    if kind == "attend":
        def unit(gain):
            x = _normal(gen, batch, heads, length, DIM)
            return (x * (gain * torch.rsqrt(x.square().mean(-1, keepdim=True)))).to(torch.bfloat16)
        return {"q": unit(GAIN), "k": unit(1.0), "v": _normal(gen, batch, heads, length, DIM).to(torch.bfloat16)}
    if kind == "qk_prep":
        return {"qkv": _normal(gen, batch, length, WIDTH).to(torch.bfloat16), "scales": _scales(gen)}
    if kind == "double8":
        return {"txt": _activation(gen, batch, text), "img": _activation(gen, batch, length - text),
                "txt_w": _weight(gen), "img_w": _weight(gen), "txt_scales": _scales(gen), "img_scales": _scales(gen),
                "modulation": (_modulation(gen, batch), _modulation(gen, batch))}
    d = {"x": _activation(gen, batch, length), "w": _weight(gen)}
    if kind == "qkv8":
        d.update(scales=_scales(gen), modulation=_modulation(gen, batch))
    return d


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("double", "single", "double8", "qkv8"):
        s["freqs"] = rope.rope_lanes(_ids(case), GAIN, device="cuda")
    if kind == "qk_prep":
        if case["rope"] == "pe":
            s["pe"] = rope.embed_nd(_ids(case), device="cuda")
        elif case["rope"] == "ids":
            s["freqs"] = rope.position_ids(_ids(case), GAIN, device="cuda")
        else:
            s["freqs"] = rope.rope_lanes(_ids(case), GAIN, device="cuda")
    if kind in ("linear8", "qkv8"):
        stats = _absmax(s["x"] if kind == "linear8" else _modulate(s["x"], *s["modulation"]))
        s["qw"] = w8a8.quantize_linear(s.pop("w"), stats)
    if kind == "double8":
        for n, m in zip(("txt", "img"), s["modulation"]):
            s[n + "_qw"] = w8a8.quantize_linear(s.pop(n + "_w"), _absmax(_modulate(s[n], *m)))
    s["case"] = case
    return s


def run(s):
    kind, heads = s["case"]["kind"], s["case"]["heads"]
    if kind == "double":
        return modules.double_attention(s["txt"], s["img"], s["txt_scales"], s["img_scales"], s["freqs"], heads)
    if kind == "single":
        return modules.single_attention(s["linear1"], *s["scales"], s["freqs"], heads, HIDDEN)
    if kind == "attend":
        return kernels.attend_merged(s["q"], s["k"], s["v"])
    if kind == "qk_prep":
        if "pe" in s:
            return modules.qkv_prep(s["qkv"], *s["scales"], s["pe"], None, heads)
        return kernels.qk_prep(s["qkv"], *s["scales"], s["freqs"], heads)
    if kind == "linear8":
        return w8a8.linear(s["x"], s["qw"])
    if kind == "qkv8":
        return w8a8.qk_prep(s["x"], s["qw"], *s["scales"], s["freqs"], heads, modulation=s["modulation"])
    if kind == "double8":
        return modules.double_attention_int8(s["txt"], s["img"], s["txt_qw"], s["img_qw"], s["txt_scales"],
                                             s["img_scales"], s["freqs"], heads, modulation=s["modulation"])
    return tuple(w8a8.quantize_linear(s["w"], w8a8.absmax_cols(s["x"])))


# ---------------------------------------------------------------- 64 bits ---------------


def _modulate(x, shift, scale):
    """The projection's input (1 + scale) * layer_norm(x) + shift, at its bfloat16 steps."""
    bf = lambda t: t.to(torch.bfloat16).double()   # noqa: E731
    x = x.double()
    d = x - x.mean(-1, keepdim=True)
    norm = bf(d / torch.sqrt(d.square().mean(-1, keepdim=True) + 1e-6))
    return bf(bf(bf(1 + scale.double())[:, None] * norm) + shift.double()[:, None]).to(torch.bfloat16)


def _lanes64(case):
    ids = torch.as_tensor(_ids(case), device="cuda", dtype=torch.float64)
    omega = 2000.0 ** -(torch.arange(16, device="cuda", dtype=torch.float64) / 16)
    angle = (ids[:, :, None] * omega).reshape(ids.shape[0], DIM // 2)
    return torch.cos(angle), torch.sin(angle)


def _prep64(qkv, scales, lanes, heads, gain):
    """(B, L, 3 H D) in 64 bits -> q, k, v (B, H, L, D): RMSNorm, scale and rotation."""
    batch, length, _ = qkv.shape
    q, k, v = qkv.reshape(batch, length, 3, heads, DIM).permute(2, 0, 3, 1, 4)
    cos, sin = lanes

    def rotate(t, scale, by):
        t = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * scale.double()
        a, b = t[..., 0::2], t[..., 1::2]
        return by * torch.stack((cos * a - sin * b, sin * a + cos * b), -1).flatten(-2)

    return rotate(q, scales[0], gain), rotate(k, scales[1], 1.0), v


def _attend64(q, k, v):
    """softmax(q k^T) v, merged to (B, L, H D); 2048 queries of one head at a time."""
    batch, heads, length, dim = q.shape
    out = torch.empty((batch, length, heads, dim), device=q.device, dtype=torch.float64)
    for b in range(batch):
        for h in range(heads):
            kt, vh = k[b, h].double().t().contiguous(), v[b, h].double().contiguous()
            for i in range(0, length, 2048):
                p = torch.exp(q[b, h, i:i + 2048].double() @ kt)
                out[b, i:i + 2048, h] = (p @ vh) / p.sum(-1, keepdim=True)
    return out.reshape(batch, length, heads * dim)


def _smooth64(x_absmax, w):
    xa, wa = x_absmax.double(), w.abs().amax(1).double()
    return torch.where((xa > 0) & (wa > 0), torch.sqrt(xa) / torch.sqrt(wa), torch.ones_like(xa))


def _linear64(x, w, x_absmax):
    """x @ w with both operands rounded to their int8 codes, products and scales in 64 bits."""
    s = _smooth64(x_absmax, w)
    wh, xh = w.double() * s[:, None], x.reshape(-1, HIDDEN).double() / s
    wo, at = wh.abs().amax(0) / 127, xh.abs().amax(1, keepdim=True) / 127
    wo, at = torch.where(wo > 0, wo, 1.0), torch.where(at > 0, at, 1.0)
    y = (torch.round(xh / at) @ torch.round(wh / wo)) * at * wo
    return y.reshape(*x.shape[:-1], WIDTH)


def exact(case, seed):
    kind, heads, text = case["kind"], case["heads"], case["text"]
    s = _inputs(case, seed)
    if kind == "attend":
        return _attend64(s["q"], s["k"], s["v"])
    if kind == "qk_prep":
        return _prep64(s["qkv"].double(), s["scales"], _lanes64(case), heads, 1.0 if case["rope"] == "pe" else GAIN)
    if kind == "linear8":
        return _linear64(s["x"], s["w"], _absmax(s["x"]))
    if kind == "calibrate":
        stats = _absmax(s["x"])
        smooth = _smooth64(stats, s["w"])
        return None, (s["w"].double() * smooth[:, None]).abs().amax(0) / 127, smooth, 1 / smooth
    if kind == "qkv8":
        x = _modulate(s["x"], *s["modulation"])
        return _prep64(_linear64(x, s["w"], _absmax(x)), s["scales"], _lanes64(case), heads, GAIN)
    if kind == "single":
        qkv = s["linear1"][..., :WIDTH].double()
        return _attend64(*_prep64(qkv, s["scales"], _lanes64(case), heads, GAIN)), s["linear1"][..., WIDTH:].double()
    cos, sin = _lanes64(case)
    parts = []
    for n, rows in (("txt", slice(0, text)), ("img", slice(text, None))):
        if kind == "double":
            qkv = s[n].double()
        else:
            x = _modulate(s[n], *s["modulation"][n == "img"])
            qkv = _linear64(x, s[n + "_w"], _absmax(x))
        parts.append(_prep64(qkv, s[n + "_scales"], (cos[rows], sin[rows]), heads, GAIN))
    out = _attend64(*(torch.cat(p, 2) for p in zip(*parts)))
    return out[:, :text], out[:, text:]
