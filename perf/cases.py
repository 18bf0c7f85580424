"""The measured work of this framework: what a LoRA fine-tuning program has it
do, through its public entry points, over the sizes it meets.

A case is one pass of one of these kinds:

  fwd    one adapted linear, forward only (``device.lora_fwd``): sampling with
         an adapter, a few tokens at a time
  layer  one adapted linear, forward and backward (``device.lora_fwd``,
         ``device.lora_bwd``): y, t, dx, dA, dB, as a host program that calls
         the C ABI trains a site
  site   the same through ``adapters.site`` and torch autograd (f32 factors)
  base   a frozen linear without an adapter, with its bias: forward and input
         gradient through ``adapters.QuantLinear`` and autograd
  load   a frozen weight brought into the layout the kernels read: quantized
         from f32 (``quant.quantize_linear_weight``), from an fp8 checkpoint
         tensor to int4 (``device.requantize_fp8_int4``), or to fp8
  glue   an MMDiT block's elementwise kernels, forward and gradient
         (``mmdit_ops``): attention inputs, modulated norm, gated residual, GELU
  step   a whole block-checkpointed training step of a one-block MMDiT
         (``mmdit.checkpointed_step``): the loss and every adapter's gradients

Sizes are those of the repository's benchmark (the 3072-wide MMDiT with 4096
image and 512 text tokens, the 2560-wide decoder, the 3072 -> 3072 and
3072 -> 12288 layers) and ragged ones around them.
"""

import math

import torch
import torch.nn.functional as F

from loractl_amd import device as D
from loractl_amd.adapters import LoraAdapters, QuantLinear, site
from loractl_amd.lora import LoraDelta
from loractl_amd.mmdit import Mmdit, MmditConfig, build_mmdit_adapters, checkpointed_step
from loractl_amd.mmdit_ops import attn_prep, gated_residual, gelu_tanh, modnorm, rope_tables
from loractl_amd.quant import QuantValue, quantize_linear_weight

DEV = "cuda"
W_STD = 0.02  # frozen weights ~ N(0, 0.02)


def _linear(kind, fmt, m, k, n, r=0, group=64):
    return {"kind": kind, "fmt": fmt, "m": m, "k": k, "n": n, "r": r, "group": group}


def listed():
    return [
        # sampling with an adapter at a handful of tokens: one short launch
        {"name": "forward_16_tokens", **_linear("fwd", "int4", 16, 3072, 12288, 32)},
        # the MMDiT's modulation linear in training: one conditioning row per
        # batch element, through autograd as the trainer runs it
        {"name": "modulation_site_1_token", **_linear("site", "int4", 1, 3072, 18432, 32)},
        # decoder MLP at a short sequence
        {"name": "decoder_gate_256_tokens", **_linear("layer", "int4", 256, 2560, 9728, 16)},
        # the text stream's MLP down projection: few tokens, deep reduction
        {"name": "text_down_512_tokens", **_linear("layer", "int4", 512, 12288, 3072, 32)},
        # the reference configuration's square layer
        {"name": "square_1024_tokens", **_linear("layer", "int4", 1024, 3072, 3072, 16)},
        # an int8 base, quant block 32, token count and rank off every tile
        {"name": "int8_ragged_1999_tokens", **_linear("layer", "int8", 1999, 2560, 4096, 24, 32)},
        # the headline layer: the image stream's MLP up projection
        {"name": "mlp_up_4096_tokens", **_linear("layer", "int4", 4096, 3072, 12288, 32)},
        # an fp8 checkpoint's linear at the image stream's length
        {"name": "fp8_qkv_4096_tokens", **_linear("layer", "fp8", 4096, 3072, 9216, 32)},
        # a site no adapter targets: frozen base with its bias, odd token count
        {"name": "frozen_bias_777_tokens", **_linear("base", "int4", 777, 3072, 9216)},
        # quantizing one frozen weight when a model is loaded
        {"name": "load_int4_from_f32", **_linear("load", "int4", 0, 3072, 12288)},
        # the block's elementwise kernels over the joint sequence
        {"name": "block_glue", "kind": "glue", "img": 4096, "txt": 512, "h": 3072, "heads": 24},
        # one training step of one block: every kernel in its place
        {"name": "train_step_one_block", "kind": "step", "img": 4096, "txt": 512, "h": 3072, "heads": 24, "r": 32},
    ]


def _logint(rng, lo, hi, mult=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / mult)) * mult))


def draw(rng):
    kind = rng.choices(["layer", "fwd", "site", "base", "load", "glue", "step"], [8, 4, 1, 2, 3, 2, 1])[0]
    if kind == "glue":
        hd = rng.choice([64, 128])
        heads = _logint(rng, 512, 4096, hd) // hd
        return {"kind": kind, "img": _logint(rng, 64, 4096), "txt": rng.randint(0, 512), "h": heads * hd, "heads": heads}
    if kind == "step":
        heads = rng.choice([8, 12, 16, 24])
        return {"kind": kind, "img": _logint(rng, 256, 4096, 8), "txt": 8 * rng.randint(2, 64), "h": 128 * heads,
                "heads": heads, "r": rng.choice([8, 16, 32, 64])}
    fmt = rng.choice(["int4", "int4", "int8", "fp8", "fp8_scalar"])
    group = rng.choice([32, 64, 64, 128])
    k = _logint(rng, 512, 12288, group if fmt.startswith("int") else 32)
    n = _logint(rng, 512, 18432, 8)
    if kind == "load":
        fmt = rng.choice(["int4", "int8", "fp8", "fp8_scalar", "fp8_to_int4", "fp8_scalar_to_int4"])
        k = _logint(rng, 512, 12288, 128)
        return _linear(kind, fmt, 0, k, _logint(rng, 512, 12288, 8), 0, group)
    if kind == "fwd":
        return _linear(kind, fmt, rng.randint(1, 16), k, n, rng.choice([4, 8, 16, 32, 64]), group)
    if kind == "site":
        return _linear(kind, fmt, _logint(rng, 1, 512), k, n, rng.choice([8, 16, 32]), group)
    # at most the 4096-token headline layer's work
    m = _logint(rng, 17, min(4096, max(17, 4096 * 3072 * 12288 // (k * n))))
    return _linear(kind, fmt, m, k, n, 0 if kind == "base" else rng.choice([4, 8, 16, 16, 24, 32, 32, 64]), group)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(dtype)


def _factors(g, k, r, n):
    """LoRA factors as training meets them: A Kaiming-uniform, B ~ N(0, 0.01)."""
    a = (torch.rand(k, r, device=DEV, generator=g) * 2 - 1) / math.sqrt(k)
    return a, _randn(g, r, n, std=1e-2)


def _raw(c, seed):
    """One linear's f32 weight and bf16 activations, from the seed alone."""
    g = _gen(seed)
    w = _randn(g, c["n"], c["k"], std=W_STD)
    if c["kind"] == "load":
        return {"w": w}
    bf = torch.bfloat16
    d = {"w": w, "x": _randn(g, c["m"], c["k"], dtype=bf)}
    if c["kind"] != "fwd":
        d["dy"] = _randn(g, c["m"], c["n"], dtype=bf)
    if c["r"]:
        d["a"], d["b"] = _factors(g, c["k"], c["r"], c["n"])
        if c["kind"] != "site":
            d["a"], d["b"] = d["a"].to(bf), d["b"].to(bf)
    else:
        d["bias"] = _randn(g, c["n"], std=0.1)
    return d


def _pack(c, w):
    if c["fmt"] == "int4":
        return D.quantize_int4(w, c["group"])
    if c["fmt"] == "int8":
        return D.quantize_int8(w, c["group"])
    return D.quantize_fp8(w, c["fmt"] == "fp8")


def _glue_raw(c, seed):
    g, bf = _gen(seed), torch.bfloat16
    li, lt, h = c["img"], c["txt"], c["h"]
    ins = {"x": _randn(g, li, h, dtype=bf), "scale": _randn(g, 1, h, std=0.3, dtype=bf),
           "shift": _randn(g, 1, h, std=0.3, dtype=bf), "gate": _randn(g, 1, h, std=0.3, dtype=bf),
           "o": _randn(g, li, h, dtype=bf), "u": _randn(g, li, 4 * h, dtype=bf),
           "qkv_txt": _randn(g, lt, 3 * h, dtype=bf), "qkv_img": _randn(g, li, 3 * h, dtype=bf)}
    hd = h // c["heads"]
    cot = [_randn(g, li, h, dtype=bf)] + [_randn(g, lt + li, c["heads"], hd, dtype=bf) for _ in range(3)]
    cot += [_randn(g, li, h, dtype=bf), _randn(g, li, 4 * h, dtype=bf)]
    return ins, cot


def _step_raw(c, seed):
    """The step's frozen weights (block linears f32, embedders and head bf16),
    adapter factors and flow-matching batch."""
    g, bf = _gen(seed), torch.bfloat16
    cfg = MmditConfig(hidden=c["h"], heads=c["heads"], layers=1, rank=c["r"], alpha=float(c["r"]))
    h = c["h"]
    bases, factors = {}, {}
    for path in cfg.site_paths():
        k, n = cfg.site_shapes()[path.rsplit(".", 1)[1]]
        bases[path] = _randn(g, n, k, std=W_STD)
        factors[path] = _factors(g, k, c["r"], n)
    plain = {}
    for name, k, n in (("img_in", cfg.patch_dim, h), ("txt_in", cfg.txt_dim, h), ("t_in", cfg.tdim, h),
                       ("t_out", h, h), ("final_mod", h, 2 * h), ("final", h, cfg.patch_dim)):
        plain[name] = (_randn(g, n, k, std=1 / math.sqrt(k), dtype=bf), _randn(g, n, std=0.02, dtype=bf))
    x0 = _randn(g, c["img"], cfg.patch_dim)
    eps = _randn(g, c["img"], cfg.patch_dim)
    txt = _randn(g, c["txt"], cfg.txt_dim, dtype=bf)
    t = torch.rand(1, device=DEV, generator=g)
    return cfg, bases, factors, plain, (((1 - t) * x0 + t * eps).to(bf), txt, t, eps - x0)


def prepare(case, seed):
    c = case
    if c["kind"] == "glue":
        ins, cot = _glue_raw(c, seed)
        ins = {k: v.requires_grad_() for k, v in ins.items()}
        return {"case": c, "ins": ins, "cot": cot, "rope": rope_tables(c["img"] + c["txt"], c["h"] // c["heads"], DEV)}
    if c["kind"] == "step":
        cfg, bases, factors, plain, batch = _step_raw(c, seed)
        cfg.layers = 0
        model = Mmdit(cfg, DEV)
        cfg.layers = 1
        for path, w in bases.items():
            model.bases[path] = QuantLinear([D.quantize_int4(w, cfg.group)])
        for name, wb in plain.items():
            setattr(model, name, wb)
        adapters = build_mmdit_adapters(cfg, DEV)
        with torch.no_grad():
            for path, (a, b) in factors.items():
                delta = adapters.get(path)
                delta.lora_a.copy_(a)
                delta.lora_b.copy_(b)
        return {"case": c, "model": model, "adapters": adapters, "batch": batch}
    d = _raw(c, seed)
    if c["kind"] == "load":
        s = {"case": c, "w": d["w"]}
        if c["fmt"].endswith("_to_int4"):  # an fp8 checkpoint's tensor
            s["w"] = D.quantize_fp8(d["w"], c["fmt"] == "fp8_to_int4")
        return s
    s = {"case": c, **{k: v for k, v in d.items() if k != "w"}}
    packed = _pack(c, d["w"])
    if c["kind"] in ("site", "base"):
        s["x"].requires_grad_()
        s["base"] = QuantLinear([packed], d.get("bias"))
        if c["kind"] == "site":
            delta = LoraDelta(c["k"], c["n"], c["r"], float(c["r"]), device=DEV)
            with torch.no_grad():
                delta.lora_a.copy_(d["a"])
                delta.lora_b.copy_(d["b"])
            s["adapters"] = LoraAdapters([delta], ["blocks.0.img.mod"])
    else:
        s["wq"] = D.compute_weight(packed)
    return s


# ------------------------------------------------------------------ the pass
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "fwd":
        return D.lora_fwd(s["x"], s["wq"], s["a"], s["b"], 1.0)
    if kind == "layer":
        y, t = D.lora_fwd(s["x"], s["wq"], s["a"], s["b"], 1.0)
        return (y, t) + tuple(D.lora_bwd(s["x"], s["dy"], s["wq"], s["a"], s["b"], 1.0, t))
    if kind == "site":
        delta = s["adapters"].deltas[0]
        y = site(s["adapters"], "blocks.0.img.mod", s["base"], s["x"])
        return (y,) + torch.autograd.grad(y, [s["x"], delta.lora_a, delta.lora_b], s["dy"])
    if kind == "base":
        y = s["base"].forward(s["x"])
        return (y,) + torch.autograd.grad(y, [s["x"]], s["dy"])
    if kind == "load":
        fmt = c["fmt"]
        if fmt.endswith("_to_int4"):
            w = D.block(D.requantize_fp8_int4(s["w"], c["group"]))
        elif fmt.startswith("fp8"):
            w = D.block(D.quantize_fp8(s["w"], fmt == "fp8"))
        else:
            w = quantize_linear_weight(s["w"], QuantValue.Q4S if fmt == "int4" else QuantValue.Q8S, c["group"])
        return {"data": w.data, "scales": w.scales}
    if kind == "glue":
        i = s["ins"]
        outs = [modnorm(i["x"], i["scale"], i["shift"])]
        outs += attn_prep(i["qkv_txt"], i["qkv_img"], s["rope"], c["heads"])
        outs += [gated_residual(i["x"], i["gate"], i["o"]), gelu_tanh(i["u"])]
        return outs + list(torch.autograd.grad(outs, list(i.values()), s["cot"]))
    ad = s["adapters"]
    for p in ad.parameters():
        p.grad = None
    loss = checkpointed_step(s["model"], ad, s["batch"])
    return {"loss": loss, "grads": [p.grad for p in ad.parameters()]}


# ------------------------------------------------------------------ what a pass needs
def _packed_bytes(c):
    per = 0.5 if c["fmt"] == "int4" else 1.0
    scales = c["n"] * (c["k"] // c["group"]) if c["fmt"].startswith("int") else (c["n"] if c["fmt"] == "fp8" else 1)
    return c["n"] * c["k"] * per + 4 * scales


def work(case):
    c = case
    kind = c["kind"]
    if kind == "glue":
        rows, h, L = c["img"], c["h"], c["img"] + c["txt"]
        # bf16 reads and writes: norm, residual and GELU, forward and
        # gradient; attention inputs
        return {"bytes": 2 * rows * h * (5 + 6 + 20) + 2 * L * h * 14, "flops": 40 * rows * h * 6 + 60 * L * h * 3}
    if kind == "step":
        h, L = c["h"], c["img"] + c["txt"]
        block = 12 * h * h  # qkv, out, up, down
        proj = 2 * L * block + 2 * 2 * 6 * h * h
        lora = 2 * c["r"] * L * (4 * h + 2 * h + 5 * h + 5 * h)
        attn = 4 * L * L * h
        # capture, replay and input gradients; the factors' gradients too
        weights = 2 * (block + 6 * h * h) * (0.5 + 4 / 64)
        adapters = 2 * c["r"] * (4 + 2 + 5 + 5 + 7) * h
        return {"bytes": weights + 2 * 4 * adapters + 2 * L * h * 4, "flops": 3 * proj + 4 * lora + 4 * attn}
    m, k, n, r = c["m"], c["k"], c["n"], c["r"]
    if kind == "load":
        pad = 64 * 64 * (-(-n // 64)) * (-(-k // 64))
        f8 = c["fmt"].endswith("_to_int4")
        out4 = f8 or c["fmt"] == "int4"
        scales = 0 if c["fmt"] in ("fp8", "fp8_scalar") else 2 * pad // c["group"]
        return {"bytes": n * k * (1 if f8 else 4) + 2 * pad * (0.5 if out4 else 1) + 4 * scales, "flops": 4 * n * k}
    factors = (2 if kind in ("fwd", "layer") else 4) * r * (k + n)
    if kind == "fwd":
        return {"bytes": _packed_bytes(c) + factors + 2 * m * (k + n + r), "flops": 2 * m * k * n + 2 * m * r * (k + n)}
    grads = 4 * r * (k + n)
    return {"bytes": _packed_bytes(c) + factors + grads + 2 * m * (2 * k + 2 * n + r),
            "flops": 4 * m * k * n + 6 * m * r * (k + n)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"  # packed bytes and their f32 scales
    if case["kind"] == "glue":
        return {"rel": 8e-3}  # one bf16 rounding per output: 2e-3 off the f64 result
    if case["kind"] == "step":
        return {"rel": 3e-2}  # bf16 roundings of a whole block travel into every gradient
    return {"rel": 1.2e-2}    # bf16 operands and outputs: 2e-3 to 3e-3 off the f64 result


# ------------------------------------------------------------------ the same in 64 bits
def _scales(w, fmt, group):
    """The f32 scales [n, k/group], [n, 1] or [1, 1] a format gives w."""
    n, k = w.shape
    if fmt.startswith("int"):
        return w.view(n, k // group, group).abs().amax(2) / (7 if fmt == "int4" else 127)
    amax = w.abs().amax(1, keepdim=True) if fmt == "fp8" else w.abs().amax().view(1, 1)
    return torch.clamp(amax / 448, min=1e-12)


def _quantized(w, fmt, group):
    """The f64 values a frozen weight holds after quantization."""
    n, k = w.shape
    s = _scales(w, fmt, group)
    if fmt.startswith("int"):
        qmax = 7 if fmt == "int4" else 127
        t = (w.view(n, k // group, group) / s[..., None]).double()
        q = torch.clamp(torch.sign(t) * torch.floor(t.abs() + 0.5), -qmax, qmax)
        return (q * s[..., None].double()).view(n, k)
    return (w / s).to(torch.float8_e4m3fn).double() * s.double()


def _exact_load(c, seed):
    """The scales as the blocked layout holds them: [n/64][k/group][64] and
    its transpose's [k/group][n]; the packed bytes have no 64-bit value."""
    w = _raw(c, seed)["w"]
    fmt, group = c["fmt"], c["group"]
    if fmt in ("fp8", "fp8_scalar"):
        return {"data": None, "scales": _scales(w, fmt, group).double().view(-1)}
    if fmt.endswith("_to_int4"):
        f8 = fmt[:-len("_to_int4")]
        s8 = _scales(w, f8, group)
        w, fmt = (w / s8).to(torch.float8_e4m3fn).float() * s8, "int4"
    n, k = w.shape
    NB, KB = -(-n // 64), -(-k // 64)
    s = torch.zeros(NB * 64, max(KB * 64 // group, -(-KB * 64 // group)), dtype=torch.float64, device=DEV)
    s[:n, :k // group] = _scales(w, fmt, group).double()
    rows = s[:, :KB * 64 // group].view(NB, 64, -1).transpose(1, 2).reshape(-1)
    return {"data": None, "scales": torch.cat([rows, s.t().reshape(-1)])}


def _norm(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5)


def _rope64(L, hd):
    inv = 10000.0 ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd)
    ang = torch.arange(L, dtype=torch.float64, device=DEV)[:, None] * inv[None]
    return torch.cos(ang)[:, None], torch.sin(ang)[:, None]


def _qkv(txt, img, heads, rope):
    """q, k, v [L, heads, head_dim]: per-head norm and rotation of q and k."""
    qkv = torch.cat([txt, img], 0)
    L, h = qkv.shape[0], qkv.shape[1] // 3
    q, k, v = (p.view(L, heads, h // heads) for p in qkv.split(h, 1))

    def turn(x):
        x = _norm(x)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * rope[0] - b * rope[1], a * rope[1] + b * rope[0]], -1).flatten(-2)

    return turn(q), turn(k), v


def _exact_glue(c, seed):
    ins, cot = _glue_raw(c, seed)
    i = {k: v.double().requires_grad_() for k, v in ins.items()}
    rope = _rope64(c["img"] + c["txt"], c["h"] // c["heads"])
    outs = [(i["scale"] + 1) * _norm(i["x"]) + i["shift"]]
    outs += _qkv(i["qkv_txt"], i["qkv_img"], c["heads"], rope)
    outs += [i["x"] + i["gate"] * i["o"], F.gelu(i["u"], approximate="tanh")]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, list(i.values()), [g.double() for g in cot]))


def _exact_step(c, seed):
    cfg, bases, factors, plain, (img, txt, t, target) = _step_raw(c, seed)
    W = {p: _quantized(w, "int4", cfg.group) for p, w in bases.items()}
    AB = {p: [f.double().requires_grad_() for f in ab] for p, ab in factors.items()}
    P = {name: [v.double() for v in wb] for name, wb in plain.items()}

    def at(p, x):
        return x @ W[p].t() + (x @ AB[p][0]) @ AB[p][1]

    lin = lambda x, wb: F.linear(x, wb[0], wb[1])  # noqa: E731
    half = cfg.tdim // 2
    freqs = torch.exp(-math.log(10000.0) * torch.arange(half, dtype=torch.float64, device=DEV) / half)
    e = (t.double() * 1000.0)[:, None] * freqs[None]
    e = torch.cat([torch.cos(e), torch.sin(e)], -1)
    vec = lin(F.silu(lin(e, P["t_in"])), P["t_out"])
    xs = {"img": lin(img.double(), P["img_in"]), "txt": lin(txt.double(), P["txt_in"])}
    L, heads = c["img"] + c["txt"], c["heads"]
    cvec, mods, qkv = F.silu(vec), {}, {}
    for s in ("txt", "img"):
        mods[s] = at(f"blocks.0.{s}.mod", cvec).chunk(6, -1)
        qkv[s] = at(f"blocks.0.{s}.qkv", (mods[s][1] + 1) * _norm(xs[s]) + mods[s][0])
    q, k, v = _qkv(qkv["txt"], qkv["img"], heads, _rope64(L, c["h"] // heads))
    heads_out = []
    for j in range(heads):
        p = torch.softmax(q[:, j] @ k[:, j].t() / math.sqrt(c["h"] // heads), -1)
        heads_out.append(p @ v[:, j])
    o = torch.cat(heads_out, 1)
    s, oo = "img", o[c["txt"]:]  # the text stream's own output feeds no loss
    _, _, g1, sh2, sc2, g2 = mods[s]
    x = xs[s] + g1 * at(f"blocks.0.{s}.out", oo)
    up = at(f"blocks.0.{s}.up", (sc2 + 1) * _norm(x) + sh2)
    x = x + g2 * at(f"blocks.0.{s}.down", F.gelu(up, approximate="tanh"))
    scale, shift = lin(F.silu(vec), P["final_mod"]).chunk(2, -1)
    pred = lin((scale + 1) * _norm(x) + shift, P["final"])
    loss = (pred - target.double()).square().mean()
    order = [f for p in cfg.site_paths() for f in AB[p]]
    grads = torch.autograd.grad(loss, order, allow_unused=True)
    # a factor that feeds no loss has a zero gradient
    return {"loss": float(loss), "grads": [torch.zeros_like(f) if g is None else g for f, g in zip(order, grads)]}


def exact(case, seed):
    c = case
    if c["kind"] == "load":
        return _exact_load(c, seed)
    if c["kind"] == "glue":
        return _exact_glue(c, seed)
    if c["kind"] == "step":
        return _exact_step(c, seed)
    d = _raw(c, seed)
    W = _quantized(d["w"], c["fmt"], c["group"])
    x = d["x"].double()
    y = x @ W.t()
    if c["r"]:
        a, b = d["a"].double(), d["b"].double()
        t = x @ a
        y = y + t @ b
    else:
        y = y + d["bias"].double()
    if c["kind"] == "fwd":
        return y, t
    dy = d["dy"].double()
    dx = dy @ W
    if c["kind"] == "base":
        return y, dx
    u = dy @ b.t()
    grads = (dx + u @ a.t(), x.t() @ u, t.t() @ dy)
    return ((y, t) if c["kind"] == "layer" else (y,)) + grads
