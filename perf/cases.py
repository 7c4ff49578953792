"""The work that a user of this package has it do, as cases that can be timed and compared.

Six kinds of call, each through the package's public entry points:

* ``block``    one training step of the FP8 MLP sub-block: forward and backward
               through ``fp8_mlp_block``, then the post-step hook
               ``fp8_update_scales`` (scale roll, re-quantization of the masters)
* ``norm``     forward and backward of ``_NormSwiGLU``, the bf16 sub-block that
               runs when FP8 is off
* ``experts``  one training step of the FP8 experts: ``_FP8Experts`` forward and
               backward, then the post-step hook
* ``grouped``  forward and backward of the bf16 experts' ``_FusedSwiGLU``
* ``mlp``      ``MLP.forward`` of bf16 weights without gradients: generation
               (a few tokens) and evaluation (a prompt or a batch of them)
* ``quant``    the standalone row / column quantizer ``ops.quant_e4m3_rowcol``
"""
import math

import torch

import spark_gpt_amd as sg

EPS = 1e-6
E4M3_MAX, E5M2_MAX = 448.0, 57344.0
LARGEST = 18.0 * 65536 * 1024 * 3072  # flops of the largest listed case


def listed():
    return [
        # generation, eight sequences at once: one token each through a 0.6B-width MLP
        {"name": "mlp_decode", "kind": "mlp", "T": 8, "D": 1024, "I": 3072},
        # evaluation of one prompt of uneven length
        {"name": "mlp_prefill", "kind": "mlp", "T": 2017, "D": 1024, "I": 3072},
        # the muP base width, the smallest that is trained: launches and host time count
        {"name": "block_base", "kind": "block", "T": 8192, "D": 256, "I": 1024},
        # a short, ragged micro-batch at the 0.6B width
        {"name": "block_ragged", "kind": "block", "T": 5003, "D": 1024, "I": 3072},
        # a layer of the 50M model at its batch
        {"name": "block_50m", "kind": "block", "T": 49152, "D": 512, "I": 1536},
        # a layer of the 0.6B model at the benchmark's batch
        {"name": "block_0.6b", "kind": "block", "T": 65536, "D": 1024, "I": 3072},
        # a wide layer at the stack benchmark's batch
        {"name": "block_wide", "kind": "block", "T": 16384, "D": 2048, "I": 6144},
        # the 50M layer without FP8 (the default path)
        {"name": "norm_50m", "kind": "norm", "T": 49152, "D": 512, "I": 1536},
        # a small ragged batch at a width that is no power of two
        {"name": "norm_ragged", "kind": "norm", "T": 4099, "D": 768, "I": 2048},
        # the benchmark's experts: top-2 of 8 at half the dense ffn
        {"name": "experts_8x2", "kind": "experts", "T": 65536, "D": 1024, "I": 1536, "E": 8, "k": 2},
        # the 50M model's width with bf16 experts, a micro-batch
        {"name": "grouped_8x2", "kind": "grouped", "T": 8192, "D": 512, "I": 768, "E": 8, "k": 2},
        # the quantizer benchmark: a 65536 x 4096 activation
        {"name": "quant_64k", "kind": "quant", "T": 65536, "D": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "norm", "norm", "experts", "grouped", "mlp", "mlp", "quant"])
    if kind == "quant":
        return {"kind": kind, "T": _log(rng, 512, 65536), "D": 128 * rng.randint(2, 32)}
    if kind == "mlp":
        D = 64 * rng.randint(4, 32)
        return {"kind": kind, "T": _log(rng, 1, 4096), "D": D, "I": 64 * rng.randint(2 * D // 64, 4 * D // 64)}
    E = rng.choice([4, 8, 16]) if kind in ("experts", "grouped") else 0
    k = rng.choice([1, 2]) if E else 1
    if kind in ("block", "experts"):  # the FP8 recipe's widths are powers of two
        D = rng.choice([256, 512, 1024] if E else [256, 512, 1024, 2048])
        I = 128 * rng.randint(D // 128, (2 if E else 4) * D // 128)
    else:
        D = 64 * rng.randint(4, 16)
        I = 64 * rng.randint(D // 64, (2 if E else 4) * D // 64)
    most = min(65536, int(LARGEST / (18.0 * D * I * k)))
    case = {"kind": kind, "T": _log(rng, 1024, most), "D": D, "I": I}
    if E:
        case.update(E=E, k=k)
    return case


# ------------------------------------------------------------------ inputs
def _pow2(v):
    return 2.0 ** math.floor(math.log2(v))


def _scales(case):
    """The five delayed scales (x, gu, h, d_gu, dy) that a run with these
    distributions settles at: a binade below the format's range over the
    largest of T * D or T * I normal values."""
    D, I = case["D"], case["I"]
    d = 1e-3 * math.sqrt(D / I)
    return [_pow2(E4M3_MAX / 2 / 6.5), _pow2(E4M3_MAX / 2 / 6.5), _pow2(E4M3_MAX / 2 / 22.0),
            _pow2(E5M2_MAX / 2 / (22.0 * d)), _pow2(E5M2_MAX / 2 / 6.5e-3)]


def _inputs(case, seed):
    """Activations N(0, 1), weights N(0, 1 / fan_in), upstream gradients
    N(0, 1e-3), a norm weight near one and, for experts, random routing."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, device=dev, generator=gen).mul_(std)

    kind, T, D = case["kind"], case["T"], case["D"]
    v = {"x": normal(T, D).to(torch.bfloat16)}
    if kind == "quant":  # a few outlier columns, as activations have them
        v["x"][:, torch.randperm(D, device=dev, generator=gen)[:max(1, D // 1024)]] *= 50
        return v
    I, E = case["I"], case.get("E", 0)
    lead = (E,) if E else ()
    v["w_gu"] = normal(*lead, 2 * I, D, std=D ** -0.5)
    if kind in ("block", "experts", "mlp"):
        v["w_down"] = normal(*lead, D, I, std=I ** -0.5)
    if kind in ("block", "norm"):
        v["norm_w"] = 1.0 + normal(D, std=0.1)
    if E:
        k = case["k"]
        chosen = torch.rand(T, E, device=dev, generator=gen).topk(k, dim=-1).indices
        experts, perm = torch.sort(chosen.reshape(-1), stable=True)
        v["token_index"] = perm // k
        v["inverse"] = torch.empty_like(perm)
        v["inverse"][perm] = torch.arange(perm.numel(), device=dev)
        v["offsets"] = torch.cumsum(torch.bincount(experts, minlength=E), 0, dtype=torch.int32)
    rows = T * case.get("k", 1)
    if kind != "mlp":
        v["dy"] = normal(rows, D if kind in ("block", "experts") else I, std=1e-3).to(torch.bfloat16)
    if kind == "grouped":  # bf16 weights, and the rows in the experts' order
        v["w_gu"] = v["w_gu"].to(torch.bfloat16)
        v["x"] = v["x"][v["token_index"]]
    return v


class _Norm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight, self.eps = torch.nn.Parameter(weight), EPS


class _Experts(torch.nn.Module):
    """The state that FP8 experts read: packed masters, scales and maxima."""

    def __init__(self, w_gu, w_down, scale):
        super().__init__()
        self.gate_up_proj, self.down_proj = torch.nn.Parameter(w_gu), torch.nn.Parameter(w_down)
        self.register_buffer("fp8_scale", scale, persistent=False)
        self.register_buffer("fp8_amax", torch.zeros_like(scale), persistent=False)


def prepare(case, seed):
    v, kind = _inputs(case, seed), case["kind"]
    v["kind"], v["k"] = kind, case.get("k", 1)
    if kind in ("block", "mlp"):
        with torch.device("meta"):
            mlp = sg.MLP(case["D"], case["I"])
        mlp.to_empty(device="cuda")
        with torch.no_grad():
            mlp.gate_up_proj.weight.copy_(v.pop("w_gu"))
            mlp.down_proj.weight.copy_(v.pop("w_down"))
            mlp.fp8_scale.copy_(torch.tensor(_scales(case)))
            mlp.fp8_amax.zero_()
        v["mlp"] = mlp.train() if kind == "block" else mlp.to(torch.bfloat16).eval()
    if kind == "block":
        v["norm"] = _Norm(v.pop("norm_w"))
    if kind == "experts":
        v["experts"] = _Experts(v.pop("w_gu"), v.pop("w_down"), torch.tensor(_scales(case), device="cuda"))
    for name in ("w_gu", "norm_w"):
        if name in v:
            v[name].requires_grad_(True)
    if kind != "mlp":
        v["x"].requires_grad_(kind != "quant")
    if kind == "quant":
        v["scale"] = torch.tensor([_pow2(E4M3_MAX / 2 / 300.0)], device="cuda")
        v["amax"] = torch.zeros(1, device="cuda")
    return v


# ------------------------------------------------------------------ one pass
def run(s):
    kind, x = s["kind"], s["x"]
    if kind == "mlp":
        with torch.no_grad():
            return {"y": s["mlp"](x)}
    if kind == "quant":
        x8, x8t = sg.ops.quant_e4m3_rowcol(x, s["scale"], s["amax"])
        return {"x8": x8.view(torch.uint8), "x8t": x8t.view(torch.uint8), "amax": s["amax"]}
    if kind == "norm":
        y = sg._NormSwiGLU.apply(x, s["norm_w"], s["w_gu"], EPS)
        wrt = [x, s["norm_w"], s["w_gu"]]
    elif kind == "grouped":
        y = sg._FusedSwiGLU.apply(x, s["w_gu"], s["offsets"])
        wrt = [x, s["w_gu"]]
    elif kind == "block":
        y = sg.fp8_mlp_block(x, s["norm"], s["mlp"])
        wrt = [x, s["norm"].weight, s["mlp"].gate_up_proj.weight, s["mlp"].down_proj.weight]
    else:
        m = s["experts"]
        y = sg._FP8Experts.apply(x, m.gate_up_proj, m.down_proj, s["token_index"], s["inverse"], s["offsets"], s["k"],
                                 m.fp8_scale, m.fp8_amax)
        wrt = [x, m.gate_up_proj, m.down_proj]
    grads = torch.autograd.grad(y, wrt, s["dy"])
    out = {"y": y.detach(), "grads": list(grads)}
    if kind in ("block", "experts"):
        module = s["mlp"] if kind == "block" else s["experts"]
        sg.fp8_update_scales(module)
        out["scale"] = module.fp8_scale
    return out


# ------------------------------------------------------------------ what a pass needs
def work(case):
    kind, T, D = case["kind"], case["T"], case["D"]
    if kind == "quant":
        return {"bytes": 4.0 * T * D, "flops": 0.0}
    I, E, R = case["I"], max(1, case.get("E", 0)), T * case.get("k", 1)
    W = 3.0 * E * D * I  # elements of gate, up and down
    if kind == "mlp":  # x, y and the bf16 weights
        return {"bytes": 4.0 * T * D + 2 * W, "flops": 6.0 * T * D * I}
    if kind == "norm":  # h, dh; out, dout; fp32 gate/up master and gradient
        return {"bytes": 4.0 * T * D + 4.0 * T * I + 16.0 * D * I, "flops": 12.0 * T * D * I}
    if kind == "grouped":  # x, dx; h, dh; bf16 gate/up weights and gradient
        return {"bytes": 4.0 * R * D + 4.0 * R * I + 8.0 * E * D * I, "flops": 12.0 * R * D * I}
    # x, dx; y, dy; fp32 masters and gradients
    return {"bytes": 4.0 * T * D + 4.0 * R * D + 8 * W, "flops": 18.0 * R * D * I}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":
        return "exact"
    if kind in ("block", "experts"):
        # an fp8 code that flips where a product's last bits differ moves its value by up to a quarter
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------ the same in 64 bits
def _f8(v, scale, dtype=torch.float8_e4m3fn):
    """v as its fp8 storage at a power-of-two scale keeps it, in 64 bits."""
    top = E4M3_MAX if dtype == torch.float8_e4m3fn else E5M2_MAX
    return (v * scale).clamp(-top, top).float().to(dtype).double() / scale


def _w8(w):
    return _f8(w.double(), _pow2(E4M3_MAX / float(w.abs().max())))


def _silu_grad(g):
    sig = torch.sigmoid(g)
    return sig * (1 + g * (1 - sig))


def _fp8_mlp(n, w_gu, w_down, dy, s):
    """(out, dn, dW_gu, dW_down) of the FP8 recipe: its fp8 storage, all else in 64 bits."""
    e5 = torch.float8_e5m2
    x, wg = _f8(n, s[0]), _w8(w_gu)
    g, u = (x @ wg.t()).chunk(2, dim=-1)
    h = _f8(g * torch.sigmoid(g) * u, s[2])
    out = h @ _w8(w_down).t()
    g, u = _f8(g, s[1]), _f8(u, s[1])
    dh = dy @ w_down.to(torch.bfloat16).double()
    d = _f8(torch.cat([dh * u * _silu_grad(g), dh * g * torch.sigmoid(g)], 1), s[3], e5)
    return out, d @ wg, d.t() @ x, _f8(dy, s[4], e5).t() @ h


def _bf16_swiglu(x, w, dy):
    """(out, dx, dW) of silu(x Wg^T) * (x Wu^T)."""
    g, u = (x @ w.t()).chunk(2, dim=-1)
    out = g * torch.sigmoid(g) * u
    d = torch.cat([dy * u * _silu_grad(g), dy * g * torch.sigmoid(g)], 1)
    return out, d @ w, d.t() @ x


def exact(case, seed):
    v, kind = _inputs(case, seed), case["kind"]
    x = v["x"].double()
    if kind == "quant":
        return None
    if kind == "mlp":
        g, u = (x @ v["w_gu"].to(torch.bfloat16).double().t()).chunk(2, dim=-1)
        return {"y": (g * torch.sigmoid(g) * u) @ v["w_down"].to(torch.bfloat16).double().t()}
    dy = v["dy"].double()
    if kind in ("block", "norm"):
        r = torch.rsqrt(x.square().mean(1, keepdim=True) + EPS)
        w = v["norm_w"].double()
        if kind == "block":
            y, dn, dwgu, dwd = _fp8_mlp(x * r * w, v["w_gu"], v["w_down"], dy, _scales(case))
        else:
            y, dn, dwgu = _bf16_swiglu(x * r * w, v["w_gu"].double(), dy)
        dx = dn * w * r - x * r ** 3 * (dn * w * x).mean(1, keepdim=True)
        dw = (dn * x * r).sum(0)
        if kind == "norm":
            return {"y": y, "grads": [dx, dw, dwgu]}
        return {"y": x + y, "grads": [dx + dy, dw, dwgu, dwd], "scale": None}
    ends = [0] + v["offsets"].tolist()
    parts = []
    for e, (a, b) in enumerate(zip(ends, ends[1:])):
        if kind == "grouped":
            parts.append(_bf16_swiglu(x[a:b], v["w_gu"][e].double(), dy[a:b]))
        else:
            parts.append(_fp8_mlp(x[v["token_index"][a:b]], v["w_gu"][e], v["w_down"][e], dy[a:b], _scales(case)))
    y, dx = (torch.cat([p[i] for p in parts]) for i in (0, 1))
    dws = [torch.stack([p[i] for p in parts]) for i in range(2, len(parts[0]))]
    if kind == "grouped":
        return {"y": y, "grads": [dx] + dws}
    dx = dx[v["inverse"]].view(case["T"], case["k"], -1).sum(1)
    return {"y": y, "grads": [dx] + dws, "scale": None}
