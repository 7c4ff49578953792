"""Benchmark: FP8 SwiGLU MLP block fwd+bwd on one MI355X.

Workload (default): tokens=65536, d_model=1024, ffn=3072 (Qwen3-0.6B width),
bf16 inputs ~N(0,1), weights ~N(0,1/fan_in), upstream grads ~N(0,1e-3),
seed-fixed, after one prewarm step + scale roll.  A step is one training
step of the block: forward and backward through the 7-argument autograd
Function, then the post-step hook ``fp8_update_scales`` (the delayed-scale
roll and the once-per-optimizer-step re-quantization of the fp32 masters),
all on the current stream.  Value = 18*T*D*I FLOP / step time, in TFLOP/s.

Also reported on the same JSON line:
  kernels_in_step  per-kernel mean duration inside the step: a second pass of
                the same steps with HIP events recorded on the launch stream
                around every C-ABI launch
  roofline      the kernel taking the most time per step (from that pass):
                algorithmic FLOP (or bytes) per launch / mean in-step duration
                vs the dense MFMA peak of its input type (or HBM); `traffic` =
                HBM bytes per launch from the committed rocprofv3 FETCH_SIZE /
                WRITE_SIZE summary
                (profiles/traffic_fwd_bwd_T65536_D1024_I3072.md), null for
                other workloads
  quantizer     the standalone quantizer (bf16 65536x4096 with 0.1% x50 outlier
                columns -> e4m3 row-major + transposed + amax): 4 B/element
                algorithmic traffic / mean duration vs 8 TB/s HBM
  kernels       per-kernel mean durations (each kernel alone, 10 launches),
                with TFLOP/s or algorithmic GB/s
  other_workloads  on the GPU, wall clock after warm-up steps: the muP base
                block (T=8192, D=256, I=1024); the wide block with
                heavy-tailed activations (T=65536, D=2048, I=6144, Student-t
                with 3 degrees of freedom); the stack of 28 blocks (T=16384,
                D=4096, I=12288, each block's RMSNorm between layers, full
                forward + backward in one step); the FP8 MoE experts
                (``_FP8Experts`` fwd+bwd + post-step hook) on 65536 tokens
                routed top-2 over 8 experts, D=1024, I=1536 (131072 expert
                rows: the dense headline's FLOP); and the reference's default
                bf16 sub-block at the headline shape (h +
                down_proj(_NormSwiGLU(h)) under bf16 autocast, the down
                projection on torch).  All but the muP base block carry their
                in-step kernels and the roofline of the dominant one (the
                MoE and bf16 `traffic` from their committed counter
                summaries); `fp8_block_speedup` = bf16 step / FP8 step
  cpu_baseline  the same FP8 recipe emulated in torch on the host cores (the
                CPU oracle) at the headline's full 65536 tokens, in TFLOP/s;
                under `other_workloads` the oracle on the muP base block and
                on the full 65536 x 4096 quantizer input, and on a token
                sample of the MoE workload

``--trace`` runs only the headline steps (prewarm, warm-up, timed and
instrumented passes), so that a ``rocprofv3 --kernel-trace --stats`` summary
of it averages in-step launches of the headline shape only; ``--trace moe``
and ``--trace bf16`` do the same for the MoE and the bf16 workloads.

``--probe`` runs, instead of the benchmark, one calibration copy (fp32 negate
of 256 Mi elements: 1 GiB read + 1 GiB written) and then every kernel of the
step once, for ``rocprofv3 --pmc FETCH_SIZE`` / ``--pmc WRITE_SIZE`` passes.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

FP8_PEAK_TFLOPS = 5033.0   # MI355X dense FP8 MFMA (256 CU x 2.4 GHz x 8192 FLOP/clk)
BF16_PEAK_TFLOPS = 2516.5  # MI355X dense bf16 MFMA
HBM_PEAK_GBPS = 8000.0     # MI355X HBM3E
TRAFFIC_PROFILE = os.path.join(ROOT, "profiles", "traffic_fwd_bwd_T65536_D1024_I3072.md")
TRAFFIC_WORKLOAD = (65536, 1024, 3072)
# counter summaries of the MoE and bf16 workloads (the same table layout)
TRAFFIC_PROFILE_MOE = os.path.join(ROOT, "profiles", "traffic_moe_fwd_bwd_T65536_E8_top2_D1024_I1536.md")
TRAFFIC_PROFILE_BF16 = os.path.join(ROOT, "profiles", "traffic_bf16_norm_swiglu_fwd_bwd_T65536_D1024_I3072.md")
# the compute-matched MoE of the headline width: top-2 of 8 experts at half the
# dense ffn (the same 18*T*k*D*I FLOP per step as the dense block)
MOE_WORKLOAD = {"T": 65536, "D": 1024, "I": 1536, "E": 8, "k": 2}


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=20)
    p.add_argument("--warmup", type=int, default=5)
    p.add_argument("--tokens", type=int, default=65536)
    p.add_argument("--d-model", type=int, default=1024)
    p.add_argument("--ffn", type=int, default=3072)
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--cpu-tokens", type=int, default=65536)
    p.add_argument("--quant-rows", type=int, default=65536)
    p.add_argument("--quant-cols", type=int, default=4096)
    p.add_argument("--probe", action="store_true", help="one launch of each kernel, for counter passes")
    p.add_argument("--trace", nargs="?", const="dense", choices=("dense", "moe", "bf16"), default=None,
                   help="steps of one workload only (no standalone kernels, quantizer, other shapes or CPU "
                        "leg): the headline block (default), the MoE experts or the bf16 sub-block")
    p.add_argument("--dist", choices=("normal", "student-t"), default="normal",
                   help="activations: N(0,1), or Student-t with 3 degrees of freedom (heavy tails)")
    return p.parse_args()


def read_traffic(kernel: str, profile: str = TRAFFIC_PROFILE):
    """HBM bytes per launch of `kernel` from a committed counter summary: the
    table row `| kernel | ... | traffic_bytes |` (last column)."""
    try:
        with open(profile) as fh:
            for line in fh:
                cells = [c.strip() for c in line.strip().strip("|").split("|")]
                if len(cells) >= 2 and cells[0] == kernel:
                    return int(float(cells[-1]))
    except (OSError, ValueError):
        return None
    return None


def timed_launches(fn, reps: int, stream) -> float:
    """Mean ms per call of fn() over reps calls, HIP events on `stream`."""
    import torch

    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    fn()
    torch.cuda.synchronize()
    start.record(stream)
    for _ in range(reps):
        fn()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) / reps


def cpu_baseline(T: int, D: int, I: int) -> dict:
    """The reference recipe emulated on the host (CPU oracle), T tokens."""
    import torch

    from oracle import fp8_mlp as O

    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    g = torch.Generator().manual_seed(2)
    h = torch.randn(T, D, generator=g).to(torch.bfloat16)
    nw = torch.ones(D)
    wgu = torch.randn(2 * I, D, generator=g) * D ** -0.5
    wd = torch.randn(D, I, generator=g) * I ** -0.5
    dy = (torch.randn(T, D, generator=g) * 1e-3).to(torch.bfloat16)
    scale, amax = torch.ones(5), torch.zeros(5)

    def step():
        y, saved = O.block_forward(h, nw, wgu, wd, scale, amax, 1e-6)
        O.block_backward(dy, saved, scale, amax)

    step()
    O.update_scales(scale, amax)
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        step()
        times.append(time.perf_counter() - t0)
    med = sorted(times)[1]
    cpu_model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    cpu_model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {
        "value": round(18.0 * T * D * I / med / 1e12, 4),
        "unit": "TFLOP/s",
        "cores": torch.get_num_threads(),
        "kind": "port",
        "sample": f"torch-CPU emulation of the FP8 recipe (oracle), fwd+bwd at tokens={T}, "
                  f"d_model={D}, ffn={I}; median of 3 steps after 1 warm-up; {med:.2f} s/step; "
                  f"cpu={cpu_model}",
    }


def cpu_extra(quant_rows: int, quant_cols: int) -> dict:
    """The CPU oracle on the other measured workloads: the muP base block
    (T=8192, D=256, I=1024) and the standalone quantizer (65536 x 4096), both
    at full size, and the MoE experts on a token sample."""
    import torch

    from oracle import fp8_mlp as O

    out = {}
    T, D, I = 8192, 256, 1024
    g = torch.Generator().manual_seed(1)
    h = torch.randn(T, D, generator=g).to(torch.bfloat16)
    nw = torch.ones(D)
    wgu = torch.randn(2 * I, D, generator=g) * D ** -0.5
    wd = torch.randn(D, I, generator=g) * I ** -0.5
    dy = (torch.randn(T, D, generator=g) * 1e-3).to(torch.bfloat16)
    scale, amax = torch.ones(5), torch.zeros(5)

    def step():
        _, saved = O.block_forward(h, nw, wgu, wd, scale, amax, 1e-6)
        O.block_backward(dy, saved, scale, amax)

    step()
    O.update_scales(scale, amax)
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        step()
        times.append(time.perf_counter() - t0)
    med = sorted(times)[1]
    out["muP_base_T8192_D256_I1024"] = {"TFLOP/s": round(18.0 * T * D * I / med / 1e12, 4),
                                        "s_per_step": round(med, 4)}
    R = quant_rows
    x = torch.randn(R, quant_cols, generator=g)
    x[:, : max(1, quant_cols // 1000)] *= 50.0
    x = x.to(torch.bfloat16)
    s0 = torch.tensor(1.0)
    O.quant_rowcol(x, s0)
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        O.quant_rowcol(x, s0)
        times.append(time.perf_counter() - t0)
    med = sorted(times)[1]
    out["quantizer"] = {"GB/s": round(4.0 * R * quant_cols / med / 1e9, 2), "s_per_call": round(med, 4),
                        "sample": f"{R} x {quant_cols} rows of the quantizer input (4 B/elem)"}
    del x
    out["moe"] = cpu_moe(8192)
    return out


def cpu_moe(T: int) -> dict:
    """The CPU oracle's FP8 experts (fwd+bwd) on T tokens of the MoE workload
    (top-2 of 8 experts, D=1024, I=1536), median of 3 steps after a prewarm
    step and scale roll."""
    import torch

    from oracle import fp8_mlp as O
    from oracle import fp8_moe as OM

    mw = MOE_WORKLOAD
    D, I, E, k = mw["D"], mw["I"], mw["E"], mw["k"]
    g = torch.Generator().manual_seed(5)
    x = torch.randn(T, D, generator=g).to(torch.bfloat16)
    wgu = torch.randn(E, 2 * I, D, generator=g) * D ** -0.5
    wd = torch.randn(E, D, I, generator=g) * I ** -0.5
    selected = torch.rand(T, E, generator=g).topk(k, dim=-1).indices
    token_index, inverse_permutation, offsets, _ = OM.route(selected, E)
    dout = (torch.randn(T * k, D, generator=g) * 1e-3).to(torch.bfloat16)
    scale, amax = torch.ones(5), torch.zeros(5)

    def step():
        _, saved = OM.moe_forward(x, wgu, wd, token_index, offsets, scale, amax)
        OM.moe_backward(dout, saved, scale, amax, inverse_permutation, k)

    step()
    O.update_scales(scale, amax)
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        step()
        times.append(time.perf_counter() - t0)
    med = sorted(times)[1]
    flop = 18.0 * T * k * D * I
    return {"TFLOP/s": round(flop / med / 1e12, 4), "s_per_step": round(med, 4),
            "sample": f"{T} tokens top-{k} of {E} experts, d_model={D}, ffn={I}"}


class _Norm:
    """The RMSNorm parameters the block reads (weight, eps)."""

    def __init__(self, weight, eps=1e-6):
        self.weight, self.eps = weight, eps


def make_block(T: int, D: int, I: int, dist: str = "normal", seed: int = 1):
    """(h, dy, norm, mlp, step): synthetic inputs of the workload and one
    training step of the block (forward, backward, post-step hook)."""
    import torch

    import spark_gpt_amd as sg

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    if dist == "normal":
        h = torch.randn(T, D, device=dev, generator=g).to(torch.bfloat16)
    else:  # Student-t, 3 degrees of freedom: z / sqrt(chi2_3 / 3)
        z = torch.randn(T, D, device=dev, generator=g)
        chi = sum(torch.randn(T, D, device=dev, generator=g) ** 2 for _ in range(3))
        h = (z / torch.sqrt(chi / 3)).to(torch.bfloat16)
        del z, chi
    mlp = sg.MLP(D, I).to(dev).train()
    with torch.no_grad():
        mlp.gate_up_proj.weight.copy_(torch.randn(2 * I, D, device=dev, generator=g) * D ** -0.5)
        mlp.down_proj.weight.copy_(torch.randn(D, I, device=dev, generator=g) * I ** -0.5)
    norm = _Norm(torch.ones(D, device=dev, requires_grad=True))
    dy = (torch.randn(T, D, device=dev, generator=g) * 1e-3).to(torch.bfloat16)
    params = [norm.weight, mlp.gate_up_proj.weight, mlp.down_proj.weight]

    def step():
        x = h.detach().requires_grad_(True)
        y = sg.fp8_mlp_block(x, norm, mlp)
        torch.autograd.backward(y, dy, inputs=[x] + params)
        for p in params:
            p.grad = None
        # post-step hook (train.py:4049-4050): scale roll + weight re-quantization
        sg.fp8_update_scales(mlp)

    return h, dy, norm, mlp, step


def block_work(T: int, D: int, I: int) -> dict:
    """FLOP (or algorithmic bytes) per launch of each kernel of one block."""
    return {
        "norm_quant": (None, T * (3.0 * D + 4)),
        # the post-step hook: scale roll + both weight quantizations (fp32
        # masters read twice, e4m3 copies, W_gu^T e4m3, W_down^T bf16)
        "post_step_quant": (None, 10.0 * 2 * I * D + 11.0 * D * I + 40.0),
        "gateup_swiglu_fwd": (4.0 * T * D * I, None),
        "down_fwd": (2.0 * T * D * I, None),
        "down_dgrad_swiglu_bf16": (2.0 * T * D * I, None),
        "gateup_dgrad": (4.0 * T * D * I, None),
        "norm_bwd": (None, T * (9.0 * D + 4)),
        "wgrad_down": (2.0 * T * D * I, None),
        "wgrad_gateup": (4.0 * T * D * I, None),
    }


def timed_steps(step, steps: int, warmup: int) -> float:
    """Wall-clock ms per step over `steps` steps after `warmup` untimed ones,
    bracketed by device synchronisations."""
    import torch

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) * 1e3 / steps


def time_block(T: int, D: int, I: int, steps: int, warmup: int, dist: str = "normal", trace: bool = False,
               workload: str = "fp8_swiglu_mlp_block_fwd_bwd") -> dict:
    """GPU training-step time of the block at another shape (prewarm step and
    scale roll first, as for the headline workload); with `trace`, also its
    in-step kernels and the roofline of the dominant one."""
    import torch

    _h, _dy, _norm, _mlp, step = make_block(T, D, I, dist)
    step()
    ms = timed_steps(step, steps, warmup)
    flop = 18.0 * T * D * I
    out = {"workload": workload, "tokens": T, "d_model": D, "ffn": I, "activations": dist,
           "flop_per_step": flop, "ms_per_step": round(ms, 4),
           "TFLOP/s": round(flop / (ms * 1e-3) / 1e12, 2),
           "frac_fp8_peak": round(flop / (ms * 1e-3) / 1e12 / FP8_PEAK_TFLOPS, 4)}
    if trace:
        per = trace_steps(step, steps, torch.cuda.current_stream(), lambda sym, a: launch_name(sym, a, D, I))
        out["kernels_in_step"], out["roofline"] = in_step_summary(per, steps, block_work(T, D, I))
    return out


def time_stack(T: int, D: int, I: int, L: int, steps: int, warmup: int) -> dict:
    """A stack of L blocks, each with its own RMSNorm (y = h + MLP(norm(h)),
    chained), full forward + backward in one step, then the post-step hook on
    every block; in-step kernels averaged over the layers."""
    import torch

    import spark_gpt_amd as sg

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(7)
    layers = []
    for _ in range(L):
        mlp = sg.MLP(D, I).to(dev).train()
        with torch.no_grad():
            mlp.gate_up_proj.weight.copy_(torch.randn(2 * I, D, device=dev, generator=g) * D ** -0.5)
            mlp.down_proj.weight.copy_(torch.randn(D, I, device=dev, generator=g) * I ** -0.5)
        layers.append((_Norm(torch.ones(D, device=dev, requires_grad=True)), mlp))
    h = torch.randn(T, D, device=dev, generator=g).to(torch.bfloat16)
    dy = (torch.randn(T, D, device=dev, generator=g) * 1e-3).to(torch.bfloat16)
    params = [p for norm, mlp in layers for p in (norm.weight, mlp.gate_up_proj.weight, mlp.down_proj.weight)]

    def step():
        x = h.detach().requires_grad_(True)
        y = x
        for norm, mlp in layers:
            y = sg.fp8_mlp_block(y, norm, mlp)
        torch.autograd.backward(y, dy, inputs=[x] + params)
        for p in params:
            p.grad = None
        for _, mlp in layers:
            sg.fp8_update_scales(mlp)

    step()
    ms = timed_steps(step, steps, warmup)
    flop = 18.0 * T * D * I * L
    per = trace_steps(step, steps, torch.cuda.current_stream(), lambda sym, a: launch_name(sym, a, D, I))
    in_step, roofline = in_step_summary(per, steps, block_work(T, D, I))
    return {"workload": f"fp8_swiglu_mlp_stack{L}_fwd_bwd", "layers": L, "tokens": T, "d_model": D, "ffn": I,
            "flop_per_step": flop, "ms_per_step": round(ms, 3), "TFLOP/s": round(flop / (ms * 1e-3) / 1e12, 2),
            "frac_fp8_peak": round(flop / (ms * 1e-3) / 1e12 / FP8_PEAK_TFLOPS, 4),
            "roofline": roofline, "kernels_in_step": in_step}


def launch_name(sym: str, a, D: int, I: int) -> str:
    """Kernel name of a launch: a C-ABI symbol, or an ``ops`` wrapper, and its
    positional arguments."""
    if sym == "wgrad_rows":
        return "wgrad_down" if a[2] == D else "wgrad_gateup"
    if sym == "weight_quant_experts":
        return "weight_quant_gu" if a[0].shape[1] == 2 * I else "weight_quant_down"
    if sym == "moe_wgrad_rows":
        return "moe_wgrad_down" if a[2] == D else "moe_wgrad_gateup"
    if sym == "moe_rows_quant":
        return "moe_gather_quant_x" if a[8] == 0 else "moe_quant_dout"
    return {"down_dgrad_swiglu": "down_dgrad_swiglu_bf16", "sfp8_update_scales": "update_scales",
            "block_weight_quant": "post_step_quant", "moe_down_dgrad_swiglu": "moe_down_dgrad_swiglu_bf16"}.get(sym, sym)


def rates(work: dict, name: str, ms: float) -> dict:
    """Mean duration of a kernel with its TFLOP/s or algorithmic GB/s."""
    fl, by = work.get(name, (None, None))
    rec = {"ms": round(ms, 4)}
    if fl:
        rec["tflops"] = round(fl / (ms * 1e-3) / 1e12, 1)
    if by:
        rec["GB/s"] = round(by / (ms * 1e-3) / 1e9, 1)
    return rec


def trace_steps(step, steps: int, stream, namer) -> dict:
    """`steps` more steps with HIP events recorded on `stream` around every
    native wrapper's and every C-ABI launch: {kernel name: [ms per launch, ...]}."""
    import torch

    from spark_gpt_amd import _lib, ops

    marks = []

    def traced(fn, name=None):
        def call(*a, **kw):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            out = fn(*a, **kw)
            e1.record(stream)
            marks.append((namer(name, a) if name else namer(a[0], a[1:]), e0, e1))
            return out

        return call

    plain = {n: getattr(ops, n) for n in ops._NATIVE}
    plain_call = _lib.call
    _lib.call = traced(plain_call)
    for n, fn in plain.items():
        setattr(ops, n, traced(fn, n))
    try:
        for _ in range(steps):
            step()
        torch.cuda.synchronize()
    finally:
        _lib.call = plain_call
        for n, fn in plain.items():
            setattr(ops, n, fn)
    per = {}
    for name, e0, e1 in marks:
        per.setdefault(name, []).append(e0.elapsed_time(e1))
    return per


def in_step_summary(per: dict, steps: int, work: dict, traffic_of=lambda k: None):
    """(per-kernel in-step means, roofline of the kernel taking the most time
    per step): algorithmic FLOP (or bytes) per launch / mean in-step duration
    vs the dense MFMA peak of its input type (or HBM)."""
    in_step = {n: dict(rates(work, n, sum(v) / len(v)), launches_per_step=len(v) / steps) for n, v in per.items()}
    dom = max(in_step, key=lambda n: in_step[n]["ms"] * in_step[n]["launches_per_step"])
    dom_ms = in_step[dom]["ms"]
    dom_flop, dom_bytes = work[dom]
    if dom_flop:
        achieved = dom_flop / (dom_ms * 1e-3) / 1e12
        peak = BF16_PEAK_TFLOPS if "bf16" in dom else FP8_PEAK_TFLOPS
        roofline = {"bound": "mfma", "kernel": dom, "achieved": round(achieved, 1), "peak": peak,
                    "unit": "TFLOP/s", "frac": round(achieved / peak, 4), "traffic": traffic_of(dom),
                    "flop_per_launch": dom_flop, "launches_timed": len(per[dom]), "ms_per_launch": round(dom_ms, 4)}
    else:
        achieved = dom_bytes / (dom_ms * 1e-3) / 1e9
        roofline = {"bound": "hbm", "kernel": dom, "achieved": round(achieved, 1), "peak": HBM_PEAK_GBPS,
                    "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBPS, 4), "traffic": traffic_of(dom),
                    "bytes_per_launch": dom_bytes, "launches_timed": len(per[dom]), "ms_per_launch": round(dom_ms, 4)}
    return in_step, roofline


def make_moe(T: int, D: int, I: int, E: int, k: int, seed: int = 4):
    """(step, rows per expert): one training step of the FP8 experts
    (``_FP8Experts`` forward and backward, then the post-step hook) on T
    tokens routed to k distinct experts each (random router logits, the
    expert-order bookkeeping of train.py:2268-2290), seed-fixed."""
    import torch

    import spark_gpt_amd as sg

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)

    class _ExpertWeights(torch.nn.Module):
        """The state the experts read: packed fp32 masters and the 5-slot
        scale / amax buffers (train.py:2252-2260)."""

        def __init__(self):
            super().__init__()
            self.gate_up_proj = torch.nn.Parameter(torch.randn(E, 2 * I, D, device=dev, generator=g) * D ** -0.5)
            self.down_proj = torch.nn.Parameter(torch.randn(E, D, I, device=dev, generator=g) * I ** -0.5)
            self.register_buffer("fp8_scale", torch.ones(5, device=dev), persistent=False)
            self.register_buffer("fp8_amax", torch.zeros(5, device=dev), persistent=False)

    m = _ExpertWeights().train()
    x = torch.randn(T, D, device=dev, generator=g).to(torch.bfloat16)
    selected = torch.rand(T, E, device=dev, generator=g).topk(k, dim=-1).indices
    sorted_experts, permutation = torch.sort(selected.reshape(-1))
    token_index = permutation // k
    inverse_permutation = torch.empty_like(permutation)
    inverse_permutation[permutation] = torch.arange(permutation.numel(), device=dev)
    counts = torch.bincount(sorted_experts, minlength=E)
    offsets = torch.cumsum(counts, dim=0, dtype=torch.int32)
    dout = (torch.randn(T * k, D, device=dev, generator=g) * 1e-3).to(torch.bfloat16)
    params = [m.gate_up_proj, m.down_proj]

    def step():
        xx = x.detach().requires_grad_(True)
        out = sg._FP8Experts.apply(xx, m.gate_up_proj, m.down_proj, token_index, inverse_permutation, offsets, k,
                                   m.fp8_scale, m.fp8_amax)
        torch.autograd.backward(out, dout, inputs=[xx] + params)
        for p in params:
            p.grad = None
        sg.fp8_update_scales(m)

    return step, counts.tolist()


def bf16_launch_name(sym: str, a) -> str:
    """Kernel name of a launch of the bf16 SwiGLU path."""
    return {"bf16_weight_slabs": "bf16_weight_fold", "bf16_swiglu_fwd": "bf16_gateup_swiglu_fwd",
            "bf16_swiglu_bwd": "bf16_swiglu_bwd_rows", "bf16_gemm": "bf16_gateup_dgrad",
            "bf16_norm_dh": "bf16_norm_bwd", "bf16_wgrad_rows": "bf16_wgrad_gateup"}.get(sym, sym)


def time_bf16(T: int, D: int, I: int, steps: int, warmup: int) -> dict:
    """The reference's default (bf16) dense MLP sub-block at the same shape:
    y = h + down_proj(_NormSwiGLU(h, norm_w, w_gu, eps)) under bf16 autocast
    (train.py:2366-2369), forward + backward; _NormSwiGLU on the HIP
    kernels of libsparkfp8, the down projection on torch (hipBLASLt).  18*T*D*I FLOP per
    step, 12*T*D*I of them in _NormSwiGLU."""
    import torch

    import spark_gpt_amd as sg

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(6)
    h = torch.randn(T, D, device=dev, generator=g).to(torch.bfloat16)
    dy = (torch.randn(T, D, device=dev, generator=g) * 1e-3).to(torch.bfloat16)
    mlp = sg.MLP(D, I).to(dev).train()
    with torch.no_grad():
        mlp.gate_up_proj.weight.copy_(torch.randn(2 * I, D, device=dev, generator=g) * D ** -0.5)
        mlp.down_proj.weight.copy_(torch.randn(D, I, device=dev, generator=g) * I ** -0.5)
    norm_w = torch.ones(D, device=dev, requires_grad=True)
    params = [norm_w, mlp.gate_up_proj.weight, mlp.down_proj.weight]

    def step():
        x = h.detach().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = x + mlp.down_proj(sg._NormSwiGLU.apply(x, norm_w, mlp.gate_up_proj.weight, 1e-6))
        torch.autograd.backward(y, dy, inputs=[x] + params)
        for p in params:
            p.grad = None

    stream = torch.cuda.current_stream()
    for _ in range(warmup + 1):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    work = {
        "bf16_weight_fold": (None, 16.0 * I * D),
        "bf16_rows_prep": (None, 4.0 * T * D + 4 * T),
        "bf16_gateup_swiglu_fwd": (4.0 * T * D * I, None),
        "bf16_swiglu_bwd_rows": (None, 10.0 * T * I),
        "bf16_gateup_dgrad": (4.0 * T * D * I, None),
        "bf16_norm_bwd": (None, 6.0 * T * D),
        "bf16_wgrad_gateup": (4.0 * T * D * I, None),
        "bf16_fold_grads": (None, 20.0 * I * D),
    }
    per = trace_steps(step, steps, stream, bf16_launch_name)
    in_step, roofline = in_step_summary(
        per, steps, work, lambda k: read_traffic(k, TRAFFIC_PROFILE_BF16) if (T, D, I) == TRAFFIC_WORKLOAD else None)
    roofline["peak"] = BF16_PEAK_TFLOPS if roofline["bound"] == "mfma" else HBM_PEAK_GBPS
    roofline["frac"] = round(roofline["achieved"] / roofline["peak"], 4)
    flop = 18.0 * T * D * I
    return {"workload": "bf16_norm_swiglu_mlp_fwd_bwd", "tokens": T, "d_model": D, "ffn": I, "flop_per_step": flop,
            "ms_per_step": round(ms, 4), "TFLOP/s": round(flop / (ms * 1e-3) / 1e12, 2),
            "frac_bf16_peak": round(flop / (ms * 1e-3) / 1e12 / BF16_PEAK_TFLOPS, 4),
            "norm_swiglu_ms_in_step": round(sum(v["ms"] * v["launches_per_step"] for v in in_step.values()), 4),
            "roofline": roofline, "kernels_in_step": in_step}


def time_moe(T: int, D: int, I: int, E: int, k: int, steps: int, warmup: int) -> dict:
    """GPU training-step time of the FP8 experts (prewarm step and scale roll
    first), its in-step kernels and the roofline of the dominant one.  The
    routed rows R = T*k carry 18*R*D*I FLOP per step."""
    import torch

    step, counts = make_moe(T, D, I, E, k)
    stream = torch.cuda.current_stream()
    step()
    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    R = T * k
    flop = 18.0 * R * D * I
    work = {
        "moe_plan": (None, 4.0 * E),
        "moe_gather_quant_x": (None, 3.0 * R * D),
        "moe_quant_dout": (None, 3.0 * R * D),
        "weight_quant_gu": (None, 10.0 * E * 2 * I * D),
        "weight_quant_down": (None, 11.0 * E * D * I),
        "moe_gateup_swiglu_fwd": (4.0 * R * D * I, None),
        "moe_down_fwd": (2.0 * R * D * I, None),
        "moe_down_dgrad_swiglu_bf16": (2.0 * R * D * I, None),
        "moe_gateup_dgrad": (4.0 * R * D * I, None),
        "moe_wgrad_gateup": (4.0 * R * D * I, None),
        "moe_wgrad_down": (2.0 * R * D * I, None),
        "moe_topk_sum": (None, 2.0 * R * D + 2.0 * T * D),
        "update_scales": (None, 40.0),
    }
    per = trace_steps(step, steps, stream, lambda sym, a: launch_name(sym, a, D, I))
    mw = MOE_WORKLOAD
    in_step, roofline = in_step_summary(
        per, steps, work,
        lambda kern: read_traffic(kern, TRAFFIC_PROFILE_MOE)
        if (T, D, I, E, k) == (mw["T"], mw["D"], mw["I"], mw["E"], mw["k"]) else None)
    return {"workload": "fp8_moe_experts_fwd_bwd", "tokens": T, "top_k": k, "experts": E, "d_model": D, "ffn": I,
            "routed_rows": R, "rows_per_expert": counts, "flop_per_step": flop, "ms_per_step": round(ms, 4),
            "TFLOP/s": round(flop / (ms * 1e-3) / 1e12, 2),
            "frac_fp8_peak": round(flop / (ms * 1e-3) / 1e12 / FP8_PEAK_TFLOPS, 4),
            "roofline": roofline, "kernels_in_step": in_step}


def main() -> None:
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported (the FP8 MLP path "
              "runs data-parallel with one block per GPU and no collective inside it)", file=sys.stderr)
        sys.exit(2)

    import torch

    from spark_gpt_amd import ops

    if args.trace == "moe":
        mw = MOE_WORKLOAD
        print(json.dumps({"moe": time_moe(mw["T"], mw["D"], mw["I"], mw["E"], mw["k"], args.steps, args.warmup)}),
              flush=True)
        return
    if args.trace == "bf16":
        print(json.dumps({"bf16": time_bf16(args.tokens, args.d_model, args.ffn, args.steps, args.warmup)}),
              flush=True)
        return
    dev = torch.device("cuda:0")
    T, D, I = args.tokens, args.d_model, args.ffn
    h, dy, norm, mlp, step = make_block(T, D, I, args.dist)
    scale, amax = mlp.fp8_scale, mlp.fp8_amax
    step()  # prewarm: records amax under scale 1, then the roll (as the trainer does)
    stream = torch.cuda.current_stream(dev)

    # FLOP or algorithmic bytes per launch of each kernel
    work = block_work(T, D, I)

    out_extra = {}
    if args.probe or not args.trace:
        # every kernel of the step alone (HIP events on the current stream)
        nwd = norm.weight.detach()
        x8, _, rstd = ops.norm_quant(h, nwd, scale, amax, 1e-6, copy=False)
        wscale = torch.empty(2, device=dev)
        w8, w8t, _ = ops.weight_quant(mlp.gate_up_proj.weight.detach(), wscale[0:1], w8=True, w8t=True)
        wd8, _, wdt = ops.weight_quant(mlp.down_proj.weight.detach(), wscale[1:2], w8=True, bf16t=True)
        gu8, h8, _ = ops.gateup_swiglu_fwd(x8, w8, scale, wscale, amax, T, I, copy=False)
        dgu8, _ = ops.down_dgrad_swiglu(dy, wdt, gu8, scale, amax, copy=False)
        dxn = ops.gateup_dgrad(dgu8, w8t, scale, wscale, T, D)
        dh, dnw, dy8t = ops.norm_bwd(h, rstd, dxn, dy, nwd, scale, amax)

        # saturation per fp8 site after the scale roll: codes at the format's
        # largest magnitude (e4m3 448 = 0x7E, e5m2 57344 = 0x7B, either sign)
        def at_max(t, code):
            return int(((t.view(torch.uint8) & 0x7F) == code).sum())

        out_extra["saturation"] = {
            "x": at_max(x8, 0x7E), "gu": at_max(gu8, 0x7E), "h": at_max(h8, 0x7E), "d_gu": at_max(dgu8, 0x7B),
            "dy": at_max(dy8t, 0x7B),
            "elements": {"x": T * D, "gu": 2 * T * I, "h": T * I, "d_gu": 2 * T * I, "dy": T * D}}
        kern = {
            "norm_quant": lambda: ops.norm_quant(h, nwd, scale, amax, 1e-6, copy=False),
            "post_step_quant": lambda: ops.block_weight_quant(mlp.gate_up_proj.weight.detach(),
                                                             mlp.down_proj.weight.detach()),
            "gateup_swiglu_fwd": lambda: ops.gateup_swiglu_fwd(x8, w8, scale, wscale, amax, T, I, copy=False),
            "down_fwd": lambda: ops.down_fwd(h8, wd8, h, scale, wscale),
            "down_dgrad_swiglu_bf16": lambda: ops.down_dgrad_swiglu(dy, wdt, gu8, scale, amax, copy=False),
            "gateup_dgrad": lambda: ops.gateup_dgrad(dgu8, w8t, scale, wscale, T, D),
            "norm_bwd": lambda: ops.norm_bwd(h, rstd, dxn, dy, nwd, scale, amax),
            "wgrad_down": lambda: ops.wgrad_rows(dy8t, h8, D, I, scale[4:5], scale[2:3], a_rows=False),
            "wgrad_gateup": lambda: ops.wgrad_rows(dgu8, x8, 2 * I, D, scale[3:4], scale[0:1]),
        }
        if args.probe:
            # calibration copy of known size, then one launch of each kernel
            src = torch.ones(256 << 20, device=dev)
            dst = torch.empty_like(src)
            torch.cuda.synchronize()
            torch.neg(src, out=dst)
            torch.cuda.synchronize()
            del src, dst
            for name, fn in kern.items():
                fn()
                torch.cuda.synchronize()
                print(f"probe {name} done", flush=True)
            xq = torch.randn(args.quant_rows, args.quant_cols, device=dev).to(torch.bfloat16)
            torch.cuda.synchronize()
            ops.quant_e4m3_rowcol(xq, scale, amax)
            torch.cuda.synchronize()
            print("probe quantizer done", flush=True)
            print(json.dumps({"probe": list(kern) + ["quantizer"], "copy_bytes_read": 1 << 30,
                              "copy_bytes_written": 1 << 30}))
            return
        out_extra["kernels"] = {name: rates(work, name, timed_launches(fn, 10, stream)) for name, fn in kern.items()}
        # the consumer of the gate/up weight gradient: the Muon momentum stage,
        # after the gradient (two kernels, dW written and read back) or fused
        # into its split reduction
        v_mom = torch.zeros(2 * I, D, device=dev)
        u_mom = torch.empty(2 * I, D, dtype=torch.bfloat16, device=dev)

        def separate():
            dw = ops.wgrad_rows(dgu8, x8, 2 * I, D, scale[3:4], scale[0:1])
            ops.momentum_stage(dw.view(-1), v_mom.view(-1), u_mom.view(-1), 0.95)

        sep_ms = timed_launches(separate, 10, stream)
        fused_ms = timed_launches(lambda: ops.wgrad_momentum(dgu8, x8, 2 * I, D, scale[3:4], scale[0:1], v_mom,
                                                             u_mom, 0.95, a_rows=True, b_rows=True), 10, stream)
        g_mom = torch.randn(2 * I * D, device=dev)
        stage_ms = timed_launches(lambda: ops.momentum_stage(g_mom, v_mom.view(-1), u_mom.view(-1), 0.95), 10,
                                  stream)
        out_extra["momentum_fusion"] = {
            "wgrad_gateup_then_momentum_stage_ms": round(sep_ms, 4), "fused_ms": round(fused_ms, 4),
            "saved_ms": round(sep_ms - fused_ms, 4),
            "momentum_stage_alone": rates({"m": (None, 14.0 * 2 * I * D)}, "m", stage_ms)}
        del v_mom, u_mom, g_mom
        del x8, rstd, w8, w8t, wd8, wdt, gu8, h8, dgu8, dxn, dh, dnw, dy8t

    # ---- timed steps (clean: nothing but the step's own launches) ----
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.steps
    flop = 18.0 * T * D * I
    tflops = flop / (ms * 1e-3) / 1e12

    # ---- the same steps again, HIP events around every C-ABI launch ----
    per = trace_steps(step, args.steps, stream, lambda sym, a: launch_name(sym, a, D, I))
    in_step, roofline = in_step_summary(
        per, args.steps, work, lambda k: read_traffic(k) if (T, D, I) == TRAFFIC_WORKLOAD else None)

    out = {
        "metric": "FP8 MLP fwd+bwd TFLOP/s (% FP8 MFMA peak); quantize GB/s (% HBM peak)",
        "value": round(tflops, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp8-e4m3/e5m2 (bf16 down dgrad)",
        "data": ("synthetic: seed-fixed " + ("N(0,1)" if args.dist == "normal" else "Student-t(3)")
                 + " bf16 activations, N(0,1/fan_in) fp32 weights, N(0,1e-3) bf16 grads"),
        "config": {"workload": "fp8_swiglu_mlp_block_fwd_bwd", "tokens": T, "d_model": D, "ffn": I,
                   "flop_per_step": flop, "frac_fp8_peak": round(tflops / FP8_PEAK_TFLOPS, 4)},
        "roofline": roofline,
        "kernels_in_step": in_step,
    }
    out.update(out_extra)
    if not args.trace:
        # ---- standalone quantizer (HBM-bound) ----
        R, C = args.quant_rows, args.quant_cols
        gq = torch.Generator(device=dev).manual_seed(3)
        xq = torch.randn(R, C, device=dev, generator=gq)
        cols = torch.randperm(C, device=dev, generator=gq)[: max(1, C // 1000)]
        xq[:, cols] *= 50.0
        xq = xq.to(torch.bfloat16)
        qs, qa = torch.ones(5, device=dev), torch.zeros(5, device=dev)
        ops.quant_e4m3_rowcol(xq, qs, qa)
        ops.update_scales(qs, qa)
        qms = timed_launches(lambda: ops.quant_e4m3_rowcol(xq, qs, qa), 20, stream)
        qbytes = 4.0 * R * C
        qgbps = qbytes / (qms * 1e-3) / 1e9
        out["quantizer"] = {"rows": R, "cols": C, "ms": round(qms, 4), "GB/s": round(qgbps, 1),
                            "frac_hbm": round(qgbps / HBM_PEAK_GBPS, 4), "bytes_per_launch": qbytes}
        del xq
        # the muP base block (T=8192, D=256, I=1024): timed, not targeted
        del h, dy, norm, mlp, step
        mw = MOE_WORKLOAD
        out["other_workloads"] = {
            "muP_base": time_block(8192, 256, 1024, 20, 5),
            "wide_student_t": time_block(65536, 2048, 6144, 10, 3, dist="student-t", trace=True),
            "stack28": time_stack(16384, 4096, 12288, 28, 5, 2),
            "moe": time_moe(mw["T"], mw["D"], mw["I"], mw["E"], mw["k"], 20, 5),
            "bf16": time_bf16(T, D, I, 20, 5)}
        out["other_workloads"]["bf16"]["fp8_block_speedup"] = round(
            out["other_workloads"]["bf16"]["ms_per_step"] / ms, 3)
        if not args.no_cpu_baseline:
            out["cpu_baseline"] = cpu_baseline(args.cpu_tokens, D, I)
            out["cpu_baseline"]["other_workloads"] = cpu_extra(args.quant_rows, args.quant_cols)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
