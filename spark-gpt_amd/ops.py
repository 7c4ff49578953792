"""Torch-facing wrappers of the libsparkfp8 kernels.

Each wrapper validates shapes/dtypes, allocates its outputs with torch's
caching allocator (as the reference allocates with ``torch.empty``), and
launches on torch's current stream.  Nothing here synchronises the device or
reads device values back.

The wrappers that a step of the block, the experts or the bf16 path calls are
native (``_native.so``, csrc/native.cpp: the same checks, allocations and
launches; a step of the block at T = 8192, D = 256, I = 1024, bound by host
time: 309 us through ctypes wrappers, 200 with these); the others are here.
"""
from __future__ import annotations

import torch

from . import _lib

# the native wrappers; without the built module each raises when it is called
_NATIVE = ("norm_quant", "block_weight_quant", "weight_quant_experts", "gateup_swiglu_fwd", "down_fwd",
           "down_dgrad_swiglu", "gateup_dgrad", "wgrad_rows", "norm_bwd", "moe_plan", "moe_rows_quant",
           "moe_gateup_swiglu_fwd", "moe_down_fwd", "moe_down_dgrad_swiglu", "moe_gateup_dgrad", "moe_wgrad_rows",
           "moe_topk_sum", "bf16_weight_slabs", "bf16_rows_prep", "bf16_swiglu_fwd", "bf16_swiglu_eval",
           "bf16_swiglu_bwd", "bf16_gemm", "bf16_norm_dh", "bf16_wgrad_rows", "bf16_fold_grads")


def _missing(name: str, why: str):
    def raises(*_args, **_kwargs):
        raise RuntimeError(f"{name} needs _native.so: build it with __graft_entry__.build() "
                           f"(there is no non-HIP fallback): {why}")

    return raises


try:
    from . import _native
except ImportError as _e:
    globals().update({_n: _missing(_n, str(_e)) for _n in _NATIVE})
else:
    globals().update({_n: getattr(_native, _n) for _n in _NATIVE})

E4M3 = torch.float8_e4m3fn
E5M2 = torch.float8_e5m2
FMT_E4M3 = 0
FMT_E5M2 = 1
TOKEN_ALIGN = 256  # leading dimension of token-contiguous fp8 copies


def ldt_of(T: int) -> int:
    """Tokens covered by the token-contiguous copies (x8t, h8t, d_gu8t, dy8t):
    T rounded up to a multiple of 256, zero past T."""
    return -(-T // TOKEN_ALIGN) * TOKEN_ALIGN


SLAB = 64  # bytes of K per slab row
# bytes per element of the dtypes the K-slabs hold
_ESIZE = {torch.float8_e4m3fn: 1, torch.float8_e5m2: 1, torch.uint8: 1, torch.bfloat16: 2, torch.float16: 2,
          torch.float32: 4}


def _esize(dtype) -> int:
    n = _ESIZE.get(dtype)
    return n if n is not None else torch.empty((), dtype=dtype).element_size()


def slab_rows(R: int) -> int:
    """Rows of a K-slab: R rounded up to the 256-row GEMM tile."""
    return -(-R // 256) * 256


def kslab_empty(R: int, L: int, dtype, device) -> torch.Tensor:
    """A K-slab of a row-major [R, L] matrix (L elements of K per row):
    [L*size/64, slab_rows(R), 64/size] for elements of `size` bytes; element
    (r, l) at [l // n, r, l % n] with n = 64 / size.  Every FP8 GEMM operand
    (and the bf16 W_down^T) uses this layout; one 64-byte K stage of a
    256-row tile is one contiguous 16 KiB block."""
    n = SLAB // _esize(dtype)
    _need(L % n == 0, f"K extent {L} must be a multiple of {n}")
    return torch.empty(L // n, slab_rows(R), n, dtype=dtype, device=device)


def kslab_shape(R: int, L: int, dtype) -> tuple:
    """Shape of kslab_empty(R, L, dtype)."""
    n = SLAB // _esize(dtype)
    _need(L % n == 0, f"K extent {L} must be a multiple of {n}")
    return (L // n, slab_rows(R), n)


def slab_empty(R: int, T: int, dtype, device) -> torch.Tensor:
    """A token-contiguous K-slab copy of R feature rows over ldt_of(T) tokens
    (the weight gradients' operands): [ldt / 64, slab_rows(R), 64]; element
    (r, t) at [t // 64, r, t % 64]."""
    return kslab_empty(R, ldt_of(T), dtype, device)


def unslab(t: torch.Tensor, R: int) -> torch.Tensor:
    """The plain [R, L] matrix of a K-slab tensor (for inspection and tests)."""
    n, rp, _ = t.shape
    return t.view(torch.uint8).permute(1, 0, 2).reshape(rp, n * SLAB)[:R].view(t.dtype)


def to_slab(x: torch.Tensor) -> torch.Tensor:
    """K-slab of a plain [R, L] tensor (64-byte multiple rows); padding rows zero."""
    R, L = x.shape
    nb = L * x.element_size()
    _need(nb % SLAB == 0, "row length must be a multiple of 64 bytes")
    out = torch.zeros(nb // SLAB, slab_rows(R), SLAB, dtype=torch.uint8, device=x.device)
    out[:, :R] = x.contiguous().view(torch.uint8).view(R, nb // SLAB, SLAB).permute(1, 0, 2)
    return out.view(x.dtype)


def _need(cond: bool, msg: str) -> None:
    if not cond:
        raise ValueError(msg)


def _cuda_contig(name: str, t: torch.Tensor, dtype: torch.dtype, ndim: int) -> None:
    _need(t.is_cuda, f"{name} must be a ROCm device tensor")
    _need(t.dtype == dtype, f"{name} must be {dtype}, got {t.dtype}")
    _need(t.dim() == ndim, f"{name} must be {ndim}-D, got shape {tuple(t.shape)}")
    _need(t.is_contiguous(), f"{name} must be contiguous")


# ------------------------------------------------------------------ quantizers
def quant_e4m3_rowcol(x: torch.Tensor, scale: torch.Tensor, amax: torch.Tensor):
    """x8 = e4m3(x * scale[0]) row-major [rows, cols]; x8t = the token-contiguous
    K-slab copy of x8^T over ldt_of(rows) tokens ([ldt / 64, slab_rows(cols),
    64], zeros past rows and cols); amax[0] max|x|."""
    _cuda_contig("x", x, torch.bfloat16, 2)
    R, C = x.shape
    _need(C % 128 == 0, "cols must be a multiple of 128")
    ldt = ldt_of(R)
    x8 = torch.empty(R, C, dtype=E4M3, device=x.device)
    x8t = slab_empty(C, R, E4M3, x.device)
    _lib.call("sfp8_quant_e4m3_rowcol", x.data_ptr(), R, C, scale.data_ptr(), amax.data_ptr(),
              x8.data_ptr(), x8t.data_ptr(), ldt, _lib.stream_of(x))
    return x8, x8t


def weight_quant(w: torch.Tensor, q_out: torch.Tensor, *, w8: bool = True, w8t: bool = False,
                 bf16t: bool = False):
    """Just-in-time e4m3 copy of an fp32 master [R, C]: returns (w8 K-slab of
    [R, C], w8t K-slab of [C, R], bf16 K-slab of W^T [C, R]), unrequested
    outputs None; the pow2 scale lands in q_out[0] (device)."""
    _cuda_contig("w", w, torch.float32, 2)
    R, C = w.shape
    _need(C % 64 == 0, "weight columns must be a multiple of 64")
    _need(not w8t or R % 64 == 0, "weight rows must be a multiple of 64 for the transposed copy")
    _need(not bf16t or R % 32 == 0, "weight rows must be a multiple of 32 for the bf16 copy")
    dev = w.device
    o8 = kslab_empty(R, C, E4M3, dev) if w8 else None
    o8t = kslab_empty(C, R, E4M3, dev) if w8t else None
    obt = kslab_empty(C, R, torch.bfloat16, dev) if bf16t else None
    parts = torch.empty(512, dtype=torch.float32, device=dev)
    _lib.call("sfp8_weight_quant", w.data_ptr(), R, C, parts.data_ptr(), parts.numel(), q_out.data_ptr(),
              _lib.ptr(o8), _lib.ptr(o8t), _lib.ptr(obt), _lib.stream_of(w))
    return o8, o8t, obt


def update_scales(scale: torch.Tensor, amax: torch.Tensor) -> None:
    """In-place delayed-scale roll of one or more contiguous 5-slot sets."""
    _need(scale.is_cuda and amax.is_cuda, "scale/amax must be device tensors")
    _need(scale.dtype == torch.float32 and amax.dtype == torch.float32, "scale/amax must be fp32")
    _need(scale.is_contiguous() and amax.is_contiguous(), "scale/amax must be contiguous")
    _need(scale.numel() == amax.numel() and scale.numel() % 5 == 0, "scale/amax: 5 slots per set")
    _lib.call("sfp8_update_scales", scale.data_ptr(), amax.data_ptr(), scale.numel() // 5,
              _lib.stream_of(scale))


# ------------------------------------------------------------------ GEMMs
def wgrad(at, bt, M: int, N: int, sa, sb):
    """out[m, n] = sum_t at[m, t] bt[n, t] / (sa * sb), fp32 [M, N]; at e5m2
    and bt e4m3 are K-slab token-contiguous copies of M and N rows (zeros past
    the last token)."""
    _cuda_contig("at", at, E5M2, 3)
    _cuda_contig("bt", bt, E4M3, 3)
    ldt = at.shape[0] * SLAB
    _need(at.shape == (ldt // SLAB, slab_rows(M), SLAB), "at must be a K-slab copy of M rows")
    _need(bt.shape == (ldt // SLAB, slab_rows(N), SLAB), "bt must be a K-slab copy of N rows over the same tokens")
    _need(ldt % TOKEN_ALIGN == 0, "token count must be a multiple of 256")
    out = torch.empty(M, N, dtype=torch.float32, device=at.device)
    nws = _lib.query("sfp8_wgrad_workspace_floats", M, N, ldt)
    ws = torch.empty(max(nws, 1), dtype=torch.float32, device=at.device)
    _lib.call("sfp8_gemm_wgrad", at.data_ptr(), FMT_E5M2, bt.data_ptr(), FMT_E4M3, M, N, ldt, sa.data_ptr(),
              sb.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(at))
    return out




# ------------------------------------------------------------------ MoE experts (grouped)
def moe_padded_rows(R: int, E: int) -> int:
    """Rows of the padded expert order (every expert's rows from a 256-row
    boundary): the worst case for R rows over E experts."""
    return _lib.query("sfp8_moe_padded_rows", R, E)


def moe_wgrad(at, bt, M: int, N: int, E: int, plan, sa, sb):
    """out[e] = sum over expert e's rows of at^T bt / (sa * sb), fp32 [E, M, N];
    at (e5m2) and bt (e4m3) token-contiguous K-slab copies over padded expert order."""
    _cuda_contig("at", at, E5M2, 3)
    _cuda_contig("bt", bt, E4M3, 3)
    ldp = at.shape[0] * SLAB
    out = torch.empty(E, M, N, dtype=torch.float32, device=at.device)
    nws = _lib.query("sfp8_moe_wgrad_workspace_floats", M, N, E)
    ws = torch.empty(max(nws, 1), dtype=torch.float32, device=at.device)
    _lib.call("sfp8_moe_gemm_wgrad", at.data_ptr(), FMT_E5M2, bt.data_ptr(), FMT_E4M3, M, N, E, plan.data_ptr(), ldp,
              sa.data_ptr(), sb.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(at))
    return out


# ----------------------------------------------------- bf16 SwiGLU path
# The default (non-FP8) MLP path: bf16 K-slabs (32 elements of K per 64-byte
# row), rows dense (no plan) or in padded expert order (a MoE plan).
BF16 = torch.bfloat16


def bf16_wgrad(at: torch.Tensor, bt: torch.Tensor, M: int, N: int, plan=None, E: int = 1):
    """bf16(A^T B) over the padded rows: [M, N] (dense) or [E, M, N] (per
    expert, with a plan); at, bt the token-contiguous bf16 K-slabs of [M, ldp]
    and [N, ldp]."""
    ldp = at.shape[0] * (SLAB // 2)
    dev = at.device
    if plan is None:
        out = torch.empty(M, N, dtype=BF16, device=dev)
        nws = _lib.query("sfp8_bf16_wgrad_workspace_floats", M, N, ldp)
        ws = torch.empty(max(nws, 1), dtype=torch.float32, device=dev)
        _lib.call("sfp8_bf16_gemm_wgrad", at.data_ptr(), bt.data_ptr(), M, N, ldp, out.data_ptr(), ws.data_ptr(),
                  ws.numel(), _lib.stream_of(at))
    else:
        out = torch.empty(E, M, N, dtype=BF16, device=dev)
        nws = _lib.query("sfp8_bf16_moe_wgrad_workspace_floats", M, N, E)
        ws = torch.empty(max(nws, 1), dtype=torch.float32, device=dev)
        _lib.call("sfp8_bf16_moe_gemm_wgrad", at.data_ptr(), bt.data_ptr(), M, N, E, plan.data_ptr(), ldp,
                  out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(at))
    return out


# ----------------------------------------------------- the optimizer's momentum stage
def _flat_state(name: str, t, dtype: torch.dtype, numel: int, device, align: int) -> None:
    """t is a contiguous `dtype` tensor of `numel` elements on `device` whose
    data pointer is `align`-byte aligned (what the kernels' vector accesses
    need); raises ValueError before anything is launched."""
    _need(isinstance(t, torch.Tensor), f"{name} must be a tensor")
    _need(t.is_cuda and t.device == device, f"{name} must be a ROCm device tensor on {device}")
    _need(t.dtype == dtype, f"{name} must be {dtype}, got {t.dtype}")
    _need(t.is_contiguous(), f"{name} must be contiguous")
    _need(t.numel() == numel, f"{name} must have {numel} elements, got {t.numel()}")
    _need(t.data_ptr() % align == 0, f"{name} must be {align}-byte aligned")


def _momentum_weights(momentum: float) -> None:
    """The kernels take w_v = 1 - momentum and w_u = momentum as fp32 values
    (ctypes rounds them as the reference's launch does) with
    -0.5 < w_v < 0.5 <= w_u."""
    import numpy as np

    w_v, w_u = np.float32(1.0 - momentum), np.float32(momentum)
    _need(bool(-0.5 < w_v < 0.5 <= w_u), f"momentum {momentum} outside the kernel's range (0.5 <= momentum < 1.5)")


def momentum_stage(g: torch.Tensor, v: torch.Tensor, u: torch.Tensor, momentum: float) -> None:
    """v <- lerp(v, g, 1 - momentum) in place; u <- bf16(lerp(g, v, momentum))."""
    _need(isinstance(g, torch.Tensor) and g.is_cuda, "g must be a ROCm device tensor")
    n = g.numel()
    _need(n % 4 == 0, "g, v, u need a multiple of 4 elements")
    _flat_state("g", g, torch.float32, n, g.device, 16)
    _flat_state("v", v, torch.float32, n, g.device, 16)
    _flat_state("u", u, BF16, n, g.device, 8)
    _momentum_weights(momentum)
    _lib.call("sfp8_momentum_stage", g.data_ptr(), v.data_ptr(), u.data_ptr(), n, 1.0 - momentum, momentum,
              _lib.stream_of(g))


def wgrad_momentum(a8, b8, M: int, N: int, sa, sb, v: torch.Tensor, u: torch.Tensor, momentum: float, grad=None, *,
                   a_rows: bool = False, b_rows: bool = False):
    """wgrad (a_rows = b_rows = False) or wgrad_rows of the same operands
    handed straight to the momentum stage: v <- lerp(v, dW, 1 - momentum),
    u <- bf16(lerp(dW, v, momentum)); dW is also written to `grad` when
    given.  v and grad are fp32, u bf16, each [M, N] on the operands' device;
    sa and sb are fp32 scales there."""
    _cuda_contig("a8", a8, E5M2, 3)
    _cuda_contig("b8", b8, E4M3, 3)
    _need(b8.device == a8.device, "a8, b8 must be on the same device")
    _flat_state("v", v, torch.float32, M * N, a8.device, 16)
    _flat_state("u", u, BF16, M * N, a8.device, 8)
    if grad is not None:
        _flat_state("grad", grad, torch.float32, M * N, a8.device, 16)
    for name, t in (("sa", sa), ("sb", sb)):
        _need(isinstance(t, torch.Tensor) and t.is_cuda and t.device == a8.device and t.dtype == torch.float32
              and t.numel() >= 1, f"{name} must be an fp32 scale on {a8.device}")
    _momentum_weights(momentum)
    ldt = a8.shape[1] if a_rows else a8.shape[0] * SLAB
    _need((b8.shape[1] if b_rows else b8.shape[0] * SLAB) == ldt, "a8, b8 must cover the same tokens")
    nws = _lib.query("sfp8_wgrad_momentum_workspace_floats", M, N, ldt)
    ws = torch.empty(max(nws, 1), dtype=torch.float32, device=a8.device)
    _lib.call("sfp8_gemm_wgrad_momentum", a8.data_ptr(), FMT_E5M2, int(a_rows), b8.data_ptr(), FMT_E4M3, int(b_rows),
              M, N, ldt, sa.data_ptr(), sb.data_ptr(), _lib.ptr(grad), v.data_ptr(), u.data_ptr(), 1.0 - momentum,
              momentum, ws.data_ptr(), ws.numel(), _lib.stream_of(a8))
