"""GPU parity of each GEMM kernel against the oracle on identical inputs.

* exact-integer operands (every partial sum exact in fp32, so accumulation
  order cannot matter): outputs bit-exact wherever no transcendental is
  involved, fp8 epilogue outputs after a sigmoid within one code;
* random operands: outputs within tolerance.  The gfx950 FP8 MFMA does not
  accumulate exactly in fp32: products are summed in groups aligned to the
  group's largest product, so a product about 2^17 times smaller than the
  largest one in its group is dropped.  Accumulators that cancel to small
  values can therefore move by a couple of fp8 codes; the bf16 MFMA is exact.
"""
import pytest
import torch

import spark_gpt_amd as sg
from oracle import fp8_mlp as O

pytestmark = pytest.mark.gpu

E4 = torch.float8_e4m3fn
E5 = torch.float8_e5m2


def u8(t):
    return t.contiguous().view(torch.uint8).cpu()


def code_dist(a, b):
    """Distance in fp8 codes (sign-magnitude ordinal) between two byte tensors."""
    def ordinal(x):
        x = x.to(torch.int32)
        return torch.where(x >= 128, -(x - 128), x)
    return (ordinal(u8(a)) - ordinal(u8(b))).abs()


def slab(x, dev):
    """K-slab device copy of a plain [R, K] operand (zero padding rows)."""
    return sg.ops.to_slab(x.contiguous()).to(dev)


def int_fp8(shape, dtype, g, lo=-8, hi=8):
    return torch.randint(lo, hi + 1, shape, generator=g).float().to(dtype)


SHAPES = [(1000, 256, 768), (257, 128, 384), (512, 512, 256), (1, 256, 128)]
# D = 1024 runs the persistent SwiGLU kernel whose epilogue of one tile is
# overlapped with the next tile's K loop: fewer tiles than CUs (one each),
# slightly more (some work-groups take two), several per work-group; ragged T.
SHAPES_PIPE = [(1000, 1024, 768), (2049, 1024, 1920), (4099, 1024, 3072), (1, 1024, 128)]


@pytest.mark.parametrize("T,D,I", SHAPES + SHAPES_PIPE)
def test_swiglu_fwd_integer_operands(dev, T, D, I):
    g = torch.Generator().manual_seed(T + D + I)
    x8 = int_fp8((T, D), E4, g)
    w8 = int_fp8((2 * I, D), E4, g)
    s = torch.tensor([0.5, 2.0 ** -6, 4.0, 1, 1])
    ws = torch.tensor([2.0 ** -3, 1.0])
    amax = torch.zeros(5, device=dev)
    gu8s, h8s, h8t = sg.ops.gateup_swiglu_fwd(slab(x8, dev), slab(w8, dev), s.to(dev), ws.to(dev), amax, T, I)
    rgu8, rh8, ra1, ra2 = O.swiglu_fwd(x8, w8, s, ws, I)
    ldt = sg.ops.ldt_of(T)
    assert gu8s.shape == (2 * I // 64, ldt, 64)
    assert torch.equal(u8(sg.ops.unslab(gu8s, T)), u8(rgu8))
    assert torch.all(u8(sg.ops.unslab(gu8s, ldt))[T:] == 0)
    assert h8s.shape == (I // 64, ldt, 64)
    h8 = sg.ops.unslab(h8s, T)
    assert torch.all(u8(sg.ops.unslab(h8s, ldt))[T:] == 0)
    assert int(code_dist(h8, rh8).max()) <= 1
    assert float((code_dist(h8, rh8) > 0).float().mean()) < 0.01
    assert h8t.shape == (ldt // 64, sg.ops.slab_rows(I), 64)
    ht = u8(sg.ops.unslab(h8t, I))
    assert torch.equal(ht[:, :T], u8(h8).t())
    assert torch.all(ht[:, T:] == 0)
    assert amax[1].item() == ra1.item()
    torch.testing.assert_close(amax[2].cpu(), ra2, rtol=1e-5, atol=0)
    # without the token-contiguous copy: the same rows and amax
    amax2 = torch.zeros(5, device=dev)
    gu8b, h8b, none = sg.ops.gateup_swiglu_fwd(slab(x8, dev), slab(w8, dev), s.to(dev), ws.to(dev), amax2, T, I,
                                               copy=False)
    assert none is None
    assert torch.equal(u8(gu8b), u8(gu8s)) and torch.equal(u8(h8b), u8(h8s))
    assert torch.equal(amax2, amax)


@pytest.mark.parametrize("T,D,I", [(300, 256, 256), (300, 1024, 256)])
def test_swiglu_fwd_nan_rows(dev, T, D, I):
    """A NaN code in a token's x8 row makes that token's gate, up and h all
    NaN: they must carry NaN codes, the other rows must be unaffected, and
    NaN values do not enter the amax slots."""
    g = torch.Generator().manual_seed(21 + D)
    x8 = int_fp8((T, D), E4, g)
    w8 = int_fp8((2 * I, D), E4, g)
    bad = torch.tensor([0, 77, T - 1])
    xb = x8.view(torch.uint8).clone()
    xb[bad, 5] = 0x7F
    x8n = xb.view(E4)
    s = torch.tensor([1.0, 2.0 ** -8, 2.0 ** -12, 1, 1])
    ws = torch.tensor([1.0, 1.0])
    amax = torch.zeros(5, device=dev)
    gu8s, h8s, _ = sg.ops.gateup_swiglu_fwd(slab(x8n, dev), slab(w8, dev), s.to(dev), ws.to(dev), amax, T, I)
    h8 = u8(sg.ops.unslab(h8s, T))
    gu = u8(sg.ops.unslab(gu8s, T))
    assert torch.all((gu[bad] & 0x7F) == 0x7F) and torch.all((h8[bad] & 0x7F) == 0x7F)
    keep = torch.ones(T, dtype=torch.bool)
    keep[bad] = False
    rgu8, rh8, ra1, ra2 = O.swiglu_fwd(x8[keep], w8, s, ws, I)
    assert torch.equal(gu[keep], u8(rgu8))
    assert int(code_dist(h8[keep].view(E4), rh8).max()) <= 1
    assert amax[1].item() == ra1.item()
    torch.testing.assert_close(amax[2].cpu(), ra2, rtol=1e-5, atol=0)


@pytest.mark.parametrize("T,D,I", SHAPES[:3])
def test_swiglu_fwd_random(dev, T, D, I):
    g = torch.Generator().manual_seed(1 + T + D + I)
    h = torch.randn(T, D, generator=g).to(torch.bfloat16)
    nw = torch.ones(D)
    s = torch.tensor([32.0, 64.0, 128.0, 1, 1])
    x8, _, _, _ = O.norm_quant(h, nw, s[0], 1e-6)
    w8, q = O.quantize_weight(torch.randn(2 * I, D, generator=g) * D ** -0.5)
    ws = torch.stack([q, torch.tensor(1.0)])
    amax = torch.zeros(5, device=dev)
    gu8s, h8s, _ = sg.ops.gateup_swiglu_fwd(slab(x8, dev), slab(w8, dev), s.to(dev), ws.to(dev), amax, T, I)
    gu8, h8 = sg.ops.unslab(gu8s, T), sg.ops.unslab(h8s, T)
    rgu8, rh8, ra1, ra2 = O.swiglu_fwd(x8, w8, s, ws, I)
    for got, ref in ((gu8, rgu8), (h8, rh8)):
        d = code_dist(got, ref)
        # one code wherever the value is clear of the e4m3 subnormal range;
        # near zero the MFMA's group truncation can move a cancelled
        # accumulator by a few subnormal steps
        clear = ref.float().abs() >= 2.0 ** -4
        assert int(d[clear].max()) <= 1 and int(d.max()) <= 8
        assert float((d > 0).float().mean()) < 0.005
        assert O.rel_l2(got.cpu().float(), ref.float()) < 2e-3
    torch.testing.assert_close(amax[1:3].cpu(), torch.stack([ra1, ra2]), rtol=1e-2, atol=0)


@pytest.mark.parametrize("T,D,I", SHAPES)
def test_down_fwd_integer_operands(dev, T, D, I):
    g = torch.Generator().manual_seed(2 + T + D + I)
    h8 = int_fp8((T, I), E4, g)
    wd8 = int_fp8((D, I), E4, g)
    res = torch.randn(T, D, generator=g).to(torch.bfloat16)
    s = torch.tensor([1, 1, 2.0 ** 4, 1, 1])
    ws = torch.tensor([1.0, 2.0 ** 3])
    y = sg.ops.down_fwd(slab(h8, dev), slab(wd8, dev), res.to(dev), s.to(dev), ws.to(dev))
    ry = O.down_fwd(h8, wd8, res, s, ws)
    assert torch.equal(y.cpu(), ry)


# The headline width D = 1024: the persistent dgrad with fewer tiles than CUs
# and with three tiles per work-group (T = 16384); ragged T.
SHAPES_DGRAD_PIPE = [(1000, 1024, 768), (1, 1024, 128), (4099, 1024, 3072), (16384, 1024, 3072)]


@pytest.mark.parametrize("T,D,I", SHAPES + SHAPES_DGRAD_PIPE)
def test_down_dgrad_swiglu_integer_operands(dev, T, D, I):
    g = torch.Generator().manual_seed(3 + T + D + I)
    dy = torch.randint(-8, 9, (T, D), generator=g).float().to(torch.bfloat16)
    wd = torch.randint(-8, 9, (D, I), generator=g).float().to(torch.bfloat16)
    gu8 = O.e4m3(torch.randn(T, 2 * I, generator=g) * 64)
    s = torch.tensor([1, 64.0, 1, 2.0 ** -12, 1])
    amax = torch.zeros(5, device=dev)
    dgu8s, dgu8t = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax)
    dgu8 = sg.ops.unslab(dgu8s, T)
    assert torch.all(u8(sg.ops.unslab(dgu8s, sg.ops.ldt_of(T)))[T:] == 0)
    rdgu8, ra3, _ = O.down_dgrad_swiglu(dy, wd, gu8, s, I)
    d = code_dist(dgu8, rdgu8)
    assert int(d.max()) <= 1 and float((d > 0).float().mean()) < 0.01
    dt = u8(sg.ops.unslab(dgu8t, 2 * I))
    assert torch.equal(dt[:, :T], u8(dgu8).t())
    assert torch.all(dt[:, T:] == 0)
    torch.testing.assert_close(amax[3].cpu(), ra3, rtol=1e-5, atol=0)
    # without the token-contiguous copy: the same rows and amax
    amax2 = torch.zeros(5, device=dev)
    dgu8b, none = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax2,
                                           copy=False)
    assert none is None
    assert torch.equal(u8(dgu8b), u8(dgu8s))
    assert torch.equal(amax2, amax)


@pytest.mark.parametrize("T,D,I", [(512, 256, 256), (8192, 1024, 3072)])
def test_down_dgrad_swiglu_every_gate_code(dev, T, D, I):
    """Every e4m3 code as gate and as up value, the two NaN codes included.
    The kernel takes sigmoid(g) and sig*(1 + g*(1 - sig)) from a table over
    the 256 gate codes and multiplies in the reference's order, so only a
    sigmoid that differs from torch's by an ulp can move a byte.  NaN outputs
    must carry a NaN code (the sign of a NaN is not specified)."""
    g = torch.Generator().manual_seed(11)
    dy = torch.randint(-8, 9, (T, D), generator=g).float().to(torch.bfloat16)
    wd = torch.randint(-8, 9, (D, I), generator=g).float().to(torch.bfloat16)
    codes = torch.arange(T * I, dtype=torch.int64)
    gate = (codes % 256).to(torch.uint8).view(T, I)
    up = ((codes * 97 + codes // 256) % 256).to(torch.uint8).view(T, I)
    gu8 = torch.cat([gate, up], dim=1).view(E4)
    s = torch.tensor([1, 64.0, 1, 2.0 ** -6, 1])
    amax = torch.zeros(5, device=dev)
    dgu8s, dgu8t = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax)
    dgu8 = sg.ops.unslab(dgu8s, T)
    rdgu8, _, _ = O.down_dgrad_swiglu(dy, wd, gu8, s, I)
    nan = torch.isnan(rdgu8.float())
    assert int(nan.sum()) > 0
    got = u8(dgu8)
    assert torch.all((got[nan] & 0x7F) == 0x7F)
    d = code_dist(dgu8, rdgu8)[~nan]
    assert int(d.max()) <= 1 and float((d > 0).float().mean()) < 1e-3
    dt = u8(sg.ops.unslab(dgu8t, 2 * I))
    assert torch.equal(dt[:, :T], got.t())
    # without the token-contiguous copy (at D = 1024 the persistent 256 x 128
    # kernel with the deferred epilogue): the same bytes, NaN codes and
    # exact-path blocks included, and the same amax
    amax2 = torch.zeros(5, device=dev)
    dgu8b, _ = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax2,
                                        copy=False)
    assert torch.equal(u8(dgu8b), u8(dgu8s))
    assert torch.equal(amax2, amax)


@pytest.mark.parametrize("T,D,I", SHAPES[:3] + SHAPES_DGRAD_PIPE[2:])
def test_down_dgrad_swiglu_random(dev, T, D, I):
    g = torch.Generator().manual_seed(4 + T + D + I)
    dy = (torch.randn(T, D, generator=g) * 1e-3).to(torch.bfloat16)
    wd = (torch.randn(D, I, generator=g) * I ** -0.5).to(torch.bfloat16)
    gu8 = O.e4m3(torch.randn(T, 2 * I, generator=g) * 64)
    s = torch.tensor([1, 64.0, 1, 2.0 ** 18, 1])
    amax = torch.zeros(5, device=dev)
    dgu8s, _ = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax)
    dgu8 = sg.ops.unslab(dgu8s, T)
    rdgu8, ra3, _ = O.down_dgrad_swiglu(dy, wd, gu8, s, I)
    d = code_dist(dgu8, rdgu8)
    # Where dh = dy @ Wd cancels, the oracle's own fp32 sum can be more than
    # half a bf16 ulp from the exact (fp64) value; its byte there is not
    # pinned (any fp32 order, the kernel's included, may round elsewhere).
    # Such elements must be rare; every other byte is within one code.
    dh32, dh64 = dy.float() @ wd.float(), dy.double() @ wd.double()
    unpinned = (dh32.double() - dh64).abs() > dh64.abs() * 2.0 ** -9
    unpinned = torch.cat([unpinned, unpinned], dim=1)
    assert float(unpinned.float().mean()) < 1e-3
    assert int(d[~unpinned].max()) <= 1 and float((d > 0).float().mean()) < 0.02
    torch.testing.assert_close(amax[3].cpu(), ra3, rtol=1e-2, atol=0)
    amax2 = torch.zeros(5, device=dev)
    dgu8b, _ = sg.ops.down_dgrad_swiglu(dy.to(dev), slab(wd.t(), dev), slab(gu8, dev), s.to(dev), amax2,
                                        copy=False)
    assert torch.equal(u8(dgu8b), u8(dgu8s))
    assert torch.equal(amax2, amax)


@pytest.mark.parametrize("T,D,I", SHAPES)
def test_gateup_dgrad_integer_operands(dev, T, D, I):
    g = torch.Generator().manual_seed(5 + T + D + I)
    dgu8 = int_fp8((T, 2 * I), E5, g)
    w8 = int_fp8((2 * I, D), E4, g)
    s = torch.tensor([1, 1, 1, 2.0 ** 5, 1])
    ws = torch.tensor([2.0 ** 2, 1.0])
    dxn = sg.ops.gateup_dgrad(slab(dgu8, dev), slab(w8.t(), dev), s.to(dev), ws.to(dev), T, D)
    rdxn = O.gateup_dgrad(dgu8, w8, s, ws)
    assert torch.equal(dxn.cpu(), rdxn)


@pytest.mark.parametrize("T,M,N", [(1000, 256, 768), (257, 768, 128), (4099, 1024, 512), (65536, 256, 256)])
def test_wgrad_integer_operands(dev, T, M, N):
    g = torch.Generator().manual_seed(6 + T + M + N)
    ldt = sg.ops.ldt_of(T)
    a = int_fp8((T, M), E5, g, -4, 4)
    b = int_fp8((T, N), E4, g, -4, 4)
    at = torch.zeros(M, ldt, dtype=torch.uint8)
    bt = torch.zeros(N, ldt, dtype=torch.uint8)
    at[:, :T] = u8(a).t()
    bt[:, :T] = u8(b).t()
    sa, sb = torch.tensor([2.0 ** 3]), torch.tensor([0.5])
    at_s = sg.ops.to_slab(at.view(E5)).view(torch.uint8)
    bt_s = sg.ops.to_slab(bt.view(E4)).view(torch.uint8)
    # padding rows (beyond M, N) hold NaN codes: they must not reach the output
    at_s[:, M:] = 0x7F
    bt_s[:, N:] = 0x7F
    out = sg.ops.wgrad(at_s.view(E5).to(dev), bt_s.view(E4).to(dev), M, N, sa.to(dev), sb.to(dev))
    ref = (a.float().t() @ b.float()) / (sa * sb)
    assert torch.equal(out.cpu(), ref)


def test_wgrad_matches_oracle_forms(dev):
    """Both weight gradients of the block through the kernel vs the oracle's
    reference-shaped formulas (down: dy quantized e5m2 in 2 token splits;
    gate/up: d_gu8^T x8)."""
    T, D, I = 1000, 256, 768
    g = torch.Generator().manual_seed(7)
    dy = (torch.randn(T, D, generator=g) * 1e-3).to(torch.bfloat16)
    h8 = O.e4m3(torch.randn(T, I, generator=g) * 30)
    dgu8 = O.e5m2(torch.randn(T, 2 * I, generator=g) * 1000)
    x8 = O.e4m3(torch.randn(T, D, generator=g) * 30)
    s = torch.tensor([16.0, 1, 32.0, 2.0 ** 10, 2.0 ** 15])
    ldt = sg.ops.ldt_of(T)

    def tpad(t8):
        out = torch.zeros(t8.shape[1], ldt, dtype=torch.uint8)
        out[:, :T] = u8(t8).t()
        return sg.ops.to_slab(out.view(t8.dtype)).to(dev)

    dy8 = O.e5m2(dy.float() * s[4])
    sd = s.to(dev)
    dwd = sg.ops.wgrad(tpad(dy8), tpad(h8), D, I, sd[4:5], sd[2:3])
    dwgu = sg.ops.wgrad(tpad(dgu8), tpad(x8), 2 * I, D, sd[3:4], sd[0:1])
    for got, ref in ((dwd, O.down_wgrad(dy, h8, s)), (dwgu, O.gateup_wgrad(dgu8, x8, s))):
        torch.testing.assert_close(got.cpu(), ref, rtol=1e-4, atol=1e-4 * float(ref.abs().max()))
        assert O.rel_l2(got.cpu(), ref) < 1e-4


@pytest.mark.parametrize("M,N", [(256, 100), (300, 36), (64, 4)])
def test_wgrad_ragged_columns_stay_in_bounds(dev, M, N):
    """N % 16 != 0 with one K split (the kernel's own epilogue writes [M, N]):
    every float4 past column N is skipped, so a guard region right after the
    output is untouched and the output equals a float32 matmul."""
    from spark_gpt_amd import _lib

    T = 200
    ldt = sg.ops.ldt_of(T)
    assert _lib.query("sfp8_wgrad_splits", M, N, ldt) == 1
    g = torch.Generator().manual_seed(M + N)
    a = int_fp8((T, M), E5, g, -4, 4)
    b = int_fp8((T, N), E4, g, -4, 4)
    at = torch.zeros(M, ldt, dtype=torch.uint8)
    bt = torch.zeros(N, ldt, dtype=torch.uint8)
    at[:, :T] = u8(a).t()
    bt[:, :T] = u8(b).t()
    at_s = sg.ops.to_slab(at.view(E5)).to(dev)
    bt_s = sg.ops.to_slab(bt.view(E4)).to(dev)
    sa, sb = torch.tensor([1.0], device=dev), torch.tensor([1.0], device=dev)
    guard = 1 << 16
    buf = torch.full((M * N + guard,), 12345.0, device=dev)
    _lib.call("sfp8_gemm_wgrad", at_s.data_ptr(), 1, bt_s.data_ptr(), 0, M, N, ldt, sa.data_ptr(), sb.data_ptr(),
              buf.data_ptr(), None, 0, _lib.stream_of(buf))
    torch.cuda.synchronize()
    ref = a.float().t() @ b.float()
    assert torch.equal(buf[: M * N].view(M, N).cpu(), ref)
    assert bool((buf[M * N:] == 12345.0).all())


@pytest.mark.parametrize("M,N,T,splits,taken", [(6144, 1024, 4096, 2, 1), (2048, 3072, 32768, 5, 2),
                                                (1024, 3072, 16384, 5, 5), (1024, 1024, 8192, 4, 4),
                                                (1024, 1024, 16384, 8, 8), (320, 192, 1000, 1, 1),
                                                (256, 256, 65536, 32, 32)])
def test_wgrad_rows_equals_token_contiguous(dev, M, N, T, splits, taken):
    """The weight gradient read from the row K-slabs through transposing LDS
    reads gives the bytes of the one read from the token-contiguous copies
    (same values in the same MFMA K positions, same split sums): one split,
    also where the workspace has room for more, and several (2 and 4 splits:
    each split on 8 / splits XCDs; 5: uneven splits, the last shorter, runs of
    the split-major order crossing split boundaries; 8 and 32: whole splits per
    XCD; 2 and 5 in 256 x 256 tiles, the others in 128 x 128), ragged tiles,
    and the same operands in both layouts.  The result is also checked against a float64
    matmul of the same operands, which no split mapping shares."""
    from spark_gpt_amd import _lib

    ops = sg.ops
    assert _lib.query("sfp8_wgrad_splits", M, N, ops.ldt_of(T)) == splits
    assert _lib.query("sfp8_wgrad_splits_of", M, N, 0, ops.ldt_of(T), 0, 0) == taken
    g = torch.Generator(device=dev).manual_seed(M + N + T)
    a = (torch.randn(T, M, device=dev, generator=g) * 8).to(ops.E5M2)
    b = (torch.randn(T, N, device=dev, generator=g) * 8).to(ops.E4M3)
    ldt = ops.ldt_of(T)
    pad = lambda x: torch.cat([x, torch.zeros(ldt - T, x.shape[1], dtype=x.dtype, device=dev)])
    a_rows, b_rows = ops.to_slab(pad(a)), ops.to_slab(pad(b))      # [M/64, ldt, 64]
    a_t, b_t = ops.to_slab(pad(a).t().contiguous()), ops.to_slab(pad(b).t().contiguous())  # [ldt/64, M, 64]
    sa = torch.tensor([2.0 ** 4], device=dev)
    sb = torch.tensor([2.0 ** -2], device=dev)
    ref = ops.wgrad(a_t, b_t, M, N, sa, sb)
    exact = (a.double().t() @ b.double()) / (sa.double() * sb.double())
    # fp32 accumulation over T products: rel-L2 about 1e-5 at T = 65536
    assert float((ref.double() - exact).norm() / exact.norm()) < 1e-4
    assert torch.equal(ops.wgrad_rows(a_rows, b_rows, M, N, sa, sb), ref)
    assert torch.equal(ops.wgrad_rows(a_rows, b_t, M, N, sa, sb, b_rows=False), ref)
    assert torch.equal(ops.wgrad_rows(a_t, b_rows, M, N, sa, sb, a_rows=False), ref)


# The bf16-output GEMMs run 128 x 128 tiles up to 128 tiles of 256 x 256, then
# 192 x 256 (K of 48 stages or more, where they take fewer rounds) or 256 x 256
# ones, a last round of up to 128 of these in halves: both sides of those lines in rows and in columns,
# one row past a tile of either shape, widths that end inside one, the shortest
# K.  The FP8 dgrad has 2I bytes of K, the bf16 GEMM 4I, the forward I.
@pytest.mark.parametrize("T,D,I", [(1, 128, 128), (128, 272, 128), (129, 128, 384), (257, 400, 256),
                                   (8192, 1024, 128), (8193, 1040, 128),
                                   (32768, 256, 128), (32769, 256, 128), (33000, 256, 3072), (9217, 1024, 1536),
                                   (65537, 256, 768), (66000, 256, 1536),
                                   (16641, 1024, 128), (24321, 1040, 128)])
def test_tile_shapes_of_bf16_outputs(dev, T, D, I):
    """Integer operands: every product and sum is exact in fp32 (at most
    64 * 6144 < 2^24), so the rounded result of every tile shape is known."""
    g = torch.Generator(device=dev).manual_seed(T + D + I)
    ldt = sg.ops.ldt_of(T)

    def ints(rows, cols, dtype):
        return torch.randint(-8, 9, (rows, cols), generator=g, device=dev).float().to(dtype)

    def padded(x):
        return sg.ops.to_slab(torch.cat([x, torch.zeros(ldt - T, x.shape[1], device=dev).to(x.dtype)]))

    one = torch.ones(5, device=dev)
    h8, wd8, res = ints(T, I, E4), ints(D, I, E4), ints(T, D, torch.bfloat16)
    y = sg.ops.down_fwd(padded(h8), sg.ops.to_slab(wd8), res, one, one[:2])
    prod = (h8.float() @ wd8.float().t()).bfloat16()
    assert torch.equal(y, (res.float() + prod.float()).bfloat16())
    dgu8, w8t = ints(T, 2 * I, E5), ints(D, 2 * I, E4)
    dxn = sg.ops.gateup_dgrad(padded(dgu8), sg.ops.to_slab(w8t), one, one[:2], T, D)
    assert torch.equal(dxn, (dgu8.float() @ w8t.float().t()).bfloat16())
    a, b = ints(T, 2 * I, torch.bfloat16), ints(D, 2 * I, torch.bfloat16)
    out = sg.ops.bf16_gemm(padded(a), sg.ops.to_slab(b), T, D, 2 * I)
    assert torch.equal(out, (a.float() @ b.float().t()).bfloat16())


# The SwiGLU forwards and the down dgrad run 128-row tiles up to 128 tiles of
# 256 rows and again from 257 to 384, the forwards at some widths
# persistent kernels from 640 tiles of 64 column pairs, the dgrad a last round of
# up to 128 tiles in halves: both sides of each line, with one row in
# the last tile of either shape (whose padding rows the K-slabs keep as zeros)
# and columns that end inside one.
@pytest.mark.parametrize("T,D,I", [(1, 128, 128), (129, 256, 384), (4099, 256, 256), (4097, 128, 1024),
                                   (16385, 128, 256), (32768, 128, 384), (33025, 128, 384), (12289, 256, 1024), (16641, 128, 1024), (25089, 128, 1408),
                                   (9984, 256, 1024), (9985, 256, 1024), (5121, 512, 1920), (5121, 512, 2048),
                                   (5121, 384, 2048), (5121, 640, 2048), (5121, 768, 2048), (4097, 1024, 2560)])
def test_tile_shapes_of_swiglu(dev, T, D, I):
    """FP8 forward and dgrad against the oracle's formulas on the device:
    integer operands make gate, up and dh exact; codes of h and of d_gu may
    differ by one where the sigmoids differ by an ulp."""
    g = torch.Generator(device=dev).manual_seed(T + D + I)
    ldt = sg.ops.ldt_of(T)

    def ints(rows, cols, dtype, n=2):
        return torch.randint(-n, n + 1, (rows, cols), generator=g, device=dev).float().to(dtype)

    def padded(x):
        return sg.ops.to_slab(torch.cat([x, torch.zeros(ldt - T, x.shape[1], device=dev).to(x.dtype)]))

    def close(got, want, fmt, top):
        got, ref = sg.ops.unslab(got, ldt), want.clamp(-top, top).to(fmt)
        assert torch.all(got.view(torch.uint8)[T:] == 0)
        a, b = (v.contiguous().view(torch.uint8).int() for v in (got[:T], ref))
        a, b = (torch.where(v >= 128, 128 - v, v) for v in (a, b))
        assert int((a - b).abs().max()) <= 1 and float((a != b).float().mean()) < 1e-3

    x8, w8 = ints(T, D, E4), ints(2 * I, D, E4)
    s = torch.tensor([1, 2.0 ** -2, 2.0 ** -4, 1, 1], device=dev)
    one, amax = torch.ones(2, device=dev), torch.zeros(5, device=dev)
    gu8, h8, h8t = sg.ops.gateup_swiglu_fwd(padded(x8), sg.ops.to_slab(w8), s, one, amax, T, I)
    gu = x8.float() @ w8.float().t()  # integers below 2^8 * 4: exact in bf16 up to 256, rounded above
    gu = gu.bfloat16().float()
    gate, up = gu.chunk(2, dim=1)
    close(gu8, gu * s[1], E4, 448.0)
    close(h8, gate * torch.sigmoid(gate) * up * s[2], E4, 448.0)
    assert torch.equal(sg.ops.unslab(h8t, I), sg.ops.unslab(h8, ldt).t())
    assert amax[1].item() == gu.abs().max().item()
    dy, wdt = ints(T, D, torch.bfloat16), ints(I, D, torch.bfloat16)
    dgu8, _ = sg.ops.down_dgrad_swiglu(dy, sg.ops.to_slab(wdt), gu8, s, amax, copy=False)
    dh = (dy.float() @ wdt.float().t()).bfloat16().float()
    gate, up = (sg.ops.unslab(gu8, T).float() / s[1]).chunk(2, dim=1)
    sig = torch.sigmoid(gate)
    close(dgu8, torch.cat([dh * up * (sig * (1 + gate * (1 - sig))), dh * gate * sig], 1),
          torch.float8_e5m2, 57344.0)
    # the bf16 forward, from row-major x and from its row K-slab
    xb, wb = x8.float().bfloat16(), w8.float().bfloat16()
    ws, _ = sg.ops.bf16_weight_slabs(wb[None], transposed=False)
    rstd, _, xs = sg.ops.bf16_rows_prep(xb, None, ldt, 1e-6, copy=False, rows=True)
    ones = torch.ones(T, device=dev)
    gub, hb = sg.ops.bf16_swiglu_fwd(xb, ws, I)
    assert torch.equal(gub, gu.bfloat16())
    gate, up = gu.chunk(2, dim=1)
    ref = (gate * torch.sigmoid(gate) * up)
    assert float((hb.float() - ref).norm() / ref.norm().clamp(min=1e-30)) < 2 ** -8  # one bf16 rounding
    for a, b in zip(sg.ops.bf16_swiglu_fwd(xb, ws, I, rstd=ones, xs=xs), (gub, hb)):
        assert torch.equal(a, b)
    pow2 = 2.0 ** torch.randint(-3, 4, (T,), generator=g, device=dev).float()  # rows scaled exactly
    gub, hb = sg.ops.bf16_swiglu_fwd(xb, ws, I, rstd=pow2, xs=xs)
    assert torch.equal(gub.float(), gu * pow2[:, None])
    gate, up = gub.float().chunk(2, dim=1)
    ref = gate * torch.sigmoid(gate) * up
    assert float((hb.float() - ref).norm() / ref.norm().clamp(min=1e-30)) < 2 ** -8


@pytest.mark.parametrize("D", [256, 512, 640])
def test_persistent_bf16_swiglu_grouped(dev, D):
    """The grouped bf16 forward on the persistent kernel has, for each
    expert's rows, the bytes of the dense forward of those rows alone (the
    one-tile kernel): ragged, full-tile, single-row and empty experts."""
    counts, I = [3000, 0, 1, 2049, 256, 700], 1536
    E, R = len(counts), sum(counts)
    g = torch.Generator(device=dev).manual_seed(D)
    x = torch.randn(R, D, generator=g, device=dev).bfloat16()
    w = (torch.randn(E, 2 * I, D, generator=g, device=dev) * D ** -0.5).bfloat16()
    plan = sg.ops.moe_plan(torch.cumsum(torch.tensor(counts), 0).to(torch.int32).to(dev), R)
    ws, _ = sg.ops.bf16_weight_slabs(w, transposed=False)
    gu, h = sg.ops.bf16_swiglu_fwd(x, ws, I, plan=plan, ldp=sg.ops.moe_padded_rows(R, E))
    row = 0
    for e, c in enumerate(counts):
        if c:
            a, b = sg.ops.bf16_swiglu_fwd(x[row:row + c].contiguous(), ws[e:e + 1], I)
            assert torch.equal(gu[row:row + c], a) and torch.equal(h[row:row + c], b)
        row += c


@pytest.mark.parametrize("T,D,I", [(16384, 256, 1024), (10241, 512, 1152), (4099, 1024, 2688)])
def test_persistent_swiglu_exact_path(dev, T, D, I):
    """Rows are independent: NaN, saturating and ordinary rows through the
    persistent kernel (several tiles per work-group) have the bytes that the
    one-tile kernel gives each of them in a batch of a few hundred rows, and
    the maxima are the larger of the batches'."""
    g = torch.Generator(device=dev).manual_seed(T + D)
    x8 = torch.randint(-8, 9, (T, D), generator=g, device=dev).float().to(E4)
    x8.view(torch.uint8)[::97, 3] = 0x7F          # NaN rows
    x8[5::89] = (x8[5::89].float() * 32).to(E4)   # rows beyond the e4m3 range of gu and h
    w8 = torch.randint(-8, 9, (2 * I, D), generator=g, device=dev).float().to(E4)
    s = torch.tensor([1.0, 2.0 ** -4, 2.0 ** -8, 1, 1], device=dev)
    ws, ws8 = torch.ones(2, device=dev), sg.ops.to_slab(w8)

    def run(x):
        n = x.shape[0]
        ldt = sg.ops.ldt_of(n)
        amax = torch.zeros(5, device=dev)
        pad = torch.zeros(ldt - n, D, device=dev).to(E4)
        gu8, h8, _ = sg.ops.gateup_swiglu_fwd(sg.ops.to_slab(torch.cat([x, pad])), ws8, s, ws, amax, n, I, copy=False)
        return u8(sg.ops.unslab(gu8, n)), u8(sg.ops.unslab(h8, n)), amax

    gu, h, amax = run(x8)
    most = torch.zeros(5, device=dev)
    for i in range(0, T, 512):
        a, b, m = run(x8[i:i + 512])
        assert torch.equal(a, gu[i:i + 512]) and torch.equal(b, h[i:i + 512])
        most = torch.maximum(most, m)
    assert torch.equal(most, amax) and amax[1] > 0 and amax[2] > 0


# With one split (few tokens) the gradient is written from its tile:
# 128 x 128 tiles up to 128 work-groups of 256 x 256 (32 x 4 of them at 8192 x
# 1024), 256 x 256 above, a last round of up to 128 in halves;
# M and N that end inside a tile, a half, a pass or a wave; from
# 5003 tokens on sizes that take fewer splits than the most.
@pytest.mark.parametrize("M,N,T", [(64, 64, 1), (192, 320, 257), (448, 192, 900), (8192, 1024, 130),
                                   (8256, 1088, 300), (8448, 1024, 3840), (6144, 1024, 5003),
                                   (1024, 3072, 5003), (6144, 1024, 16384), (12288, 2048, 16384),
                                   (16448, 1088, 300), (8256, 2304, 200)])
def test_one_split_gradients(dev, M, N, T):
    """Integer operands (at most 64 * 16384 < 2^24, exact in fp32): fp8 in every
    layout pair and bf16, and nothing written past the gradient."""
    from spark_gpt_amd import _lib

    ops = sg.ops
    g = torch.Generator(device=dev).manual_seed(M + N + T)
    ldt = ops.ldt_of(T)
    a, b = (torch.zeros(ldt, n, device=dev) for n in (M, N))
    for v in (a, b):
        v[:T] = torch.randint(-8, 9, (T, v.shape[1]), generator=g, device=dev).float()
    ref, s = a.t() @ b, torch.tensor([4.0], device=dev)
    rows = [ops.to_slab(a.to(E5)), ops.to_slab(b.to(E4))]
    cols = [ops.to_slab(a.to(E5).t().contiguous()), ops.to_slab(b.to(E4).t().contiguous())]
    for ar, br in ((True, True), (True, False), (False, True)):
        out = ops.wgrad_rows(rows[0] if ar else cols[0], rows[1] if br else cols[1], M, N, s, s, a_rows=ar, b_rows=br)
        assert torch.equal(out, ref / 16)
    assert torch.equal(ops.wgrad(cols[0], cols[1], M, N, s, s), ref / 16)
    buf = torch.full((M * N + 256,), 12345.0, device=dev)
    ws = torch.empty(max(1, _lib.query("sfp8_wgrad_rows_workspace_floats", M, N, ldt)), device=dev)
    _lib.call("sfp8_gemm_wgrad_rows", rows[0].data_ptr(), 1, 1, rows[1].data_ptr(), 0, 1, M, N, ldt, s.data_ptr(),
              s.data_ptr(), buf.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(buf))
    assert torch.equal(buf[: M * N].view(M, N), ref / 16) and bool((buf[M * N:] == 12345.0).all())
    gs, x = ops.to_slab(a.bfloat16()), b[:T].bfloat16().contiguous()
    assert torch.equal(ops.bf16_wgrad_rows(gs, x, M, N), ref.bfloat16())
    at, bt = (ops.to_slab(v.bfloat16().t().contiguous()) for v in (a, b))
    assert torch.equal(ops.bf16_wgrad(at, bt, M, N), ref.bfloat16())


def test_wgrads_without_workspace(dev):
    """Where the size query says 0 floats a null workspace is taken."""
    from spark_gpt_amd import _lib

    ops = sg.ops
    M, N, ldt = 128, 192, 512
    g = torch.Generator(device=dev).manual_seed(3)
    a, b = (torch.randint(-8, 9, (ldt, n), generator=g, device=dev).float() for n in (M, N))
    ref, one, st = a.t() @ b, torch.ones(1, device=dev), _lib.stream_of(a)
    for q in ("sfp8_wgrad_workspace_floats", "sfp8_wgrad_rows_workspace_floats", "sfp8_bf16_wgrad_workspace_floats"):
        assert _lib.query(q, M, N, ldt) == 0
    f = torch.empty(M, N, device=dev)
    h = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    a8, b8 = ops.to_slab(a.to(E5)), ops.to_slab(b.to(E4))
    _lib.call("sfp8_gemm_wgrad_rows", a8.data_ptr(), 1, 1, b8.data_ptr(), 0, 1, M, N, ldt, one.data_ptr(),
              one.data_ptr(), f.data_ptr(), None, 0, st)
    assert torch.equal(f, ref)
    at, bt = ops.to_slab(a.to(E5).t().contiguous()), ops.to_slab(b.to(E4).t().contiguous())
    _lib.call("sfp8_gemm_wgrad", at.data_ptr(), 1, bt.data_ptr(), 0, M, N, ldt, one.data_ptr(), one.data_ptr(),
              f.zero_().data_ptr(), None, 0, st)
    assert torch.equal(f, ref)
    at, bt = ops.to_slab(a.bfloat16().t().contiguous()), ops.to_slab(b.bfloat16().t().contiguous())
    _lib.call("sfp8_bf16_gemm_wgrad", at.data_ptr(), bt.data_ptr(), M, N, ldt, h.data_ptr(), None, 0, st)
    assert torch.equal(h, ref.bfloat16())
    gs, x = ops.to_slab(a.bfloat16()), b.bfloat16()
    _lib.call("sfp8_bf16_gemm_wgrad_rows", gs.data_ptr(), x.data_ptr(), 1, M, N, ldt, ldt, h.zero_().data_ptr(), None,
              0, st)
    assert torch.equal(h, ref.bfloat16())


@pytest.mark.parametrize("M,N,T,fp8,bf16", [(1600, 2880, 20300, 3, 3), (3136, 1984, 6001, 1, 2),
                                            (1024, 3072, 16384, 5, 5)])
def test_split_gradients_of_large_tiles(dev, M, N, T, fp8, bf16):
    """Several splits in 256 x 256 tiles, fp8 and bf16, ragged in both widths
    and in the tokens: integer operands (at most 64 * 20300 < 2^24, exact in
    fp32), so every partial and every sum is known."""
    from spark_gpt_amd import _lib

    ops = sg.ops
    ldt = ops.ldt_of(T)
    assert [_lib.query("sfp8_wgrad_splits_of", M, N, 0, ldt, b, 0) for b in (0, 1)] == [fp8, bf16]
    g = torch.Generator(device=dev).manual_seed(M + N + T)
    a, b = (torch.zeros(ldt, n, device=dev) for n in (M, N))
    for v in (a, b):
        v[:T] = torch.randint(-8, 9, (T, v.shape[1]), generator=g, device=dev).float()
    ref, one = a.t() @ b, torch.ones(1, device=dev)
    assert torch.equal(ops.wgrad_rows(ops.to_slab(a.to(E5)), ops.to_slab(b.to(E4)), M, N, one, one), ref)
    gs, x = ops.to_slab(a.bfloat16()), b[:T].bfloat16().contiguous()
    assert torch.equal(ops.bf16_wgrad_rows(gs, x, M, N), ref.bfloat16())
    xt = ops.to_slab(b.bfloat16().t().contiguous())
    assert torch.equal(ops.bf16_wgrad_rows(gs, xt, M, N, T=T), ref.bfloat16())
