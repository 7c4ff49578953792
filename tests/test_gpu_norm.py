"""GPU parity: norm-fused quantizer (bit-exact) and norm backward."""
import pytest
import torch

import spark_gpt_amd as sg
from oracle import fp8_mlp as O

pytestmark = pytest.mark.gpu


def u8(t):
    return t.contiguous().view(torch.uint8).cpu()


CASES = [(1, 128), (257, 256), (1000, 256), (333, 512), (1000, 1024), (4099, 1024), (300, 2048),
         (200, 4096), (300, 8192), (1, 8192), (129, 16384)]


@pytest.mark.parametrize("T,D", CASES)
def test_norm_quant_bit_exact(dev, T, D):
    g = torch.Generator().manual_seed(T + D)
    h = (torch.randn(T, D, generator=g) * 3).to(torch.bfloat16)
    nw = torch.empty(D).uniform_(0.5, 1.5, generator=g)
    s0 = 16.0
    scale = torch.tensor([s0, 1, 1, 1, 1], device=dev)
    amax = torch.zeros(5, device=dev)
    x8, x8t, rstd = sg.ops.norm_quant(h.to(dev), nw.to(dev), scale, amax, 1e-6)
    r8, r8t, rr, ra = O.norm_quant(h, nw, torch.tensor(s0), 1e-6)
    assert torch.equal(rstd.cpu(), rr)
    ldt = sg.ops.ldt_of(T)
    assert x8.shape == (D // 64, ldt, 64)
    assert torch.equal(u8(sg.ops.unslab(x8, T)), u8(r8))
    assert torch.all(u8(sg.ops.unslab(x8, ldt))[T:] == 0)
    assert x8t.shape == (ldt // 64, sg.ops.slab_rows(D), 64)
    xt = u8(sg.ops.unslab(x8t, D))
    assert torch.equal(xt[:, :T], u8(r8t))
    assert torch.all(xt[:, T:] == 0)
    assert amax[0].item() == ra.item()
    # without the token-contiguous copy: the same x8 (padding included), rstd and amax
    amax2 = torch.zeros(5, device=dev)
    x8b, none, rstd2 = sg.ops.norm_quant(h.to(dev), nw.to(dev), scale, amax2, 1e-6, copy=False)
    assert none is None
    assert torch.equal(u8(x8b), u8(x8)) and torch.equal(rstd2, rstd) and torch.equal(amax2, amax)


def test_norm_quant_heavy_tails(dev):
    """Student-t(3) activations: saturation at +-448 and tiny values."""
    T, D = 2048, 2048
    g = torch.Generator().manual_seed(11)
    z = torch.randn(T, D, generator=g)
    chi = (torch.randn(T, D, 3, generator=g) ** 2).sum(-1)  # chi-square, 3 dof
    h = (z / torch.sqrt(chi / 3)).to(torch.bfloat16)
    nw = torch.ones(D)
    scale = torch.tensor([64.0, 1, 1, 1, 1], device=dev)
    amax = torch.zeros(5, device=dev)
    x8, x8t, rstd = sg.ops.norm_quant(h.to(dev), nw.to(dev), scale, amax, 1e-6)
    r8, r8t, rr, ra = O.norm_quant(h, nw, torch.tensor(64.0), 1e-6)
    assert torch.equal(rstd.cpu(), rr)
    assert torch.equal(u8(sg.ops.unslab(x8, T)), u8(r8))
    assert amax[0].item() == ra.item()
    assert (u8(r8) & 0x7F).eq(0x7E).any()  # some saturate


@pytest.mark.parametrize("T,D", [(1000, 256), (257, 1024), (4099, 1024), (300, 4096), (300, 8192),
                                 (65, 16384)])
def test_norm_bwd(dev, T, D):
    g = torch.Generator().manual_seed(T * D)
    h = torch.randn(T, D, generator=g).to(torch.bfloat16)
    nw = torch.empty(D).uniform_(0.5, 1.5, generator=g)
    dxn = torch.randn(T, D, generator=g).to(torch.bfloat16)
    dy = (torch.randn(T, D, generator=g) * 1e-3).to(torch.bfloat16)
    rstd = O.norm_stats(h, 1e-6)
    scale = torch.tensor([1, 1, 1, 1, 2.0 ** 15], device=dev)
    amax = torch.zeros(5, device=dev)
    dh, dnw, dy8t = sg.ops.norm_bwd(h.to(dev), rstd.to(dev), dxn.to(dev), dy.to(dev), nw.to(dev), scale, amax)
    rdh, rdnw = O.norm_bwd(h, rstd, dxn, dy, nw)
    # sums over D/T in a different order: dh within one bf16 ulp, dnw to fp32 rounding
    torch.testing.assert_close(dh.cpu().float(), rdh.float(), rtol=8e-3, atol=1e-6)
    assert O.rel_l2(dh.cpu().float(), rdh.float()) < 1e-3
    torch.testing.assert_close(dnw.cpu(), rdnw, rtol=1e-4, atol=1e-4)
    ref8 = O.e5m2(dy.float() * 2.0 ** 15)
    yt = u8(sg.ops.unslab(dy8t, D))
    assert torch.equal(yt[:, :T], u8(ref8).t())
    assert torch.all(yt[:, T:] == 0)
    assert amax[4].item() == dy.float().abs().max().item()
    # dy8 as the K-slab of [T, D] instead: the same dh, dnw and amax
    amax2 = torch.zeros(5, device=dev)
    dh2, dnw2, dy8 = sg.ops.norm_bwd(h.to(dev), rstd.to(dev), dxn.to(dev), dy.to(dev), nw.to(dev), scale, amax2,
                                     rows=True)
    assert torch.equal(dh2, dh) and torch.equal(dnw2, dnw) and torch.equal(amax2, amax)
    ldt = sg.ops.ldt_of(T)
    assert dy8.shape == (D // 64, ldt, 64)
    y8 = u8(sg.ops.unslab(dy8, ldt))
    assert torch.equal(y8[:T], u8(ref8))
    assert torch.all(y8[T:] == 0)


@pytest.mark.parametrize("T,D", [(16385, 1024), (8192, 2048)])
def test_row_block_sizes_agree(dev, T, D):
    """At these widths the norm kernels take 64 (32 at D = 2048) rows a
    work-group from 256 row blocks on, below 16: a row's bytes do not depend on it, nor the maxima;
    the norm weight's gradient is an fp32 sum of T rows in another order
    (relative error of a pairwise-like sum over 16 to 64 rows a block: 1e-5)."""
    from spark_gpt_amd import _lib

    ops = sg.ops
    ldt, few = ops.ldt_of(T), ops.ldt_of(T) // 2 // 256 * 256
    blocks = lambda n: _lib.query("sfp8_norm_bwd_partials", D, n) - 32
    assert blocks(ldt) == ldt // (64 if D < 2048 else 32) and blocks(few) == few // 16
    g = torch.Generator(device=dev).manual_seed(T + D)
    h, dxn = (torch.randn(T, D, generator=g, device=dev).bfloat16() for _ in range(2))
    dy = (torch.randn(T, D, generator=g, device=dev) * 1e-3).bfloat16()
    nw = torch.rand(D, generator=g, device=dev) + 0.5
    scale = torch.tensor([32.0, 1, 1, 1, 2.0 ** 20], device=dev)

    def run(a, b):
        amax = torch.zeros(5, device=dev)
        n = b - a
        x8, x8t, rstd = ops.norm_quant(h[a:b], nw, scale, amax, 1e-6)
        dh, dnw, dy8t = ops.norm_bwd(h[a:b], rstd, dxn[a:b], dy[a:b], nw, scale, amax)
        assert torch.equal(ops.unslab(x8t, D).view(torch.uint8)[:, :n], ops.unslab(x8, n).view(torch.uint8).t())
        return (ops.unslab(x8, n).view(torch.uint8), rstd, dh, ops.unslab(dy8t, D).view(torch.uint8)[:, :n].t()), dnw, amax

    whole, dnw, amax = run(0, T)
    parts = [run(a, min(T, a + few)) for a in range(0, T, few)]
    for i, w in enumerate(whole):
        assert torch.equal(torch.cat([p[0][i] for p in parts]), w)
    assert torch.equal(torch.stack([p[2] for p in parts]).amax(0), amax)
    exact = (dxn.double() * h.double() * whole[1].double()[:, None]).sum(0)
    for got in (dnw.double(), sum(p[1].double() for p in parts)):
        assert float((got - exact).norm() / exact.norm()) < 1e-5


@pytest.mark.parametrize("T,D", [(1, 64), (17, 320), (4099, 768), (300, 1024)])
def test_bf16_rows_slab(dev, T, D):
    """rstd and the row K-slab of dense rows without the transposed copy: the
    slab is x's bytes with zero padding rows, rstd the fp32 rounding of the
    exact sum of squares (one more rounding each for the mean and the root)."""
    ops = sg.ops
    x = torch.randn(T, D, device=dev).bfloat16()
    ldt = ops.ldt_of(T)
    rstd, none, xs = ops.bf16_rows_prep(x, None, ldt, 1e-6, copy=False, rows=True)
    assert none is None
    ref = torch.cat([x, torch.zeros(ldt - T, D, device=dev, dtype=x.dtype)])
    assert torch.equal(ops.unslab(xs, ldt).view(torch.uint8), ref.view(torch.uint8).view(ldt, 2 * D))
    want = torch.rsqrt(x.double().square().mean(1) + 1e-6)
    assert float(((rstd.double() - want) / want).abs().max()) < 2 ** -22
    only, _, _ = ops.bf16_rows_prep(x, None, ldt, 1e-6, copy=False)
    both, xt, xs2 = ops.bf16_rows_prep(x, None, ldt, 1e-6, rows=True)
    assert torch.equal(only, rstd) and torch.equal(both, rstd) and torch.equal(xs2, xs)
    assert torch.equal(ops.unslab(xt, D).view(torch.int16), ref.t().contiguous().view(torch.int16))
