"""Stride-1 3x3x3 convolutions on 64-pixel column blocks at output widths other than 64, 128 and 256: integer
accumulators exactly, and fp16 results within the rounding of their sums, against a float64 convolution."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _conv64(x, w, d, h, wd):
    """Valid 3x3x3 conv of NDHWC x with w [O, 27 * C], k = (kd, kh, kw, c), in float64."""
    b, c, o = x.shape[0], x.shape[-1], w.shape[0]
    w = w.double().view(o, 27, c)
    out = torch.zeros(b, d, h, wd, o, dtype=torch.float64, device=DEV)
    for t in range(27):
        kd, kh, kw = t // 9, t // 3 % 3, t % 3
        part = x[:, kd:kd + d, kh:kh + h, kw:kw + wd].double().reshape(-1, c)
        out.view(-1, o).addmm_(part, w[:, t].t().contiguous())
    return out


# (batch, Cin, Cout, D, H, W): at least 128 tiles of 8 x 64 pixels x 128 channels, the edges of the tile order
# (one column block of 64, odd counts of blocks and row groups, one row group), both channel counts
SHAPES = [(1, 128, 128, 3, 120, 192), (1, 128, 128, 2, 136, 320), (1, 256, 128, 5, 8, 1664), (1, 128, 256, 3, 72, 192),
          (2, 128, 256, 1, 64, 576), (1, 256, 256, 4, 40, 320)]


@pytest.mark.parametrize("b,cin,cout,d,h,w", SHAPES)
def test_int8_exact(ops, b, cin, cout, d, h, w):
    print(f"cols int8 {b} x {cin} -> {cout}, {d} x {h} x {w}", flush=True)
    gen = torch.Generator(DEV).manual_seed(b + cin + d + h + w)
    x = torch.randint(-127, 128, (b, d + 2, h + 2, w + 2, cin), generator=gen, dtype=torch.int8, device=DEV)
    x[:, :2] = 0
    wt = torch.randint(-127, 128, (cout, 27 * cin), generator=gen, dtype=torch.int8, device=DEV)
    acc = torch.empty(b, d, h, w, cout, dtype=torch.int32, device=DEV)
    p, hip = ops.hip.ptr, ops.hip
    hip.call("h3v_conv3d_i8_i32", p(x), p(wt), p(acc), b, cin, d + 2, h + 2, w + 2, cout, 3, 3, 3, 1, 1, 1, 1,
             hip.stream(DEV))
    want = _conv64(x, wt, d, h, w)
    assert torch.equal(acc, want.to(torch.int32))
    # dequant with bias and residual: fp16(fp32(res) + fp16(fma(acc * sx, sw, bias))) around the exact sums
    sx, sw = torch.tensor(0.03, device=DEV), torch.rand(cout, generator=gen, device=DEV) * 1e-3 + 1e-4
    bias = torch.randn(cout, generator=gen, device=DEV).half()
    res = torch.randn(b, d, h, w, cout, generator=gen, device=DEV).half()
    out = torch.empty_like(res)
    hip.call("h3v_conv3d_i8_residual", p(x), p(sx), p(wt), p(sw), p(bias), p(res), p(out), b, cin, d + 2, h + 2, w + 2,
             cout, 3, 3, 3, 1, 1, 1, 1, hip.stream(DEV))
    y = want * sx.double() * sw.double() + bias.double()
    # one fp16 rounding of y (2^-11 |y|), fp32 roundings far below it, one of the sum
    bound = 2.0 ** -11 * (1.01 * y.abs() + (y + res.double()).abs()) + 1e-6
    assert bool(((out.double() - (y + res.double())).abs() <= bound).all())


@pytest.mark.parametrize("b,cin,cout,d,h,w", [(1, 64, 128, 3, 120, 192), (1, 128, 128, 2, 64, 640), (1, 256, 256, 3, 40, 320),
                                              (2, 128, 256, 2, 64, 192), (1, 128, 128, 3, 64, 256),
                                              (1, 128, 256, 2, 64, 128)])
def test_f16_within_rounding(ops, b, cin, cout, d, h, w):
    print(f"cols fp16 {b} x {cin} -> {cout}, {d} x {h} x {w}", flush=True)
    gen = torch.Generator(DEV).manual_seed(b + cin + d + h + w)
    x = torch.randn(b, d + 2, h + 2, w + 2, cin, generator=gen, device=DEV).half()
    x[:, :2] = 0
    wt = (0.02 * torch.randn(cout, 27 * cin, generator=gen, device=DEV)).half()
    bias = torch.randn(cout, generator=gen, device=DEV).half()
    out = torch.empty(b, d, h, w, cout, dtype=torch.float16, device=DEV)
    p, hip = ops.hip.ptr, ops.hip
    hip.call("h3v_conv3d_f16", p(x), p(wt), p(bias), None, p(out), b, cin, d + 2, h + 2, w + 2, cout, 3, 3, 3, 1, 1, 1,
             1, hip.stream(DEV))
    want = _conv64(x, wt, d, h, w) + bias.double()
    # fp32 sums of 27 * cin products: at most n * 2^-24 of the sum of magnitudes; one fp16 rounding
    mags = _conv64(x.abs(), wt.abs(), d, h, w)
    bound = 27 * cin * 2.0 ** -24 * mags + 2.0 ** -11 * 1.01 * want.abs() + 1e-6
    assert bool(((out.double() - want).abs() <= bound).all())
