"""Stride-1 3x3x3 convolutions on 64-pixel column blocks at output widths other than 64, 128 and 256: integer
accumulators exactly, and fp16 results within the rounding of their sums, against a float64 convolution."""
from __future__ import annotations

import numpy as np
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


def _operands(cin, cout, d, h, w, seed):
    gen = torch.Generator(DEV).manual_seed(seed)
    x = torch.randint(-127, 128, (1, d + 2, h + 2, w + 2, cin), generator=gen, dtype=torch.int8, device=DEV)
    x[:, :2] = 0
    wt = torch.randint(-127, 128, (cout, 27 * cin), generator=gen, dtype=torch.int8, device=DEV)
    sx, sw = torch.tensor(0.004, device=DEV), torch.rand(cout, generator=gen, device=DEV) * 2e-3 + 1e-4
    bias = (0.2 * torch.randn(cout, generator=gen, device=DEV)).half()
    res = torch.randn(1, d, h, w, cout, generator=gen, device=DEV).half()
    return x, wt, sx, sw, bias, res, (0.5 * torch.randn(cout, generator=gen, device=DEV)).half()


@pytest.mark.parametrize("cin,cout,d,h,w,with_res,with_bias", [(128, 128, 2, 16, 192, True, False),
                                                               (128, 256, 3, 8, 64, False, True),
                                                               (256, 256, 1, 24, 320, True, True),
                                                               (256, 128, 2, 8, 640, False, False)])
def test_statistics_at_other_widths(ops, oracle, cin, cout, d, h, w, with_res, with_bias):
    """h3v_conv3d_i8_cols: the output of the plain conv, and the tile statistics of the oracle, bit for bit."""
    print(f"cols statistics {cin} -> {cout}, {d} x {h} x {w}", flush=True)
    hip, p = ops.hip, ops.hip.ptr
    x, wt, sx, sw, bias, res, gb = _operands(cin, cout, d, h, w, cin + cout + w)
    res, gb = res if with_res else None, gb if with_bias else None
    head, geo, st = (p(x), p(sx), p(wt), p(sw), p(bias)), (cin, d + 2, h + 2, w + 2, cout), hip.stream(DEV)
    plain = torch.empty(1, d, h, w, cout, dtype=torch.float16, device=DEV)
    if with_res:
        hip.call("h3v_conv3d_i8_residual", *head, p(res), p(plain), 1, *geo, 3, 3, 3, 1, 1, 1, 1, st)
    else:
        hip.call("h3v_conv3d_i8", *head, p(plain), 1, *geo, 3, 3, 3, 1, 1, 1, 1, st)
    out = torch.full_like(plain, float("nan"))
    ws = torch.full((int(hip.lib().h3v_gn_norm_pack_workspace_floats(d, h, w)),), float("nan"), device=DEV)
    hip.call("h3v_conv3d_i8_cols", *head, p(res), None, p(out), *geo, 1, 0, 0, 0, 0, 0, 0, p(gb), p(ws), st)
    torch.cuda.synchronize()
    assert torch.equal(out, plain)
    n = (h // 8) * (w // 64)
    k, flat = d * 32 * n, ws.cpu().numpy()
    avg, m2, ext = oracle.gn_partials_tiled(plain.cpu().numpy()[0], None if gb is None else gb.cpu().numpy())
    assert np.array_equal(flat[:k].view(np.uint32), avg.reshape(-1).view(np.uint32))
    assert np.array_equal(flat[k:2 * k].view(np.uint32), m2.reshape(-1).view(np.uint32))
    assert np.array_equal(flat[2 * k:2 * k + d * n * cout].view(np.uint32), ext.reshape(-1))


@pytest.mark.parametrize("cin,cout,d,h,w,front,border,pack_bias", [
    (128, 128, 2, 8, 192, 2, (1, 1, 1, 1), False), (256, 256, 1, 16, 320, 2, (0, 1, 0, 1), True),
    (128, 256, 3, 8, 64, 1, (1, 0, 0, 1), True), (128, 128, 1, 24, 640, 0, (0, 0, 0, 0), False)])
def test_padded_output_at_other_widths(ops, cin, cout, d, h, w, front, border, pack_bias):
    """h3v_conv3d_i8_cols: the plain conv's output padded as the downsample reads it, bit for bit."""
    print(f"cols padded {cin} -> {cout}, {d} x {h} x {w}, front {front}, border {border}", flush=True)
    hip, p = ops.hip, ops.hip.ptr
    x, wt, sx, sw, bias, res, rb = _operands(cin, cout, d, h, w, cin + cout + w + front)
    bias, rb = (None, rb) if pack_bias else (bias, None)
    head, geo, st = (p(x), p(sx), p(wt), p(sw), p(bias)), (cin, d + 2, h + 2, w + 2, cout), hip.stream(DEV)
    y = torch.empty(1, d, h, w, cout, dtype=torch.float16, device=DEV)
    hip.call("h3v_conv3d_i8", *head, p(y), 1, *geo, 3, 3, 3, 1, 1, 1, 1, st)
    v = (res.float() + (y.float() + rb.float())).half() if pack_bias else res + y
    top, bottom, left, right = border
    rows = [1] * top + list(range(h)) + [h - 2] * bottom
    cols = [1] * left + list(range(w)) + [w - 2] * right
    want = v[:, :, rows][:, :, :, cols]
    out = torch.full((1, d + front, h + top + bottom, w + left + right, cout), 7.5, dtype=torch.float16, device=DEV)
    hip.call("h3v_conv3d_i8_cols", *head, p(res), p(rb), p(out), *geo, 1, 1, front, *border, None, None, st)
    torch.cuda.synchronize()
    assert torch.equal(out[:, front:], want)
    assert bool((out[:, :front] == 7.5).all())     # the frames in front are the caller's


def _between_boundaries(t):
    """The same values and strides, starting 2 bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    view = flat[1:].as_strided(t.shape, t.stride(), 1)
    assert view.copy_(t).data_ptr() % 16 == 2
    return view


@pytest.mark.parametrize("padded", [False, True])
def test_residual_and_biases_between_16_byte_boundaries(ops, padded):
    """The Python entries take such views at these widths as they do where the plain conv runs."""
    print(f"cols unaligned views, padded {padded}", flush=True)
    e8 = ops.encoder_int8
    x, wt, sx, sw, bias, res, gb = _operands(128, 128, 6, 64, 192, 5)
    qx, res = x.permute(0, 4, 1, 2, 3), res.permute(0, 4, 1, 2, 3)

    def run(res, extra):
        if padded:
            return e8._conv3d_from_quantized_padded(qx, sx, wt, sw, bias=None, residual=res, residual_bias=extra, front=2,
                                                    border=(0, 1, 0, 1))
        ws = torch.zeros(e8.gn_workspace_floats(6, 64, 192), device=DEV)
        config = e8.Int8Conv3DConfig(128, 128, (3, 3, 3), (1, 1, 1))
        out = e8._conv3d_from_quantized(qx, sx, wt, sw, config=config, bias=bias, tile_variant="64x64x64",
                                        causal_prefix_zero=True, residual=res, gn_workspace=ws, gn_bias=extra)
        return torch.cat([out.flatten().float(), ws[:2 * 6 * 32 * 24]])
    with torch.inference_mode():
        want, got = run(res, gb), run(_between_boundaries(res), _between_boundaries(gb))
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_cols_refuses_other_calls(ops):
    z = torch.zeros(64, device=DEV)
    p, geo = ops.hip.ptr(z), (128, 4, 10, 66, 128)

    def call(geometry=geo, res=None, rb=None, padded=0, front=0, border=(0, 0, 0, 0), ws=p):
        ops.hip.call("h3v_conv3d_i8_cols", p, p, p, p, None, res, rb, p, *geometry, 1, padded, front, *border, None, ws,
                     ops.hip.stream(DEV))
    for match, kwargs in (("multiple of 64", {"geometry": (128, 4, 10, 98, 128)}),
                          ("multiple of 8", {"geometry": (128, 4, 14, 66, 128)}),
                          ("Cin % 128", {"geometry": (64, 4, 10, 66, 128)}),
                          ("128 or 256", {"geometry": (128, 4, 10, 66, 384)}),
                          ("either", {"padded": 1}), ("either", {"ws": None}),
                          ("needs a residual", {"rb": p}), ("alias", {"res": p}),
                          ("front", {"padded": 1, "ws": None, "front": 17}),
                          ("border", {"padded": 1, "ws": None, "border": (0, 2, 0, 0)})):
        with pytest.raises(ValueError, match=match):
            call(**kwargs)


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
