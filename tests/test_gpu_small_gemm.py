"""The INT8 GEMM's tiles for outputs that do not fill the chip, and its split of the last rows: integer sums
exactly against a float64 product (every sum is below 2^53), the fp16 epilogue bit for bit against the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import assert_bitwise, np_

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# K steps of 128: 1 ... 4 fill the ring, odd and even counts end on either fragment buffer
SIZES = [
    # 64 x 64 tiles (up to 512 of them)
    (1, 1, 128, True), (63, 65, 256, True), (64, 64, 384, False), (65, 200, 512, True), (129, 37, 640, False),
    (453, 2048, 768, True), (1013, 2048, 1152, True), (128, 16384, 128, False),
    # 128 x 128 tiles, one per CU (more than 512 tiles of 64 x 64, up to 256 of 128 x 128)
    (453, 6144, 128, True), (1797, 2048, 640, False), (2048, 2048, 512, True), (1100, 2050, 384, True),
    # 128 x 128 tiles, two per CU (257 to 512)
    (453, 16384, 256, True), (3594, 2047, 128, False), (2049, 2049, 896, True),
    # ping-pong tiles with the last rows split off (to each small tile) or kept
    (4225, 4224, 128, True), (8405, 2048, 256, True), (4609, 4096, 384, False), (3000, 6144, 128, True),
    (4100, 2048, 128, True),
]


@pytest.mark.parametrize("m,n,k,with_bias", SIZES)
def test_gemm_tiles_exact(oracle, m, n, k, with_bias):
    from h3_arch import _pkg
    hip = _pkg._hip
    print(f"small gemm m={m} n={n} k={k}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m * 7 + n * 3 + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, dtype=torch.int8, device=DEV)
    w = torch.randint(-127, 128, (n, k), generator=gen, dtype=torch.int8, device=DEV)
    sx = torch.rand(m, generator=gen, device=DEV) * 0.02 + 0.001
    sw = torch.rand(n, generator=gen, device=DEV) * 0.02 + 0.001
    bias = torch.randn(n, generator=gen, device=DEV).half() if with_bias else None
    acc = torch.full((m, n), 7, dtype=torch.int32, device=DEV)
    out = torch.empty((m, n), dtype=torch.float16, device=DEV)
    hip.call("h3v_gemm_i8_i32", hip.ptr(a), hip.ptr(w), hip.ptr(acc), m, n, k, hip.stream(DEV))
    hip.call("h3v_gemm_i8_dequant", hip.ptr(a), hip.ptr(sx), hip.ptr(w), hip.ptr(sw), hip.ptr(bias), hip.ptr(out),
             m, n, k, hip.stream(DEV))
    side, other = torch.cuda.Stream(), torch.full_like(acc, 7)   # on another stream the choice of tiles is narrower
    side.wait_stream(torch.cuda.current_stream())
    hip.call("h3v_gemm_i8_i32", hip.ptr(a), hip.ptr(w), hip.ptr(other), m, n, k, side.cuda_stream)
    torch.cuda.synchronize()
    want = (a.double() @ w.double().t()).to(torch.int32)
    assert torch.equal(acc, want) and torch.equal(other, want)
    assert_bitwise(np_(out), oracle.gemm_dequant(np_(want), np_(sx), np_(sw), None if bias is None else np_(bias)), "out")
    assert np.isfinite(np_(out)).all()
