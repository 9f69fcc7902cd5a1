"""GPU parity: decoder attention (h3v_attention_d64) against the float64 oracle.

Tolerance: the kernel rounds the softmax weights to fp16 for the P.V product and
the output to fp16; against float64 it stays within |err| <= 2e-3 + 4e-3 |ref|
for N(0, 1) values (half an fp16 ulp of the output is 2.4e-4 |ref|).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
ATOL, RTOL = 2e-3, 4e-3


def _qkv(b, n, h, seed, qk_scale=1.0):
    """q, k [B, N, H, 64] contiguous and v as the strided slice of a [B, N, H*192] projection."""
    gen = torch.Generator().manual_seed(seed)
    qkv = torch.randn(b, n, h * 192, generator=gen).half()
    q = (torch.randn(b, n, h, 64, generator=gen) * qk_scale).half()
    k = (torch.randn(b, n, h, 64, generator=gen) * qk_scale).half()
    qkv_d = qkv.to(DEV)
    v_d = qkv_d.view(b, n, h, 192)[..., 128:]
    v = qkv.view(b, n, h, 192)[..., 128:]
    return q, k, v, q.to(DEV), k.to(DEV), v_d


def _check(ops, oracle, q, k, v, out, queries=None):
    ref = oracle.attention(q.numpy(), k.numpy(), v.numpy(), 0.125, queries)
    got = out.cpu().numpy().astype(np.float64)
    if queries is not None:
        got = got[:, queries]
    err = np.abs(got - ref)
    bound = ATOL + RTOL * np.abs(ref)
    worst = float((err / bound).max())
    assert worst <= 1.0, f"max err {err.max():.3e} ({worst:.2f} of the bound)"


@pytest.mark.parametrize("b,n,h", [(1, 1, 1), (1, 2, 2), (2, 63, 1), (1, 64, 2), (3, 65, 1), (1, 129, 2),
                                   (2, 200, 3), (1, 513, 1), (2, 1025, 1), (1, 1100, 2), (1, 1537, 1)])
def test_attention_small_shapes_match_oracle(ops, oracle, b, n, h):
    """Key-block (64) and wave (64 queries) edges, and the workgroup edges: a workgroup holds 8 waves of 64
    queries (512), so 513, 1025, 1100 and 1537 tokens put ragged workgroups after full ones; one token, odd
    batches and heads.  Every query is checked."""
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=b * 1000 + n * 10 + h)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
    torch.cuda.synchronize()
    assert out.shape == (b, n, h, 64) and out.is_contiguous()
    _check(ops, oracle, q, k, v, out)


def test_attention_h3_shape_sampled(ops, oracle):
    """H3 decoder call: B4 x 1797 tokens x 32 heads; the last query and key blocks are ragged."""
    print("attention H3 [4, 1797, 32, 64]", flush=True)
    b, n, h = 4, 1797, 32
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=1797)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
    torch.cuda.synchronize()
    rng = np.random.default_rng(5)
    # workgroup (512-query) and wave (64-query) edges, the ragged tail, random others
    edges = [0, 1, 63, 64, 127, 128, 511, 512, 1023, 1024, 1535, 1536, 1791, 1792, 1795, 1796]
    queries = np.unique(np.concatenate([edges, rng.integers(0, n, 40)]))
    _check(ops, oracle, q, k, v, out, queries)


def test_attention_large_scores_online_max(ops, oracle):
    """Scores ~ N(0, 64): the running maximum changes across key blocks and exp would overflow without it."""
    q, k, v, qd, kd, vd = _qkv(2, 300, 2, seed=77, qk_scale=2.83)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    _check(ops, oracle, q, k, v, out)


@pytest.mark.parametrize("direction", [1, -1])
def test_attention_score_ramp_moves_the_lazy_maximum(ops, oracle, direction):
    """The kernel's reference maximum moves only when a score exceeds it by more than 8 / (scale * log2 e)
    (a weight above 2^8).  Key norms growing with the key index make the maximum jump past that margin in
    many blocks (the O and l rescale runs repeatedly); the reverse ramp sets it in the first block and
    leaves later weights tiny (no rescale after block 0, deep exponents)."""
    b, n, h = 1, 700, 2
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=91 + direction)
    ramp = torch.linspace(0.2, 6.0, n) if direction > 0 else torch.linspace(6.0, 0.2, n)
    k = (k.float() * ramp.view(1, n, 1, 1)).half()
    kd = k.to(DEV)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    _check(ops, oracle, q, k, v, out)


def test_attention_cfg4_sampled_and_against_torch_sdpa(ops, oracle):
    """one 256x256 tile, 16384 tokens x 16 heads; also compared with torch's SDPA."""
    print("attention cfg4 [1, 16384, 16, 64]", flush=True)
    b, n, h = 1, 16384, 16
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=4)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
        sdpa = torch.nn.functional.scaled_dot_product_attention(
            qd.transpose(1, 2), kd.transpose(1, 2), vd.transpose(1, 2).contiguous(), scale=0.125).transpose(1, 2)
    torch.cuda.synchronize()
    rng = np.random.default_rng(6)
    edges = [0, 511, 512, 8191, 8192, 16383]
    queries = np.unique(np.concatenate([edges, rng.integers(0, n, 24)]))
    _check(ops, oracle, q, k, v, out, queries)
    assert float((out.float() - sdpa.float()).abs().max()) < 4e-3


def test_attention_rejects_bad_layouts(ops):
    qd = torch.zeros(1, 8, 2, 64, dtype=torch.float16, device=DEV)
    att = ops.decoder_fused_qk_rope.attention_d64
    with pytest.raises(ValueError, match="one shape"):
        att(qd, qd[:, :4], qd, 0.125)
    with pytest.raises(ValueError, match="FP16"):
        att(qd.float(), qd.float(), qd.float(), 0.125)
    odd = torch.zeros(1, 8, 2, 68, dtype=torch.float16, device=DEV)[..., :64]    # head stride 68
    with pytest.raises(ValueError, match="strides"):
        att(odd, odd, odd, 0.125)
    with pytest.raises(ValueError, match="scale"):
        att(qd, qd, qd, 0.0)


# (batch, tokens, heads) per workgroup shape and split, at the edges of the rule that picks them; `head`: the queries
# before those past the full rounds, which take the key-split kernel and its merge (all of them where nothing splits)
@pytest.mark.parametrize("b,n,h,head", [
    (1, 65, 64, 65), (1, 1025, 21, 1025),                  # 128-query workgroups
    (1, 64, 65, 64), (2, 453, 40, 453),                    # 256 queries
    (1, 300, 129, 300), (2, 513, 64, 513),                 # 512 queries, one full round
    (1, 600, 150, 600), (5, 520, 30, 520),                 # 4-wave workgroups
    (4, 1025, 32, 1024), (2, 2049, 32, 2048), (2, 2300, 32, 2048), (1, 4097, 32, 4096), (1, 4101, 31, 4096),
    (1, 8250, 16, 8192),
])
def test_attention_workgroup_shapes_and_key_splits(ops, oracle, b, n, h, head):
    print(f"attention shapes [{b}, {n}, {h}, 64]", flush=True)
    floats = int(ops.hip.lib().h3v_attention_d64_workspace_floats(b, n, h))
    # fp32 rows of 64 outputs, a maximum and a sum, per split and split query
    assert floats == 0 if head == n else floats > 0 and floats % (b * h * (n - head) * 66) == 0
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=b * 100 + n + h)
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
        plain = torch.empty_like(out)
        ops.hip.call("h3v_attention_d64", ops.hip.ptr(qd), qd.stride(1), qd.stride(2), ops.hip.ptr(kd), kd.stride(1),
                     kd.stride(2), ops.hip.ptr(vd), vd.stride(1), vd.stride(2), ops.hip.ptr(plain), out.stride(1),
                     out.stride(2), b, n, h, 0.125, ops.hip.stream(DEV))
    torch.cuda.synchronize()
    # a few heads against the oracle (every path sees every head alike), the last queries and the edges
    heads = sorted({0, h // 2, h - 1})
    rng = np.random.default_rng(n)
    queries = np.unique(np.concatenate([[0, 31, 32, 63], np.arange(max(0, n - 6), n), rng.integers(0, n, 24)]) % n)
    for got in (out, plain):
        _check(ops, oracle, q[:, :, heads], k[:, :, heads], v[:, :, heads].contiguous(), got[:, :, heads], queries)
    # the two entries differ in the split queries only, by the order of fp32 sums
    same = (out == plain).all(dim=3).all(dim=2).all(dim=0)
    assert bool(same[:head].all())
    assert float((out.float() - plain.float()).abs().max()) < 2e-3


# last rounds of 512-query workgroups half full, 5/8 full, and after four rounds; a key split
@pytest.mark.parametrize("b,n,h", [(12, 453, 32), (13, 453, 32), (33, 453, 32), (2, 2049, 32)])
def test_attention_on_another_stream(ops, b, n, h):
    """A call on another stream than the default one may take larger workgroups; every query keeps its wave's 64."""
    print(f"attention on another stream [{b}, {n}, {h}, 64]", flush=True)
    _, _, _, qd, kd, vd = _qkv(b, n, h, seed=b + n)
    att, side = ops.decoder_fused_qk_rope.attention_d64, torch.cuda.Stream()
    with torch.inference_mode():
        out = att(qd, kd, vd, 0.125)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            other = att(qd, kd, vd, 0.125)
        torch.cuda.synchronize()
    assert torch.equal(other, out)


@pytest.mark.parametrize("ramp", [False, True])
@pytest.mark.parametrize("b", [4, 8, 10])    # 256 queries per workgroup, 512, 256 on four waves; one item alone: 128
def test_attention_of_an_item_alone_and_in_a_batch(ops, b, ramp):
    """The queries of a wave move their reference maximum together, so a workgroup shape may weigh a query's keys
    against another reference: the fp16 weights then round differently (2^-11 each), in the sum and in the product,
    on either side.  4 * 2^-11 of the weighted |v|, and the output's own rounding."""
    n, h = 453, 32
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=31 + b)
    if ramp:
        kd = (k.float() * torch.linspace(0.2, 6.0, n).view(1, n, 1, 1)).half().to(DEV)
    att = ops.decoder_fused_qk_rope.attention_d64
    with torch.inference_mode():
        out, mag = att(qd, kd, vd, 0.125).float(), att(qd, kd, vd.abs(), 0.125).float()
        for i in (0, b - 1):
            alone = att(qd[i:i + 1].contiguous(), kd[i:i + 1].contiguous(), vd[i:i + 1], 0.125)[0].float()
            assert bool(((out[i] - alone).abs() <= 2.0 ** -9 * mag[i] + 2.0 ** -10 * alone.abs() + 2.0 ** -24).all())


def test_attention_key_splits_carry_large_scores(ops, oracle):
    """Splits whose reference maxima differ by far more than 2^8: key norms rise along the sequence, so the last
    split holds nearly all the weight and the others' outputs are scaled to nothing."""
    b, n, h = 2, 2100, 32
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=17)
    k = (k.float() * torch.linspace(0.2, 6.0, n).view(1, n, 1, 1)).half()
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, k.to(DEV), vd, 0.125)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    queries = np.arange(2040, n)
    _check(ops, oracle, q[:, :, :2], k[:, :, :2], v[:, :, :2].contiguous(), out[:, :, :2], queries)


@pytest.mark.parametrize("first,last", [(1024, 2049), (512, 1600)])
def test_attention_key_splits_without_a_finite_score(ops, first, last):
    """Keys of minus infinite score over whole splits weigh nothing, in the split queries as in the others."""
    b, n, h = 2, 2049, 32
    q, k, v, qd, kd, vd = _qkv(b, n, h, seed=23)
    qd, kd = qd.clone(), kd.clone()
    qd[..., 0] = qd[..., 0].abs() + 0.1
    kd[:, first:last, :, 0] = -float("inf")
    with torch.inference_mode():
        out = ops.decoder_fused_qk_rope.attention_d64(qd, kd, vd, 0.125)
    torch.cuda.synchronize()
    keep = [t for t in range(n) if not first <= t < last]
    for i in (0, 2000, 2047, 2048):
        qs, ks, vs = (x.double().cpu().transpose(1, 2) for x in (qd[:, i:i + 1], kd[:, keep], vd[:, keep]))
        want = torch.softmax(qs @ ks.transpose(2, 3).contiguous() * 0.125, dim=-1) @ vs
        err = (out[:, i:i + 1].double().cpu().transpose(1, 2) - want).abs()
        assert bool((err <= 2e-3 + 4e-3 * want.abs()).all())


def test_attention_workspace_is_required_for_splits(ops):
    b, n, h = 4, 1025, 32
    x = torch.zeros(b, n, h, 64, dtype=torch.float16, device=DEV)
    need = int(ops.hip.lib().h3v_attention_d64_workspace_floats(b, n, h))
    ws = torch.empty(need, dtype=torch.float32, device=DEV)
    args = (ops.hip.ptr(x), x.stride(1), x.stride(2)) * 4 + (b, n, h, 0.125)
    for bad in ((None, 0), (ops.hip.ptr(ws), need - 1)):
        with pytest.raises(ValueError, match="workspace"):
            ops.hip.call("h3v_attention_d64_ws", *args, *bad, ops.hip.stream(DEV))
