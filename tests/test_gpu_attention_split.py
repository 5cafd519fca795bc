"""fp32 attention on bf16 parts (attention_split.hip) against float64 on the same inputs.

Sizes at the edges of its tiles (64 keys, 32 queries a wavefront, 64 or 128 a workgroup), every mask form
it takes, strided and broadcast operands, extreme values.  Bound: a score is off by at most D = (64 + 8)
2^-24 scale sum |q| |k| (its products exact or off by under 2^-24 each, 64-term fp32 sums), a
probability by 2 D + 2^-21 of itself (exp2, the normalisation), and the sum over n keys by n 2^-24 more.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(got, q, k, v, allowed, scale=0.125):
    """(B, H, L, 64) fp32 against float64; allowed (B, 1, L, E) bool or None."""
    q, k, v = q.double(), k.double(), v.double()
    kt = k.transpose(-1, -2).contiguous()
    s = torch.matmul(q, kt) * scale
    d = torch.matmul(q.abs(), k.abs().transpose(-1, -2).contiguous()) * abs(scale) * 72 * 2.0 ** -24
    if allowed is not None:
        s = s.masked_fill(~allowed, float("-inf"))
        d = d.masked_fill(~allowed, 0.0)
    p = s.softmax(-1).nan_to_num(0.0)
    want = torch.matmul(p, v)
    tol = (2 * d.amax(-1, keepdim=True) + 2.0 ** -21 + k.shape[2] * 2.0 ** -24) * torch.matmul(p, v.abs())
    assert got.dtype == torch.float32
    assert ((got - want).abs() <= tol + 1e-30).all(), float(((got - want).abs() / (tol + 1e-30)).max())


@pytest.mark.parametrize("L,E", [(1, 1), (2, 63), (31, 64), (33, 65), (64, 200), (129, 129), (200, 1000), (256, 256)])
@pytest.mark.parametrize("B,H", [(2, 3), (43, 8)])
@pytest.mark.parametrize("mask", ["none", "lengths", "keys", "tiles", "tiles+keys"])
def test_sizes_and_masks(L, E, B, H, mask):
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(L * 1000 + E + B)
    q, k, v = (torch.randn(B, H, n, 64, generator=g, device=DEV) for n in (L, E, E))
    kw, allowed = {}, torch.ones(B, 1, L, E, dtype=torch.bool, device=DEV)
    ar = torch.arange(E, device=DEV)
    if mask == "lengths":
        n = torch.randint(0, E + 1, (B,), generator=g, device=DEV)
        kw["kv_lengths"] = n
        allowed = allowed & (ar < n[:, None])[:, None, None, :]
    if "keys" in mask:
        m = torch.rand(B, E, generator=g, device=DEV) < 0.4
        m[0] = False
        kw["key_mask"] = m
        allowed = allowed & m[:, None, None, :]
    if "tiles" in mask:
        bl, be = 24, 128
        t = torch.rand(B, -(-L // bl), -(-E // be), generator=g, device=DEV) < 0.5
        kw.update(block_mask=t, block_l=bl, block_e=be)
        allowed = allowed & t.repeat_interleave(bl, 1)[:, :L].repeat_interleave(be, 2)[:, None, :, :E]
    _check(ops.attention(q, k, v, **kw), q, k, v, allowed)


def test_csr_broadcast_queries_and_merged_heads():
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(3)
    H, L, lens = 4, 96, [70, 0, 1, 300]
    off = torch.tensor([0, 70, 70, 71, 371], device=DEV)
    q = torch.randn(L, H * 64, generator=g, device=DEV)
    kv = torch.randn(371, 2 * H * 64, generator=g, device=DEV)
    buf, o = ops.merge_heads_out(4, L, H, 64, torch.float32, torch.device(DEV))
    ops.attention(ops.heads_view(q, 1, L, H), ops.heads_view(kv, 1, 371, H, 0, H * 64),
                  ops.heads_view(kv, 1, 371, H, H * 64, H * 64), kv_offsets=off, out=o, batch=4)
    for b, n in enumerate(lens):
        rows = kv[off[b]:off[b + 1]].reshape(n, 2, H, 64).permute(1, 2, 0, 3)[:, None]
        if n == 0:
            assert (o[b] == 0).all()
        else:
            _check(o[b:b + 1], ops.heads_view(q, 1, L, H), rows[0], rows[1], None)


@pytest.mark.parametrize("scale", [0.125, 8.0, -1.0])
def test_extremes(scale):
    """Peaked and negative scales, large values, an infinite value behind a zero and a non-zero weight."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(4)
    q, k, v = (torch.randn(1, 2, 130, 64, generator=g, device=DEV) for _ in range(3))
    _check(ops.attention(q, k, v, scale=scale), q, k, v, None, scale)
    v[0, 0] *= 1e36
    _check(ops.attention(q, k, v, scale=scale), q, k, v, None, scale)
    v[0, 1, 5, 7] = float("inf")
    v[0, 1, 6, 8] = float("nan")
    got = ops.attention(q, k, v, scale=0.01)[0, 1]
    assert torch.isposinf(got[:, 7]).all() and torch.isnan(got[:, 8]).all()
    rest = torch.cat([got[:, :7], got[:, 9:]], 1)
    assert torch.isfinite(rest).all()


@pytest.mark.parametrize("L", [40, 8192])
def test_infinite_operands(L):
    """An infinite query component on an infinite key of the other sign is a score of -inf: that key drops out."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(5)
    q, k, v = (torch.randn(1, 4, n, 64, generator=g, device=DEV) for n in (L, 70, 70))
    q[0, 0, :, 3] = float("inf")
    k[0, 0, :, 3] = float("-inf")
    k[0, 0, 5:9, 3] = 0.0  # inf * 0: NaN
    q[0, 1, :, 3] = float("inf")
    k[0, 1, :, 3] = float("-inf")
    got = ops.attention(q, k, v)
    assert torch.isnan(got[0, 0]).all()
    assert (got[0, 1] == 0).all()  # every score -inf: no key counts
    q[0, 1, 1:, 3] = 1.0
    k[0, 1, :9, 3] = torch.randn(9, generator=g, device=DEV)
    got = ops.attention(q[:, 1:2], k[:, 1:2], v[:, 1:2])
    assert torch.isnan(got[0, 0, 0]).all() or L == 1
    _check(got[:, :, 1:], q[:, 1:2, 1:], k[:, 1:2, :9], v[:, 1:2, :9], None)


@pytest.mark.parametrize("L", [40, 8192])
@pytest.mark.parametrize("E", [1, 70, 150])
def test_infinite_last_value(L, E):
    """An infinite value in the last row, whose tile has rows past the end, stays infinite with its sign."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(6)
    q, k, v = (torch.randn(1, 4, n, 64, generator=g, device=DEV) for n in (L, E, E))
    v[0, 0, -1, 7] = float("inf")
    v[0, 1, -1, 8] = float("-inf")
    got = ops.attention(q, k, v, scale=0.01)
    assert torch.isposinf(got[0, 0, :, 7]).all() and torch.isneginf(got[0, 1, :, 8]).all()
    got[0, 0, :, 7] = got[0, 1, :, 8] = 0
    assert torch.isfinite(got).all()
