"""The fp32 linear on bf16 parts (gemm_split.hip) against 64-bit products.

Sizes at the edges of its tiles (64, 128), K blocks (32), register-held rows (K 1024) and row chunks, all
operand forms, and values at the ends of the fp32 range.  The bound is elementwise: every product is
exact or off by under 2^-24 of itself, and a sum of n terms of magnitude S = sum |a| |w| is off by at
most n 2^-24 S per accumulation chain; a normalised row carries 8 roundings of its own.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ops():
    from cortex.kernels import ops

    return ops


def _bound(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    K = a.shape[1]
    return (12 * (K // 32 + 1) + 16) * 2.0 ** -24 * (a.abs() @ w.abs().t().contiguous()) + 1e-30


def _weight(ops, form, N, K, g):
    w = torch.randn(N, K, generator=g, device=DEV) * 0.05
    if form == "int8":
        q, s = ops.quantize_int8(w)
        return dict(weight_int8=q, weight_scale=s), q.double() * s.double()[:, None]
    if form == "kn":
        return dict(weight=w.t().contiguous(), w_layout="kn"), w.double()
    return dict(weight=w), w.double()


@pytest.mark.parametrize("form", ["int8", "nk", "kn"])
@pytest.mark.parametrize("M,N,K", [(1, 9, 1), (1, 33, 31), (31, 64, 33), (65, 130, 100), (127, 17, 520), (129, 129, 1056),
                                   (600, 512, 512), (2100, 2050, 96), (4097, 1024, 64)])
@pytest.mark.parametrize("norm", [None, "layer", "rms"])
def test_split_linear_sizes(form, M, N, K, norm):
    ops = _ops()
    g = torch.Generator(DEV).manual_seed(M * 7 + N + K)
    x = torch.randn(M, K, generator=g, device=DEV) + 0.5
    kw, wd = _weight(ops, form, N, K, g)
    a = x.double()
    if norm:
        gm = 1 + 0.1 * torch.randn(K, generator=g, device=DEV)
        kw.update(norm=norm, gamma=gm, eps=1e-5)
        if norm == "layer":
            bt = 0.1 * torch.randn(K, generator=g, device=DEV)
            kw.update(beta=bt)
            a = (a - a.mean(1, keepdim=True)) / (a.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt() * gm + bt
        else:
            a = a / (a.square().mean(1, keepdim=True) + 1e-5).sqrt() * gm
    got = ops.norm_linear(x, **kw, compute_dtype=torch.float32)
    if norm == "layer" and K == 1:
        a = bt.double().expand(M, 1)  # (x - mean is 0)
    # a LayerNorm with a mean that cancels: x - mean is off by 2^-24 (|x| + |mean|), then scaled
    slack = a.abs() + (4.0 if norm == "layer" else 0.0)
    assert ((got - a @ wd.t().contiguous()).abs() <= _bound(slack, wd)).all()


@pytest.mark.parametrize("form", ["int8", "nk"])
def test_split_linear_epilogue_and_views(form):
    """Bias, GELU, a broadcast residual and one updated in place, rows and outputs at odd strides."""
    ops = _ops()
    g = torch.Generator(DEV).manual_seed(5)
    M, N, K = 200, 70, 77
    xs = torch.randn(M, K + 3, generator=g, device=DEV)[:, 1:K + 1]  # unaligned rows
    kw, wd = _weight(ops, form, N, K, g)
    bias = torch.randn(N, generator=g, device=DEV)
    res = torch.randn(40, N, generator=g, device=DEV)
    y = xs.double() @ wd.t().contiguous() + bias.double()
    want = torch.nn.functional.gelu(y) + res.double().repeat(5, 1)
    got = ops.norm_linear(xs, **kw, bias=bias, act="gelu", residual=res, res_rows=40, compute_dtype=torch.float32)
    tol = 1.13 * (_bound(xs.double(), wd) + 2.0 ** -23 * y.abs()) + 2.0 ** -22 * (y.abs() + want.abs() + 1)
    assert ((got - want).abs() <= tol).all()
    buf = torch.randn(M, N + 5, generator=g, device=DEV)
    before = buf.clone()
    ops.norm_linear(xs, **kw, residual=buf[:, :N], out=buf[:, :N], compute_dtype=torch.float32)
    want = before[:, :N].double() + xs.double() @ wd.t().contiguous()
    assert ((buf[:, :N] - want).abs() <= _bound(xs.double(), wd) + 2.0 ** -22 * want.abs()).all()
    assert torch.equal(buf[:, N:], before[:, N:])


@pytest.mark.parametrize("form", ["int8", "kn"])
def test_split_linear_row_chunks(form):
    """A workspace of 128 rows gives bit for bit what one of all rows gives."""
    from cortex import _native as nat

    g = torch.Generator(DEV).manual_seed(6)
    M, N, K = 400, 96, 64
    x = torch.randn(M, K, generator=g, device=DEV)
    gm = torch.rand(K, generator=g, device=DEV)
    kw, _ = _weight(_ops(), form, N, K, g)
    w, scale = kw.get("weight_int8", kw.get("weight")), kw.get("weight_scale")
    res = torch.randn(130, N, generator=g, device=DEV)
    full = nat.load().cortex_norm_linear_split_workspace_bytes(M, N, K, nat.code(w.dtype))
    one = nat.load().cortex_norm_linear_split_workspace_bytes(1, N, K, nat.code(w.dtype))
    outs = []
    for size in (full, one):
        ws = torch.empty(size, dtype=torch.uint8, device=DEV)
        out = torch.empty(M, N, device=DEV)
        nat.call("cortex_norm_linear_split", M, N, K, nat.ptr(x), K, 2, nat.ptr(gm), None, 0, 1e-6, nat.code(w.dtype),
                 int(form == "kn"), nat.ptr(w), w.stride(0), nat.ptr(scale), None, 0, nat.ptr(res), N, 130, nat.ptr(out), N,
                 nat.ptr(ws), size, nat.stream_of(torch.device(DEV)))
        outs.append(out)
    assert torch.equal(*outs)
    rc = nat.load().cortex_norm_linear_split(M, N, K, nat.ptr(x), K, 0, None, None, 0, 0.0, nat.code(w.dtype),
                                             int(form == "kn"), nat.ptr(w), w.stride(0), None, None, 0, None, 0, 0,
                                             nat.ptr(out), N, nat.ptr(ws), one - 1, None)
    assert rc == -4 and b"workspace" in nat.load().cortex_last_error()


@pytest.mark.parametrize("form", ["int8", "nk"])
def test_split_linear_special_values(form):
    """Infinities and NaN stay in their row (or column) with their sign; the largest and small values."""
    ops = _ops()
    x = torch.ones(8, 64, device=DEV)
    x[0, 3], x[1, 3], x[2, 3], x[3, 3] = float("inf"), float("-inf"), float("nan"), 3.4028e38
    x[4] *= 1e-30
    x[5] *= 3.39e38 / 64
    w = torch.full((16, 64), 0.5, device=DEV)
    if form == "int8":
        kw = dict(weight_int8=torch.full((16, 64), 1, dtype=torch.int8, device=DEV),
                  weight_scale=torch.full((16,), 0.5, device=DEV))
    else:
        w[15, 0] = float("inf")
        kw = dict(weight=w)
    got = ops.norm_linear(x, **kw, compute_dtype=torch.float32).cpu()
    want = (x.cpu().double() @ w.cpu().double().t()).float()
    for fn in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(fn(got), fn(want))
    ok = torch.isfinite(want)
    assert ((got - want).abs()[ok] <= 2.0 ** -20 * want.abs()[ok]).all()


def test_split_linear_infinities_that_meet():
    """Infinities of x and of the weight at the same k: their signed product, as the fp32 product gives it."""
    ops = _ops()
    inf = float("inf")
    x = torch.ones(4, 64, device=DEV)
    x[0, 5], x[1, 5], x[2, 5], x[3, 5] = inf, -inf, 0.0, float("nan")
    w = torch.full((16, 64), 0.5, device=DEV)
    w[1, 5], w[2, 5], w[3, 5] = inf, -inf, 0.0
    got = ops.norm_linear(x, weight=w, compute_dtype=torch.float32).cpu()
    want = (x.cpu().double() @ w.cpu().double().t()).float()
    for fn in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(fn(got), fn(want))
    ok = torch.isfinite(want)
    assert torch.equal(got[ok], want[ok])


@pytest.mark.parametrize("form", ["int8", "nk"])
@pytest.mark.parametrize("power", [-100, -110, -114, -118, -126])
def test_split_linear_smallest_values(form, power):
    """Rows near the bottom of the range: full precision down to 2^-110, below that every operand value off
    by at most 2^-134 (half of the smallest bf16 step)."""
    ops = _ops()
    g = torch.Generator(DEV).manual_seed(8)
    x = torch.randn(64, 256, generator=g, device=DEV) * 2.0 ** power
    kw, wd = _weight(ops, form, 128, 256, g)
    want = x.double() @ wd.t().contiguous()
    got = ops.norm_linear(x, **kw, compute_dtype=torch.float32)
    step = 2.0 ** -149 * (1 + got.shape[1])  # (the sums' own denormals)
    slack = 0 if power >= -100 else 2.0 ** -134 * wd.abs().sum(1)
    rel = (12 * 9 + 16) * 2.0 ** -24 * (x.double().abs() @ wd.abs().t().contiguous())
    assert ((got.double() - want).abs() <= rel + slack + step).all()
    if power >= -110:
        assert ((got.double() - want).norm() <= 4e-7 * want.norm())


@pytest.mark.parametrize("form", ["int8", "nk"])
@pytest.mark.parametrize("M,N,K", [(7424, 512, 2048), (1661, 2048, 2075), (1920, 2048, 96), (2049, 2048, 96), (2049, 2048, 1056),
                                   (2600, 2050, 96), (3201, 2048, 96)])
@pytest.mark.parametrize("residual", [False, True])
def test_split_linear_tile_rule(form, M, N, K, residual):
    """Either side of the rule for the tile, in 128 x 128 tiles on 256 CUs: 232, 208, 240, 272 (twice), 357 and 416,
    without a residual (64 x 64 tiles up to 224 or 256, and from 257 to 320) and with one (up to 384)."""
    ops = _ops()
    if not residual:
        return test_split_linear_sizes(form, M, N, K, None)
    g = torch.Generator(DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV)
    kw, wd = _weight(ops, form, N, K, g)
    buf = torch.randn(M, N, generator=g, device=DEV)
    want = buf.double() + x.double() @ wd.t().contiguous()
    ops.norm_linear(x, **kw, residual=buf, out=buf, compute_dtype=torch.float32)
    assert ((buf - want).abs() <= _bound(x.double(), wd) + 2.0 ** -22 * want.abs() + 2.0 ** -22).all()
