"""The tiled bf16 GEMMs where a launch has more tiles than CUs."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,N,K", [(11008, 1536, 256), (22016, 768, 128), (9216, 2304, 128), (6144, 3072, 128),
                                   (17000, 1280, 128)])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_large_linear_column_parameters(M, N, K, act):
    """Scales and biases of linears with more 256 x 256 tiles than CUs whose column count does not divide the
    tile step (N / 256 = 6, 3, 9, 12, 5): every tile uses its own columns' (against 64 bits, 2^-8)."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    s = torch.rand(N, generator=g, device=DEV) + 0.5
    b = torch.randn(N, generator=g, device=DEV) * 3
    got = ops.norm_linear(x, weight=w, weight_scale=s, bias=b, act=act, out_dtype=torch.bfloat16)
    want = x.double() @ w.double().t().contiguous() * s.double() + b.double()
    if act:
        want = torch.nn.functional.gelu(want)
    assert ((got.double() - want).norm() <= 2.0 ** -8 * want.norm())
    assert ((got.double() - want).abs().amax() <= 2.0 ** -8 * want.abs().amax() + 2.0 ** -8)


@pytest.mark.parametrize("M,N,K", [(26000, 1280, 128), (33000, 2304, 128), (64000, 768, 128), (15000, 3072, 256)])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_persistent_linear_column_parameters(M, N, K, act):
    """The same where the persistent tiles take the call (N / 256 = 5, 9, 3, 12 does not divide the tile step of
    32, so that the next tile of a workgroup has other columns)."""
    from cortex import _native as nat

    assert nat.load().cortex_bf16_gemm_form(M, N, K, nat.BF16, nat.BF16) == 4
    test_large_linear_column_parameters(M, N, K, act)


@pytest.mark.parametrize("M,N,K", [(65536, 256, 2048), (65300, 256, 2112), (32769, 512, 2048), (21900, 768, 3072),
                                   (98400, 256, 2048)])
@pytest.mark.parametrize("res_rows", [0, 384])
def test_wide_residual_linear(M, N, K, res_rows):
    """The persistent 256 x 256 residual GEMM (long K, rounds of tiles that fill the CUs): partial last rows,
    one to two rounds, an odd number of K stages, a broadcast residual and one updated in place; sampled
    rows against 64 bits (K / 16 + 8 accumulations of 2^-24 of sum |a| |w|)."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(M + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    s = torch.rand(N, generator=g, device=DEV) + 0.5
    b = torch.randn(N, generator=g, device=DEV)
    rows = torch.cat([torch.randint(0, M, (500,), generator=g, device=DEV), torch.arange(M - 300, M, device=DEV)])
    y = x[rows].double() @ w.double().t().contiguous() * s.double()
    mag = x[rows].double().abs() @ w.double().abs().t().contiguous() * s.double() + 8
    if res_rows:
        res = torch.randn(res_rows, N, generator=g, device=DEV)
        got = ops.norm_linear(x, weight=w, weight_scale=s, residual=res, res_rows=res_rows, out_dtype=torch.float32)
        want = y + res[rows % res_rows].double()
    else:
        got = torch.randn(M, N, generator=g, device=DEV)
        want = y + b.double() + got[rows].double()
        ops.norm_linear(x, weight=w, weight_scale=s, bias=b, residual=got, out=got, out_dtype=torch.float32)
    assert ((got[rows] - want).abs() <= (K / 16 + 8) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M", [8192, 8193, 8250, 8256, 16385, 20001])
@pytest.mark.parametrize("N,K", [(256, 256), (256, 512), (512, 256), (512, 512)])
@pytest.mark.parametrize("res_rows", [0, 256])
def test_tall_residual_layer_norm_equals_ring(M, N, K, res_rows):
    """The 64-row direct-weight form (past 8192 rows) gives the plain-row kernel's bits, at partial last
    workgroups, with a broadcast residual and in place."""
    from cortex.kernels import ops

    g = torch.Generator(DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    s, b, gm, bt = (torch.rand(N, generator=g, device=DEV) + 0.5 for _ in range(4))
    res = torch.randn(res_rows or M, N, generator=g, device=DEV)
    ln = (gm, bt, 1e-5)
    want = ops.linear_residual_ln(x, w, s, b, residual=res, ln=ln, res_rows=res_rows)
    out = None if res_rows else res.clone()
    got = ops.linear_residual_ln(x, ops.frag_weight(w), s, b, residual=res if out is None else out, ln=ln,
                                 res_rows=res_rows, out=out, frag=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("M,N", [(3069, 2304), (4093, 2304), (6141, 2304), (7679, 2304), (9213, 2304), (4605, 2048),
                                 (12285, 768), (12285, 1536), (9213, 2048), (16381, 2304), (16381, 2048), (24573, 2304),
                                 (33001, 1024)])
@pytest.mark.parametrize("form", ["image", "int8", "rms"])
def test_tile_rule(M, N, form):
    """Row counts on every side of the tile rule (128 x 128, 256 x 192 in one to three rounds, 256 x 256 in one
    to four), partial last tiles: sampled and last rows against 64 bits, 2^-8."""
    from cortex.kernels import ops
    from cortex.kernels.fused_rmsnorm import norm_linear_int8

    K = 128
    g = torch.Generator(DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    q, s = ops.quantize_int8(torch.randn(N, K, generator=g, device=DEV) * 0.05)
    wd = q.double() * s.double()[:, None]
    rows = torch.cat([torch.randint(0, M, (400,), generator=g, device=DEV), torch.arange(M - 260, M, device=DEV)])
    a = x[rows].double()
    if form == "rms":
        got = norm_linear_int8(x, q, s, gamma=torch.ones(K, device=DEV))
        a = a / (a.square().mean(1, keepdim=True) + 1e-6).sqrt()
    elif form == "int8":
        got = ops.norm_linear(x, weight_int8=q, weight_scale=s, act="gelu", out_dtype=torch.bfloat16)
    else:
        got = ops.norm_linear(x, weight=ops.convert(q, torch.bfloat16), weight_scale=s, act="gelu",
                              out_dtype=torch.bfloat16)
    want = a @ wd.t().contiguous()
    if form != "rms":
        want = torch.nn.functional.gelu(want)
    err = (got[rows].double() - want).abs()
    assert (err.norm() <= 2.0 ** -8 * want.norm()) and (err.amax() <= 2.0 ** -7 * want.abs().amax())


def test_tile_rule_shapes_take_every_tiling():
    """The shapes of ``test_tile_rule`` reach each tiling, the large ones in more than one round."""
    from cortex import _native as nat

    shapes = next(m for m in test_tile_rule.pytestmark if m.args[0] == "M,N").args[1]
    rounds = {}
    for M, N in shapes:
        form = nat.load().cortex_bf16_gemm_form(M, N, 128, nat.BF16, nat.BF16)
        width = {1: 128, 2: 192, 3: 256, 4: 256}[form]
        tiles = -(-M // (128 if form == 1 else 256)) * -(-N // width)
        rounds.setdefault(form, set()).add(-(-tiles // (512 if form == 1 else 256)))
    assert set(rounds) == {1, 2, 3, 4} and {1, 2, 3} <= rounds[2] and max(rounds[4]) >= 4 and max(rounds[1]) >= 4
