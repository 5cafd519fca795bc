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
