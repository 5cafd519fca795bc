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
