"""The few-row bf16 linear (gemm_small.hip) against 64-bit products of the same bf16 operands.

Row counts around its 32-row tiles and 16-row fragment blocks, every K it takes, both operand and output
orders.  fp32 outputs: at most K / 32 + 16 accumulations of 2^-24 of sum |a| |w|; bf16 outputs and the
LayerNorm'd operand add half a bf16 step (2^-9) each.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _unfrag(t: torch.Tensor, rows: int) -> torch.Tensor:
    """Rows of a fragment-order (R, N) tensor (R a multiple of 16)."""
    R, N = t.shape
    return t.reshape(R // 16, N // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(R, N)[:rows]


def _case(M, N, K, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    s = torch.rand(N, generator=g, device=DEV) + 0.5
    b = torch.randn(N, generator=g, device=DEV)
    return g, x, w, s, b


@pytest.mark.parametrize("K", [256, 512, 768, 1024, 2048, 3072])
@pytest.mark.parametrize("M,N", [(1, 32), (15, 64), (16, 96), (17, 32), (33, 160), (129, 64)])
def test_bf16_rows_residual_and_orders(M, N, K):
    from cortex.kernels import ops

    g, x, w, s, b = _case(M, N, K, M + N + K)
    xb, wf = x.bfloat16(), ops.frag_weight(w)
    res = torch.randn(7, N, generator=g, device=DEV)
    y = xb.double() @ w.double().t().contiguous() * s.double() + b.double()
    acc = (K / 32 + 16) * 2.0 ** -24 * (xb.double().abs() @ w.double().abs().t().contiguous() * s.double() + y.abs() + 8)
    want = y + res.double().repeat(M // 7 + 1, 1)[:M]
    got = ops.linear_small(xb, wf, s, b, residual=res, res_rows=7, out_dtype=torch.float32)
    assert ((got - want).abs() <= acc).all()
    buf = torch.randn(M, N, generator=g, device=DEV)
    want = buf.double() + y
    ops.linear_small(xb, wf, s, b, residual=buf, out=buf)
    assert ((buf - want).abs() <= acc).all()
    q, qs = ops.quantize_int8(w.float())  # int8 rows: bit for bit their bf16 image
    a8 = ops.linear_small(xb, q, qs, b, act="gelu")
    assert torch.equal(a8, ops.linear_small(xb, ops.frag_weight(q), qs, b, act="gelu"))
    # GELU to bf16 rows, the same in fragment order, and that order as the operand of the next linear
    act = torch.nn.functional.gelu(y)
    rows = ops.linear_small(xb, wf, s, b, act="gelu")
    assert ((rows.double() - act).abs() <= 1.13 * acc + 2.0 ** -8 * act.abs() + 1e-6).all()
    h = ops.linear_small(xb, wf, s, b, act="gelu", out_frag=True)
    assert h.shape[0] % 16 == 0 and torch.equal(_unfrag(h, M), rows)
    xf = torch.zeros((M + 15) // 16 * 16, K, dtype=torch.bfloat16, device=DEV)
    xf[:M] = xb
    again = ops.linear_small(ops.frag_weight(xf), wf, s, b, rows=M, out_dtype=torch.float32)
    assert torch.equal(again, ops.linear_small(xb, wf, s, b, out_dtype=torch.float32))


@pytest.mark.parametrize("K", [256, 512, 768, 1024])
@pytest.mark.parametrize("M", [1, 31, 64, 100])
def test_layer_norm_inside(M, K):
    from cortex.kernels import ops

    g, x, w, s, _ = _case(M, 96, K, M + K)
    x = torch.cat([x * 3 + 1, x], 1)[:, :K]  # rows at a stride of 2 K
    gm, bt = 1 + 0.1 * torch.randn(K, generator=g, device=DEV), 0.1 * torch.randn(K, generator=g, device=DEV)
    a = torch.nn.functional.layer_norm(x.double(), (K,), gm.double(), bt.double(), 1e-5)
    want = a @ w.double().t().contiguous() * s.double()
    mag = (a.abs() + 0.1) @ w.double().abs().t().contiguous() * s.double()
    got = ops.linear_small(x, ops.frag_weight(w), s, ln=(gm, bt, 1e-5), out_dtype=torch.float32)
    assert ((got - want).abs() <= (2.0 ** -9 + (K / 32 + 40) * 2.0 ** -24) * mag).all()
    assert ((got - want).norm() <= 2.0 ** -9 * want.norm())


@pytest.mark.parametrize("model", ["xs", "s", "m"])
@pytest.mark.parametrize("batch", [1, 2, 3, 5, 9])
def test_block_around_the_few_row_rule(model, batch):
    """A block on either side of the few-row rules against the same block in fp32 compute."""
    from cortex.models import config
    from cortex.models.perceiver import SelfAttentionBlock

    cfg = getattr(config, "CORTEX_" + model.upper())
    torch.manual_seed(0)
    blk = SelfAttentionBlock(cfg).to(DEV).eval()
    ref = SelfAttentionBlock(cfg.model_copy(update={"dtype": "float32"})).to(DEV).eval()
    ref.load_state_dict(blk.state_dict())
    x = torch.randn(batch, cfg.num_latents, cfg.latent_dim, device=DEV)
    with torch.no_grad():
        got, want = blk(x), ref(x)
    # (bf16 operands, and a float weight rounded to bf16: a few bf16 steps of the branches' size)
    assert ((got - want).norm() <= 1e-2 * (want - x).norm())


@pytest.mark.parametrize("batch", [1, 3])
def test_float16_weights_at_few_rows(batch):
    """float16 nn.Linear weights run as their bf16 rounding, which fp32 weights of the same values have too."""
    from cortex.kernels import ops
    from cortex.models import config
    from cortex.models.perceiver import CrossAttentionBlock, SelfAttentionBlock

    cfg = config.CORTEX_S
    torch.manual_seed(1)
    for cls in (SelfAttentionBlock, CrossAttentionBlock):
        blk, ref = cls(cfg).to(DEV).eval(), cls(cfg).to(DEV).eval()
        for a, b in zip(blk.modules(), ref.modules()):
            if isinstance(a, torch.nn.Linear):
                a.weight.data = a.weight.data.half()
                b.weight.data = a.weight.data.float()
            elif isinstance(a, torch.nn.LayerNorm):
                b.load_state_dict(a.state_dict())
        args = [torch.randn(batch, cfg.num_latents, cfg.latent_dim, device=DEV)]
        if cls is CrossAttentionBlock:
            args.append(torch.randn(batch, 70, cfg.hidden_dim, device=DEV))
        with torch.no_grad():
            assert torch.equal(blk(*args), ref(*args))
    w = torch.randn(64, 96, device=DEV).half()
    assert torch.equal(ops.frag_weight(w), ops.frag_weight(w.bfloat16()))


def _lin(N, K, bias=True):
    torch.manual_seed(N + K)
    return torch.nn.Linear(K, N, bias=bias).to(DEV)


@pytest.mark.parametrize("M", [2, 40])
def test_expanded_rows_and_residual(M):
    """Rows and residuals that share memory (expanded), of a stride below their width or of a transposed
    matrix give what their copies give."""
    from cortex.models._layers import apply_linear

    K = N = 256
    lin, norm = _lin(N, K), torch.nn.LayerNorm(K).to(DEV)
    kw = dict(out_dtype=torch.float32, compute=torch.bfloat16)
    views = [((1, K), lambda t: t.expand(M, K)), ((M + K,), lambda t: t.as_strided((M, K), (1, 1))),
             ((K, M), lambda t: t.t()), ((M, 1, K), lambda t: t.expand(M, 3, K))]
    with torch.no_grad():
        for shape, view in views:
            base = torch.randn(shape, device=DEV)
            x, xb = view(base), view(base.bfloat16())
            assert torch.equal(apply_linear(lin, xb, **kw), apply_linear(lin, xb.contiguous(), **kw))
            assert torch.equal(apply_linear(lin, x, norm=norm, **kw), apply_linear(lin, x.contiguous(), norm=norm, **kw))
        x = torch.randn(M, K, device=DEV).bfloat16()
        for res in (torch.randn(1, N, device=DEV).expand(M, N), torch.randn(M + N, device=DEV).as_strided((M, N), (1, 1)),
                    torch.randn(N, M, device=DEV).t()):
            assert torch.equal(apply_linear(lin, x, residual=res, **kw), apply_linear(lin, x, residual=res.contiguous(), **kw))
    from cortex.quantization.calibrate import QuantizedLinear

    q8 = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV)
    scale = torch.rand(N, 2, device=DEV)[:, 0]  # every second value
    got, want = (apply_linear(QuantizedLinear(q8, s, None), x, **kw) for s in (scale, scale.contiguous()))
    assert ((got - want).norm() <= 1e-5 * want.norm())  # (another order of the K sums)


@pytest.mark.parametrize("M", [1, 30, 3000])
def test_output_buffer_with_more_rows(M):
    """An output of more rows than the result keeps the rest of its rows."""
    from cortex.kernels import ops
    from cortex.models._layers import apply_linear

    K = N = 256
    lin = _lin(N, K, bias=False)
    x = torch.randn(M, K, device=DEV).bfloat16()
    with torch.no_grad():
        for dtype in (torch.bfloat16, torch.float32):
            want = apply_linear(lin, x, out_dtype=dtype, compute=torch.bfloat16)
            out = torch.full((M + 5, N), 7.0, dtype=dtype, device=DEV)
            apply_linear(lin, x, out_dtype=dtype, compute=torch.bfloat16, out=out)
            assert (out[M:] == 7).all()
            assert ((out[:M] - want).abs() <= 2.0 ** -7 * want.abs() + 1e-4).all()
            w = lin.weight.bfloat16()
            want = ops.norm_linear(x, weight=w, out_dtype=dtype)
            out = torch.full((M + 5, N), 7.0, dtype=dtype, device=DEV)
            ops.norm_linear(x, weight=w, out_dtype=dtype, out=out)
            assert torch.equal(out[:M], want) and (out[M:] == 7).all()
            with pytest.raises((ValueError, RuntimeError)):
                ops.norm_linear(x, weight=w, out_dtype=dtype, out=out[:0])
            with pytest.raises((ValueError, RuntimeError)):
                ops.norm_linear(x, weight=lin.weight, out_dtype=dtype, out=out[:M - 1])


def test_buffers_too_small_are_refused():
    """Outputs, and rows in fragment order, of fewer rows than a launch writes or reads."""
    from cortex.kernels import ops

    _, x, w, s, _ = _case(20, 64, 256, 0)
    xb, wf = x.bfloat16(), ops.frag_weight(w)
    xf = ops.frag_weight(torch.zeros(32, 256, dtype=torch.bfloat16, device=DEV))
    with pytest.raises(ValueError):
        ops.linear_small(xb, wf, s, out=torch.empty(19, 64, device=DEV))
    with pytest.raises(ValueError):
        ops.linear_small(xb, wf, s, out=torch.empty(20, 64, dtype=torch.bfloat16, device=DEV), out_frag=True)
    with pytest.raises(ValueError):
        ops.linear_small(xf[:16], wf, s, rows=20)
    assert ops.linear_small(xf, wf, s, rows=20).shape == (20, 64)
