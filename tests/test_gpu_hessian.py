"""exl3_gram and the damping kernel at the edges of their tiles (128, 192),
token chunks (64) and shares, against float64."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,d", [(1, 8), (7, 40), (64, 128), (65, 136), (500, 192),
                                      (513, 328), (1000, 520), (4097, 1024), (700, 3968)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_gram(tokens, d, dtype):
    import torch

    from exl3_intel_arc_quantizer_amd._native import gram
    g = torch.Generator(device="cuda").manual_seed(tokens + d)
    x = torch.randn(tokens, d + 8, generator=g, device="cuda").to(getattr(torch, dtype))
    for view in (x[:, :d], x[:, :d].contiguous()):      # a row stride, and none
        h = gram(view, 0.5)
        want = 0.5 * (view.double().T @ view.double())
        assert torch.equal(h, h.T)
        # Exact products; each sum of `tokens` of them rounds at most that
        # often at the size of the sum of magnitudes.
        bound = 0.5 * (view.double().abs().T @ view.double().abs()) * (tokens + 2) * 2.0 ** -24
        assert bool(((h.double() - want).abs() <= bound + 1e-30).all())
        if tokens >= 64:
            assert float((h.double() - want).norm() / want.norm()) < 1e-6


@pytest.mark.parametrize("d", [1, 64, 1025, 3000])
def test_damping(d):
    import torch

    from exl3_intel_arc_quantizer_amd._native import damp_diagonal
    rng = np.random.default_rng(d)
    h = torch.from_numpy(rng.standard_normal((d, d)).astype(np.float32)).cuda()
    h.diagonal().abs_()
    h[d // 2, d // 2] = 0.0
    before = h.clone()
    mean = damp_diagonal(h, 0.01, 0.25)
    diag = before.diagonal().cpu().numpy().astype(np.float64)
    assert float(mean) == pytest.approx(diag.mean(), rel=2.0 ** -23)
    add = np.float32(max(1e-8, 0.01 * float(mean)))
    want = before.diagonal().cpu().numpy() + add
    want = np.where(np.abs(want) < np.float32(0.25), np.float32(0.25), want)
    np.testing.assert_array_equal(h.diagonal().cpu().numpy(), want)
    h.diagonal().zero_()
    before.diagonal().zero_()
    assert torch.equal(h, before)


def test_layouts_of_hessian_from_activations():
    """Widths and strides that exl3_gram does not take give the same Hessian
    as those it takes, up to summation order."""
    import torch

    from exl3_intel_arc_quantizer_amd._native import gram_takes
    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(3, 300, 264, device="cuda").to(torch.bfloat16)
    cases = [x[..., :260], x[..., :255], x[..., 1:257], x.reshape(-1, 264).T.contiguous().T]
    assert not any(gram_takes(c.reshape(-1, c.shape[-1])) for c in cases)
    for c in cases:
        flat = c.reshape(-1, c.shape[-1]).double()
        want = flat.T @ flat / flat.shape[0]
        h, damp = hessian_from_activations(c)
        assert damp == pytest.approx(0.01 * float(want.diagonal().mean()), rel=1e-6)
        want.diagonal().add_(damp)
        assert float((h.double() - want).norm() / want.norm()) < 1e-6
    with pytest.raises(ValueError):
        hessian_from_activations(x[..., :256].contiguous(), chunk_tokens=0)
