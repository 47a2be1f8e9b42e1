"""Host-side pieces of the layer driver (exl3_intel_arc_quantizer_amd/
layer_quant.py) on CPU tensors."""

from __future__ import annotations

import pytest
import torch


@pytest.mark.parametrize("n,block", [(64, 16), (300, 128), (1100, 256), (1100, 4096)])
def test_factorization_residual_matches_full_product(n, block):
    """The row-blocked residual (layer_quant.py:95-101) over a lower
    triangular factor equals ||H - L L^T||_F / ||H||_F computed with the
    full product, for a factor perturbed well above rounding level."""
    from exl3_intel_arc_quantizer_amd.layer_quant import compute_factorization_residual
    g = torch.Generator().manual_seed(n)
    X = torch.randn(n + 10, n, generator=g, dtype=torch.float64)
    H = (X.T @ X) / n + 0.1 * torch.eye(n, dtype=torch.float64)
    L = torch.linalg.cholesky(H)
    L += torch.tril(torch.randn(n, n, generator=g, dtype=torch.float64)) * 1e-4
    H32, L32 = H.float(), L.float()
    got = compute_factorization_residual(H32, L32, block_rows=block)
    want = float(torch.linalg.norm(H - L @ L.T) / torch.linalg.norm(H))
    assert got == pytest.approx(want, rel=1e-4)


@pytest.mark.parametrize("chunk", [64, 8192])
def test_hessian_is_summed_in_float32_under_autocast(chunk):
    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(300, 96, generator=torch.Generator().manual_seed(2))
    with torch.autocast("cpu", dtype=torch.bfloat16):
        h, damp = hessian_from_activations(x, chunk_tokens=chunk)
    want = x.double().T @ x.double() / 300
    want.diagonal().add_(damp)
    assert h.dtype == torch.float32
    # Inputs and products rounded to 8 bits, the sums not.
    assert float((h.double() - want).norm() / want.norm()) < 3 * 2.0 ** -8


@pytest.mark.parametrize("tokens,chunk", [(300, 8192), (300, 64), (5, 1), (0, 8)])
def test_hessian_on_the_cpu(tokens, chunk):
    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(tokens, 96, generator=torch.Generator().manual_seed(3))
    h, damp = hessian_from_activations(x, chunk_tokens=chunk)
    want = x.double().T @ x.double() / max(1, tokens)
    want.diagonal().add_(damp)
    want.diagonal().clamp_(min=1e-7)
    torch.testing.assert_close(h.double(), want, rtol=1e-5, atol=1e-6)
