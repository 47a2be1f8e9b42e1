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


@pytest.mark.parametrize("tokens,d", [(65536, 4096), (70001, 4096), (131072, 2048)])
def test_long_sums_are_no_worse_than_chunked_ones(tokens, d):
    """The error against float64 is that of float32 sums over at most 8192
    tokens, added in float32, whatever the token count and the width's share
    of the GPU: the diagonal (growing sums) and the rest."""
    import torch

    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    g = torch.Generator(device="cuda").manual_seed(d)
    x = torch.randn(tokens, d, generator=g, device="cuda").to(torch.bfloat16)
    chunked = torch.zeros(d, d, device="cuda")
    want = torch.zeros(d, d, dtype=torch.float64, device="cuda")
    for s in range(0, tokens, 8192):
        part = x[s:s + 8192]
        chunked += torch.mm(part.T, part, out_dtype=torch.float32)
        wide = part.double()
        want += wide.T @ wide
    chunked /= tokens
    want /= tokens
    # The damping, here 1e-8, is far below a rounding of the diagonal (1).
    h, _ = hessian_from_activations(x, damping_lambda=0.0, zero_floor=0.0)
    eye = torch.eye(d, dtype=torch.bool, device="cuda")
    for mask in (eye, ~eye):
        # As many roundings in another order: 1.25 for the spread of a root
        # mean square over thousands of entries.
        ours, theirs = (float((v.double() - want)[mask].square().mean().sqrt())
                        for v in (h, chunked))
        assert ours <= 1.25 * theirs, (ours, theirs)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("d", [8, 4096])
def test_chunk_tokens_have_sums_of_their_own(d, dtype):
    """2^30 from the first token swallows products of 1 (its last place is
    128), but not the sums that chunks of 1024 tokens bring: one float32
    sum over all tokens would stay at 2^30."""
    import torch

    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.ones(4096, d, device="cuda", dtype=getattr(torch, dtype))
    x[0] = 2.0 ** 15
    h, damp = hessian_from_activations(x, damping_lambda=0.0, chunk_tokens=1024)
    assert damp == 1e-8
    exact = 2.0 ** 30 + 4095.0
    # The first chunk may lose its other 1023 tokens; a half rounding (64) for
    # each of the three additions.
    assert bool(((h.double() * 4096 - exact).abs() <= 1023 + 3 * 64).all())


@pytest.mark.parametrize("tokens,d,chunk", [(64, 136, 64), (129, 136, 64), (1000, 520, 100),
                                            (4097, 328, 192), (2000, 4096, 640), (700, 4096, 1)])
def test_chunk_edges(tokens, d, chunk):
    """Chunks that end inside and at the ends of shares, a ragged last one,
    lengths that are no multiple of the kernel's 64 tokens."""
    import torch

    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn(tokens, d, generator=g, device="cuda").to(torch.bfloat16)
    wide = x.double()
    h, damp = hessian_from_activations(x, zero_floor=0.0, chunk_tokens=chunk)
    assert torch.equal(h, h.T)
    h = h.double()
    h.diagonal().sub_(damp)
    # Each sum of `tokens` exact products rounds at most that often at the
    # size of the sum of magnitudes, and at the division and the damping.
    bound = (wide.abs().T @ wide.abs()) / tokens * (tokens + 4) * 2.0 ** -24
    assert bool(((h - wide.T @ wide / tokens).abs() <= bound + 1e-7 * damp).all())


def test_two_rounds_of_workgroups():
    """A width whose tiles (378) are more than the GPU's compute units."""
    import torch

    from exl3_intel_arc_quantizer_amd._native import gram
    x = torch.randn(300, 5000, device="cuda").to(torch.bfloat16)
    h, wide = gram(x, 1.0), x.double()
    assert torch.equal(h, h.T)
    bound = (wide.abs().T @ wide.abs()) * 302 * 2.0 ** -24
    assert bool(((h.double() - wide.T @ wide).abs() <= bound).all())


@pytest.mark.parametrize("width", [260, 255])
def test_chunks_of_other_layouts(width):
    import torch

    from exl3_intel_arc_quantizer_amd._native import gram_takes
    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(900, 264, device="cuda").to(torch.bfloat16)[:, :width]
    assert not gram_takes(x)
    h, damp = hessian_from_activations(x, chunk_tokens=256)     # three and a part
    want = x.double().T @ x.double() / 900
    want.diagonal().add_(damp)
    assert float((h.double() - want).norm() / want.norm()) < 1e-6


def test_float32_sums_under_autocast():
    """Autocast chooses the products' precision, never the sum's, which is
    what the damping and the caller take."""
    import torch

    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(900, 256, device="cuda")

    def error(h, damp, x):
        assert h.dtype == torch.float32
        want = x.double().T @ x.double() / 900
        want.diagonal().add_(damp)
        return float((h.double() - want).norm() / want.norm())

    with torch.autocast("cuda", dtype=torch.bfloat16):
        for chunk in (256, 8192):
            # Inputs and products rounded to 8 bits.
            assert error(*hessian_from_activations(x, chunk_tokens=chunk), x) < 3 * 2.0 ** -8
        half = x.to(torch.float16)      # products in float32 there, autocast or not
        assert error(*hessian_from_activations(half), half) < 1e-6


def test_followed_activations():
    """Activations that torch follows go through torch's products: float32
    ones carry gradients and tangents, half-precision ones, whose products
    have no derivatives, are refused and not passed on without them."""
    import torch
    import torch.autograd.forward_ad as forward_ad

    from exl3_intel_arc_quantizer_amd.layer_quant import hessian_from_activations
    x = torch.randn(300, 128, device="cuda")
    t = torch.randn(300, 128, device="cuda")
    cross = x.double().T @ t.double() / 300
    with forward_ad.dual_level():
        h, _ = hessian_from_activations(forward_ad.make_dual(x, t))
        tangent = forward_ad.unpack_dual(h).tangent.double()
        assert float((tangent - cross - cross.T).norm() / cross.norm()) < 1e-5
        with pytest.raises((NotImplementedError, RuntimeError)):
            hessian_from_activations(forward_ad.make_dual(x.bfloat16(), t.bfloat16()))
    leaf = x.clone().requires_grad_()
    h, _ = hessian_from_activations(leaf)
    h.sum().backward()
    want = 2.0 * x.double().sum(dim=1, keepdim=True).expand(-1, 128) / 300
    assert float((leaf.grad.double() - want).norm() / want.norm()) < 1e-5
