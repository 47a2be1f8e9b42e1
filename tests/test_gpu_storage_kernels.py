"""The one-pass storage kernels against the separate steps they replace, bit
for bit: exl3_unrotate and exl3_decode_weight against the unpack kernel, the
codebook table, the un-permutation and exl3_hadamard128 with torch scalings
in between (the same fp32 operations); the wide packing kernel against the
span-by-span one, which misaligned buffers take."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _scales(torch, k, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(k, generator=g, device="cuda"),
            torch.rand(n, generator=g, device="cuda") + 0.5)


def _separate(w_hat, su, sv):
    from exl3_intel_arc_quantizer_amd.hadamard import preapply_had_l, preapply_had_r
    w = preapply_had_l(w_hat) * su[:, None]
    return preapply_had_r(w) * sv[None, :]


@pytest.mark.parametrize("k,n", [(128, 128), (128, 640), (384, 256)])
def test_unrotate(k, n):
    import torch

    from exl3_intel_arc_quantizer_amd.hadamard import weight_from_quantized
    w_hat = torch.randn(k, n, device="cuda")
    su, sv = _scales(torch, k, n, 1)
    assert torch.equal(weight_from_quantized(w_hat, su, sv), _separate(w_hat, su, sv))
    # A strided matrix and a scale vector off the 8-byte grid.
    wide = torch.randn(k, n + 8, device="cuda")[:, 3:n + 3]
    off = torch.cat([sv[:1], sv])[1:]
    assert torch.equal(weight_from_quantized(wide, su, off), _separate(wide, su, sv))


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8])
def test_decode_weight(K):
    import torch

    from exl3_intel_arc_quantizer_amd.serialization import (decode_weight_from_storage,
                                                            unpack_module_trellis)
    from exl3_intel_arc_quantizer_amd.trellis_format import codebook_lut, tensor_core_perm
    for cb, (k, n) in enumerate([(128, 256), (256, 128), (384, 384)]):
        g = torch.Generator(device="cuda").manual_seed(10 * K + cb)
        words = torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), generator=g,
                              device="cuda", dtype=torch.int32).to(torch.int16)
        su, sv = _scales(torch, k, n, K)
        lut = torch.from_numpy(codebook_lut(cb)).cuda().float()
        vals = lut[unpack_module_trellis(words, K).long() & 0xFFFF]
        tiles = torch.empty_like(vals)
        tiles[..., torch.as_tensor(tensor_core_perm()).long().cuda()] = vals
        w_hat = tiles.view(k // 16, n // 16, 16, 16).permute(0, 2, 1, 3).reshape(k, n)
        got = decode_weight_from_storage(words, su, sv, K, cb)
        assert torch.equal(got, _separate(w_hat, su, sv)), (K, cb)


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8])
def test_pack_alignments(K):
    import torch

    from exl3_intel_arc_quantizer_amd._native import extension
    for n in (1, 33):
        buf = torch.randint(-32768, 32768, (n * 256 + 8,), device="cuda",
                            dtype=torch.int32).to(torch.int16)
        aligned = buf[8:].view(n, 256)
        shifted = torch.cat([buf[:1], aligned.reshape(-1)])[1:].view(n, 256)
        assert aligned.data_ptr() % 16 == 0 and shifted.data_ptr() % 16
        out = torch.zeros((n, 16 * K), dtype=torch.int16, device="cuda")
        ref = torch.zeros(n * 16 * K + 1, dtype=torch.int16, device="cuda")[1:].view(n, 16 * K)
        extension().pack_trellis(aligned, out, K)
        extension().pack_trellis(shifted, ref, K)
        assert torch.equal(out, ref)


def test_gradient_of_output_scales():
    """A recorded sv gives the same weight and its gradient, the column sums
    of the weight before the last scaling."""
    import torch

    from exl3_intel_arc_quantizer_amd.hadamard import weight_from_quantized
    from exl3_intel_arc_quantizer_amd.serialization import (decode_weight_from_storage,
                                                            pack_module_trellis)
    g = torch.Generator(device="cuda").manual_seed(5)
    su = torch.rand(128, generator=g, device="cuda") + 0.5
    sv = torch.rand(256, generator=g, device="cuda") + 0.5
    w = torch.randn(128, 256, generator=g, device="cuda")
    states = torch.randint(-32768, 32768, (8, 16, 256), generator=g, device="cuda",
                           dtype=torch.int32).to(torch.int16)
    trellis = pack_module_trellis(states, 4)
    for decode in (lambda v: weight_from_quantized(w, su, v),
                   lambda v: decode_weight_from_storage(trellis, su, v, 4)):
        plain = decode(sv)
        leaf = sv.clone().requires_grad_()
        out = decode(leaf)
        assert torch.equal(out, plain) and not plain.requires_grad
        out.sum().backward()
        # Sums of 128 float32 terms.
        want, size = (plain.double() / sv).sum(dim=0), (plain.double() / sv).abs().sum(dim=0)
        assert bool(((leaf.grad - want).abs() <= 140 * 2.0 ** -24 * size).all())


def _decoders(torch, g):
    from exl3_intel_arc_quantizer_amd.hadamard import weight_from_quantized
    from exl3_intel_arc_quantizer_amd.serialization import (decode_weight_from_storage,
                                                            pack_module_trellis)
    w = torch.randn(128, 256, generator=g, device="cuda")
    states = torch.randint(-32768, 32768, (8, 16, 256), generator=g, device="cuda",
                           dtype=torch.int32).to(torch.int16)
    trellis = pack_module_trellis(states, 4)
    return (lambda su, sv: weight_from_quantized(w, su, sv),
            lambda su, sv: decode_weight_from_storage(trellis, su, sv, 4))


def test_tangent_of_output_scales():
    """A forward-mode sv gives the same weight and carries its tangent."""
    import torch
    import torch.autograd.forward_ad as forward_ad
    g = torch.Generator(device="cuda").manual_seed(6)
    su, sv, t = (torch.rand(n, generator=g, device="cuda") + 0.5 for n in (128, 256, 256))
    for decode in _decoders(torch, g):
        plain = decode(su, sv)
        with forward_ad.dual_level():
            out, tangent = forward_ad.unpack_dual(decode(su, forward_ad.make_dual(sv, t)))
            assert torch.equal(out, plain) and tangent is not None
            # One product an element, one rounding; the weight's own is one more.
            torch.testing.assert_close(tangent.double(), plain.double() / sv * t,
                                       rtol=4 * 2.0 ** -24, atol=0.0)


def test_derivatives_of_input_scales():
    """A recorded or forward-mode su, alone or beside a recorded sv, gives the
    same weight, and its derivatives are those of a product that is linear in
    su."""
    import torch
    import torch.autograd.forward_ad as forward_ad
    g = torch.Generator(device="cuda").manual_seed(7)
    su, sv, t = (torch.rand(n, generator=g, device="cuda") + 0.5 for n in (128, 256, 128))
    pull = torch.randn(128, 256, generator=g, device="cuda")
    for decode in _decoders(torch, g):
        plain = decode(su, sv)
        # d/d su[r] of sum(pull * weight): row r of a weight with su = 1.
        rows = decode(torch.ones_like(su), sv).double() * pull.double()
        for with_sv in (False, True):
            leaf = su.clone().requires_grad_()
            col = sv.clone().requires_grad_(with_sv)
            out = decode(leaf, col)
            assert torch.equal(out, plain)
            out.backward(pull)
            # 256 products a sum, behind three transforms of 7 levels.
            size = decode(torch.ones_like(su), sv).double().norm(dim=1) * pull.double().norm(dim=1)
            err = (leaf.grad.double() - rows.sum(dim=1)).abs()
            assert bool((err <= 64 * 2.0 ** -24 * size).all()), float((err / size).max())
            assert (col.grad is not None) == with_sv
        with forward_ad.dual_level():
            out, tangent = forward_ad.unpack_dual(decode(forward_ad.make_dual(su, t), sv))
            assert torch.equal(out, plain)
            want = decode(t, sv).double()
            assert float((tangent.double() - want).norm() / want.norm()) < 64 * 2.0 ** -24
