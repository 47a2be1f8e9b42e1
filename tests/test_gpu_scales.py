"""The scale kernels of regularize at the ends of their ranges: the skew by
radix selection against a float64 sort (ties at the threshold, lengths
around the 1/50 cut, a strided diagonal, NaN), the scale vectors against
float64, the row RMS at slice counts around the chunk and batch sizes, and the
two passes over the matrix against the single transforms."""

from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS32 = 2.0 ** -24


def _run(torch, x, diag, decide=2, forced=False, sv=None):
    from exl3_intel_arc_quantizer_amd._native import output_scales
    n = x.shape[1]
    sv = torch.ones(n, device="cuda") if sv is None else sv
    out = [torch.empty(n, device="cuda") for _ in range(3)]
    flags = torch.zeros(3, dtype=torch.float64, device="cuda")
    output_scales(x, sv, decide, forced, *out, flags, diag)
    return [t.cpu().numpy().astype(np.float64) for t in out], flags.tolist()


@pytest.mark.parametrize("length", [1, 49, 50, 99, 100, 1023, 4097, 12288])
def test_skew(length):
    import torch
    rng = np.random.default_rng(length)
    x = torch.randn(128, 128, device="cuda")
    for case in ("random", "ties", "strided"):
        d = (rng.random(length) * 4.0).astype(np.float32)
        if case == "ties":
            d = np.round(d)
        if case == "strided":
            host = np.zeros((length, 3), dtype=np.float32)
            host[:, 1] = d
            diag = torch.from_numpy(host).cuda()[:, 1]
        else:
            diag = torch.from_numpy(d).cuda()
        root = np.sort(np.sqrt(d).astype(np.float64))[::-1]
        want = root[:length // 50].sum() / root.sum()
        _, flags = _run(torch, x, diag)
        # Double sums of the same float32 roots, two roundings to float32 and
        # a division (one more each for the roots).
        assert flags[1] == pytest.approx(want, rel=4 * EPS32, abs=0.0), case
        assert flags[2] == float(np.float32(flags[1]) < np.float32(0.15))
    d[0] = np.nan
    assert math.isnan(_run(torch, x, torch.from_numpy(d).cuda())[1][1])


@pytest.mark.parametrize("k,n", [(32, 1), (128, 63), (1056, 65), (4128, 1100)])
def test_output_scales(k, n):
    import torch
    rng = np.random.default_rng(n)
    w = rng.standard_normal((k, n)).astype(np.float32)
    if n > 8:
        w[:, 5] = 0.0
    sv = (rng.random(n) + 0.5).astype(np.float32)
    col = np.sqrt((w.astype(np.float64) ** 2).mean(axis=0))
    v = col / col.mean()
    dead = v < 1e-30
    floored = np.where(dead, 0.1, v)
    x, svd = torch.from_numpy(w).cuda(), torch.from_numpy(sv).cuda()
    # Sums of k squares in float32, slice by slice: relative error below
    # (32 + k / 32 + 4) roundings on the sum, half of that on its root.
    tol = (36 + k / 32) * EPS32
    (scales, div, out), flags = _run(torch, x, None, decide=1, sv=svd)
    np.testing.assert_allclose(scales, floored, rtol=tol)
    np.testing.assert_allclose(div, sv * floored + 1e-10, rtol=tol)
    np.testing.assert_allclose(out, np.where(dead, 0.0, sv * floored + 1e-10), rtol=tol)
    assert flags[0] == 1.0 and flags[2] == 1.0
    (scales, div, out), flags = _run(torch, x, None, decide=0, sv=svd)
    np.testing.assert_allclose(scales, v, rtol=tol, atol=0)
    np.testing.assert_array_equal(div, sv.astype(np.float64))
    np.testing.assert_array_equal(out, np.where(dead, 0.0, sv.astype(np.float64)))
    assert flags[2] == 0.0
    # A matrix without energy: the scales apply only where the choice is forced.
    for forced in (False, True):
        (scales, div, out), flags = _run(torch, torch.zeros_like(x), None, 0, forced, svd)
        assert flags[0] == 0.0 and flags[2] == float(forced) and not out.any()
        np.testing.assert_allclose(scales, 0.1 if forced else 0.0, rtol=EPS32)


@pytest.mark.parametrize("rows,slices", [(1, 1), (63, 2), (64, 127), (65, 128), (130, 129),
                                         (70, 300)])
def test_row_reduction(rows, slices):
    import torch

    from exl3_intel_arc_quantizer_amd._native import block_rms, block_rms_from_slices, input_scales
    g = torch.Generator(device="cuda").manual_seed(rows)
    sq = torch.rand(rows, slices, generator=g, device="cuda")
    sq[rows // 2] = 0.0
    n = 32 * slices
    ref = np.zeros(rows, dtype=np.float32)
    host = sq.cpu().numpy()
    for s in range(slices):     # slice order, float32
        ref = host[:, 0].copy() if s == 0 else ref + host[:, s]
    ref = np.sqrt(ref / np.float32(n))
    out = torch.empty(rows, device="cuda")
    block_rms_from_slices(sq, out, n)
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    su = torch.rand(rows, generator=g, device="cuda") + 0.5
    scales, su_out = torch.empty_like(su), torch.empty_like(su)
    input_scales(sq, su, scales, su_out, n)
    want = np.where(ref < 1e-30, np.float32(0.1), ref)
    np.testing.assert_array_equal(scales.cpu().numpy(), want)
    np.testing.assert_allclose(su_out.cpu().numpy(),
                               su.cpu().numpy().astype(np.float64) * want / -1.24371088 + 1e-10,
                               rtol=4 * EPS32)
    # Both dimensions of block_rms go through the same reductions.
    x = torch.randn(n, rows, generator=g, device="cuda")
    for dim in (0, 1):
        y = x if dim == 0 else x.t().contiguous()
        block_rms(y, out, dim)
        np.testing.assert_allclose(out.cpu().numpy(),
                                   np.sqrt((x.cpu().numpy().astype(np.float64) ** 2).mean(0)),
                                   rtol=(36 + slices) * EPS32)


@pytest.mark.parametrize("k,n", [(128, 128), (128, 1152), (640, 128), (384, 1024)])
@pytest.mark.parametrize("offset", [0, 1])
def test_rotation_passes(k, n, offset):
    """The rotation is bit for bit the two scaled transforms and the row
    energies are those of the first, also from a matrix that is only 4-byte
    aligned; infinities and NaN land in the same places."""
    import torch

    from exl3_intel_arc_quantizer_amd._native import hadamard128_scaled, rotate, row_energy
    g = torch.Generator(device="cuda").manual_seed(k + n)
    x = torch.randn(k * n + offset, generator=g, device="cuda")[offset:].view(k, n)
    sv = torch.rand(n, generator=g, device="cuda") * 3 + 0.1
    su = torch.rand(k, generator=g, device="cuda") * 3 - 1.6
    for special in (False, True):
        if special:
            x[1, 5], x[k - 1, n - 1], x[k // 2] = float("inf"), float("nan"), 0.0
            x[6, 0] = x[6, 127] = float("-inf")
            x[8, 64] = float("-inf")
        before = x.clone()
        mid, want = torch.empty(k, n, device="cuda"), torch.empty(k, n, device="cuda")
        hadamard128_scaled(before, mid, 1, divisor=sv)
        hadamard128_scaled(mid, want, 0, divisor=su)
        out, energy = torch.empty_like(want), torch.empty(k, n // 128, device="cuda")
        row_energy(x, sv, energy)
        rotate(x, sv, su, out)
        for got, ref in ((out, want), (x, before)):
            assert torch.equal(got.isnan(), ref.isnan())
            assert torch.equal(got.nan_to_num(), ref.nan_to_num())
        wide = mid.double().square().view(k, n // 128, 128).sum(dim=2)
        assert torch.equal(energy.isnan(), wide.isnan())
        assert torch.equal(energy.isinf(), wide.isinf())
        # A quotient, a square and seven additions here; seven additions, a
        # scaling, and the quotient in the transform.
        torch.testing.assert_close(energy.double().nan_to_num(posinf=0.0),
                                   wide.nan_to_num(posinf=0.0), rtol=32 * EPS32, atol=0.0)
    with pytest.raises(RuntimeError):
        rotate(x, sv[:-1], su, out)


@pytest.mark.parametrize("apply", [None, False, True])
@pytest.mark.parametrize("skewed", [False, True])
def test_recorded_scales(apply, skewed):
    """regularize's su and sv keep the gradient and the tangent of those given:
    both are affine in what they come from (regularize.py:159-181), at the same
    values as without."""
    import torch
    import torch.autograd.forward_ad as forward_ad

    from exl3_intel_arc_quantizer_amd.regularize import regularize
    k, n = 256, 384
    g = torch.Generator(device="cuda").manual_seed(9)
    w = torch.randn(k, n, generator=g, device="cuda")
    w[:, 7] = 0.0
    w[9] = 0.0
    su = torch.rand(k, 1, generator=g, device="cuda") + 0.5
    sv = torch.rand(1, n, generator=g, device="cuda") + 0.5
    sv[0, 3] = 0.1
    diag = torch.rand(k, generator=g, device="cuda") + 0.1
    if skewed:
        diag[:2] = 1e6
    args = lambda: None if apply is None else {"apply_out_scales": apply}
    plain = regularize(w, su, sv, quant_args=args(), H_diag=diag)
    assert not plain.su.requires_grad and not plain.sv.requires_grad
    a, b = su.clone().requires_grad_(), sv.clone().requires_grad_()
    for pair in ((a, sv), (su, b), (a, b)):
        a.grad = b.grad = None
        r = regularize(w, *pair, quant_args=args(), H_diag=diag)
        for name in ("weight", "su", "sv", "out_channel_scales", "in_channel_scales"):
            assert torch.equal(getattr(r, name), getattr(plain, name)), name
        assert r.apply_out_scales == plain.apply_out_scales
        assert r.su.requires_grad == pair[0].requires_grad
        assert r.sv.requires_grad == pair[1].requires_grad and not r.weight.requires_grad
        (r.su.sum() + r.sv.sum()).backward() if r.su.requires_grad and r.sv.requires_grad else \
            (r.su if r.su.requires_grad else r.sv).sum().backward()
        if r.su.requires_grad:
            torch.testing.assert_close(a.grad, plain.in_channel_scales / -1.24371088,
                                       rtol=4 * EPS32, atol=0.0)
        if r.sv.requires_grad:
            want = plain.out_channel_scales.clone() if plain.apply_out_scales \
                else torch.ones_like(sv)
            want[0, 7] = 0.0
            torch.testing.assert_close(b.grad, want, rtol=4 * EPS32, atol=0.0)
    with forward_ad.dual_level():
        r = regularize(w, forward_ad.make_dual(su, 2 * su), forward_ad.make_dual(sv, 3 * sv),
                       quant_args=args(), H_diag=diag)
        (s0, st), (v0, vt) = (forward_ad.unpack_dual(x) for x in (r.su, r.sv))
        assert torch.equal(s0, plain.su) and torch.equal(v0, plain.sv)
        # The added 1e-10 is below a rounding.
        torch.testing.assert_close(st, 2 * plain.su, rtol=4 * EPS32, atol=0.0)
        torch.testing.assert_close(vt, 3 * plain.sv, rtol=4 * EPS32, atol=0.0)
