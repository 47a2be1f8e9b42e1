"""The blocked Cholesky factorisation and the fold of a block LDL at the
edges of their tiles (16) and panels (128) against float64."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spd(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((2 * n + 8, n))
    a = x.T @ x / (2 * n + 8) + 0.1 * np.eye(n)
    return a.astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 143, 144, 256, 257, 400, 645])
def test_factor_and_tile_inverses(n):
    import torch

    from exl3_intel_arc_quantizer_amd.ldlq import _cholesky
    a = _spd(n, n)
    noise = np.triu(np.full((n, n), np.nan, dtype=np.float32), 1)   # above: not read
    L, inv, info = _cholesky(torch.from_numpy(a + noise).cuda())
    L, inv = L.cpu().numpy().astype(np.float64), inv.cpu().numpy().astype(np.float64)
    assert int(info.item()) == 0 and inv.shape == (-(-n // 16), 16, 16)
    assert not np.triu(L, 1).any() and not np.triu(inv, 1).any()
    want = np.linalg.cholesky(a.astype(np.float64))
    # Backward error of a float32 factorisation, n + 1 roundings an entry.
    eps = 2.0 ** -24
    assert np.abs(L @ L.T - a).max() <= 4 * (n + 1) * eps * np.abs(a).max()
    np.testing.assert_allclose(L, want, rtol=0, atol=1e-4 * np.abs(want).max())
    for t in range(inv.shape[0]):
        m = min(16, n - 16 * t)
        blk = L[16 * t:16 * t + m, 16 * t:16 * t + m]
        np.testing.assert_allclose(inv[t, :m, :m] @ blk, np.eye(m), rtol=0,
                                   atol=64 * eps * np.linalg.cond(blk))


@pytest.mark.parametrize("n", [16, 48, 128, 144, 272, 656])
def test_fold(n):
    import torch

    from exl3_intel_arc_quantizer_amd.ldlq import block_ldl
    a = _spd(n, 3 * n)
    res = block_ldl(torch.from_numpy(a).cuda())
    L = res.cholesky.cpu().numpy().astype(np.float64)
    inv = res.block_inverses.cpu().numpy().astype(np.float64)
    want = np.zeros((n, n))
    for b in range(n // 16):
        cols = slice(16 * b, 16 * b + 16)
        want[:, cols] = L[:, cols] @ inv[b]
        want[cols, cols] = np.eye(16)
    got = res.transformed.cpu().numpy()
    # Sixteen float32 products and sums an entry.
    bound = 32 * 2.0 ** -24 * (np.abs(L).max() * np.abs(inv).max() * 16)
    np.testing.assert_allclose(got, want, rtol=0, atol=bound)
    assert not np.triu(got, 1).any()
    np.testing.assert_array_equal(np.diagonal(got), 1.0)


@pytest.mark.parametrize("j", [0, 3, 5, 17, 130, 300, 399])
def test_infinite_pivot(j):
    """An infinite diagonal entry is a pivot with an infinite root: its column
    is zero below, and the rest is the factor of the matrix without it."""
    import torch

    from exl3_intel_arc_quantizer_amd.ldlq import cholesky_ex
    n = 400
    a = _spd(n, j)
    a[j, j] = np.inf
    L, info = cholesky_ex(torch.from_numpy(a).cuda())
    L = L.cpu().numpy()
    assert int(info.item()) == 0
    assert L[j, j] == np.inf and not L[j + 1:, j].any()
    keep = np.arange(n) != j
    want = np.linalg.cholesky(a[np.ix_(keep, keep)].astype(np.float64))
    np.testing.assert_allclose(L[np.ix_(keep, keep)], want, rtol=0,
                               atol=1e-4 * np.abs(want).max())


@pytest.mark.parametrize("n", [160, 520])
def test_ill_conditioned(n):
    """Eigenvalues over 2^18 (float32 still factors it): the backward error
    stays that of n + 1 roundings an entry."""
    import torch

    from exl3_intel_arc_quantizer_amd.ldlq import cholesky_ex
    rng = np.random.default_rng(n)
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    a = ((q * 2.0 ** -rng.uniform(0.0, 18.0, n)) @ q.T)
    a = (0.5 * (a + a.T)).astype(np.float32)
    L, info = cholesky_ex(torch.from_numpy(a).cuda())
    L = L.cpu().numpy().astype(np.float64)
    assert int(info.item()) == 0
    assert np.abs(L @ L.T - a).max() <= 4 * (n + 1) * 2.0 ** -24 * np.abs(a).max()
