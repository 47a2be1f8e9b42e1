"""GPU parity of the traceback walks at the ends of their ranges: rotations
that leave a walk one row, part of a row or every row but one, tiles whose
candidates all tie and tiles with infinite costs, both traceback kernels
against the numpy restatement of the reference, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from oracle.reference_encoder import ReferenceTrellisEncoder

pytestmark = pytest.mark.gpu

L = 160


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8])
def test_walk_edges(K):
    import torch

    from exl3_intel_arc_quantizer_amd import _native
    from exl3_intel_arc_quantizer_amd._native import edges_shape
    from exl3_intel_arc_quantizer_amd.gpu_quantizer import build_quantize_extension
    ext = build_quantize_extension()
    rng = np.random.default_rng(700 + K)
    tiles = rng.normal(0.0, 1.2, size=(3, L)).astype(np.float16)
    tiles[1] = 0.0
    tiles[2, 60:63] = np.inf
    n, E = len(tiles), 65536 >> K
    ref = ReferenceTrellisEncoder(K=K, tile_len=L)
    x = torch.from_numpy(tiles.astype(np.float32)).cuda()
    for roll in (1, 77, L - 1):
        # The reference's end state and path for every tile.
        want = []
        for t in tiles:
            preds = np.zeros((L, E), dtype=np.uint16)
            with np.errstate(invalid="ignore", over="ignore"):
                best = ref.argmin_cost(ref.forward(t, roll, -1, preds))
            end, _, _ = ref.backward(preds, roll, False, best)
            _, idx, _ = ref.backward(preds, roll, True, end)
            want.append((end, idx))
        costs = torch.zeros((n, 2, E), dtype=torch.float16, device="cuda")
        edges = torch.zeros(edges_shape(n, K, L), dtype=torch.uint8, device="cuda")
        pre = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        ext.quantize_tiles_forward_pass(x, costs, edges, pre, K, False, True, roll, 0)
        previous = _native.set_traceback_policy("auto")
        try:
            for policy in ("rows", "stream"):
                _native.set_traceback_policy(policy)
                print(f"K={K} roll={roll} {policy}", flush=True)
                ends = torch.zeros((n,), dtype=torch.int32, device="cuda")
                w = torch.zeros((n, L), dtype=torch.float32, device="cuda")
                idx = torch.zeros((n, L), dtype=torch.int16, device="cuda")
                ext.quantize_tiles_backward_pass(costs, edges, w, idx, ends, n, K, False, True,
                                                 roll, 0, False)
                got_end = ends.cpu().numpy()
                ext.quantize_tiles_backward_pass(costs, edges, w, idx, ends, n, K, False, True,
                                                 roll, 0, True)
                got = idx.cpu().numpy().view(np.uint16)
                for t in range(n):
                    assert int(got_end[t]) == want[t][0], (policy, t)
                    np.testing.assert_array_equal(got[t], want[t][1], err_msg=f"{policy} {t}")
        finally:
            _native.set_traceback_policy(previous)
