"""mi_gelu_mlp_f32 at the edges of its tiles, at the fp32 bar (1e-5 of the
largest value) against the float64 oracle; calls share one workspace, so its
counters have to be zero again after each."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import rng, to_np, to_torch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from autotuner_runtime import ops  # noqa: E402


@pytest.mark.parametrize("M,K,H,N", [
    (1, 4, 4, 1),          # one chunk of everything
    (9, 256, 64, 17),      # one hidden chunk, a second row block of one row, N off 4
    (3, 260, 1028, 260),   # K and N past one batch, 17 chunks with 4 units in the last
    (20, 1024, 2048, 68),  # 32 chunks, four batches of W1
    (8, 20, 100, 321),     # N past 256 and off 4
    (50, 128, 128, 30),    # the last rows of the small-network form at H = 128
    (51, 128, 128, 30),    # ... and one past it
    (8, 56, 288, 259),     # ... past H = 128
    (9, 56, 288, 259),
    (3, 164, 8, 5),        # rows too long for it
])
def test_tiny_mlp_tile_edges(M, K, H, N):
    r = rng(6000 + M + K + H + N)
    x, w1, b1 = (r.normal(0, s, n).astype(np.float32) for s, n in ((1, (M, K)), (K ** -0.5, (H, K)), (1, H)))
    w2, b2 = (r.normal(0, s, n).astype(np.float32) for s, n in ((H ** -0.5, (N, H)), (1, N)))
    args = [to_torch(a, "float32") for a in (x, w1, b1, w2, b2)]
    want = oracle.tiny_mlp(x, w1, b1, w2, b2)
    for _ in range(2):
        got = to_np(ops.gelu_mlp_f32(*args)).astype(np.float64)
        err = np.abs(got - want).max() / np.abs(want).max()
        assert err <= 1e-5, err
