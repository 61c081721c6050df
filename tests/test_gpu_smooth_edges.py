"""Edge weights at the edges of the kernel's tiling (256-row workgroups, chunks that end inside
one, each neighbour-count variant) and where the bisection has no root to find early: equal
distances, zero distances, too few neighbours for the target."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n,k,chunk,lc", [
    (1, 11, 1000, 1.0), (255, 2, 100, 1.0), (256, 12, 256, 1.0), (257, 13, 7, 1.0),
    (700, 16, 1, 1.0), (1000, 17, 300, 0.5), (513, 24, 5000, 1.5), (300, 33, 256, 1.0),
    (600, 49, 250, 2.5), (400, 64, 100, 1.0)])
def test_smooth_edges(cuda, n, k, chunk, lc):
    import torch
    from oracle import smooth as osmooth
    from scarf_amd.smooth import smooth_knn
    say("smooth edges", n, k, chunk, lc)
    rng = np.random.default_rng(n + k)
    d = np.sort(rng.gamma(4.0, 5.0, (n, k)), axis=1).astype(np.float32)
    if n > 50:
        d[3] = 7.5                       # all equal
        d[5] = 0.0                       # all zero: no rho
        d[8, :k // 2] = 0.0              # duplicates of the row
        d[20] *= 1e-6
        d[21] *= 1e6
        d[22, 1:] = d[22, 1]             # one near, the rest level
    idx = rng.integers(0, max(n, 2), (n, k))
    idx[::9, 0] = (np.arange(n) % chunk)[::9]  # some neighbours at the row's chunk position
    _, want = osmooth.smoothen_dists(idx, d, lc, 1.5, chunk)
    _, _, w = smooth_knn(torch.from_numpy(d).cuda(), torch.from_numpy(idx).cuda(), chunk, lc, 1.5)
    assert np.abs(w.cpu().numpy() - np.asarray(want, dtype=np.float32)).max() <= 1e-5
