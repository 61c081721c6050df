"""Small FP64 products of the subspace iteration at the edges of their tiles: the tall GEMM
(16 x 16 tiles, 32-step batches), the block Gram's slice sum and the merge matrix."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("m,n,k", [(256, 1, 1), (257, 16, 32), (300, 17, 33), (2000, 94, 94),
                                   (1001, 65, 31), (511, 256, 256), (255, 40, 40)])
def test_tall_gemm(cuda, m, n, k):
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    say("tall gemm", m, n, k)
    rng = np.random.default_rng(m + n + k)
    A = rng.standard_normal((m, k + 3))
    B = rng.standard_normal((k, n + 5))
    C = rng.standard_normal((m, n + 2))
    a, b, c = (torch.from_numpy(x).cuda() for x in (A, B, C))
    _lib.call("sh_dgemm", 0, m, n, k, 1.5, ptr(a), k + 3, ptr(b), n + 5, -0.5, ptr(c), n + 2,
              stream_handle())
    got = c.cpu().numpy()
    want = 1.5 * A[:, :k] @ B[:, :n] - 0.5 * C[:, :n]
    # k products and two more terms, each within an ulp of the running magnitude
    tol = (k + 4) * 2.0 ** -52 * (1.5 * np.abs(A[:, :k]) @ np.abs(B[:, :n]) + np.abs(C[:, :n]))
    assert np.all(np.abs(got[:, :n] - want) <= tol)
    assert np.array_equal(got[:, n:], C[:, n:])


@pytest.mark.parametrize("d,na,nb", [(5, 3, 2), (130, 33, 31), (2000, 94, 94)])
def test_block_gram_edges(cuda, d, na, nb):
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    say("block gram", d, na, nb)
    rng = np.random.default_rng(d)
    A, B = rng.standard_normal((d, na)), rng.standard_normal((d, nb))
    a, b = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    c = torch.empty((na, nb), dtype=torch.float64, device="cuda")
    nbytes = _lib.lib().sh_block_gram_workspace(d, na, nb)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    _lib.call("sh_block_gram", ptr(a), na, na, ptr(b), nb, nb, d, ptr(c), ptr(ws), nbytes,
              stream_handle())
    tol = (d + 2) * 2.0 ** -52 * (np.abs(A).T @ np.abs(B))
    assert np.all(np.abs(c.cpu().numpy() - A.T @ B) <= tol)


@pytest.mark.parametrize("d,nc", [(1, 1), (63, 5), (64, 32), (65, 33), (200, 51)])
@pytest.mark.parametrize("first", [True, False])
def test_merge_matrix_edges(cuda, d, nc, first):
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    say("merge matrix", d, nc, first)
    rng = np.random.default_rng(d + nc)
    G = rng.standard_normal((d, d))
    G = G + G.T
    bm, mc = rng.standard_normal(d), rng.standard_normal(d)
    V, s2 = rng.standard_normal((nc, d)), rng.uniform(1, 9, nc)
    t = [torch.from_numpy(x).cuda() for x in (G, bm, V, s2, mc)]
    M = torch.empty((d, d), dtype=torch.float64, device="cuda")
    _lib.call("sh_merge_matrix", ptr(t[0]), d, 7.0, ptr(t[1]), None if first else ptr(t[2]),
              None if first else ptr(t[3]), 0 if first else nc, None if first else ptr(t[4]),
              ptr(M), stream_handle())
    got = M.cpu().numpy()
    want = G - 7.0 * np.outer(bm, bm)
    mag = np.abs(G) + 7.0 * np.outer(np.abs(bm), np.abs(bm))
    if not first:
        want = want + (V.T * s2) @ V + np.outer(mc, mc)
        mag = mag + (np.abs(V).T * s2) @ np.abs(V) + np.outer(np.abs(mc), np.abs(mc))
    assert np.all(np.abs(got - want) <= (nc + 6) * 2.0 ** -52 * mag)
    assert np.array_equal(got, got.T)


@pytest.mark.parametrize("d,nc", [(401, 51), (640, 9), (640, 10), (1200, 3)])
def test_merge_matrix_tiles(cuda, d, nc):
    """Past 400 features and a few million products the tiled kernel, on both sides of the line."""
    test_merge_matrix_edges(cuda, d, nc, False)


@pytest.mark.parametrize("m,n,k", [(12_800, 64, 64), (12_801, 64, 64), (20_000, 94, 94),
                                   (20_000, 200, 16), (20_000, 200, 17)])
def test_gemm_of_many_rows(cuda, m, n, k):
    """Both kernels' sides of the lines in tiles, padding and depth."""
    test_tall_gemm(cuda, m, n, k)
