"""Statistics and projection kernels at the edges of their tiling: slabs of few rows, empty
and very long rows, column blocks, row batches of 64, one and two column passes."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _csr(n, d, lens, seed):
    """Host CSR whose row i holds lens[i % len(lens)] non-zeros at random columns."""
    from scarf_amd.synth import CSR
    rng = np.random.default_rng(seed)
    ln = np.array([min(lens[i % len(lens)], d) for i in range(n)], dtype=np.int64)
    cols = [np.sort(rng.choice(d, m, replace=False)) for m in ln]
    rp = np.concatenate([[0], np.cumsum(ln)])
    vals = rng.integers(1, 40, int(rp[-1])).astype(np.uint32)
    return CSR(vals, np.concatenate(cols + [np.zeros(0, np.int64)]).astype(np.int32), rp, d)


@pytest.mark.parametrize("n,chunk,d,lens", [
    (1, 1000, 30, (7,)), (15, 4, 30, (0, 1, 30)), (385, 384, 64, (3, 0, 64)),
    (4097, 1000, 100, (0, 5, 100)), (700, 700, 2048, (512, 513, 1, 1030)),
    (333, 100, 5000, (0, 700, 2500))])
def test_stats_edges(cuda, n, chunk, d, lens):
    from scarf_amd.device import DeviceCSR
    from scarf_amd.normalize import NormParams, feature_stats
    say("stats edges", n, chunk, d)
    h = _csr(n, d, lens, 3)
    st = feature_stats(DeviceCSR.from_host(h), chunk, NormParams())
    X = h.to_dense()
    lib = X.sum(1)
    lib[lib == 0] = 1
    assert np.array_equal(st.libsize.cpu().numpy(), lib)
    x = np.log1p(1000.0 * X / lib[:, None])
    for c, (a, b) in enumerate(st.chunk_bounds):
        # a sum of m positive terms is within (m + 2) half-ulps of itself
        tol = (b - a + 2) * 2.0 ** -53
        np.testing.assert_allclose(st.chunk_sums[c].cpu().numpy(), x[a:b].sum(0), rtol=2 * tol)
        np.testing.assert_allclose(st.chunk_sumsq[c].cpu().numpy(), (x[a:b] ** 2).sum(0),
                                   rtol=4 * tol)
    again = feature_stats(DeviceCSR.from_host(h), chunk, NormParams())
    assert bool((again.chunk_sums == st.chunk_sums).all())
    assert bool((again.chunk_sumsq == st.chunk_sumsq).all())


@pytest.mark.parametrize("D", [1, 4, 50, 64, 65, 128])
@pytest.mark.parametrize("mapped", [False, True])
def test_project_edges(cuda, D, mapped):
    from scarf_amd.device import DeviceCSR, col_map_tensor
    from scarf_amd.normalize import NormParams
    from scarf_amd.pca import Projector
    say("project edges", D, mapped)
    d_in = 400
    h = _csr(203, d_in, (0, 1, 3, 4, 63, 64, 65, 127, 128, 129, 400), 5)
    rng = np.random.default_rng(6)
    keep = np.sort(rng.choice(d_in, 250, replace=False)) if mapped else np.arange(d_in)
    d = keep.shape[0]
    W = rng.standard_normal((d, D))
    mu, sd = rng.uniform(0.1, 1.0, d), rng.uniform(0.5, 2.0, d)
    cm, _ = col_map_tensor(d_in, keep if mapped else None)
    proj = Projector.build(W, mu, sd, clip=3.0)
    E = proj.project(DeviceCSR.from_host(h), NormParams(), col_map=cm).cpu().numpy()
    X = h.to_dense()[:, keep]
    lib = X.sum(1)
    lib[lib == 0] = 1
    z = np.clip((np.log1p(1000.0 * X / lib[:, None]) - mu) / sd, -3.0, 3.0)
    # FP32 x, z and W (a few roundings each, |z| <= 3 from operands up to 8 / 0.5) and a sum
    # of at most 400 products in four chains of 100, plus the constant
    tol = (100 + 60) * 2.0 ** -24 * (6.0 * np.abs(W).sum(0) + 1.0)
    assert np.all(np.abs(E - z @ W) <= tol[None, :])
