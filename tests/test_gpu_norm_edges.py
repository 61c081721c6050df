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


@pytest.mark.parametrize("d_in,D,clip,mapped", [
    (3, 1, 0.0, False), (40, 64, 3.0, False), (2500, 50, 3.0, True), (2500, 33, 0.0, False),
    (8192, 64, 3.0, False)])
def test_project_tables_equal_general_path(cuda, d_in, D, clip, mapped):
    """From 131,072 rows on, the most used rows of W come from LDS: the same bits as the general
    kernel gives for pieces of fewer rows, with all of W in the table and with part of it,
    empty and long rows, counts on both sides of 64 and an infinity in W."""
    import torch

    from scarf_amd.device import DeviceCSR, col_map_tensor
    from scarf_amd.normalize import NormParams
    from scarf_amd.pca import Projector
    from scarf_amd.synth import CSR
    say("project tables", d_in, D, clip, mapped)
    rng = np.random.default_rng(8)
    n = 131072 + 5
    ln = np.minimum(np.array([0, 1, 31, 33, 64, 65, 5, 2, 9, 20])[np.arange(n) % 10], d_in)
    ln[[7, 70_000, n - 1]] = min(d_in, 1000)
    rp = np.concatenate([[0], np.cumsum(ln)]).astype(np.int64)
    within = np.arange(rp[-1]) - np.repeat(rp[:-1], ln)
    # distinct sorted columns of a row, the low ones the more frequent
    gap = np.maximum(d_in // np.maximum(np.repeat(ln, ln), 1), 1)
    cols = np.minimum(within * gap + (rng.random(rp[-1]) ** 3 * gap).astype(np.int64), d_in - 1)
    vals = np.where(rng.random(rp[-1]) < 0.02, rng.integers(60, 5000, rp[-1]),
                    rng.integers(1, 8, rp[-1])).astype(np.uint32)
    csr = DeviceCSR.from_host(CSR(vals, cols.astype(np.int32), rp, d_in))
    keep = np.sort(rng.choice(d_in, d_in // 2, replace=False)) if mapped else np.arange(d_in)
    d = keep.shape[0]
    W = rng.standard_normal((d, D))
    W[d // 2, 0] = np.inf
    cm, _ = col_map_tensor(d_in, keep if mapped else None)
    proj = Projector.build(W, rng.uniform(0.1, 1.0, d), rng.uniform(0.5, 2.0, d), clip=clip)
    proj.c.zero_()  # finite: the infinity of W stays in the rows that use it
    E = proj.project(csr, NormParams(), col_map=cm)
    for a in range(0, n, 50_000):
        m = min(50_000, n - a)
        part = proj.project(csr, NormParams(), col_map=cm, row_start=a, n_rows=m)
        assert torch.equal(E[a:a + m].view(torch.int32), part.view(torch.int32))
    assert bool(torch.isfinite(E[:, 0]).any()) and not bool(torch.isfinite(E[:, 0]).all())


@pytest.mark.parametrize("sf", [1e-6, 1.0, 1000.0, 1e12])
def test_stats_values_over_the_range(cuda, sf):
    """One row a chunk, so that a sum is one value: counts over all of uint32 and stored zeros,
    library sizes from 0 over 1e-300 and 1e300 to infinity, where the quotient's correction and
    the logarithm's table hand over to the general way."""
    import torch

    from scarf_amd.device import DeviceCSR
    from scarf_amd.normalize import NormParams, feature_stats
    from scarf_amd.synth import CSR
    say("stats values", sf)
    rng = np.random.default_rng(12)
    n, d = 48, 300
    vals = np.exp(rng.uniform(0, np.log(2.0 ** 32 - 1), n * d)).astype(np.uint32)
    vals[rng.random(n * d) < 0.05] = 0
    vals[5::97] = 2 ** 32 - 1
    lib = np.concatenate([[0.0, np.inf, 1e-300, 1e300, 5e-324, 1e-281, 1e281],
                          np.exp(rng.uniform(-20, 40, n - 7))])
    h = CSR(vals, np.tile(np.arange(d, dtype=np.int32), n), np.arange(n + 1, dtype=np.int64) * d, d)
    st = feature_stats(DeviceCSR.from_host(h), 1, NormParams(size_factor=sf,
                                                            renormalize_subset=False),
                       n_counts=torch.from_numpy(lib))
    with np.errstate(all="ignore"):
        x = np.log1p(sf * vals.reshape(n, d).astype(np.float64) / lib[:, None])
    # the quotient within half a unit in the last place, of which a logarithm passes on at most
    # as much, and the logarithm within one, on both sides: 3 units, each at most 2^-52
    np.testing.assert_allclose(st.chunk_sums.cpu().numpy(), x, rtol=3 * 2.0 ** -52, atol=0)


@pytest.mark.parametrize("D", [65, 128])
@pytest.mark.parametrize("mapped", [False, True])
def test_project_of_many_rows_equals_few(cuda, D, mapped):
    """Past 8192 rows the second pass of columns takes fewer steps at once: the same bits as for
    pieces of fewer rows, over rows that end in each of a batch's four blocks."""
    import torch

    from scarf_amd.device import DeviceCSR, col_map_tensor
    from scarf_amd.normalize import NormParams
    from scarf_amd.pca import Projector
    say("project rows", D, mapped)
    d_in, n = 400, 8197
    csr = DeviceCSR.from_host(_csr(n, d_in, (0, 1, 15, 16, 17, 31, 33, 47, 49, 63, 64, 65, 130), 9))
    rng = np.random.default_rng(10)
    keep = np.sort(rng.choice(d_in, 250, replace=False)) if mapped else np.arange(d_in)
    d = keep.shape[0]
    cm, _ = col_map_tensor(d_in, keep if mapped else None)
    proj = Projector.build(rng.standard_normal((d, D)), rng.uniform(0.1, 1.0, d),
                           rng.uniform(0.5, 2.0, d), clip=3.0)
    E = proj.project(csr, NormParams(), col_map=cm)
    for a in range(0, n, 4000):
        m = min(4000, n - a)
        part = proj.project(csr, NormParams(), col_map=cm, row_start=a, n_rows=m)
        assert torch.equal(E[a:a + m].view(torch.int32), part.view(torch.int32))


@pytest.mark.parametrize("d_in,D,clip,mapped,sizes", [
    (3, 1, 0.0, False, True), (40, 64, 3.0, False, False), (2500, 50, 3.0, True, False),
    (2500, 33, 0.0, False, True), (8192, 64, 3.0, False, True)])
def test_project_table_and_entries(cuda, d_in, D, clip, mapped, sizes):
    """sh_project takes the table of W's rows from 131,072 rows on; the caller's count of entries
    can say that rows are too short for it.  The same bits, with all of W in the table and with
    part of it, empty and long rows, counts on both sides of 64 and an infinity in W."""
    import torch

    from scarf_amd import _lib
    from scarf_amd.device import DeviceCSR, col_map_tensor, ptr, stream_handle
    from scarf_amd.pca import Projector
    from scarf_amd.synth import CSR
    say("project table", d_in, D, clip, mapped, sizes)
    rng = np.random.default_rng(18)
    n = 131072 + 5
    ln = np.minimum(np.array([0, 1, 31, 33, 64, 65, 5, 2, 9, 20])[np.arange(n) % 10], d_in)
    ln[[7, 70_000, n - 1]] = min(d_in, 1000)
    rp = np.concatenate([[0], np.cumsum(ln)]).astype(np.int64)
    within = np.arange(rp[-1]) - np.repeat(rp[:-1], ln)
    gap = np.maximum(d_in // np.maximum(np.repeat(ln, ln), 1), 1)
    cols = np.minimum(within * gap + (rng.random(rp[-1]) ** 3 * gap).astype(np.int64), d_in - 1)
    vals = np.where(rng.random(rp[-1]) < 0.02, rng.integers(60, 5000, rp[-1]),
                    rng.integers(1, 8, rp[-1])).astype(np.uint32)
    csr = DeviceCSR.from_host(CSR(vals, cols.astype(np.int32), rp, d_in))
    keep = np.sort(rng.choice(d_in, d_in // 2, replace=False)) if mapped else np.arange(d_in)
    d = keep.shape[0]
    W = rng.standard_normal((d, D))
    W[d // 2, 0] = np.inf
    cm, _ = col_map_tensor(d_in, keep if mapped else None)
    p = Projector.build(W, rng.uniform(0.1, 1.0, d), rng.uniform(0.5, 2.0, d), clip=clip)
    p.c.zero_()  # finite: the infinity of W stays in the rows that use it
    lib = torch.rand(n, dtype=torch.float64, device="cuda") * 900 + 100 if sizes else None
    out = []
    for name, count in (("sh_project", ()), ("sh_project_counted", (0,)),
                        ("sh_project_counted", (1 << 40,)), ("sh_project_counted", (-1,))):
        E = torch.full((n, D), -7.0, device="cuda")
        _lib.call(name, ptr(csr.vals), ptr(csr.cols), ptr(csr.rowptr), n, *count, ptr(cm), d_in, d,
                  1000.0, 1, ptr(lib), ptr(p.mu), ptr(p.inv_sigma), p.clip, ptr(p.W),
                  p.W.stride(0), D, ptr(p.c), ptr(E), D, stream_handle())
        out.append(E.view(torch.int32))
    for E in out[1:]:
        assert torch.equal(out[0], E)
