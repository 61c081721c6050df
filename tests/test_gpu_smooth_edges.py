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


def _plain_bisection(d, rho, lc, bw, n_iter=64):
    """umap's loop with the sum evaluated at every step, in float32 in column order; and per row
    how far its closest decision (step up or down, stop or go on) was from the other way, in
    units of the sum's own float32 error there."""
    import torch
    n, k = d.shape
    f32 = torch.float32
    gap = d[:, 1:] - rho[:, None]
    target = float(np.log2(k)) * float(np.float32(bw))
    lo = torch.zeros(n, dtype=f32, device=d.device)
    hi, mid = torch.full_like(lo, np.inf), torch.ones_like(lo)
    done = torch.zeros(n, dtype=torch.bool, device=d.device)
    clear = torch.full((n,), np.inf, dtype=torch.float64, device=d.device)
    for _ in range(n_iter):
        psum = torch.zeros_like(lo)
        for j in range(k - 1):
            g = gap[:, j]
            psum = psum + torch.where(g > 0, torch.exp(-(g / mid)), torch.ones_like(g))
        # k additions of half a unit each, and per term one unit of exp and the quotient's
        # rounding (a e^-a <= 0.37)
        err = (0.5 * k * psum.double() + 1.5 * k) * 2.0 ** -23
        f = psum.double() - target
        stop = f.abs() < 1e-5
        now = torch.minimum(f.abs(), (f.abs() - 1e-5).abs()) / err
        clear = torch.where(done, clear, torch.minimum(clear, now))
        done |= stop
        up = f > 0
        hi2, lo2 = torch.where(up, mid, hi), torch.where(up, lo, mid)
        new = torch.where(torch.isinf(hi2), mid * 2, (lo2 + hi2) / 2)
        hi, lo = torch.where(done, hi, hi2), torch.where(done, lo, lo2)
        mid = torch.where(done, mid, new)
    return mid, clear


@pytest.mark.parametrize("k,bw", [(2, 1.5), (4, 1.5), (12, 1.0), (13, 1.5), (21, 1.5), (33, 0.5),
                                  (64, 1.5)])
def test_sigma_is_the_plain_bisections(cuda, k, bw):
    """The steps that are not evaluated decide as the plain bisection does: sigma is the same
    float, but for rows where a decision lies within the sum's float32 error, which another
    exponential may take the other way (and those rows end where the sum is still the target,
    to the tolerance and that error)."""
    import torch
    from scarf_amd.smooth import smooth_knn
    say("sigma", k, bw)
    rng = np.random.default_rng(k)
    n = 20_000
    d = np.sort(rng.gamma(rng.uniform(0.3, 6.0, (n, 1)), 1.0, (n, k)), axis=1) + 1e-3
    d *= 10.0 ** rng.uniform(-7, 7, (n, 1))
    d[::50] = d[::50, :1]                                    # flat
    d[1::50, :max(1, k // 2)] = 0.0                          # duplicates of the row
    d[2::50, 1:] = d[2::50, -1:]                             # one near, the rest level
    d[3::50, 1:] = d[3::50, :1] * (1 + 1e-6 * np.arange(1, k))  # gaps of a few units
    d[4::50, -1] = 1e30                                      # one very far
    d = torch.from_numpy(d.astype(np.float32)).cuda()
    idx = torch.full((n, k), n, dtype=torch.int64, device="cuda")
    sigma, rho, w = smooth_knn(d, idx, 1000, 1.0, bw)
    first = torch.where(d > 0, d, torch.full_like(d, np.inf)).min(1).values
    assert torch.equal(rho, torch.where(torch.isinf(first), torch.zeros_like(first), first))
    want, clear = _plain_bisection(d, rho, 1.0, bw)
    chunk = d.double().view(n // 1000, -1).mean(1).float().repeat_interleave(1000)
    floor = torch.where(rho > 0, d.double().mean(1).float(), chunk) * np.float32(1e-3)
    floored = (want <= floor * (1 + 2.0 ** -22)) | (sigma <= floor * (1 + 2.0 ** -22))
    assert bool((sigma >= floor * (1 - 2.0 ** -22)).all())
    same = (sigma == want) | floored
    say("rows", n, "floored", int(floored.sum()), "other", int((~same).sum()))
    assert bool((clear[~same] <= 1.0).all())
    g = (d[:, 1:] - rho[:, None]).double()
    s = sigma.double()[:, None]
    psum = torch.where(g > 0, torch.exp(-g / s), torch.ones_like(g)).sum(1)
    target = float(np.log2(k)) * float(np.float32(bw))
    err = (0.5 * k * psum + 1.5 * k) * 2.0 ** -23
    assert bool((((psum - target).abs() <= 1e-5 + err) | same).all())
    # and the weights that follow from sigma
    ww = torch.where(d - rho[:, None] <= 0, torch.ones_like(d),
                     torch.exp(-((d - rho[:, None]) / sigma[:, None])))
    ww = ww.double()
    assert bool((((w.view(n, k).double() - ww).abs() <= 2.0 ** -22) | (ww == 0)).all())


@pytest.mark.parametrize("k", [2, 33])
def test_rows_without_a_root_are_not_a_slow_case(cuda, k):
    """Level rows, rows half of zeros and rows of two neighbours have no sigma that meets the
    target.  Their sums are not evaluated; where they were, at each of 64 steps, such tables took
    1.8, 2.5 and 0.54 times as long as ordinary rows of 33 neighbours (now 0.65, 0.75, 0.32)."""
    import time

    import torch
    from scarf_amd.smooth import smooth_knn
    say("smooth without a root", k)
    n = 300_000
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    d = torch.cumsum(torch.rand(n, 33, generator=g, device="cuda") + 0.02, 1) + 20
    idx = torch.randint(0, n, (n, 33), generator=g, device="cuda")
    level, zeros = d[:, :1].expand(n, 33).contiguous(), d.clone()
    zeros[:, :16] = 0.0

    def took(x):
        best = float("inf")
        ix = idx[:, :x.shape[1]].contiguous()
        for _ in range(5):
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                smooth_knn(x, ix, 20_000)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        return best

    usual = took(d)
    for x, most in ((level, 1.3), (zeros, 1.3)) if k == 33 else ((d[:, :2].contiguous(), 0.45),):
        t = took(x)
        say("times the usual", t / usual)
        assert t <= most * usual
