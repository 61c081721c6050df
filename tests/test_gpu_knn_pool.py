"""sh_knn_pool (threshold pass, sliced scan, merge) keeps the pool that the one-slice screen
with an open threshold keeps, bit for bit: it is the same set of MFMA keys, selected another
way."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _rows(n, D, seed, dup=0):
    rng = np.random.default_rng(seed)
    c = rng.standard_normal((9, D)) * 2
    E = (c[rng.integers(0, 9, n)] + rng.standard_normal((n, D))).astype(np.float32)
    if dup:
        E[rng.choice(n, min(dup, n), replace=False)] = E[0]
    return E


# query counts around a 256-query block, reference counts around the 128-row stage, the
# smallest set that takes a threshold pass (8 pools) and one below it, several slices
CASES = [("bf16", 64, 50, 1, 511), ("bf16", 64, 50, 1, 512), ("bf16", 64, 50, 33, 20001),
         ("bf16", 64, 13, 257, 4097), ("bf16", 128, 70, 255, 9000), ("bf16", 64, 125, 40, 30000),
         ("bf16", 64, 50, 3000, 60013), ("bf16", 32, 50, 9000, 9000),
         ("fp32", 64, 50, 1, 40), ("fp32", 64, 50, 300, 19001), ("fp32", 128, 7, 65, 2049),
         ("fp32", 16, 128, 31, 5000), ("fp8", 128, 100, 700, 30011), ("fp8", 64, 64, 1, 8192),
         ("fp8", 256, 100, 130, 12000)]


def _compare(Q, R, screen, pool):
    """Pools of sh_knn_pool and of the one-slice open screen, as (keys, counts) pairs."""
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    from scarf_amd.knn import pack, pack_refs
    L, code = _lib.lib(), _lib.DTYPES[screen]
    (nq, D), nr = Q.shape, R.shape[0]
    refs = pack_refs(R, screen)
    qp, _, _ = pack(Q, screen, 1)
    want = torch.full((nq, pool), -1, dtype=torch.int64, device="cuda")
    want_n = torch.empty(nq, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.sh_knn_screen_workspace(nq, pool, 1), dtype=torch.uint8, device="cuda")
    _lib.call("sh_knn_screen", ptr(qp), nq, ptr(refs.data), nr, D, code, None, None, pool, 1,
              None, ptr(want), ptr(want_n), ptr(ws), ws.numel(), stream_handle())
    got = torch.full_like(want, -1)
    got_n = torch.empty_like(want_n)
    ws = torch.empty(L.sh_knn_pool_workspace(nq, nr, D, code, pool), dtype=torch.uint8,
                     device="cuda")
    _lib.call("sh_knn_pool", ptr(qp), nq, ptr(refs.data), nr, D, code, pool, ptr(got),
              ptr(got_n), ptr(ws), ws.numel(), stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(got_n, want_n)
    assert torch.equal(got, want)


@pytest.mark.parametrize("screen,pool,D,nq,nr", CASES)
@pytest.mark.parametrize("dup", [0, 400])
def test_pool_equals_open_screen(cuda, screen, pool, D, nq, nr, dup):
    import torch
    say("knn pool", screen, "pool", pool, "D", D, nq, "x", nr, "dup", dup)
    R = torch.from_numpy(_rows(nr, D, 5, dup)).cuda()
    Q = torch.from_numpy(_rows(nq, D, 6)).cuda()
    if dup:
        Q[0] = R[0]  # a query whose nearest keys are all equal
    _compare(Q, R, screen, pool)


# over a billion pairs: the collecting scan, whose overflowing queries (a thousand equal
# references each, more of them than the first list of the second screen takes) are
# screened again
@pytest.mark.parametrize("screen,pool,D,nq,nr,equal", [
    ("bf16", 64, 50, 9001, 120_013, 0), ("bf16", 64, 50, 13_000, 100_000, 6_000),
    ("bf16", 128, 20, 20_000, 60_001, 3), ("fp32", 64, 50, 20_011, 55_000, 700),
    ("fp8", 128, 100, 9_000, 131_072, 40), ("fp8", 256, 100, 3_001, 400_000, 1)])
def test_collected_pool_equals_open_screen(cuda, screen, pool, D, nq, nr, equal):
    import torch
    say("knn collect", screen, "pool", pool, "D", D, nq, "x", nr, "equal", equal)
    R = torch.from_numpy(_rows(nr, D, 7, 3000 if equal else 0)).cuda()
    Q = torch.from_numpy(_rows(nq, D, 8)).cuda()
    Q[:equal] = R[0]
    _compare(Q, R, screen, pool)


@pytest.mark.parametrize("shift", [1, 2, 3, 4])
def test_misleading_sample(cuda, shift):
    """Near references only where the threshold pass looks: its guess is too low, the scan
    meets fewer keys than the pool, and the query is screened again."""
    import torch
    say("knn misleading sample", shift)
    nr, nq, D, near = 120_000, 9_000, 50, 60
    i = np.arange(near, dtype=np.uint64) * 31
    rows = (i << np.uint64(shift)) + ((((i * np.uint64(2654435761)) & np.uint64(0xffffffff))
                                       >> np.uint64(16)) & np.uint64((1 << shift) - 1))
    E = _rows(nr, D, 9)
    rng = np.random.default_rng(10)
    E[rows.astype(np.int64)] = 40.0 + 0.01 * rng.standard_normal((near, D))
    Q = _rows(nq, D, 11)
    Q[100:5000] = 40.0 + 0.01 * rng.standard_normal((4900, D))
    _compare(torch.from_numpy(Q.astype(np.float32)).cuda(), torch.from_numpy(E).cuda(), "bf16", 64)


@pytest.mark.parametrize("D,pool,extra", [(1, 5, 0), (4, 64, 1), (31, 64, 2), (33, 100, 0),
                                          (50, 64, 0), (64, 128, 3), (65, 200, 1), (256, 256, 0)])
def test_rerank_of_many_queries_equals_few(cuda, D, pool, extra):
    """From 1024 queries on the candidates' rows go through LDS: the same bits as for pieces of
    fewer queries, over feature counts around the 32 of a piece, rows and buffers that are
    aligned to 4 bytes only, a last row that ends the buffer, and pools from empty to full."""
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    say("rerank", D, pool, extra)
    rng = np.random.default_rng(21)
    nq, nr, ld = 1029, 900, D + extra
    k = min(11, pool)
    buf = torch.from_numpy(rng.standard_normal(nr * ld + 1).astype(np.float32)).cuda()
    R = buf[1:1 + nr * ld]
    Q = torch.from_numpy(rng.standard_normal((nq, D)).astype(np.float32)).cuda()
    cnt = rng.integers(0, pool + 1, nq).astype(np.int32)
    cnt[:4] = [0, 1, pool, pool - 1]
    idx = np.argsort(rng.random((nq, nr)), axis=1)[:, :pool].astype(np.int64)
    idx[2, 0] = nr - 1
    key = (np.arange(pool, dtype=np.int64)[None, :] + 0x40000000) << 32  # ascending, positive
    cand = torch.from_numpy(key | idx).cuda()
    cnt = torch.from_numpy(cnt).cuda()

    def rank(a, b):
        oi = torch.full((b - a, k), -7, dtype=torch.int64, device="cuda")
        od = torch.full((b - a, k), -7.0, device="cuda")
        fl = torch.full((b - a,), -7, dtype=torch.int32, device="cuda")
        _lib.call("sh_knn_rerank", ptr(Q[a:b]), b - a, D, ptr(R), nr, ld, D, ptr(cand[a:b]),
                  ptr(cnt[a:b]), pool, 1, k, -1, None, -1.0, 0.0, 0.0, ptr(oi), ptr(od), ptr(fl),
                  stream_handle())
        return oi, od, fl

    whole = rank(0, nq)
    for a in range(0, nq, 343):
        for x, y in zip(whole, rank(a, a + 343)):
            assert torch.equal(x[a:a + 343], y)
    # and the oracle's: FP64 terms added in feature order
    i = 2
    r = R.cpu().numpy().reshape(nr, ld)[:, :D].astype(np.float64)
    df = Q[i].cpu().numpy().astype(np.float64) - r[idx[i]]
    d = np.zeros(pool)
    for t in range(D):
        d += df[:, t] ** 2
    order = np.lexsort((idx[i], d))[:k]
    assert np.array_equal(whole[0][i].cpu().numpy(), idx[i][order])
    assert np.array_equal(whole[1][i].cpu().numpy(), d[order].astype(np.float32))


def test_threads_on_one_stream(cuda):
    """Four threads search on the default stream, with their own sizes (the workspace grows) and
    queries: the neighbours of a search alone."""
    import threading

    import torch
    from scarf_amd.knn import pack_refs, search
    say("knn threads on one stream")
    R = torch.from_numpy(_rows(60_000, 50, 41)).cuda()
    refs = pack_refs(R, "bf16")
    Q = [torch.from_numpy(_rows(n, 50, 42 + n)).cuda() for n in (300, 2000, 4500, 9000)]
    want = [search(q, R, refs, 11) for q in Q]
    torch.cuda.synchronize()
    got = [[] for _ in Q]
    start = threading.Barrier(len(Q))

    def work(i):
        start.wait()
        for _ in range(20):
            got[i].append(search(Q[i], R, refs, 11))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(Q))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, w in enumerate(want):
        assert len(got[i]) == 20
        for g in got[i]:
            assert torch.equal(g[0], w[0]) and torch.equal(g[1], w[1])


@pytest.mark.parametrize("nq,nr", [(100, 30_000), (500, 25_000), (40, 17_000)])
def test_pool_of_many_slots(cuda, nq, nr):
    """A pool of 256 in more slices than eight minima a lane half leave slots for."""
    import torch
    say("knn pool of many slots", nq, nr)
    _compare(torch.from_numpy(_rows(nq, 100, 13)).cuda(),
             torch.from_numpy(_rows(nr, 100, 14)).cuda(), "fp8", 256)


@pytest.mark.parametrize("screen,pool,D,nq,nr,equal", [
    ("bf16", 64, 50, 1, 3000, 200), ("bf16", 64, 50, 300, 20_000, 10_000),
    ("bf16", 64, 50, 700, 300_000, 150_000), ("bf16", 128, 50, 9000, 60_000, 5000),
    ("fp32", 64, 50, 500, 30_000, 15_000), ("fp8", 256, 100, 300, 40_000, 9000)])
def test_equal_references_keep_the_lowest_indices(cuda, screen, pool, D, nq, nr, equal):
    """Queries that are one of many equal references: its pool is the lowest-indexed of them,
    whichever of the scan's ways it takes (the second screen, ties in every slice, one slice)."""
    import torch
    from scarf_amd import _lib
    from scarf_amd.device import ptr, stream_handle
    from scarf_amd.knn import pack, pack_refs
    say("knn equal references", screen, pool, nq, nr, equal)
    L, code = _lib.lib(), _lib.DTYPES[screen]
    R = _rows(nr, D, 31)
    at = np.sort(np.random.default_rng(32).choice(nr, equal, replace=False))
    R[at] = 3.0 * R[at[0]]  # far out, so that nothing else is near
    R = torch.from_numpy(R).cuda()
    Q = torch.from_numpy(_rows(nq, D, 33)).cuda()
    Q[::2] = R[int(at[0])]
    refs = pack_refs(R, screen)
    qp, _, _ = pack(Q, screen, 1)
    want = torch.from_numpy(at[:pool].astype(np.int64)).cuda()
    for name in ("sh_knn_pool", "sh_knn_screen"):
        cand = torch.full((nq, pool), -1, dtype=torch.int64, device="cuda")
        cnt = torch.empty(nq, dtype=torch.int32, device="cuda")
        need = (L.sh_knn_pool_workspace(nq, nr, D, code, pool) if name == "sh_knn_pool" else
                L.sh_knn_screen_workspace(nq, pool, 1))
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        extra = () if name == "sh_knn_pool" else (1, None)
        aux = () if name == "sh_knn_pool" else (None, None)
        _lib.call(name, ptr(qp), nq, ptr(refs.data), nr, D, code, *aux, pool, *extra, ptr(cand),
                  ptr(cnt), ptr(ws), need, stream_handle())
        assert bool((cnt == pool).all())
        assert bool(((cand[::2] & 0xffffffff) == want[None, :]).all())


def test_equal_references_are_not_a_slow_case(cuda):
    """100,000 cells of which half are one row, against the same number without equal ones:
    about 2.2 times the time where every tie was inserted, twice, it was 57 times."""
    import time

    import torch
    from scarf_amd.knn import pack_refs, search
    say("knn time with equal references")
    E = torch.from_numpy(_rows(100_000, 50, 34)).cuda()
    T = E.clone()
    T[torch.randperm(100_000, device="cuda")[:50_000]] = E[0]
    took = []
    for x in (E, T):
        refs = pack_refs(x, "bf16")
        best = float("inf")
        for _ in range(4):
            torch.cuda.synchronize()
            t = time.perf_counter()
            search(x, x, refs, 11, self_offset=0)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        took.append(best)
    say("ms", [1e3 * t for t in took])
    assert took[1] < 10.0 * took[0]
