"""CPU-only: searches of several threads on one stream.  sh_knn_pool and sh_locality_order queue
several kernels that hand results on in a workspace, and the stream's workspace is one: another
thread's call on the same buffer must not come between them."""
import functools
import os
import threading
import time
import types

import pytest
import torch

from scarf_amd import _lib, device, knn

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH),
                                reason="libscarfhip.so not built")


@pytest.fixture
def recorded(monkeypatch):
    """The library's calls on CPU tensors: each takes a while, and calls that share a buffer at
    the same time are noted."""
    busy, overlaps, lock = {}, [], threading.Lock()

    def call(name, *args):
        at = {"sh_knn_pool": 9, "sh_knn_screen": 13, "sh_locality_order": 5}.get(name)
        if at is None:
            return
        buf = args[at].value
        with lock:
            if buf in busy:
                overlaps.append((name, busy[buf]))
            busy[buf] = name
        time.sleep(0.02)
        with lock:
            busy.pop(buf, None)

    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(knn, "require_gpu", lambda: None)
    monkeypatch.setattr(knn, "stream_handle", lambda stream=None: None)
    monkeypatch.setattr(knn, "pack", lambda E, *a: (E, E[:, 0], 64))
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda *a: types.SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(device, "_workspaces", {})
    monkeypatch.setattr(device, "Workspace", functools.partial(device.Workspace, device="cpu"))
    return overlaps


@pytest.mark.parametrize("n_slices", [None, 2])
@pytest.mark.parametrize("ordered", [False, True])
def test_threads_on_one_stream_do_not_share_a_workspace_at_once(recorded, n_slices, ordered):
    R = torch.randn(4000, 50)
    refs = knn.PackedRefs("bf16", 50, 64, R, R[:, 0], 1.0)
    start = threading.Barrier(4)
    errors = []

    def work(i):
        try:
            start.wait()
            for _ in range(3):
                knn.search(torch.randn(8 + 40 * i, 50), R, refs, 5, n_slices=n_slices,
                           order=ordered)
        except BaseException as e:  # a thread's failure is the test's
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    assert recorded == []
