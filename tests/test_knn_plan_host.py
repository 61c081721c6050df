"""CPU-only: how sh_knn_pool plans a search.  A width or size that is not built is an error of
the call, as for sh_knn_screen, whatever the size of the search."""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

import pytest

from scarf_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "scarf_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# packed widths that sh_knn_{bf16,fp8,f32}.hip build
WIDTHS = {"SH_BF16": {16 * i for i in range(1, 9)}, "SH_FP8": {64, 128},
          "SH_F32": {8 * i for i in range(1, 18)}}

# in a process of its own: an arithmetic trap must not take the test run with it
SWEEP = """
from scarf_amd import _lib
L = _lib.lib()
for name in ("SH_BF16", "SH_FP8", "SH_F32"):
    code = getattr(_lib, name)
    for D in range(1, 257):
        for nq, nr in ((1, 1), (1, 500_000), (4700, 4700), (10_000, 10_000), (16_384, 500_000),
                       (1_000_000, 1_000_000), (1 << 53, 1_000_000), (1000, 1 << 40)):
            for pool in (1, 64, 128, 256):
                ws = L.sh_knn_pool_workspace(nq, nr, D, code, pool)
                print(name, L.sh_knn_pack_k(code, D), nq, nr, pool, ws)
print(L.sh_knn_pool_workspace(10, 10, 8, 77, 64))
"""


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libscarfhip.so not built")
def test_workspace_of_every_width():
    r = subprocess.run([sys.executable, "-c", SWEEP], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, f"exit status {r.returncode}: {r.stderr[-500:]}"
    *lines, unknown = r.stdout.splitlines()
    assert unknown == "0"
    for line in lines:
        name, K, nq, nr, pool, ws = line.split()
        built = int(K) in WIDTHS[name] and (int(pool) <= 128 or name == "SH_FP8")
        fits = int(nq) < 1 << 31 and int(nr) < (1 << 32) - 1
        assert (int(ws) > 0) == (built and fits), line


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libscarfhip.so not built")
@pytest.mark.parametrize("nq,nr", [(10, 100), (10_000, 10_000)])
def test_unbuilt_width_is_refused(nq, nr):
    """Checked before anything is launched, so the pointers are never followed."""
    L = _lib.lib()
    p = 4096
    rc = L.sh_knn_pool(p, nq, p, nr, 128, _lib.SH_BF16, 64, p, p, p, 256, None)
    assert rc == _lib.SH_EUNSUPPORTED
    assert b"packed K=144 not supported" in L.sh_last_error()


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """(plans, slots that k_tau takes): dicts over a grid of the arguments' whole range."""
    if not os.path.exists(HIPCC):
        pytest.skip("ROCm toolchain not available")
    out = tmp_path_factory.mktemp("plan")
    srcs = [os.path.join(os.path.dirname(__file__), "knn_plan_driver.hip")] + \
        [os.path.join(CSRC, f"sh_{n}.hip") for n in ("knn_bf16", "knn_fp8", "knn_f32", "common")]
    flags = ["--offload-arch=gfx950", "--cuda-host-only", "-O1", "-w", "-std=c++17", "-I",
             os.path.join(ROOT, "include"), "-I", CSRC]

    def compile_one(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        r = subprocess.run([HIPCC, *flags, "-c", src, "-o", obj], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return obj

    with cf.ThreadPoolExecutor(4) as ex:
        objs = list(ex.map(compile_one, srcs))
    exe = str(out / "plan")
    # no device code is built, so its image stays unresolved; nothing here launches a kernel
    r = subprocess.run([HIPCC, "--hip-link", "--offload-arch=gfx950", *objs,
                        "-Wl,--unresolved-symbols=ignore-all", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
    *lines, last = r.stdout.splitlines()
    names = ("dtype D pool nq nr bounded collect rank S1 per slots m S3 cap len3 bytes").split()
    return [dict(zip(names, map(int, x.split()))) for x in lines], int(last.split()[1])


def test_thresholds_take_every_slot(plans):
    """k_tau looks at all the minima that k_bound writes, and there are as many as its rank."""
    rows, tau_slots = plans
    assert len(rows) > 10_000
    for p in rows:
        if p["bounded"]:
            assert p["slots"] == p["S1"] * 2 * p["per"] <= tau_slots, p
            assert p["per"] in (1, 2, 4, 8) and p["slots"] >= p["rank"], p


def test_collected_positions_fit_32_bits(plans):
    """k_collect counts a lane half's keys in bytes from the wave's first segment, in 32 bits: the
    64 queries' segments and every second reference of a slice passing."""
    for p in plans[0]:
        if p["collect"]:
            last = 64 * p["S3"] * p["cap"] * 8 + (p["len3"] + 1) // 2 * 8
            assert last < 1 << 32, p
