"""Scene creation when its optional part, the oriented boxes, cannot be had: the scene is created without them.
Runs the library's host code against a stand-in for the HIP runtime (hip_stub.cpp) in a process of its own."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

from zombie_amd import _abi as A

HERE = Path(__file__).resolve().parent

PROGRAM = r"""
import ctypes as C, sys
import numpy as np
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for f in ("stub_live_bytes", "stub_peak_bytes"):
    getattr(stub, f).restype = C.c_int64
stub.stub_largest_launch.restype = C.c_uint64
stub.stub_reset.argtypes = [C.c_int64, C.c_int, C.c_int64]
from zombie_amd import _abi as A
L = A.lib()
NO_LIMIT = 1 << 62


def strip(n, shift):
    # n triangles of a wavy strip, so that leaves differ
    i = np.arange(n)
    V = np.stack([0.1 * np.arange(n + 2) + shift, np.arange(n + 2) % 2 + 0.0, np.sin(np.arange(n + 2))], 1)
    return V.astype(np.float32), np.stack([i, i + 1, i + 2], 1).astype(np.int32)


def create(n_abs, n_refl, limit=NO_LIMIT, refuse=0, mallocs=-1, width=8):
    Va, Ia = strip(n_abs, 0.0)
    Vr, Ir = strip(n_refl, 1000.0)
    V = np.concatenate([Va, Vr])
    I = np.concatenate([Ia, Ir + len(Va)])
    refl = np.concatenate([np.zeros(n_abs, np.uint8), np.ones(n_refl, np.uint8)])
    lo, hi = (V.min(0) - 1).copy(), (V.max(0) + 1).copy()
    opts = A.zg_build_options(width, 2, 16, 0)
    h = C.c_void_p()
    before = stub.stub_live_bytes()
    stub.stub_reset(limit, refuse, mallocs)
    rc = L.zg_scene_create(3, V.ctypes.data, len(V), I.ctypes.data, len(I), refl.ctypes.data, lo.ctypes.data,
                           hi.ctypes.data, 0, 1e-3, C.byref(opts), C.byref(h))
    launch = stub.stub_largest_launch()
    stub.stub_reset(NO_LIMIT, 0, -1)
    info = A.zg_scene_info()
    if rc == A.ZG_OK:
        assert L.zg_scene_get_info(h, C.byref(info)) == A.ZG_OK
        assert stub.stub_live_bytes() - before == info.device_bytes     # nothing else is kept
        assert info.n_absorbing_prims == n_abs and info.n_reflecting_prims == n_refl
        assert L.zg_scene_destroy(h) == A.ZG_OK
    assert stub.stub_live_bytes() == before                             # and nothing is lost
    return rc, info.device_bytes, launch


case = sys.argv[2]
rc, full, launch = create(40, 400)
assert rc == A.ZG_OK and launch > 0, rc
if case == "launch":
    rc, bare, _ = create(40, 400, refuse=1)
    assert rc == A.ZG_OK and 0 < bare < full, (rc, bare, full)
elif case == "memory":
    # what the scene needs without boxes, plus less than the boxes take: the reflecting part must still fit
    _, bare, _ = create(40, 400, refuse=1)
    for extra in (0, (full - bare) // 2, full - bare):   # the last: boxes fit, the build's inputs do not
        rc, got, _ = create(40, 400, limit=bare + extra)
        assert rc == A.ZG_OK and got == bare, (extra, rc, got, bare)
    rc, _, _ = create(40, 400, limit=bare - 1)
    assert rc != A.ZG_OK
elif case == "host":
    # the first allocation after the absorbing part's three uploads belongs to the boxes
    rc, got, _ = create(300, 0, mallocs=3)
    _, bare, _ = create(300, 0, refuse=1)
    assert rc == A.ZG_OK and got == bare, (rc, got, bare)
else:
    # threads of the largest launch stay bounded as the mesh grows
    _, _, small = create(60000, 0, width=4)
    _, _, large = create(240000, 0, width=4)
    assert large < 2 * small and large < 1 << 26, (small, large)
print("ok")
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "hip_stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(HERE / "hip_stub.cpp"), "-o", str(so)], check=True)
    return so


@pytest.mark.parametrize("case", ["launch", "memory", "host", "grid"])
def test_scene_is_created_without_boxes(stub, case):
    if not A.LIB_PATH.exists():
        pytest.fail("libzombie_amd.so is not built")
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(stub), case], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, PYTHONPATH=str(HERE.parent)))
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stderr[-2000:]
