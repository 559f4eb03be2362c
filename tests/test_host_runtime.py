"""The library's host side on a test double of the HIP runtime (fake_hip.cpp): which bytes a host-pointer call moves and when,
and what it does when the runtime refuses something.  No GPU: kernels that compute do nothing there, so a result is the
untouched device memory it was copied from, word i = i."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes as C, os, sys, time
F = C.CDLL({fake!r}, C.RTLD_GLOBAL)   # under the runtime's name: the library binds to it
for f in ("fake_inbound", "fake_pending", "fake_host_live"):
    getattr(F, f).restype = C.c_size_t
sys.path.insert(0, {root!r})
import numpy as np
import __graft_entry__ as entry
pkg, synth = entry.package(), entry.synth()
L = pkg.load_library()

def floats(n, shift=0):   # n floats in memory of their own, `shift` bytes behind a 64-byte boundary
    raw = np.zeros(n * 4 + 128, np.uint8)
    at = (-raw.ctypes.data) % 64 + shift
    return raw[at:at + n * 4].view(np.float32)

def p(a):
    return a.ctypes.data_as(C.c_void_p)

def inbound():
    out = np.zeros(F.fake_inbound(None, C.c_size_t(0)), np.uint8)
    F.fake_inbound(p(out), C.c_size_t(out.nbytes))
    return out.view(np.float32)

def untouched(y):   # what device memory holds that no kernel has written
    return np.array_equal(y.reshape(-1).view(np.uint32), np.arange(y.size, dtype=np.uint32))

def accel(K=256, N=4096):
    a = pkg.Mi355WeightAccel(0)
    assert a.upload_q8_0("w", synth.make_q8_0(N, K, 1), K, N)
    F.fake_keep_inbound(1)
    return a
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    """The test double, under the runtime's file name."""
    out = str(tmp_path_factory.mktemp("fake") / "libamdhip64.so.7")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-shared", "-fPIC", "-pthread",
                    "-Wl,-soname,libamdhip64.so.7", os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", out], check=True)
    return out


@pytest.fixture
def run(fake):
    """Runs a piece of Python in a process of its own (the library binds to one runtime per process)."""
    def go(code, **values):
        text = PRELUDE.format(fake=fake, root=ROOT) + "".join(f"{k} = {v!r}\n" for k, v in values.items()) + textwrap.dedent(code)
        r = subprocess.run([sys.executable, "-c", text], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
        assert r.returncode == 0, r.stdout
    return go


@pytest.mark.parametrize("m,K,N,behind", [(4000, 256, 2048, 0), (4000, 256, 2048, 1000), (4000, 256, 2048, -64), (1500, 4096, 2048, 333), (20, 256, 4096, 7)])
def test_rows_and_results_that_overlap(run, m, K, N, behind):
    """Every row is read before a result is written, on the small route and on the one that pipelines row groups."""
    run("""
        a = accel(K, N)
        buf = np.random.default_rng(1).random(max(behind, 0) + m * max(K, N) + 64, dtype=np.float32)
        xs, y = buf[64:64 + m * K], buf[64 + behind:64 + behind + m * N]
        want = xs.copy()
        F.fake_keep_inbound(1)
        assert L.smx_gemm(a._h, b"w", p(xs), m, K, p(y), y.size) == 1
        assert untouched(y)
        got = inbound()
        if got.size:                          # (a small call's kernels read the staging itself)
            assert np.array_equal(got, want)
    """, m=m, K=K, N=N, behind=behind)
