"""The CPython extension against a library that only records its calls (no GPU, no HIP): what the binding hands over, and that
it stays valid while a call runs."""
import ctypes as C
import importlib.util
import os
import re
import subprocess

import numpy as np
import pytest

from conftest import PKG_DIR, _load_by_path

# smx_gemv_batch_dev / smx_gemv_fused_dev pass their keys to `seen`; the batch calls also set every item's status
RECORDER = r"""
#include <stddef.h>
static int (*seen)(size_t, const char* const*);
static int statuses[80], batch_calls, batch_rc = 1;
void rec_set(int (*f)(size_t, const char* const*)) { seen = f; }
void rec_status(int rc, const int* st, size_t n) { batch_rc = rc; for (size_t i = 0; i < n; i++) statuses[i] = st[i]; }
int rec_batch_calls(void) { return batch_calls; }
int smx_gemv_batch_dev(void* c, size_t n, const char* const* keys) { return seen ? seen(n, keys) : 1; }
int smx_gemv_fused_dev(void* c, size_t n, const char* const* keys) { return seen ? seen(n, keys) : 1; }
int smx_gemv_batch(void* c, size_t n, const char* const* keys, const float* const* xs, const size_t* il, float* const* ys,
                   const size_t* oc, int* st) {
    batch_calls++;
    for (size_t i = 0; i < n; i++) {
        st[i] = statuses[i];
        if (oc[i]) ys[i][0] = xs[i][0] + (float)i;
    }
    return seen ? seen(n, keys) : batch_rc;
}
const char* smx_last_error(void* c) { return "recorded"; }
"""


@pytest.fixture(scope="module")
def rec(tmp_path_factory):
    """(extension module linked to the recorder, the recorder)"""
    d = str(tmp_path_factory.mktemp("binding"))
    with open(os.path.join(PKG_DIR, "host", "pybind.cpp")) as f:
        names = set(re.findall(r"\b(smx_[a-z0-9_]+)\b", f.read())) - {"smx_ctx", "smx_graph"}
    defined = set(re.findall(r"\b(smx_[a-z0-9_]+)\(", RECORDER))
    with open(os.path.join(d, "rec.c"), "w") as f:
        f.write(RECORDER + "".join(f"int {n}(void) {{ return 1; }}\n" for n in sorted(names - defined)))
    lib = os.path.join(d, "libsmx_recorder.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", os.path.join(d, "rec.c"), "-o", lib], check=True)
    path = _load_by_path("strix_rs_amd_build", os.path.join(PKG_DIR, "build.py")).build_pybind(d, "smx_recorder")
    spec = importlib.util.spec_from_file_location("_smx_native", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    L = C.CDLL(lib)
    yield mod, L
    L.rec_set(None)


SEEN = C.CFUNCTYPE(C.c_int, C.c_size_t, C.POINTER(C.c_char_p))


class Key(str):
    """A key whose end is noted."""
    gone = []

    def __del__(self):
        Key.gone.append(str(self))


class Fresh:
    """A sequence that makes its items when it is asked for them, as a numpy array of strings does."""

    def __init__(self, names):
        self.names = names

    def __len__(self):
        return len(self.names)

    def __getitem__(self, i):
        return Key(self.names[i])


def _call(rec, how, keys, during=None):
    """The keys the library saw, and which of them were gone while it ran."""
    mod, L = rec
    got = []

    @SEEN
    def seen(n, k):
        if during:
            during()
        got.append(([k[i].decode() for i in range(n)], list(Key.gone)))
        return 1

    L.rec_set(seen)
    n = len(keys)
    L.rec_status(1, (C.c_int * n)(*[1] * n), n)
    if how == "batch_dev":
        assert mod.gemv_batch_dev(16, keys, (256 for _ in range(n)), [512] * n) == 1
    elif how == "fused_dev":
        assert mod.gemv_fused_dev(16, keys, 0, 256, None, 0.0, [512] * n) == 1
    else:
        assert mod.gemv_batch(16, 0, keys, [np.zeros(1, np.float32) for _ in range(n)]) == 1
    L.rec_set(None)
    return got[0]


NAMES = [f"blk.{i}.ffn_gate.weight" for i in range(5)]


@pytest.mark.parametrize("how", ["batch_dev", "fused_dev"])
@pytest.mark.parametrize("make", [list, tuple, Fresh, np.array, lambda n: dict.fromkeys(n), lambda n: dict.fromkeys(n).keys()])
def test_keys_outlive_the_call(rec, how, make):
    Key.gone = []
    names, gone = _call(rec, how, make(NAMES))
    assert names == NAMES and gone == []


@pytest.mark.parametrize("how", ["batch_dev", "fused_dev", "batch"])
def test_a_list_changed_during_the_call(rec, how):
    """The lock is released while the library runs: another thread may empty the caller's list."""
    Key.gone = []
    keys = [Key(n) for n in NAMES]
    calls = [(k, np.ones(2, np.float32)) for k in keys] if how == "batch" else keys
    if how == "batch":
        del keys
    names, gone = _call(rec, how, calls, during=calls.clear)
    assert names == NAMES and gone == []
    assert sorted(Key.gone) == NAMES   # and nothing is held afterwards


def test_refused_key_sequences(rec):
    mod, _ = rec
    for keys in ((k for k in NAMES), 7, None):
        with pytest.raises(TypeError):
            mod.gemv_batch_dev(16, keys, [256] * 5, [512] * 5)
        with pytest.raises(TypeError):
            mod.gemv_fused_dev(16, keys, 0, 256, None, 0.0, [512] * 5)
    with pytest.raises(TypeError):
        mod.gemv_batch_dev(16, [b"a"], [256], [512])
    with pytest.raises(ValueError):
        mod.gemv_batch_dev(16, NAMES, [256], [512] * 5)


@pytest.fixture
def recorded(rec, pkg):
    """An accelerator object over the recorder (nothing is created or destroyed)."""
    mod, L = rec
    L.smx_last_error.restype = C.c_char_p
    a = pkg.Mi355WeightAccel.__new__(pkg.Mi355WeightAccel)
    a._L, a._n, a._a, a._h = L, mod, 16, C.c_void_p(16)
    yield a
    a._h = None


@pytest.mark.parametrize("status", [(1, 1, 1), (1, 0, 1), (0, 0, 0), (1, -1, 0)])
@pytest.mark.parametrize("layout", ["float32", "float64"])
def test_a_batch_runs_once_whatever_its_items_return(recorded, rec, pkg, status, layout):
    """A declined item is the ordinary case (a weight that is not resident): its batch must not be computed a second time."""
    L = rec[1]
    L.rec_status(1, (C.c_int * 3)(*status), 3)
    calls = [(f"k{i}", np.full(4, 10 * i, layout)) for i in range(3)]
    before = L.rec_batch_calls()
    if min(status) < 0:
        with pytest.raises(pkg.SmxError, match="recorded"):
            recorded.gemv_batch(calls, [2, 2, 2])
    else:
        got = recorded.gemv_batch(calls, [2, 2, 2])
        assert [g is not None for g in got] == [s == 1 for s in status]
        assert all(g is None or g[0] == 11 * i for i, g in enumerate(got))
    assert L.rec_batch_calls() == before + 1


def test_a_failed_batch_raises_and_runs_once(recorded, rec, pkg):
    L = rec[1]
    L.rec_status(-2, (C.c_int * 1)(1), 1)
    before = L.rec_batch_calls()
    with pytest.raises(pkg.SmxError, match="smx error -2"):
        recorded.gemv_batch([("k", np.zeros(4, np.float32))], [2])
    assert L.rec_batch_calls() == before + 1
    L.rec_status(1, (C.c_int * 1)(1), 1)


def test_a_batch_of_more_items_than_the_extension_takes(recorded, rec):
    L = rec[1]
    n = 64 + 1
    L.rec_status(1, (C.c_int * n)(*[1] * n), n)
    before = L.rec_batch_calls()
    got = recorded.gemv_batch([(f"k{i}", np.zeros(4, np.float32)) for i in range(n)], [2] * n)
    assert len(got) == n and L.rec_batch_calls() == before + 1
