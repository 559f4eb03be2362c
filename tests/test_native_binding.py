"""The CPython extension against a library that only records its calls (no GPU, no HIP): what the binding hands over, and that
it stays valid while a call runs."""
import ctypes as C
import importlib.util
import os
import re
import subprocess

import numpy as np
import pytest

from conftest import PKG_DIR, ROOT, _load_by_path

# Every entry point logs its arguments; those that take keys also pass them to `seen`, and the batch calls set their items'
# statuses and results.
HEAD = r"""
#include <stdio.h>
#include "strix_mi355.h"
static int (*seen)(size_t, const char* const*);
static int statuses[80], batch_calls, batch_rc = 1;
static char text[4096];
#define LOG(...) at += snprintf(text + at, sizeof text - at, __VA_ARGS__)
void rec_set(int (*f)(size_t, const char* const*)) { seen = f; }
void rec_status(int rc, const int* st, size_t n) { batch_rc = rc; for (size_t i = 0; i < n; i++) statuses[i] = st[i]; }
int rec_batch_calls(void) { return batch_calls; }
const char* rec_text(void) { return text; }
const char* smx_last_error(const smx_ctx* c) { return "recorded"; }
"""
BATCH = """
    batch_calls++;
    for (size_t i = 0; i < n; i++) {
        status[i] = statuses[i];
        if (out_caps[i]) ys[i][0] = xs[i][0] + (float)i;
    }
    return seen ? seen(n, keys) : batch_rc;"""


def _recorder():
    """C source of the recording library, from the prototypes of the header."""
    with open(os.path.join(ROOT, "include", "strix_mi355.h")) as f:
        header = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
    src = [HEAD]
    for name, args in re.findall(r"^int (smx_\w+)\(([^)]*)\);", header, flags=re.M):
        body = [f'int at = 0; LOG("{name}");']
        names = []
        for arg in args.split(","):
            ty, var = re.match(r"\s*(.*?)(\w+)\s*$", arg, flags=re.S).groups()
            ty = " ".join(ty.split())
            names.append(var)
            if ty == "const char* const*":
                body.append(f'for (size_t i = 0; i < n && i < 16; i++) LOG(" %s", {var}[i]);')
            elif "* const*" in ty:
                body.append(f'for (size_t i = 0; i < n && i < 16; i++) LOG(" %p", (void*){var}[i]);')
            else:
                fmt, cast = {"const char*": ("%s", ""), "size_t": ("%zu", ""), "int": ("%d", ""), "float": ("%g", "(double)")}.get(ty, ("%p", "(void*)"))
                body.append(f'LOG(" {fmt}", {cast}{var});')
        body.append(BATCH if name.endswith("_batch") else "return seen ? seen(n, keys) : 1;" if "keys" in names else "return 1;")
        src.append(f"int {name}({args}) {{ {' '.join(body)} }}")
    return "\n".join(src)


@pytest.fixture(scope="module")
def rec(tmp_path_factory):
    """(extension module linked to the recorder, the recorder)"""
    d = str(tmp_path_factory.mktemp("binding"))
    with open(os.path.join(d, "rec.c"), "w") as f:
        f.write(_recorder())
    lib = os.path.join(d, "libsmx_recorder.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-I" + os.path.join(ROOT, "include"), os.path.join(d, "rec.c"), "-o", lib], check=True)
    path = _load_by_path("strix_rs_amd_build", os.path.join(PKG_DIR, "build.py")).build_pybind(d, "smx_recorder")
    spec = importlib.util.spec_from_file_location("_smx_native", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    L = C.CDLL(lib)
    L.smx_last_error.restype = L.rec_text.restype = C.c_char_p
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


_x, _y = np.arange(8, dtype=np.float32), np.zeros(8, np.float32)
CALLS = [("gemv_dev", ("a.weight", 256, 3, 512)), ("gemm_dev", ("a.weight", 256, np.int64(30), 512)), ("gemv_noalloc_dev", ("a", 256, 8, 512)),
         ("gemv_f32_dev", ("a", 256, 512)), ("gemm_fused_dev", ("a", 1, 256, None, 7, 1e-6, 512)),
         ("ffn_gate_up_dev", ("g", "u", 2, 256, 1, C.c_void_p(768), 1e-5, 512)), ("gemv_batch_dev", (["a", "b"], [256, 512], (768, None))),
         ("gemv_fused_dev", (("a", "b", "c"), 3, 256, 512, 0.5, [1, 2, 3])), ("moe_route_dev", (256, 64, 8, 512, 768)),
         ("moe_ffn_logits_dev", (3, 256, 8, 512, 768, 1024, 1280)), ("moe_ffn_routed_dev", (3, 256, 512, 8, 768, 1024)),
         ("graph_launch", (C.c_void_p(4096),)), ("gemv", ("a", _x, _y)), ("gemv_f32", ("a", _x, _y))]


@pytest.mark.parametrize("name,args", CALLS, ids=[c[0] for c in CALLS])
def test_ctypes_calls_equal_the_extension(rec, pkg, name, args):
    """Without the extension module the package makes the same library calls."""
    mod, L = rec
    saw = []
    for calls in (mod, pkg.CtypesCalls(_typed(pkg, L))):
        assert getattr(calls, name)(16, *args) == 1
        saw.append(L.rec_text())
    assert saw[0].startswith(b"smx_" + name.encode() + b" 0x10 ") and saw[0] == saw[1]


def _typed(pkg, L):
    for n in pkg.EXPORTS:
        if hasattr(L, n):
            getattr(L, n).argtypes = getattr(pkg.load_library(), n).argtypes
    return L


def test_ctypes_calls_offer_every_function(rec, pkg):
    names = {n for n in dir(rec[0]) if not n.startswith("_")}
    assert names == {n for n in dir(pkg.CtypesCalls) if not n.startswith("_")}


def test_the_package_works_without_the_extension(pkg, monkeypatch, tmp_path):
    monkeypatch.setattr(pkg, "NATIVE_PATH", str(tmp_path / "none.so"))
    monkeypatch.setattr(pkg, "_native", None)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        assert isinstance(pkg.load_native(), pkg.CtypesCalls)


def test_a_build_without_the_headers(pkg, monkeypatch, tmp_path):
    builder = _load_by_path("strix_rs_amd_build", os.path.join(PKG_DIR, "build.py"))
    monkeypatch.setattr(builder.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    (tmp_path / "_smx_native.so").write_bytes(b"of an older build")
    assert builder.build_pybind(str(tmp_path)) is None and not (tmp_path / "_smx_native.so").exists()
