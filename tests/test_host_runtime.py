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


def test_host_calls_are_refused_during_capture(run):
    """At once, without a wait and without pulling further streams into the capture, which goes on."""
    run("""
        a = accel()
        K, N, ne, hidden, eff = 256, 4096, 4, 256, 256
        assert a.upload_moe_q8(0, *synth.make_moe_q8(ne, hidden, eff, seed=1), hidden, eff, ne)
        x, xs = synth.make_acts(1, K, seed=1)[0], synth.make_acts(300, K, seed=1)
        ids, w = synth.zipf_routing(300, ne, 2, seed=3)
        plan, tok, wslot = synth.group_by_expert(ids, w, ne)
        calls = [lambda: a.gemv("w", x, N), lambda: a.gemv_f32("w", x, N), lambda: a.gemv_rows("w", xs[:7], N), lambda: a.prefill_q8_gemm("w", xs, 300, N),
                 lambda: a.gemv_batch([("w", x)] * 2, [N] * 2), lambda: a.gemv_fused("w", 1, x, x, N), lambda: a.lm_head_argmax_rows("w", xs[:3], 3),
                 lambda: a.quantize(xs, K), lambda: a.gemv_block_dots("w", x, N, K // 32), lambda: a.moe_ffn(0, ids[0], w[0], x),
                 lambda: a.moe_route(x[:64], 8), lambda: a.moe_layer_q8_dev(0, xs, 300, plan, tok, wslot),
                 lambda: a.moe_layer_ffn(0, [(1, 300)], xs, 300)]
        for call in calls[:3]:       # (a context that has made no large call yet)
            call()
        streams = F.fake_streams()
        a.graph_begin()
        for i, call in enumerate(calls):
            t0 = time.perf_counter()
            try:
                call()
            except pkg.SmxError as e:
                assert e.code == -1 and "captured" in str(e), (i, e)
            else:
                raise AssertionError(i)
            assert time.perf_counter() - t0 < 1.0, i
        assert a.gemv("absent", x, N) is None       # a decline comes first, as ever
        assert F.fake_streams() == streams
        a.graph_end()
        for call in calls:
            call()
    """)


@pytest.mark.parametrize("call,slow,failing", [
    ("a.prefill_q8_gemm('w', xs[:70], 70, N)", "actquant", "gemm_i8"), ("a.prefill_q8_gemm('w', xs[:70], 70, N)", "gemm_i8", "span_out"),
    ("a.prefill_q8_gemm('w', xs, 300, N)", "actquant", "gemm_i8"), ("a.prefill_q8_gemm('w', xs, 300, N)", "gemm_i8", "span_out"),
    ("a.gemv('w', xs[:1], N)", "gemv_flat", "stream_flag"), ("a.gemv_f32('w', xs[:1], N)", "gemv_f32", "stream_flag"),
    ("a.gemv_rows('w', xs[:3], N)", "span_in", "gemv_"), ("a.gemv_rows('w', xs[:9], N)", "skinny_quant", "skinny_kernel"),
    ("a.gemv_batch([('w', xs[0])] * 2, [N] * 2)", "gemv_", "stream_flag"), ("a.gemv_fused('w', 1, xs[0], xs[0], N)", "gemv_", "stream_flag"),
    ("a.lm_head_argmax_rows('w', xs[:3], 3)", "gemv_", "argmax_final"), ("a.gemm_block_dots('w', xs[:70], 70, N, K // 32)", "actquant", "gemm_i8"),
    ("a.moe_ffn(0, ids[0], w[0], xs[0])", "dual", "moe_down"), ("a.moe_ffn(0, ids[0], w[0], xs[0], 0.5)", "moe_down", "shexp_add"),
    ("a.moe_layer_q8_dev(0, xs, 300, plan, tok, wslot)", "gemm_i8", "moe_combine"),
    ("a.moe_layer_ffn(0, [(1, 300)], xs, 300)", "actquant", "silu_mul")])
def test_a_failed_call_leaves_nothing_running(run, call, slow, failing):
    run("""
        a = accel()
        K, N, ne, hidden, eff = 256, 4096, 4, 256, 256
        assert a.upload_moe_q8(0, *synth.make_moe_q8(ne, hidden, eff, seed=1), hidden, eff, ne)
        for part in ("gate", "up", "down"):
            assert a.upload_q8_0(f"blk.0.ffn_{part}_shexp.weight", synth.make_q8_0(hidden, eff, 1), eff, hidden)
        xs = synth.make_acts(300, K, seed=1)
        ids, w = synth.zipf_routing(300, ne, 2, seed=3)
        plan, tok, wslot = synth.group_by_expert(ids, w, ne)
        eval(call)
        F.fake_slow_kernel(slow.encode(), 100000)
        F.fake_failing_kernel(failing.encode())
        t0 = time.perf_counter()
        try:
            eval(call)
        except pkg.SmxError as e:
            pending = F.fake_pending()
            assert e.code == -2 and "HIP error" in str(e), e
        else:
            raise AssertionError("no error")
        assert F.fake_failed_launches() > 0
        assert time.perf_counter() - t0 > 0.09      # the slow kernel did run
        assert pending == 0
        F.fake_failing_kernel(b"")
        F.fake_slow_kernel(b"", 0)
        eval(call)                                  # and the next call is an ordinary one
    """, call=call, slow=slow, failing=failing)


@pytest.mark.parametrize("refuse", [False, True])
def test_large_calls_without_the_pipe(run, refuse):
    """Where 64 MB of pinned memory are not to be had the large calls copy from and to the caller's memory; it is asked for once."""
    run("""
        a = accel()
        K, N, ne, hidden, eff = 256, 4096, 4, 1024, 256
        assert a.upload_moe_q8(0, *synth.make_moe_q8(ne, hidden, eff, seed=1), hidden, eff, ne)
        xs, xh = synth.make_acts(700, K, seed=1), synth.make_acts(700, hidden, seed=2)
        ids, w = synth.zipf_routing(700, ne, 2, seed=3)
        plan, tok, wslot = synth.group_by_expert(ids, w, ne)
        if refuse:
            F.fake_host_limit(C.c_size_t(8 << 20))
        for _ in range(2):
            F.fake_keep_inbound(1)
            assert untouched(a.prefill_q8_gemm("w", xs, 700, N)) and np.array_equal(inbound(), xs.ravel())
            F.fake_keep_inbound(1)
            assert untouched(a.moe_layer_q8_dev(0, xh, 700, plan, tok, wslot)) 
            assert xh.tobytes() in inbound().tobytes()
            F.fake_keep_inbound(1)
            y = a.moe_layer_ffn(0, [(1, 300), (2, 400)], xh, 700)
            assert np.array_equal(np.diff(y.reshape(-1).view(np.uint32)), np.ones(y.size - 1))
            assert xh.tobytes() in inbound().tobytes()
        assert F.fake_host_refused() == (1 if refuse else 0)
        assert F.fake_streams() == (1 if refuse else 3)
        if refuse:
            assert F.fake_host_live() < 8 << 20
        a.close()
        assert F.fake_host_live() == 0 and F.fake_streams() == 0
    """, refuse=refuse)


def test_workers_sleep_while_the_device_computes(run):
    """During a long kernel a large call occupies the calling thread's core (it polls) and not the workers' too."""
    run("""
        a = accel()
        xs = synth.make_acts(300, 256, seed=1)
        assert untouched(a.prefill_q8_gemm("w", xs, 300, 4096))
        F.fake_slow_kernel(b"gemm_i8", 500000)
        cpu, wall = time.process_time(), time.perf_counter()
        assert untouched(a.prefill_q8_gemm("w", xs, 300, 4096))
        cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
        assert wall > 0.5 and cpu < 1.5 * wall, (cpu, wall)
        F.fake_slow_kernel(b"", 0)
        for _ in range(200):                        # asleep or not, each call's transfers are whole
            F.fake_keep_inbound(1)
            assert untouched(a.prefill_q8_gemm("w", xs, 300, 4096)) and np.array_equal(inbound(), xs.ravel())
    """)


def test_pinned_memory_is_asked_for_as_coherent(run):
    """Whatever HIP_HOST_COHERENT says: polled words and results that kernels write with plain stores rest on it."""
    run("""
        a = accel()
        xs = synth.make_acts(300, 256, seed=1)
        a.gemv("w", xs[0], 4096)
        a.prefill_q8_gemm("w", xs[:70], 70, 4096)
        a.prefill_q8_gemm("w", xs, 300, 4096)
        assert F.fake_host_live() > 64 << 20 and F.fake_host_noncoherent() == 0
    """)


@pytest.mark.parametrize("ty,eff,refused", [(8, 8192, True), (8, 8160, False), (14, 8192, True), (14, 7936, False)])
def test_expert_tensors_beyond_the_grouped_kernels_range(run, ty, eff, refused):
    """The grouped GEMMs address an expert tensor with 32-bit offsets: 64 experts x 8192 x 4096 = 2^31 elements are refused by
    every grouped call, and one step less is served."""
    run("""
        a = pkg.Mi355WeightAccel(0)
        ne, hidden = 64, 4096
        n = ne * eff * hidden // (256 if ty == 14 else 32) * (210 if ty == 14 else 34)
        raw = np.zeros(n, np.uint8)
        assert (a.upload_moe_q6 if ty == 14 else a.upload_moe_q8)(0, raw, raw, raw, hidden, eff, ne)
        xs = np.ones((70, hidden), np.float32)
        ids, w = synth.zipf_routing(70, ne, 2, seed=3)
        plan, tok, wslot = synth.group_by_expert(ids, w, ne)
        xd, yd = a.dev_alloc(xs.nbytes), a.dev_alloc(xs.nbytes)
        for call in (lambda: a.moe_layer_q8_dev(0, xs, 70, plan, tok, wslot), lambda: a.moe_layer_ffn(0, [(63, 70)], xs, 70),
                     lambda: a.moe_expert_ffn(0, 1, xs, 70), lambda: a.moe_layer_resident(0, xd, 70, plan, tok, wslot, yd),
                     lambda: a.moe_layer_stages(0, xs, 70, plan, tok, wslot, eff)):
            try:
                call()
            except pkg.SmxError as e:
                assert refused and e.code == -3, e
            else:
                assert not refused
    """, ty=ty, eff=eff, refused=refused)


@pytest.mark.parametrize("cores", [1, 2, 8])
@pytest.mark.parametrize("shift_in,shift_out", [(0, 0), (4, 0), (0, 4), (8, 12)])
def test_workers_and_alignments(run, cores, shift_in, shift_out):
    """Transfers whole with no worker besides the calling thread, with one and with several, from and to memory of any float
    alignment; more results than the outbound ring holds (54 MB), ragged last parts."""
    run("""
        os.sched_setaffinity(0, set(sorted(os.sched_getaffinity(0))[:cores]))
        K, N = 256, 4096
        a = accel(K, N)
        for m in (300, 3301):
            xs, y = floats(m * K, shift_in), floats(m * N - 5, shift_out)
            xs[:] = np.random.default_rng(m).random(m * K, dtype=np.float32)
            F.fake_keep_inbound(1)
            assert L.smx_gemm(a._h, b"w", p(xs), m, K, p(y), m * N - 1) == -1          # one result short: refused, nothing moved
            assert inbound().size == 0 and not y.any()
            y = floats(m * N, shift_out)
            assert L.smx_gemm(a._h, b"w", p(xs), m, K, p(y), y.size) == 1
            assert untouched(y) and np.array_equal(inbound(), xs)
    """, cores=cores, shift_in=shift_in, shift_out=shift_out)


@pytest.mark.parametrize("call,slow", [("a.gemv('w', xs[0], N)", "gemv_flat"), ("a.gemv_rows('w', xs[:3], N)", "gemv_"), ("a.prefill_q8_gemm('w', xs[:70], 70, N)", "gemm_i8"),
                                       ("a.prefill_q8_gemm('w', xs, 300, N)", "gemm_i8")])
def test_work_longer_than_the_polls(run, call, slow):
    """Beyond the polled 2 ms a call waits in the runtime, and its result is whole."""
    run("""
        K, N = 256, 4096
        a = accel(K, N)
        xs = synth.make_acts(300, K, seed=1)
        F.fake_slow_kernel(slow.encode(), 50000)
        for _ in range(3):
            t0 = time.perf_counter()
            y = eval(call)
            assert time.perf_counter() - t0 > 0.05
            # (a result written by the kernel itself is the pinned buffer's filling here, one copied out the device memory's)
            assert untouched(y) or (y.view(np.uint32) == 0xeeeeeeee).all()
    """, call=call, slow=slow)
