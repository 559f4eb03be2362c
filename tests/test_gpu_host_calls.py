"""Host-pointer calls: the grouped fp32-activation batch against one call per item (same bits), the binding's handling of
arrays that are not contiguous float32, the routes of small and large transfers, and rows that are not finite."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _up(accel, ty):
    return {2: accel.upload_q4_0, 8: accel.upload_q8_0, 14: accel.upload_q6_k}[ty]


@pytest.mark.parametrize("ty,Ns,K", [(8, (2560, 640, 640), 2560), (2, (1, 9728, 3), 2560), (14, (300, 40), 1024), (2, (256, 257, 255), 256),
                                     (8, (33,) * 18, 512), (2, (65, 66), 96), (14, (130, 7), 9728), (8, (60000, 5), 512)])
def test_f32_batch_equals_single_calls(accel, synth, ty, Ns, K):
    """Shared launches with unequal heights: fewer rows than workgroups, more items than a launch takes (18), rows that the flat
    form does not serve (K = 96), several rounds of workgroups (60000 rows)."""
    calls = []
    for i, N in enumerate(Ns):
        assert _up(accel, ty)(f"hb{i}", synth.make_weight(ty, N, K, seed=i + N), K, N)
        calls.append((f"hb{i}", synth.make_acts(1, K, seed=100 + i // 2)[0]))
    got = accel.gemv_batch(calls, list(Ns), f32=True)
    for (key, x), N, y in zip(calls, Ns, got):
        assert np.array_equal(y, accel.gemv_f32(key, x, N)), (key, N)


def test_arrays_of_other_layouts(accel, synth):
    N, K = 96, 256
    assert accel.upload_q8_0("hl", synth.make_q8_0(N, K, 1), K, N)
    x = synth.make_acts(3, K, seed=2)
    x1 = x[0].copy()
    wide = np.zeros((3, 2 * K), np.float32)
    wide[:, ::2] = x
    for fn in (accel.gemv, accel.gemv_f32):
        want = fn("hl", x1, N)
        for other in (x1.astype(np.float64), wide[0, ::2], x1.reshape(1, K), list(map(float, x1))):
            assert np.array_equal(fn("hl", other, N), want)
        assert fn("absent", x1, N) is None
    want = accel.prefill_q8_gemm("hl", x, 3, N)
    assert np.array_equal(accel.prefill_q8_gemm("hl", wide[:, ::2], 3, N), want)
    assert np.array_equal(accel.prefill_q8_gemm("hl", x.astype(np.float64), 3, N), want)
    ids = accel.lm_head_argmax_rows("hl", x, 3)
    assert np.array_equal(accel.lm_head_argmax_rows("hl", wide[:, ::2], 3), ids)
    batch = accel.gemv_batch([("hl", x1), ("absent", x1), ("hl", wide[1, ::2])], [N, N, N])
    assert np.array_equal(batch[0], accel.gemv("hl", x1, N)) and batch[1] is None and np.array_equal(batch[2], accel.gemv("hl", x[1], N))


def _dev_gemm(accel, key, xs, N):
    m, K = xs.shape
    xd, yd = accel.dev_alloc(xs.nbytes), accel.dev_alloc(m * N * 4)
    accel.h2d(xd, xs)
    assert accel.gemm_dev(key, xd, m, yd)
    y = accel.d2h(np.empty((m, N), np.float32), yd)
    accel.dev_free(xd)
    accel.dev_free(yd)
    return y


@pytest.mark.parametrize("ty,m,N,K", [(8, 5, 33, 96), (2, 40, 1001, 256), (8, 64, 4096, 2048), (8, 128, 4097, 1024), (14, 383, 999, 2560), (2, 513, 777, 1024),
                                      (8, 900, 4096, 512), (8, 1500, 9001, 256), (8, 300, 256, 15360)])
def test_large_transfers_equal_the_device_call(accel, synth, ty, m, N, K):
    """Every route of a host call: the staging with whole and ragged 16 KB parts, one and several row groups through the ring, more
    results than the ring holds (54 MB), inputs larger than it.  (Row groups may take another split-K: 1e-6 instead of equal bits.)"""
    assert _up(accel, ty)("hp", synth.make_weight(ty, N, K, seed=N), K, N)
    xs = synth.make_acts(m, K, seed=m)
    want = _dev_gemm(accel, "hp", xs, N)
    for _ in range(2):
        got = accel.prefill_q8_gemm("hp", xs, m, N)
        assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()


@pytest.mark.parametrize("m,hidden", [(3, 256), (150, 512), (700, 1024)])
def test_moe_layer_host_rows_equal_resident_rows(accel, synth, m, hidden):
    ne, eff, k = 8, 256, 3
    gate, up, down = synth.make_moe_q8(ne, hidden, eff, seed=hidden)
    assert accel.upload_moe_q8(7, gate, up, down, hidden, eff, ne)
    ids, w = synth.zipf_routing(m, ne, k, seed=m)
    plan, tok, wslot = synth.group_by_expert(ids, w, ne)
    xs = synth.make_acts(m, hidden, seed=3)
    xd, yd = accel.dev_alloc(xs.nbytes), accel.dev_alloc(xs.nbytes)
    accel.h2d(xd, xs)
    assert accel.moe_layer_resident(7, xd, m, plan, tok, wslot, yd)
    want = accel.d2h(np.empty_like(xs), yd)
    accel.dev_free(xd)
    accel.dev_free(yd)
    assert np.array_equal(accel.moe_layer_q8_dev(7, xs, m, plan, tok, wslot), want)


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def test_rows_and_results_that_overlap(accel, synth):
    """A result row covers four activation rows of groups that are read later."""
    m, K, N = 4000, 256, 1024
    assert accel.upload_q8_0("ho", synth.make_q8_0(N, K, 1), K, N)
    xs = synth.make_acts(m, K, seed=1)
    want = accel.prefill_q8_gemm("ho", xs, m, N)
    buf = np.zeros(m * N + 77, np.float32)
    for at in (0, 77):
        buf[:m * K] = xs.ravel()
        assert accel._L.smx_gemm(accel._h, b"ho", _p(buf), m, K, _p(buf[at:]), m * N) == 1
        assert np.array_equal(buf[at:at + m * N].reshape(m, N), want)


@pytest.mark.parametrize("m", [70, 700])
@pytest.mark.parametrize("shift_in,shift_out", [(4, 0), (0, 4), (8, 12)])
def test_host_memory_of_any_float_alignment(accel, synth, m, shift_in, shift_out):
    K, N = 512, 4099
    assert accel.upload_q8_0("ha", synth.make_q8_0(N, K, 1), K, N)
    xs = synth.make_acts(m, K, seed=m)
    want = accel.prefill_q8_gemm("ha", xs, m, N)

    def at(n, shift):
        raw = np.zeros(n * 4 + 128, np.uint8)
        o = (-raw.ctypes.data) % 64 + shift
        return raw[o:o + n * 4].view(np.float32)
    x, y = at(m * K, shift_in), at(m * N, shift_out)
    x[:] = xs.ravel()
    assert accel._L.smx_gemm(accel._h, b"ha", _p(x), m, K, _p(y), m * N) == 1
    assert np.array_equal(y.reshape(m, N), want)


def test_large_calls_on_one_core(pkg, synth):
    """A context made where the process may use one core only: the calling thread moves every piece itself."""
    m, K, N = 1500, 256, 9001   # 54 MB of results, more than the ring
    raw, xs = synth.make_q8_0(N, K, 1), synth.make_acts(m, K, seed=1)
    got, all_cores = [], os.sched_getaffinity(0)
    for cores in (all_cores, {min(all_cores)}):
        try:
            os.sched_setaffinity(0, cores)
            with pkg.Mi355WeightAccel(0) as a:
                assert a.upload_q8_0("w", raw, K, N)
                got.append(a.prefill_q8_gemm("w", xs, m, N))
        finally:
            os.sched_setaffinity(0, all_cores)
    assert np.array_equal(got[0], got[1])


def test_a_polled_call_behind_long_work(accel, synth):
    """More than the polled 2 ms of work in front of a call: it waits in the runtime."""
    K, N, m = 2560, 9728, 1024
    assert accel.upload_q8_0("hw", synth.make_q8_0(N, K, 1), K, N)
    x = synth.make_acts(70, K, seed=2)
    one, some = accel.gemv("hw", x[0], N), accel.prefill_q8_gemm("hw", x, 70, N)
    xd, yd = accel.dev_alloc(m * K * 4), accel.dev_alloc(m * N * 4)
    accel.h2d(xd, synth.make_acts(m, K, seed=3))
    for _ in range(2):
        for _ in range(60):   # 60 x 0.1 ms
            assert accel.gemm_dev("hw", xd, m, yd)
        assert np.array_equal(accel.gemv("hw", x[0], N), one)
        for _ in range(60):
            assert accel.gemm_dev("hw", xd, m, yd)
        assert np.array_equal(accel.prefill_q8_gemm("hw", x, 70, N), some)
    accel.dev_free(xd)
    accel.dev_free(yd)


@pytest.mark.parametrize("hidden,rows", [(512, (150, 1, 33, 700)), (1024, (129, 64, 400, 7))])
def test_large_expert_ffn_equals_its_groups(accel, synth, hidden, rows):
    """Over 3 MB of expert-major rows (the transfer rings) against a call per group (the staging)."""
    ne, eff = 8, 256
    gate, up, down = synth.make_moe_q8(ne, hidden, eff, seed=hidden)
    assert accel.upload_moe_q8(9, gate, up, down, hidden, eff, ne)
    xs = synth.make_acts(sum(rows), hidden, seed=4)
    assert 2 * xs.nbytes >= 3 << 20
    plan = [(2 * i + 1, n) for i, n in enumerate(rows)]
    got = accel.moe_layer_ffn(9, plan, xs, sum(rows))
    o = 0
    for e, n in plan:
        for a in range(0, n, 128):   # whole tiles, and sizes that take the same number of K slices: the same sums
            part = xs[o + a:o + min(n, a + 128)]
            assert np.array_equal(got[o + a:o + min(n, a + 128)], accel.moe_expert_ffn(9, e, part, part.shape[0])), (e, a)
        o += n


def test_host_calls_leave_a_capture_as_it_is(accel, pkg, synth):
    K, N, m = 256, 4096, 300
    assert accel.upload_q8_0("hc", synth.make_q8_0(N, K, 1), K, N)
    xs = synth.make_acts(m, K, seed=5)
    want = [accel.gemv("hc", x, N) for x in xs[:3]]
    xd, yd = accel.dev_alloc(K * 4), accel.dev_alloc(N * 4)
    accel.gemv_dev("hc", xd, 1, yd)
    accel.graph_begin()
    for call in (lambda: accel.gemv("hc", xs[0], N), lambda: accel.prefill_q8_gemm("hc", xs, m, N), lambda: accel.gemv_f32("hc", xs[0], N)):
        with pytest.raises(pkg.SmxError, match="captured"):
            call()
    assert accel.gemv_dev("hc", xd, 1, yd)
    g = accel.graph_end()
    for x, y in zip(xs, want):
        accel.h2d(xd, x)
        accel.graph_launch(g)
        assert np.array_equal(accel.d2h(np.empty(N, np.float32), yd), y)
        assert np.array_equal(accel.gemv("hc", x, N), y)
    accel.graph_destroy(g)
    accel.dev_free(xd)
    accel.dev_free(yd)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("ty,m,N,K", [(8, 20 + 64 * 2, 130, 256), (8, 85, 300, 96), (2, 150, 130, 256), (14, 150, 130, 512), (14, 72, 300, 2560)])
def test_a_row_that_is_not_finite_stays_by_itself(accel, synth, ty, m, N, K, bad):
    """Tiles whose rows share fragments and scale registers: the other rows keep their bits.  (65..150 rows of Q8_0 end in a tile of
    at most 32, which streams its weights three stages ahead where K is a multiple of 128.)"""
    assert _up(accel, ty)("hn", synth.make_weight(ty, N, K, seed=N), K, N)
    xs = synth.make_acts(m, K, seed=m)
    want = accel.prefill_q8_gemm("hn", xs, m, N)
    assert np.isfinite(want).all()
    for row in (0, m // 2, m - 1):
        x = xs.copy()
        x[row, K // 3] = bad
        got = accel.prefill_q8_gemm("hn", x, m, N)
        rest = np.arange(m) != row
        assert np.array_equal(got[rest], want[rest]), row
        # an infinite block maximum scales its whole row; a NaN never is the maximum (fmaxf, as in kernels.rs:75-96), and the
        # quantiser gives it some integer of the block's range
        assert np.isnan(bad) or not np.isfinite(got[row]).any(), row


@pytest.mark.parametrize("ty", [8, 14])
def test_a_token_that_is_not_finite_stays_by_itself(accel, synth, ty):
    ne, hidden, eff, k, m = 8, 512, 256, 2, 90     # expert groups of 1 .. 64 rows
    gate, up, down = (synth.make_weight(ty, ne * eff, hidden, 1), synth.make_weight(ty, ne * eff, hidden, 2), synth.make_weight(ty, ne * hidden, eff, 3))
    assert (accel.upload_moe_q6 if ty == 14 else accel.upload_moe_q8)(10, gate, up, down, hidden, eff, ne)
    ids, w = synth.zipf_routing(m, ne, k, seed=m)
    plan, tok, wslot = synth.group_by_expert(ids, w, ne)
    xs = synth.make_acts(m, hidden, seed=6)
    want = accel.moe_layer_q8_dev(10, xs, m, plan, tok, wslot)
    for row in (0, m - 1):
        x = xs.copy()
        x[row, 3] = np.nan
        got = accel.moe_layer_q8_dev(10, x, m, plan, tok, wslot)
        rest = np.arange(m) != row
        assert np.array_equal(got[rest], want[rest])
