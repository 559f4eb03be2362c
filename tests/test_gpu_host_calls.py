"""Host-pointer calls: the grouped fp32-activation batch against one call per item (same bits), and the binding's handling of
arrays that are not contiguous float32."""
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
