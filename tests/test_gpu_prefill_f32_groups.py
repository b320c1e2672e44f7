"""f32 prefill attention at the edges of its key groups: query blocks of 16, 32 and 64, key tiles of 32 shared out over
four, two and one groups of waves, and the prompt lengths where the number of groups changes."""
import ctypes as C
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_past,T", [(0, 1), (0, 2), (0, 15), (0, 16), (0, 17), (0, 33), (0, 64), (0, 129), (31, 1), (1, 31),
                                      (97, 50), (1000, 156), (3, 1280), (0, 1281), (5, 3456), (0, 3457)])
def test_f32_prefill_equals_row_kernel(qa, n_past, T):
    """Against the f32 row kernel (QA_PREFILL_F32_ROWS=1: two passes, the reference's order).  Each output is a sum of
    at most 3.5k products weighted by probabilities that sum to 1: in another association, with one merge per key
    group, it moves by a few 2^-24 of the values (2e-5 absolute at |v| <= 5, 2e-6 in the 2-norm)."""
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"
    lay = qa.KvLayout(1, 1, 8, 128, n_past + T + 3, qa.QA_CACHE_F32)
    rng = np.random.default_rng(1000 * n_past + T)
    cache = qa.DeviceArray.from_numpy(rng.standard_normal((2, 8, n_past + T + 3, 128)).astype(np.float32))
    q = qa.DeviceArray.from_numpy(rng.standard_normal((T, 2048)).astype(np.float32))
    outs = []
    for rows in ("0", "1"):
        os.environ["QA_PREFILL_F32_ROWS"] = rows
        try:
            out = qa.DeviceArray((T, 2048))
            print(f"f32 prefill rows-kernel={rows} n_past={n_past} T={T}", flush=True)
            qa.check(qa.lib.qa_prefill_attn(q.ptr, cache.ptr, C.byref(lay), 0, 0, n_past, T, 16, 128 ** -0.5, out.ptr,
                                            None, 0, None))
            qa.synchronize()
            outs.append(out.numpy().astype(np.float64))
        finally:
            os.environ.pop("QA_PREFILL_F32_ROWS", None)
    d = outs[0] - outs[1]
    assert np.isfinite(d).all()
    assert np.abs(d).max() <= 2e-5 and np.linalg.norm(d) <= 2e-6 * np.linalg.norm(outs[1]), (np.abs(d).max(),)


@pytest.mark.parametrize("entry,T,bad", [("causal", 33, 32), ("causal", 97, 64), ("causal", 130, 96), ("cache", 33, 32),
                                         ("cache", 64, 5), ("cache", 1300, 32)])
def test_f32_prefill_keeps_nan(qa, entry, T, bad):
    """A NaN in key row `bad` of KV head 3 reaches every query that attends it, also the one that sees no other key of
    its key group (the query at the key's own position, where the key opens a tile); nothing else moves by a bit."""
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"
    rng = np.random.default_rng(T + bad)
    q = qa.DeviceArray.from_numpy(rng.standard_normal((T, 2048)).astype(np.float32))
    k, v = (rng.standard_normal((8, T, 128)).astype(np.float32) for _ in range(2))
    outs = []
    for poisoned in (False, True):
        if poisoned:
            k[3, bad, 17] = np.nan
        out = qa.DeviceArray((T, 2048))
        print(f"f32 prefill entry={entry} T={T} NaN key {bad if poisoned else None}", flush=True)
        if entry == "causal":
            dk, dv = (qa.DeviceArray.from_numpy(np.ascontiguousarray(a.transpose(1, 0, 2))) for a in (k, v))
            qa.check(qa.lib.qa_causal_attn_f32(q.ptr, dk.ptr, dv.ptr, T, 16, 8, 128 ** -0.5, out.ptr, None))
        else:
            lay = qa.KvLayout(1, 1, 8, 128, T, qa.QA_CACHE_F32)
            cache = qa.DeviceArray.from_numpy(np.stack([k, v]))
            qa.check(qa.lib.qa_prefill_attn(q.ptr, cache.ptr, C.byref(lay), 0, 0, 0, T, 16, 128 ** -0.5, out.ptr, None, 0,
                                            None))
        qa.synchronize()
        outs.append(out.numpy().reshape(T, 16, 128))
    clean, got = outs
    assert np.isfinite(clean).all()
    hit = np.zeros(clean.shape, bool)
    hit[bad:, 6:8] = True
    assert np.isnan(got[hit]).all(), np.argwhere(~np.isnan(got[bad:, 6:8]).all(axis=(1, 2)))[:4].ravel() + bad
    np.testing.assert_array_equal(got[~hit].view(np.uint32), clean[~hit].view(np.uint32))


def test_f32_prefill_of_one_key_tile_is_short(qa):
    """16 positions are one key tile, which no key group shares: 6.6 us against 7.9 us for 33 positions (on four groups
    both took 8.1).  A hundred launches in one graph, so that the host's launch rate is not what is measured."""
    hip = qa.lib                                       # the library's own HIP runtime

    def ok(rc):
        assert rc == 0, rc

    stream = C.c_void_p()
    ok(hip.hipStreamCreateWithFlags(C.byref(stream), 1))
    us = []
    for T in (16, 33):
        lay = qa.KvLayout(1, 1, 8, 128, T, qa.QA_CACHE_F32)
        cache, q, out = qa.DeviceArray((2, 8, T, 128)), qa.DeviceArray((T, 2048)), qa.DeviceArray((T, 2048))
        args = (q.ptr, cache.ptr, C.byref(lay), 0, 0, 0, T, 16, 128 ** -0.5, out.ptr, None, 0, stream)
        qa.synchronize()
        graph, run = C.c_void_p(), C.c_void_p()
        ok(hip.hipStreamBeginCapture(stream, 2))
        for _ in range(100):
            qa.check(qa.lib.qa_prefill_attn(*args))
        ok(hip.hipStreamEndCapture(stream, C.byref(graph)))
        ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        got = []
        for _ in range(21):
            t = time.perf_counter()
            for _ in range(5):
                ok(hip.hipGraphLaunch(run, stream))
            ok(hip.hipStreamSynchronize(stream))
            got.append((time.perf_counter() - t) / 500 * 1e6)
        us.append(sorted(got)[5])
        ok(hip.hipGraphExecDestroy(run))
        ok(hip.hipGraphDestroy(graph))
    ok(hip.hipStreamDestroy(stream))
    print(f"f32 prefill: 16 positions {us[0]:.2f} us, 33 positions {us[1]:.2f} us", flush=True)
    assert us[0] < 0.93 * us[1]
