"""Which f16 prefill attention kernel a call runs, by its tokens and the positions cached before them: key groups (32 query
tokens per workgroup) or the 128-token tiles, on either side of every line of the rule."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _attend(qa, n_past, T, reps=0):
    """One call: outputs and inputs.  reps > 0: the times of that many calls in us."""
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"
    L = n_past + T
    lay = qa.KvLayout(1, 1, 8, 128, L + 5, qa.QA_CACHE_F16)
    rng = np.random.default_rng(1000 * n_past + T)
    kv = rng.standard_normal((2, 8, L + 5, 128), np.float32).astype(np.float16)
    kv[:, :, L:] = np.nan                                  # nothing past the end is read into a result
    q = rng.standard_normal((T, 16, 128), np.float32)
    cache, dq, out = qa.DeviceArray.from_numpy(kv), qa.DeviceArray.from_numpy(q), qa.DeviceArray((T, 2048))
    nbytes = qa.lib.qa_prefill_attn_workspace_bytes(T, 16)
    ws = qa.DeviceArray((nbytes,), np.uint8)
    args = (dq.ptr, cache.ptr, C.byref(lay), 0, 0, n_past, T, 16, 128 ** -0.5, out.ptr, ws.ptr, nbytes, None)
    print(f"f16 prefill n_past={n_past} T={T}", flush=True)
    qa.check(qa.lib.qa_prefill_attn(*args))
    qa.synchronize()
    us = []
    for _ in range(reps):
        t = time.perf_counter()
        for _ in range(10):
            qa.check(qa.lib.qa_prefill_attn(*args))
        qa.synchronize()
        us.append((time.perf_counter() - t) * 1e5)
    if reps:
        return us
    return out.numpy().reshape(T, 16, 128), kv[0, :, :L].astype(np.float32), kv[1, :, :L].astype(np.float32), q


@pytest.mark.parametrize("n_past,T", [(1151, 1025), (1152, 1025), (128, 2048), (129, 2048), (11264, 1024), (11265, 1024),
                                      (12287, 1), (12287, 2), (4000, 1280)])
def test_f16_prefill_behind_cached_positions(qa, orc, n_past, T):
    got, k, v, q = _attend(qa, n_past, T)
    for t in sorted({0, 31, 127, 128, T // 2, T - 1} & set(range(T))):
        ref = orc.cache_attention(k[:, :n_past + t + 1], v[:, :n_past + t + 1], q[t:t + 1], n_past + t, True)[0]
        d = got[t].astype(np.float64) - ref
        assert np.abs(d).max() <= 2e-3 and np.linalg.norm(d) <= 1e-3 * np.linalg.norm(ref), (t, np.abs(d).max())


@pytest.mark.parametrize("n_past,more,fewer", [(4000, 2560, 2048), (8000, 2560, 2048)])
def test_f16_prefill_chunk_time_grows_with_tokens(qa, n_past, more, fewer):
    """Fewer tokens behind the same cached positions never take longer: on key groups 2048 tokens took 1.05 to
    1.11 times the 2560 tokens' time, on the 128-token tiles they take 0.65 to 0.82."""
    us = [min(_attend(qa, n_past, T, reps=20)) for T in (more, fewer)]
    print(f"n_past={n_past}: {more} tokens {us[0]:.1f} us, {fewer} tokens {us[1]:.1f} us", flush=True)
    assert us[1] < us[0]
