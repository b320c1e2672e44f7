"""f16 prefill attention with key groups (prompts up to 2048 tokens): query tiles of 32, key tiles of 32 shared out over
four groups of waves, at their edges and where the 128-token tiles take over, against the oracle's attention."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_past,T", [(0, 1), (0, 2), (0, 31), (0, 32), (0, 33), (0, 65), (0, 127), (0, 129), (1, 32), (31, 33),
                                      (127, 2), (300, 77), (1000, 156), (0, 2048), (0, 2049)])
def test_f16_prefill_matches_oracle(qa, orc, n_past, T):
    """Bars of the attention: 2e-3 max-abs and 1e-3 relative 2-norm (f16 operands).  All rows up to 500 tokens, else
    rows around the tile edges as decodes over their prefix."""
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"
    L = n_past + T
    lay = qa.KvLayout(1, 1, 8, 128, L + 5, qa.QA_CACHE_F16)
    rng = np.random.default_rng(1000 * n_past + T)
    kv = rng.standard_normal((2, 8, L + 5, 128)).astype(np.float16)
    kv[:, :, L:] = np.nan                                  # nothing past the end is read into a result
    q = rng.standard_normal((T, 16, 128)).astype(np.float32)
    cache, dq, out = qa.DeviceArray.from_numpy(kv), qa.DeviceArray.from_numpy(q), qa.DeviceArray((T, 2048))
    nbytes = qa.lib.qa_prefill_attn_workspace_bytes(T, 16)
    ws = qa.DeviceArray((nbytes,), np.uint8)
    print(f"f16 prefill n_past={n_past} T={T}", flush=True)
    qa.check(qa.lib.qa_prefill_attn(dq.ptr, cache.ptr, C.byref(lay), 0, 0, n_past, T, 16, 128 ** -0.5, out.ptr, ws.ptr,
                                    nbytes, None))
    qa.synchronize()
    got = out.numpy().reshape(T, 16, 128)
    k, v = (kv[i, :, :L].astype(np.float32) for i in (0, 1))
    if T <= 500:
        pairs = [(got, orc.cache_attention(k, v, q, n_past, True))]
    else:
        rows = (0, 31, 32, 1023, T - 33, T - 32, T - 1)
        pairs = [(got[t], orc.cache_attention(k[:, :n_past + t + 1], v[:, :n_past + t + 1], q[t:t + 1], n_past + t, True)[0])
                 for t in rows]
    for a, b in pairs:
        d = a.astype(np.float64) - b
        assert np.abs(d).max() <= 2e-3 and np.linalg.norm(d) <= 1e-3 * np.linalg.norm(b), np.abs(d).max()
