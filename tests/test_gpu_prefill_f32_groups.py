"""f32 prefill attention at the edges of its key groups: query blocks of 16, 32 and 64, key tiles of 32 shared out over
four, two and one groups of waves, and the prompt lengths where the number of groups changes."""
import ctypes as C
import os

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
