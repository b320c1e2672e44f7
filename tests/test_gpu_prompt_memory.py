"""The prompt copies of f32 weights (6 bytes per weight) are an option: what a decoder cannot do without comes first, and
they are given back when it needs the memory later."""
import contextlib
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS, VOCAB, CAPACITY = 4, 4096, 32768
MIB = 1 << 20


def _free(qa):
    free, total = C.c_size_t(), C.c_size_t()
    assert qa.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def _left(qa, nbytes):
    """All device memory but `nbytes` taken."""
    held = []
    try:
        while (more := _free(qa) - nbytes) > 4 * MIB:
            held.append(qa.DeviceArray((min(more, 16 << 30),), np.uint8, zero=False))
        print(f"{len(held)} blocks held, {_free(qa) // MIB} MiB left", flush=True)
        yield
    finally:
        del held


def _sizes(qa):
    z = qa.QWEN3_ASR_0_6B
    params = LAYERS * (4096 * z.hidden + z.hidden * 2048 + 3 * z.hidden * z.intermediate)
    lay = qa.KvLayout(LAYERS, 1, 8, 128, CAPACITY, qa.QA_CACHE_F32)
    return 4 * (params + VOCAB * z.hidden), 6 * params, qa.lib.qa_kv_cache_bytes(C.byref(lay))


@pytest.fixture(scope="module")
def model(qa):
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"
    return qa.Model(qa.QWEN3_ASR_0_6B, n_layers=LAYERS, vocab=VOCAB)


@pytest.fixture(scope="module")
def reference(qa, model):
    """Logits of the same prompts without the copies."""
    x = qa.prompt_input(model, 1990, 10)
    os.environ["QA_PROMPT_COPIES"] = "0"
    try:
        with qa.Decoder(model, 1, 2048, qa.QA_CACHE_F32) as dec:
            return x, {T: dec.forward(x[:T], 0) for T in (40, 2000)}
    finally:
        del os.environ["QA_PROMPT_COPIES"]


def _close(got, ref):
    # four layers, each four projections of at most 3072 products in another order (3.3e-6 a projection's sum)
    return np.linalg.norm(got.astype(np.float64) - ref) <= 5.6e-5 * np.linalg.norm(ref)


def test_cache_that_fits_beside_the_weights(qa, model, reference):
    weights, copies, cache = _sizes(qa)
    x, logits = reference
    slack = 250 * MIB
    assert slack < copies
    with _left(qa, weights + cache + slack):
        with qa.Decoder(model, 1, CAPACITY, qa.QA_CACHE_F32) as dec:
            assert _close(dec.forward(x[:40], 0), logits[40])


def test_copies_make_room_for_a_long_prompt(qa, model, reference):
    x, logits = reference
    with qa.Decoder(model, 1, 2048, qa.QA_CACHE_F32) as dec:
        assert _close(dec.forward(x[:40], 0), logits[40])
        with _left(qa, 150 * MIB):
            assert _close(dec.forward(x, 0), logits[2000])
        np.testing.assert_array_equal(dec.forward(x[:40], 0), logits[40])   # without the copies from here on


def test_copies_make_room_for_a_cache_upload(qa, model, reference):
    x, logits = reference
    rows = 16384
    with qa.Decoder(model, 1, rows + 64, qa.QA_CACHE_F32) as dec:
        kv = np.zeros((LAYERS, 8, rows, 128), np.float32)
        with _left(qa, 32 * MIB):
            dec.fill_cache(0, kv, kv, rows)
        assert dec.cur_len(0) == rows
        np.testing.assert_array_equal(dec.forward(x[:40], 0), logits[40])
