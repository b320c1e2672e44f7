"""Prompt projections (gemm_prefill.hip) through the decoder: one layer at prompt lengths around the edges of the
token tiles (32 rows), the K-slice plans and the row kernels, with f32 weights and with bf16 copies."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (2, 31, 32, 33, 63, 64, 65, 96, 97, 156, 160, 161, 255, 257, 300)


@pytest.fixture(scope="module", autouse=True)
def _gpu(qa):
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"


def _decoder(qa, model, max_seq, f32_weights):
    old = os.environ.pop("QA_WEIGHTS_F32", None)
    if f32_weights:
        os.environ["QA_WEIGHTS_F32"] = "1"
    try:
        return qa.Decoder(model, 1, max_seq, qa.QA_CACHE_F32)
    finally:
        os.environ.pop("QA_WEIGHTS_F32", None)
        if old is not None:
            os.environ["QA_WEIGHTS_F32"] = old


@pytest.mark.parametrize("bf16", [False, True], ids=["f32-weights", "bf16-copies"])
@pytest.mark.parametrize("cached", [False, True], ids=["nocache", "cached"])
def test_layer_matches_oracle(qa, orc, bf16, cached):
    """Four projections in sequence, each a sum of at most 3072 products (exact, or within 2^-24 on f32 weights): two orders
    of an f32 sum of n terms differ by about sqrt(n) 2^-24 = 3.3e-6 of the result, so a layer by at most 1.4e-5
    (relative 2-norm)."""
    model = qa.Model(qa.QWEN3_ASR_0_6B, n_layers=1, bf16=bf16)
    om = orc.OracleModel.from_product_model(model)
    x = qa.prompt_input(model, max(LENGTHS) - 10, 10)
    with _decoder(qa, model, max(LENGTHS), False) as dec:
        assert dec.weights_bf16 == bf16
        for T in LENGTHS:
            print(f"prompt length {T}", flush=True)
            if cached:
                got = dec.layer_forward(0, x[:T], 0)
                ref = om.layer_forward_cached(0, x[:T], 0, om.cache(max(LENGTHS), False))
            else:
                got = dec.layer_forward_nocache(0, x[:T])
                ref = om.layer_forward_nocache(0, x[:T])
            d = got.astype(np.float64) - ref
            assert np.linalg.norm(d) <= 1.4e-5 * np.linalg.norm(ref), (T, np.linalg.norm(d) / np.linalg.norm(ref))


@pytest.mark.parametrize("T", [2, 33, 100, 156, 300, 640, 1037, 2100])
def test_three_part_weights_equal_bf16_copies(qa, T):
    """f32 weights that hold bf16 values: their mid and lo parts add exact zeros, so the three-part GEMM gives the
    bits of the GEMM on the bf16 copies, whatever the plan (2100 rows: 256 columns per workgroup against 128).  Up to 32
    rows f32 weights do not run it."""
    model = qa.Model(qa.QWEN3_ASR_0_6B, n_layers=1, bf16=True)
    x = qa.prompt_input(model, T - 1, 1)
    out = []
    for f32_weights in (False, True):
        with _decoder(qa, model, T, f32_weights) as dec:
            assert dec.weights_bf16 == (not f32_weights)
            out.append(dec.layer_forward(0, x, 0))
    assert np.isfinite(out[0]).all()
    if T <= 32:   # the skinny f32 GEMM: another order of the same sums, as above
        d = out[1].astype(np.float64) - out[0]
        assert np.linalg.norm(d) <= 1.4e-5 * np.linalg.norm(out[0])
        return
    np.testing.assert_array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


@pytest.mark.parametrize("T", [2, 17, 32, 33])
def test_f32_weights_up_to_32_rows_read_the_f32_weights(qa, T):
    """Up to 32 positions the f32 rows are the shorter read (4 bytes per weight against 6): the copies change no bit."""
    model = qa.Model(qa.QWEN3_ASR_0_6B, n_layers=1)
    x = qa.prompt_input(model, T - 1, 1)
    out = []
    for copies in ("1", "0"):
        os.environ["QA_PROMPT_COPIES"] = copies
        try:
            with qa.Decoder(model, 1, 300, qa.QA_CACHE_F32) as dec:
                dec.layer_forward(0, qa.prompt_input(model, 299, 1), 0)    # activations for longer prompts too
                out.append(dec.layer_forward(0, x, 0))
        finally:
            del os.environ["QA_PROMPT_COPIES"]
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32)) == (T <= 32)
    d = out[1].astype(np.float64) - out[0]
    assert np.linalg.norm(d) <= 1.4e-5 * np.linalg.norm(out[0])
