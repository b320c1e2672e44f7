"""The three-part bf16 operands of the prompt projections (split3.hpp, gemm_prefill.hip) where single products show:
infinities, and mantissas whose parts are as large as they get."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(qa):
    assert qa.device_count() > 0, "no HIP device: GPU tests need the MI355X"


def _tensor(model, name):
    """A layer-0 tensor of a synthetic model, in place."""
    rows = {"attn_q": 2048, "attn_k": 1024, "attn_v": 1024, "attn_output": model.cfg.hidden,
            "ffn_gate": model.cfg.intermediate, "ffn_up": model.cfg.intermediate, "ffn_down": model.cfg.hidden}
    t = model.tensor(f"text.blk.0.{name}.weight")
    return t.reshape(rows[name], -1) if name in rows else t


@pytest.mark.parametrize("bf16", [False, True], ids=["f32-weights", "bf16-copies"])
@pytest.mark.parametrize("T", [40, 156, 300])
def test_infinite_input_keeps_the_sign_of_its_weight(qa, T, bf16):
    """silu(gate) * up overflows in column 5: every output is its down weight's sign times infinity, as in an f32 GEMM,
    also where the weight's smaller parts are zero (the first 64 rows: bf16 values)."""
    model = qa.Model(qa.QWEN3_ASR_0_6B, n_layers=1, vocab=4096, bf16=bf16)
    for name, w in (("ffn_gate", 1.0), ("ffn_up", 3.0e38)):
        m = _tensor(model, name)
        m[5] = 0.0
        m[5, 0] = (np.array([w], np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)[0]
    down = _tensor(model, "ffn_down")
    down[:64, 5] = (down[:64, 5].copy().view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    x = qa.prompt_input(model, T - 1, 1)
    x[:, 0] = 30.0                                    # 20 or so after the RMSNorm: 20 x 3e38 overflows
    with qa.Decoder(model, 1, T, qa.QA_CACHE_F32) as dec:
        assert dec.weights_bf16 == bf16
        got = dec.layer_forward(0, x, 0)
    want = np.broadcast_to(np.copysign(np.float32(np.inf), down[:, 5]), got.shape)
    assert (down[:, 5] != 0).all()
    np.testing.assert_array_equal(got, want)
