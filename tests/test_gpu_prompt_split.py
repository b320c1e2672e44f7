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


def _cached_v(qa, dec, T):
    """V rows [T][1024] of layer 0 of a decoder's f32 cache."""
    address, lay = dec.cache()
    host = np.empty((2, lay.n_kv_heads, lay.max_seq, 128), np.float32)
    qa.check(qa.lib.qa_copy_to_host(host.ctypes.data, address, host.nbytes))
    return host[1, :, :T].transpose(1, 0, 2).reshape(T, -1)


@pytest.mark.parametrize("size", ["0.6B", "1.7B"])
@pytest.mark.parametrize("T", [33, 64, 96, 130, 156, 200, 300, 1100])
def test_single_products_of_f32_weights(qa, size, T):
    """One weight per row of v, so that each output is one product of six part products: what is left out is at most
    2^-24 of it, and the sums round once by at most 2^-23 (a sum of parts that is below 2^-7 of the whole adds less than a
    tenth of that).  Mantissas are those whose parts are largest beside random ones; a part product that is missing is
    2^-16 of the result."""
    z = {"0.6B": qa.QWEN3_ASR_0_6B, "1.7B": qa.QWEN3_ASR_1_7B}[size]
    model = qa.Model(z, n_layers=1, vocab=4096)
    rng = np.random.default_rng(T)

    def values(n):
        low = rng.choice(np.array([0xFFFF, 0x7FFF, 0x8000, 0x8001, 0x0001, 0xFF7F, 0x0080, 0xFF80], np.uint32), n)
        low = np.where(rng.random(n) < 0.3, rng.integers(0, 1 << 16, n, dtype=np.uint32), low)
        top = np.where(rng.random(n) < 0.5, 0, rng.integers(0, 128, n)).astype(np.uint32)
        exponent = rng.integers(124, 131, n, dtype=np.uint32)
        return (rng.integers(0, 2, n, dtype=np.uint32) << 31 | exponent << 23 | top << 16 | low).view(np.float32)

    at = np.arange(1024) * (z.hidden // 1024) + np.arange(1024) % (z.hidden // 1024)
    w = values(1024)
    # past the largest bf16, where rounding would give infinity
    w[:4] = np.array([0x7F7FFFFF, 0xFF7FFFFF, 0x7F7F8000, 0x7F7F7FFF], np.uint32).view(np.float32)
    wv = _tensor(model, "attn_v")
    wv[:] = 0.0
    wv[np.arange(1024), at] = w
    nw = values(z.hidden)
    nw[at[:4]] *= np.float32(2.0 ** -20)
    model.tensor("text.blk.0.attn_norm.weight")[:] = nw
    x = rng.choice(np.array([-1.0, 1.0], np.float32), (T, z.hidden))
    # the RMSNorm of rows of ones: mean square 1, float scale, (x scale) w
    scale = np.float32(1.0) / np.sqrt(np.float32(1.0) + np.float32(model.cfg.rms_norm_eps))
    xn = (x * scale).astype(np.float32) * nw
    print(f"single products {size} T={T}", flush=True)
    with qa.Decoder(model, 1, T, qa.QA_CACHE_F32) as dec:
        assert not dec.weights_bf16
        dec.layer_forward(0, x, 0)
        got = _cached_v(qa, dec, T)
    want = xn[:, at].astype(np.float64) * w
    off = np.abs(got - want) / np.abs(want) * 2.0 ** 24
    print(f"  largest error {off.max():.2f} x 2^-24, mean of the signed error towards zero "
          f"{((np.abs(want) - np.abs(got)) / np.abs(want)).mean() * 2.0 ** 24:.3f} x 2^-24", flush=True)
    assert off.max() <= 3.2


def _layer64(model, x, T):
    """The layer in 64 bits, from position 0 (text-decoder.cpp:265-345), and its v."""
    H, eps, theta = model.cfg.hidden, model.cfg.rms_norm_eps, model.cfg.rope_theta
    mat = lambda name: _tensor(model, name).astype(np.float64)
    vec = lambda name: model.tensor(f"text.blk.0.{name}.weight").astype(np.float64)
    rms = lambda a, w: a / np.sqrt(np.square(a).mean(-1, keepdims=True) + eps) * w
    x = x.astype(np.float64)
    h = rms(x, vec("attn_norm"))
    angle = np.arange(T)[:, None] * theta ** (-np.arange(64) / 64.0)
    c, s = np.cos(angle), np.sin(angle)

    def rope(a):                                      # [heads, T, 128]
        lo, hi = a[..., :64], a[..., 64:]
        return np.concatenate([lo * c - hi * s, hi * c + lo * s], -1)

    heads = lambda name: (h @ mat(name).T).reshape(T, -1, 128).transpose(1, 0, 2)
    q, k, v = rope(rms(heads("attn_q"), vec("attn_q_norm"))), rope(rms(heads("attn_k"), vec("attn_k_norm"))), heads("attn_v")
    out = np.empty((T, 2048))
    for i in range(16):
        sc = q[i] @ k[i // 2].T / np.sqrt(128.0)
        sc[np.triu_indices(T, 1)] = -np.inf
        p = np.exp(sc - sc.max(1, keepdims=True))
        out[:, 128 * i:128 * i + 128] = p @ v[i // 2] / p.sum(1, keepdims=True)
    x = x + out @ mat("attn_output").T
    h = rms(x, vec("ffn_norm"))
    g = h @ mat("ffn_gate").T
    y = x + (g / (1.0 + np.exp(-g)) * (h @ mat("ffn_up").T)) @ mat("ffn_down").T
    return y, v.transpose(1, 0, 2).reshape(T, -1)


@pytest.mark.parametrize("bf16", [False, True], ids=["f32-weights", "bf16-copies"])
@pytest.mark.parametrize("size,T", [("0.6B", 40), ("0.6B", 156), ("1.7B", 52), ("1.7B", 156), ("1.7B", 300), ("1.7B", 700)])
def test_layer_without_residual_against_64_bits(qa, size, T, bf16):
    """o and down are scaled up, so that the residual is 1/100 of each sum and hides nothing.  The error is that of four
    projections in a row: f32 sums over 2048 k are off by 0.7e-6 and over 6144 by 1.2e-6 at most, q|k|v, o, gate and up
    (whose errors both go into down) and down together 2.0e-6, and a factor 1.3 for the seed.  A part product left out of
    any one of them moves the output by 1.0e-5; rounding towards one side in the sums is an error that all tokens share,
    which the attention's average over 700 tokens keeps (2.9e-6), and shows in the mean of v: 1e-7 of its root mean square
    in every row, where independent errors leave less than 2e-9."""
    z = {"0.6B": qa.QWEN3_ASR_0_6B, "1.7B": qa.QWEN3_ASR_1_7B}[size]
    model = qa.Model(z, n_layers=1, vocab=4096, bf16=bf16)
    _tensor(model, "attn_output")[:] *= 64.0
    _tensor(model, "ffn_down")[:] *= 8192.0
    x = qa.prompt_input(model, T - 1, 1)
    print(f"layer {size} T={T} bf16={bf16}", flush=True)
    with qa.Decoder(model, 1, T, qa.QA_CACHE_F32) as dec:
        assert dec.weights_bf16 == bf16
        got = dec.layer_forward(0, x, 0)
        v = _cached_v(qa, dec, T)
    want, want_v = _layer64(model, x, T)
    bias = (v - want_v).mean() / np.sqrt(np.square(want_v).mean())
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"  {off:.2e}, mean of v {bias:.1e}", flush=True)
    assert off <= 2.6e-6 and abs(bias) <= 1.0e-8
