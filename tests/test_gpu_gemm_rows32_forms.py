"""The forms of the 32-row projection GEMM at the edges of their rules, against float64: two 24-row tiles per workgroup
(SwiGLU of 8193 to 12288 weight rows) and the 32-row tiles on either side, 8 waves with fewer K blocks than waves, merged
K slices of row counts that are no multiple of a store, and outputs that are not 16-byte aligned."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.float32(1e-6)


def _launch(qa, b16, w, x, y, offset, accumulate, norm, stats, swiglu):
    """One call; y goes to the device `offset` floats behind an aligned address and comes back with the statistics."""
    out_dim, in_dim = w.shape
    rows = x.shape[0]
    d_w = qa.DeviceArray.from_numpy((w.view(np.uint32) >> 16).astype(np.uint16) if b16 else w)
    fn = qa.lib.qa_gemm_rows_fused_bf16 if b16 else qa.lib.qa_gemm_rows_fused
    d_x = qa.DeviceArray.from_numpy(x)
    buf = np.full(y.size + offset + 8, -7.0, np.float32)
    buf[offset:offset + y.size] = y.ravel()
    d_y = qa.DeviceArray.from_numpy(buf)
    d_nw = d_st = None
    parts = 0
    if norm is not None:
        parts = (in_dim + 31) // 32
        st = np.zeros((parts, 32))
        st[:, :rows] = np.square(x.astype(np.float64)).reshape(rows, parts, 32).sum(2).T
        d_nw, d_st = qa.DeviceArray.from_numpy(norm), qa.DeviceArray.from_numpy(st)
    d_so = qa.DeviceArray(((out_dim + 31) // 32, 32), np.float64) if stats else None
    wsb = qa.lib.qa_gemm_rows_workspace_bytes(out_dim, in_dim, rows)
    ws = qa.DeviceArray.from_numpy(np.zeros(wsb, np.uint8))
    ptr = lambda a: a.ptr if a is not None else None
    y_ptr = type(d_y.ptr)(d_y.ptr.value + 4 * offset)
    qa.check(fn(d_w.ptr, out_dim, in_dim, d_x.ptr, rows, y_ptr, accumulate, ptr(d_nw), ptr(d_st), parts, EPS, ptr(d_so),
                swiglu, ws.ptr, wsb, None))
    qa.synchronize()
    got = d_y.numpy()
    # nothing outside the rows of Y is written
    assert (got[:offset] == -7.0).all() and (got[offset + y.size:] == -7.0).all()
    return got[offset:offset + y.size].reshape(y.shape), d_so.numpy() if stats else None


def _bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


def _normed(x, nw):
    ss = np.square(x.astype(np.float64)).sum(1)
    scale = (np.float32(1.0) / np.sqrt((ss / x.shape[1]).astype(np.float32) + EPS)).astype(np.float32)
    return ((x * scale[:, None]).astype(np.float32) * nw[None, :]).astype(np.float32)


def _bound(x, w):
    # f32 sums of K products in at most K / 16 + 16 steps of one rounding each (2^-24 of the running sum, which is at
    # most the sum of magnitudes), twice for the two accumulators, and the f32 rounding of the inputs' normalisation
    k = x.shape[1]
    return (2 * (k / 16 + 16) + 4) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T)


@pytest.mark.parametrize("b16", [False, True])
@pytest.mark.parametrize("out_dim,in_dim,rows,offset", [
    (8192, 64, 32, 0), (8224, 64, 31, 0), (8256, 128, 1, 0), (12288, 576, 32, 0), (12288, 64, 9, 1), (12320, 64, 5, 0)])
def test_swiglu_forms(qa, b16, out_dim, in_dim, rows, offset):
    rng = np.random.default_rng(out_dim + in_dim + rows)
    w = _bf16(rng.standard_normal((out_dim, in_dim)) * 0.05)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    nw = (1.0 + 0.1 * rng.standard_normal(in_dim)).astype(np.float32)
    print(f"swiglu {out_dim}x{in_dim} rows={rows} offset={offset} bf16={b16}", flush=True)
    half = out_dim // 2
    y, _ = _launch(qa, b16, w, x, np.zeros((rows, half), np.float32), offset, 0, nw, False, 1)
    xn = _normed(x, nw)
    gu = xn.astype(np.float64) @ w.astype(np.float64).T
    g, u = gu[:, :half], gu[:, half:]
    b = _bound(xn, w)
    # |d silu| <= 1.1, |silu(g)| <= |g|; expf, the division and the two products round once each
    tol = 1.1 * b[:, :half] * np.abs(u) + np.abs(g) * b[:, half:] + 6 * 2.0 ** -24 * np.abs(g * u) + 1e-30
    assert (np.abs(y - g / (1.0 + np.exp(-g)) * u) <= tol).all()


@pytest.mark.parametrize("b16", [False, True])
@pytest.mark.parametrize("out_dim,in_dim,rows,offset", [
    (1024, 2048, 32, 0), (1024, 2048, 3, 1), (1001, 2048, 32, 0), (1001, 1024, 17, 3), (40, 512, 7, 0), (96, 64, 32, 0),
    (33, 4096, 1, 0), (8256, 128, 32, 0), (4096, 320, 20, 2)])
def test_accumulate_and_statistics_forms(qa, b16, out_dim, in_dim, rows, offset):
    rng = np.random.default_rng(out_dim * 5 + in_dim + rows)
    w = _bf16(rng.standard_normal((out_dim, in_dim)) * 0.05)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    y0 = rng.standard_normal((rows, out_dim)).astype(np.float32)
    print(f"accumulate {out_dim}x{in_dim} rows={rows} offset={offset} bf16={b16}", flush=True)
    y, st = _launch(qa, b16, w, x, y0, offset, 1, None, True, 0)
    ref = y0 + x.astype(np.float64) @ w.astype(np.float64).T
    assert (np.abs(y - ref) <= _bound(x, w) + 2.0 ** -24 * np.abs(ref)).all()
    pad = np.zeros((rows, st.shape[0] * 32))
    pad[:, :out_dim] = y.astype(np.float64)
    want = np.square(pad).reshape(rows, -1, 32).sum(2).T
    np.testing.assert_allclose(st[:, :rows], want, rtol=1e-12, atol=0)   # 32 squares summed in double


def test_workspace_covers_fewer_rows(qa):
    """A workspace sized for more rows serves any smaller row count of the same shape."""
    for out_dim, in_dim in ((40, 512), (1001, 2048), (1024, 3072)):
        sizes = [qa.lib.qa_gemm_rows_workspace_bytes(out_dim, in_dim, r) for r in (1, 5, 32, 33, 64)]
        assert sizes == sorted(sizes)
