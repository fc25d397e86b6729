"""The persistent LSTM recurrence with the bias apart: the same bits as with the bias added to the input half beforehand."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one to 64 rows in LDS (values awaited up to 32 rows, barriers above), sizes whose weights sit in registers; one step and many
@pytest.mark.parametrize("T,B,H", [(1, 1, 256), (9, 1, 1024), (33, 8, 1024), (12, 8, 256), (5, 9, 768), (7, 16, 512), (6, 17, 1024), (6, 32, 512), (4, 33, 256), (3, 64, 1024), (5, 7, 320), (3, 96, 640)])
def test_bias_apart(gpu, rng, T, B, H):
    hip = gpu
    pre, U = rng.randn(T, B, 4 * H).astype(np.float32), (rng.randn(H, 4 * H) / np.sqrt(H)).astype(np.float32)
    bias, h0, c0 = rng.randn(4 * H).astype(np.float32), rng.randn(B, H).astype(np.float32), rng.randn(B, H).astype(np.float32)

    def device(a):
        p = C.c_void_p()
        assert hip.dali_hip_malloc(C.byref(p), a.nbytes) == 0
        assert hip.dali_hip_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), a.nbytes) == 0
        return p
    hs, c = np.zeros((T, B, H), np.float32), np.zeros((B, H), np.float32)
    d = {k: device(v) for k, v in dict(pre=pre, both=pre + bias, U=U, bias=bias, h0=h0, c0=c0, hs=hs, c=c).items()}

    def run(first, b):
        assert hip.dali_hip_lstm_recurrent_persistent_bias(T, B, H, d[first], b, d["U"], 4 * H, d["h0"], d["c0"], d["hs"], d["c"]) == 0, hip.dali_hip_last_error()
        out = np.empty_like(hs), np.empty_like(c)
        for o, k in zip(out, ("hs", "c")):
            assert hip.dali_hip_memcpy_d2h(o.ctypes.data_as(C.c_void_p), d[k], o.nbytes) == 0, hip.dali_hip_last_error()
        return out
    try:
        want = run("both", None)
        assert np.isfinite(want[0]).all() and np.abs(want[0]).max() > 0
        for _ in range(3):
            got = run("pre", d["bias"])
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert hip.dali_hip_lstm_recurrent_persistent_bias(T, B, H, d["pre"], d["hs"], d["U"], 4 * H, d["h0"], d["c0"], d["hs"], d["c"]) != 0  # the bias inside hs
    finally:
        for p in d.values():
            hip.dali_hip_free(p)


# weights in registers: one and two 16-column tiles, one and two row tiles to a turn, one to eight turns, the last one partly filled
@pytest.mark.parametrize("T,B,H", [(3, 8, 640), (4, 64, 640), (3, 17, 320), (3, 32, 2048), (3, 33, 1536), (2, 128, 1024), (2, 100, 64), (3, 1, 1920)])
def test_bias_apart_with_weights_in_registers(gpu, rng, T, B, H):
    test_bias_apart(gpu, rng, T, B, H)
