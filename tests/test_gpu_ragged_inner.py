"""Products of at most 64 rows whose inner extent is no multiple of four: what lies behind it in memory is NaN and reaches no result."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def device(hip, a):
    p = C.c_void_p()
    assert hip.dali_hip_malloc(C.byref(p), a.nbytes) == 0
    assert hip.dali_hip_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), a.nbytes) == 0
    return p


# inner extents around the vectors, trips of 16 and groups of 64 values of a wave, one share and many; rows around the tiles of 16
@pytest.mark.parametrize("K", [65, 66, 67, 127, 129, 254, 257, 513, 1023, 4097, 15299])
@pytest.mark.parametrize("M,N", [(1, 2049), (7, 4096), (16, 3001), (17, 2048), (33, 2050), (64, 2100)])
@pytest.mark.parametrize("tb", [0, 1])
def test_at_most_64_rows(gpu, rng, M, N, K, tb):
    hip = gpu
    if K > 5000:
        N = 1025 + N % 4
    a, b = rng.randint(-8, 9, (M, K)).astype(np.float32), rng.randint(-8, 9, (K, N)).astype(np.float32)
    for pad in (0, 3):  # without: the next row's values follow a row, and nothing the last one
        lda, ldb = K + pad, (K if tb else N) + pad
        ap, bp = np.full((M, lda), np.nan, np.float32), np.full((N if tb else K, ldb), np.nan, np.float32)
        ap[:, :K], bp[:, :K if tb else N] = a, b.T if tb else b
        if pad == 0 and M > 1:
            ap[1, 0] = np.nan  # right behind the first row
        c = rng.randint(-8, 9, (M, N + 1)).astype(np.float32)
        d = [device(hip, v) for v in (ap, bp, c)]
        try:
            assert hip.dali_hip_sgemm(tb, 0, N, M, K, 1.0, d[1], ldb, d[0], lda, 2.0, d[2], N + 1) == 0, hip.dali_hip_last_error()
            out = np.empty_like(c)
            assert hip.dali_hip_memcpy_d2h(out.ctypes.data_as(C.c_void_p), d[2], out.nbytes) == 0
        finally:
            for p in d:
                hip.dali_hip_free(p)
        want = a.astype(np.float64) @ b + 2.0 * c[:, :N]  # whole numbers below 2^24: exact in any order
        rows = np.ones(M, bool)
        if pad == 0 and M > 1:
            rows[1] = False
            assert np.isnan(out[1, :N]).all()
        assert np.array_equal(out[rows, :N], want[rows])
        assert np.array_equal(out[:, N], c[:, N])


# more than 32 rows: either side of the lines between the streamed form and the tiles (rows, column blocks, shares, alignment of the right operand's rows)
@pytest.mark.parametrize("M,N", [(48, 4001), (49, 4001), (64, 4000), (33, 9601), (49, 9601), (48, 12000), (64, 12001), (49, 19265), (64, 24513)])
@pytest.mark.parametrize("K", [97, 191, 201, 255, 257, 321, 451, 513, 701, 1201, 1501])
@pytest.mark.parametrize("tb", [0, 1])
def test_33_to_64_rows(gpu, rng, M, N, K, tb):
    test_at_most_64_rows(gpu, rng, M, N, K, tb)
