"""Products of odd sizes and leading dimensions, from the smallest that go through the bf16 matrix cores on, in the four orders of operands."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def product(hip, a, b, ta, tb):
    (K, M), N = (a.shape if ta else a.shape[::-1]), (b.shape[0] if tb else b.shape[1])
    out, d = np.full((M, N), 7.0, np.float32), []
    for x in (a, b, out):
        p = C.c_void_p()
        assert hip.dali_hip_malloc(C.byref(p), x.nbytes) == 0 and hip.dali_hip_memcpy_h2d(p, x.ctypes.data_as(C.c_void_p), x.nbytes) == 0
        d.append(p)
    try:
        assert hip.dali_hip_sgemm(tb, ta, N, M, K, 1.0, d[1], b.shape[1], d[0], a.shape[1], 0.0, d[2], N) == 0, hip.dali_hip_last_error()
        assert hip.dali_hip_memcpy_d2h(out.ctypes.data_as(C.c_void_p), d[2], out.nbytes) == 0
    finally:
        for p in d:
            hip.dali_hip_free(p)
    return out


# around the line: taken in one share, in several, part tiles and part slabs of one row, column and value; too small
@pytest.mark.parametrize("M,N,K", [(1023, 1025, 1027), (4099, 515, 259), (129, 9999, 515), (2001, 2003, 301), (513, 513, 8191), (172, 30001, 425), (300, 20001, 67), (700, 701, 703), (200, 2001, 129)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_odd_sizes(gpu, ta, tb, M, N, K):
    rng = np.random.RandomState(M + N + K)
    for whole in (True, False):
        a, b = ((rng.randint(-15, 16, s) if whole else rng.randn(*s)).astype(np.float32) for s in ((M, K), (K, N)))
        got = product(gpu, np.ascontiguousarray(a.T) if ta else a, np.ascontiguousarray(b.T) if tb else b, ta, tb)
        want = a.astype(np.float64) @ b.astype(np.float64)
        if whole:
            assert np.array_equal(got, want)  # sums below 2^24
        else:
            # an fp32 product in any order: a partial sum that grows as sqrt(k) is rounded at most K / 4 times (instructions of four k)
            assert np.linalg.norm(got - want) <= (np.sqrt(K / 4.0) + 4.0) * 2.0 ** -24 * np.linalg.norm(want)
