"""Large fp32 products, which go through the bf16 matrix cores with every value cut in three (dali_amd/csrc/sgemm_split.hip),
against numpy in double precision."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(hip, a):
    p = C.c_void_p()
    assert hip.dali_hip_malloc(C.byref(p), a.nbytes) == 0
    assert hip.dali_hip_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), a.nbytes) == 0
    return p


def _product(hip, A, B, ta, tb, alpha=1.0, beta=0.0, pad=0, C0=None):
    """alpha * op(A) . op(B) + beta * C0 through the column-major entry point, operands stored with `pad` NaN behind each row."""
    K, M = A.shape if ta else A.shape[::-1]
    N = B.shape[0] if tb else B.shape[1]
    pa, pb = (np.ascontiguousarray(np.pad(x, ((0, 0), (0, pad)), constant_values=np.nan)) for x in (A, B))
    out = np.full((M, N + pad), 7.0, np.float32)
    if C0 is not None:
        out[:, :N] = C0
    da, db, dc = (_dev(hip, x) for x in (pa, pb, out))
    try:
        assert hip.dali_hip_sgemm(int(tb), int(ta), N, M, K, alpha, db, pb.shape[1], da, pa.shape[1], beta, dc, N + pad) == 0
        assert hip.dali_hip_memcpy_d2h(out.ctypes.data_as(C.c_void_p), dc, out.nbytes) == 0
    finally:
        for p in (da, db, dc):
            hip.dali_hip_free(p)
    assert np.all(out[:, N:] == 7.0)
    return out[:, :N]


def _tolerance(K):
    # Relative error in the 2-norm for operands of random sign. Each of the K / 32 additions of a chain's sum rounds a partial sum
    # that grows as sqrt(k): together at most sqrt(K / 32) half units, and the chain itself four. (Measured: about a third.)
    return (np.sqrt(K / 32.0) + 4.0) * 2.0 ** -24


def _check(got, ref, K):
    assert np.linalg.norm(got - ref) <= _tolerance(K) * np.linalg.norm(ref)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
# whole tiles and slabs; a tile row with one row, a slab with one value; odd rows and a slab one short; few rows in many shares; few slabs
@pytest.mark.parametrize("M,N,K,pad", [(2048, 2048, 2048, 0), (1985, 1923, 2049, 0), (2047, 2047, 2047, 3), (255, 1023, 30001, 1), (1023, 32001, 257, 0)])
def test_sizes(gpu, ta, tb, M, N, K, pad):
    rng = np.random.RandomState(M + N + K)
    a, b = rng.randn(M, K).astype(np.float32), rng.randn(K, N).astype(np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    _check(_product(gpu, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb, pad=pad), ref, K)


def test_whole_numbers_are_exact_and_alpha_beta(gpu):
    rng = np.random.RandomState(5)
    a, b, c = (rng.randint(-31, 32, s).astype(np.float32) for s in ((2040, 2050), (2050, 2040), (2040, 2040)))
    ref = a.astype(np.float64) @ b.astype(np.float64)  # below 2^24: every sum is exact
    assert np.array_equal(_product(gpu, a, b, 0, 0), ref)
    assert np.array_equal(_product(gpu, a, b, 0, 0, alpha=0.5, beta=2.0, C0=c), 0.5 * ref + 2.0 * c)


@pytest.mark.parametrize("shape", [(2040, 2040, 2050), (200, 1000, 32000)])
def test_values_that_three_bf16_do_not_hold(gpu, shape):
    """Infinities, NaN and values next to the largest float: what the fp32 instructions make of them. Values whose last bits would lie
    below the smallest bf16: within the fp32 instructions' tolerance as well."""
    M, N, K = shape
    rng = np.random.RandomState(6)
    a, b = rng.randn(M, K).astype(np.float32), rng.randn(K, N).astype(np.float32)
    a[3, 17], a[5, K - 1], a[140, 40] = np.inf, -np.inf, np.nan
    b[K // 2, 900] = np.inf
    a[150, :] *= np.float32(2.0 ** -125)  # denormal in part
    a[151, :] *= np.float32(2.0 ** -112)
    a[152, 7] = np.finfo(np.float32).max
    b[7, :] *= np.float32(2.0 ** -20)
    with np.errstate(all="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    got = _product(gpu, a, b, 0, 0)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
    for m in (0, 150, 151, 152):
        # (row 150: its sums are denormal or close to it, where a float resolves 2^-149: each of the K roundings adds half of that at most)
        slack = 0.5 * 2.0 ** -149 * K * np.sqrt(N) if m == 150 else 0.0
        assert np.linalg.norm((got[m] - ref[m])[fin[m]]) <= _fp32_tolerance(K) * np.linalg.norm(ref[m][fin[m]]) + slack


def _fp32_tolerance(K):
    # rows that the fp32 instructions sum two values of k at a time: sqrt(K / 2) half units by the same reasoning
    return (np.sqrt(K / 2.0) + 4.0) * 2.0 ** -24


def _split_tolerance(K):
    """Relative error in the 2-norm that the split product stays within and the fp32 kernels, two values of k at a time, do not.
    Rounding a sum to 24 bits is off by up to half a unit, evenly: 2^-24 / sqrt(6) of it in the root mean square over its leading
    digits. n = K / 32 chains are added to a sum whose variance grows as j / n: sqrt((n + 1) / 2) such errors together; four for
    the chain's own roundings. Twice that."""
    return 2.0 * 2.0 ** -24 / np.sqrt(6.0) * np.sqrt((np.ceil(K / 32.0) + 1.0) / 2.0 + 4.0)


def _norm_ratio(got, ref):
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(4000, 3999, 512), (4097, 2999, 1025), (2000, 4001, 2041)])
def test_accuracy(gpu, ta, tb, M, N, K):
    """Closer to double precision than the fp32 kernels come: also that it was this path that was taken."""
    rng = np.random.RandomState(M + N + K)
    a, b = rng.randn(M, K).astype(np.float32), rng.randn(K, N).astype(np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    got = _product(gpu, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb)
    assert _norm_ratio(got, ref) <= _split_tolerance(K)
    got = _product(gpu, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb, alpha=-0.5, beta=1.0, C0=np.float32(ref))
    # (alpha * sum + beta * C: C0 is rounded once, and so is the result, which is half as large)
    assert _norm_ratio(got, 0.5 * ref) <= _split_tolerance(K) + 3 * 2.0 ** -24


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_single_products(gpu, ta, tb):
    """A diagonal left operand, mantissas at random: every result is one product. ml + lm + ll, which is left out, is at most
    (2^-24 + 2^-34) |a b|, the last rounding at most 2^-24, and the five sums of small products (below 2^-6 |a b|) lose at most a unit each."""
    M = N = K = 2048
    rng = np.random.RandomState(10)
    values = lambda *s: ((1.0 + rng.rand(*s)) * np.where(rng.rand(*s) < 0.5, -1.0, 1.0)).astype(np.float32)
    a, b = np.diag(values(M)), values(K, N)
    ref = np.diag(a).astype(np.float64)[:, None] * b.astype(np.float64)
    got = _product(gpu, a, b.T.copy() if tb else b, ta, tb)
    assert np.max(np.abs(got - ref) / np.abs(ref)) <= 2.0 ** -23 + 2.0 ** -34 + 5 * 2.0 ** -29
    # In the 2-norm: the rounding of a product of such values, 2.49e-8, and what is left out. m is even over 2^-8 and l over 2^-17 in
    # either direction: ml and lm 2^-25 / 3 each, over values of 7 / 3 in the root mean square. A twentieth more.
    assert _norm_ratio(got, ref) <= 1.05 * np.hypot(2.49e-8, np.sqrt(2.0) * 2.0 ** -25 / 3.0 / (7.0 / 3.0))
    # one operand a power of two: nothing is left out and nothing rounded
    a = np.diag(np.ldexp(1.0, rng.randint(-60, 60, M)).astype(np.float32))
    assert np.array_equal(_product(gpu, a, b.T.copy() if tb else b, ta, tb), np.diag(a)[:, None] * b)


def test_equal_operands(gpu):
    """What is left out of every product is largest, and of the same sign, for this value: 2^-24 of the sum."""
    M, N, K = 2048, 1920, 2048
    c = np.float32(1.0 + 2.0 ** -8 - 2.0 ** -17)
    got = _product(gpu, np.full((M, K), c), np.full((K, N), c), 0, 0)
    assert np.max(np.abs(got / (K * np.float64(c) ** 2) - 1.0)) <= 2.0 ** -24 + _split_tolerance(K)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_tiny_values_do_not_send_their_tile_to_the_fp32_instructions(gpu, ta, tb):
    """A few entries far below the others, as a softmax gradient has them, and whole strips of rows whose pieces are denormal."""
    M, N, K = 2048, 1920, 2050
    rng = np.random.RandomState(8)
    a, b = rng.randn(M, K).astype(np.float32), (rng.randn(K, N) * 2.0 ** 40).astype(np.float32)
    a[:, 5::61] *= np.float32(2.0 ** -116)
    powers = {128: -105, 256: -112, 384: -124, 512: -149 + 13}  # (the last: whole multiples of the smallest float)
    for m, p in powers.items():
        a[m:m + 128] = np.ldexp(rng.randn(128, K), p).astype(np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    got = _product(gpu, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb)
    for m in [0] + sorted(powers) + [640]:
        assert _norm_ratio(got[m:m + 128], ref[m:m + 128]) <= _split_tolerance(K), m


@pytest.mark.parametrize("bits", [(17, 2), (2, 17), (12, 7)])
@pytest.mark.parametrize("powers", [(0, 0), (-149, 100), (100, -149), (-130, 60), (-70, -60)])
def test_whole_numbers_of_several_pieces_are_exact(gpu, bits, powers):
    """Whole numbers that take two or three pieces, and the same as multiples of powers of two down to the smallest float."""
    M, N, K, chosen = 2048, 1920, 2048, 16
    rng = np.random.RandomState(9)
    a, b = (rng.randint(-2 ** n + 1, 2 ** n, s).astype(np.float64) for n, s in zip(bits, ((M, K), (K, N))))
    # sixteen terms a row, so that every sum is below 2^24 and exact
    a[~(np.argsort(rng.rand(M, K), axis=1) < chosen)] = 0.0
    ref = np.ldexp(a @ b, powers[0] + powers[1])
    a, b = (np.ldexp(x, p).astype(np.float32) for x, p in zip((a, b), powers))
    assert np.array_equal(_product(gpu, a, b, 0, 0), ref.astype(np.float32))


@pytest.mark.parametrize("fmt", ["NHWC", "NCHW"])
@pytest.mark.parametrize("n,side,cin,cout,window", [(16, 58, 64, 128, 3), (9, 61, 67, 130, 5)])
def test_convolution_terms_with_a_row_map(gpu, D, fmt, n, side, cin, cout, window):
    rng = np.random.RandomState(7)
    x = rng.randn(n, side, side, cin).astype(np.float32)
    w = (rng.randn(cout, window, window, cin) / np.sqrt(window * window * cin)).astype(np.float32)
    out = side - window + 1
    ref = np.zeros((n, out, out, cout))
    for i in range(window):
        for j in range(window):
            ref += x[:, i:i + out, j:j + out, :].astype(np.float64) @ w[:, i, j, :].astype(np.float64).T
    put = (lambda t: t) if fmt == "NHWC" else (lambda t: np.ascontiguousarray(t.transpose(0, 3, 1, 2)))
    got = D.op.conv2d(D.Array.from_numpy(put(x)), D.Array.from_numpy(put(w)), 1, 1, "valid", fmt).numpy()
    # (not every layout takes this path at every size: the bound of the fp32 instructions)
    assert np.linalg.norm(got - put(ref)) <= _fp32_tolerance(window * window * cin) * np.linalg.norm(ref)


def _check_specials(got, ref, K):
    """`ref` in double precision, or what the fp32 instructions make of sums that overflow there."""
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
    fin = np.isfinite(ref)
    assert np.linalg.norm(got[fin] - ref[fin]) <= _fp32_tolerance(K) * np.linalg.norm(ref[fin])


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("shape", [(2040, 4000, 1030), (200, 1000, 32007)])  # the second in shares
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-2.0, 0.5)])
def test_tiles_redone_with_the_fp32_instructions(gpu, ta, tb, shape, alpha, beta):
    M, N, K = shape
    rng = np.random.RandomState(11)
    a, b, c = (rng.randn(*s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    a[3, K - 1], a[5, 40], a[140, K - 9], a[M - 1, K // 2] = np.inf, -np.inf, np.nan, np.float32(2.0 ** 114)
    b[K // 3, N - 2] = -np.inf
    b[K // 2, 130] = np.float32(2.0 ** 13)  # 2^127 in the corner of its tile
    with np.errstate(all="ignore"):
        ref = alpha * (a.astype(np.float64) @ b.astype(np.float64)) + beta * c.astype(np.float64)
        ref = np.where(np.abs(ref) >= 2.0 ** 128, np.copysign(np.inf, ref), ref)
    got = _product(gpu, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb, alpha, beta, pad=1, C0=c)
    for rows in (slice(0, 128), slice(128, M - 1), slice(M - 1, M)):
        _check_specials(got[rows], ref[rows], K)


def test_convolution_accuracy(gpu, D):
    """As test_accuracy: closer to double precision than the kernel that the fp32 instructions have for several terms."""
    n, side, cin, cout, window = 16, 58, 64, 128, 3
    rng = np.random.RandomState(13)
    x, w = rng.randn(n, side, side, cin).astype(np.float32), rng.randn(cout, window, window, cin).astype(np.float32)
    out = side - window + 1
    ref = np.zeros((n, out, out, cout))
    for i in range(window):
        for j in range(window):
            ref += x[:, i:i + out, j:j + out, :].astype(np.float64) @ w[:, i, j, :].astype(np.float64).T
    got = D.op.conv2d(D.Array.from_numpy(x), D.Array.from_numpy(w), 1, 1, "valid", "NHWC").numpy()
    assert _norm_ratio(got, ref) <= _split_tolerance(window * window * cin)


@pytest.mark.parametrize("value", [np.inf, np.nan, 2.0 ** 120, 2.0 ** -130])
def test_convolution_of_special_values(gpu, D, value):
    """Three terms with overlapping rows and a row map: tiles that are redone walk the same terms; tiny values need none."""
    n, side, cin, cout, window = 16, 58, 64, 128, 3
    rng = np.random.RandomState(12)
    x = rng.randn(n, side, side, cin).astype(np.float32)
    for at in ((0, 0, 0, 0), (3, 20, 31, 7), (9, 57, 57, 63), (15, 56, 2, 30)):
        x[at] = value
    w = (rng.randn(cout, window, window, cin) / np.sqrt(window * window * cin)).astype(np.float32)
    out = side - window + 1
    ref = np.zeros((n, out, out, cout))
    with np.errstate(all="ignore"):
        for i in range(window):
            for j in range(window):
                ref += x[:, i:i + out, j:j + out, :].astype(np.float64) @ w[:, i, j, :].astype(np.float64).T
    got = D.op.conv2d(D.Array.from_numpy(x), D.Array.from_numpy(w), 1, 1, "valid", "NHWC").numpy()
    ordinary = np.abs(ref) < 2.0 ** 60  # (NaN is not)
    _check_specials(got[~ordinary], ref[~ordinary], window * window * cin)
    assert _norm_ratio(got[ordinary], ref[ordinary]) <= _fp32_tolerance(window * window * cin)


# (ta, tb, M, N, K, elements behind each row, whether the split product takes it): on either side of the rule's lines
_ROUTES = [
    (0, 0, 2048, 2048, 1024, 0, False), (1, 0, 2048, 2048, 512, 0, False), (0, 1, 1024, 1024, 4096, 0, False),  # the fp32 kernels' tiles fill the chip
    (0, 0, 2048, 2048, 4096, 0, True), (0, 1, 2048, 4096, 512, 0, True),
    (0, 0, 2048, 2048, 1024, 1, True),                                # their loads cannot write LDS
    (0, 1, 1920, 4096, 1030, 1, True), (0, 0, 1000, 1000, 1000, 0, False),
    (0, 0, 3072, 4096, 1024, 0, True), (1, 0, 4096, 5120, 256, 0, True), (1, 1, 3072, 4096, 256, 0, True),  # three and five tiles a compute unit
    (0, 0, 200, 1000, 16000, 0, True), (0, 0, 256, 4096, 1024, 0, False),  # shares
    (0, 0, 64, 32000, 1024, 0, False), (0, 0, 4096, 4096, 64, 0, False),
]
# products that the kernel walking lists of 128x128 tiles had before; with the switch off it still has them
_WALKED = [(1, 0, 1024, 32000, 256, 4), (0, 0, 4096, 768, 2048, 4), (0, 1, 8192, 1024, 320, 4), (0, 0, 3072, 1536, 1024, 4), (1, 0, 1536, 2048, 544, 4),
           (0, 1, 3000, 1540, 416, 4), (0, 0, 768, 4096, 2048, 4), (1, 1, 2304, 2560, 2068, 4)]


def _case_product(hip, ta, tb, M, N, K, pad):
    rng = np.random.RandomState(M + 3 * N + 7 * K)
    a, b = rng.randn(M, K).astype(np.float32), rng.randn(K, N).astype(np.float32)
    return _product(hip, a.T.copy() if ta else a, b.T.copy() if tb else b, ta, tb, pad=pad), a, b


def fp32_products(path):
    """Run in a process that has DALI_HIP_GEMM_SPLIT=0."""
    from dali_amd._native import hip, hip_check
    hip_check(hip.dali_hip_init(0), "dali_hip_init")
    for i, case in enumerate([c[:6] for c in _ROUTES] + _WALKED):
        np.save(os.path.join(path, "%d.npy" % i), _case_product(hip, *case)[0])
        print(case, flush=True)


@pytest.fixture(scope="module")
def fp32_path(gpu, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("fp32_products"))
    here = os.path.dirname(os.path.abspath(__file__))
    code = "import sys; sys.path[:0] = %r; import test_gpu_split_product as t; t.fp32_products(%r)" % ([os.path.dirname(here), here], path)
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, DALI_HIP_GEMM_SPLIT="0"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert out.returncode == 0, out.stdout
    return path


@pytest.mark.parametrize("i", range(len(_ROUTES)), ids=["-".join(map(str, c)) for c in _ROUTES])
def test_which_products_are_split(gpu, fp32_path, i):
    """A product that stays on the fp32 kernels has the bits that it has with the switch off; one that is split has others, and is
    closer to double precision."""
    got, a, b = _case_product(gpu, *_ROUTES[i][:6])
    fp32 = np.load(os.path.join(fp32_path, "%d.npy" % i))
    assert np.array_equal(got, fp32) != _ROUTES[i][6]
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert _norm_ratio(fp32, ref) <= _fp32_tolerance(_ROUTES[i][4])
    if _ROUTES[i][6]:
        assert _norm_ratio(got, ref) < _norm_ratio(fp32, ref) and _norm_ratio(got, ref) <= _split_tolerance(_ROUTES[i][4])


@pytest.mark.parametrize("i", range(len(_WALKED)), ids=["-".join(map(str, c)) for c in _WALKED])
def test_products_of_the_tile_walking_kernel_with_the_switch_off(gpu, fp32_path, i):
    ta, tb, M, N, K, pad = _WALKED[i]
    got, a, b = _case_product(gpu, *_WALKED[i])
    fp32 = np.load(os.path.join(fp32_path, "%d.npy" % (len(_ROUTES) + i)))
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert _norm_ratio(fp32, ref) <= _fp32_tolerance(K)
    assert _norm_ratio(got, ref) <= _fp32_tolerance(K)
