"""Kernels that reduce and rewrite millions of short rows: the number of threads a row gets, over row lengths around every change of it, aligned and not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def softmax64(x):
    e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True).astype(np.float64))
    return e, e.sum(1, keepdims=True)


# one thread a row, four, eight lanes to a cache line, halves of 16, 32 and 64 lanes, and just past the 64 vectors where the rule ends; each with the rows
# (65536 threads of a thread per vector) where it begins
@pytest.mark.parametrize("cols", [2, 3, 5, 7, 8, 9, 12, 13, 15, 16, 20, 33, 40, 64, 96, 97, 100, 128, 150, 160, 200, 250, 255, 256, 257, 259, 260])
@pytest.mark.parametrize("shift", [0, 1])
def test_softmax_and_cross_entropy_over_many_short_rows(gpu, D, rng, cols, shift):
    vectors = cols if cols < 16 and (cols % 4 or shift) else cols // 4
    whole = 1
    while whole < min(vectors, 64):
        whole *= 2
    for rows in (65536 // whole - 1, 65536 // whole + 3):
        full = (rng.randn(rows, cols + shift) * 3).astype(np.float32)
        full[0, shift:] = -np.finfo(np.float32).max  # equal entries of the lowest value
        full[1, shift] = 80.0
        x = np.ascontiguousarray(full[:, shift:])
        X = D.Array.from_numpy(full)
        X = X[:, shift:] if shift else X
        t = rng.randint(0, cols, rows).astype(np.int32)
        e, s = softmax64(x)
        # the sum of n positive terms in any order: at most n 2^-24 of it; the rest a few roundings, and that of the exponent d = x - max,
        # which is at most 2^-24 |d| and goes into the exponential as a factor of 1 + 2^-24 |d|
        tol = (cols + 16) * 2.0 ** -24
        with np.errstate(over="ignore"):
            drop = np.minimum(np.abs(x.astype(np.float64) - x.max(1, keepdims=True)), 200.0) * 2.0 ** -24
        assert (np.abs(D.op.softmax(X, 1).numpy() - e / s) <= (tol + drop) * (e / s) + 1e-37).all()
        mean, loss, grad = D.op.softmax_cross_entropy(X, D.Array.from_numpy(t))
        want = np.log(s[:, 0]) + x.max(1) - x[np.arange(rows), t]
        hot = e / s
        hot[np.arange(rows), t] -= 1.0
        # (the probability's own error, tol of it, and the rounding of a difference of at most one)
        assert (np.abs(grad.numpy() - hot) <= (tol + drop) * (e / s) + 2.0 ** -24).all()
        # (the first row's values are as large as floats get: their differences are exact zeros, but log(s) is lost in adding the maximum)
        scale = np.abs(x).max(1) + 1.0
        assert (np.abs(loss.numpy() - want)[1:] <= tol * scale[1:] + tol).all()


@pytest.mark.parametrize("cols", [5, 10, 40, 96, 97, 160, 250])
def test_infinities_and_nan_stay_in_their_rows(gpu, D, rng, cols):
    rows = 20011
    x = rng.randn(rows, cols).astype(np.float32)
    x[3, 1], x[5, 0], x[7, cols - 1] = np.inf, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        e = np.exp(x[5].astype(np.float64) - x[5].max())
    got = D.op.softmax(D.Array.from_numpy(x), 1).numpy()
    assert np.isnan(got[3]).any() and np.isnan(got[7]).any()
    np.testing.assert_allclose(got[5], e / e.sum(), rtol=(cols + 16) * 2.0 ** -24, atol=1e-37)
    others = np.ones(rows, bool)
    others[[3, 7]] = False
    assert np.isfinite(got[others]).all()
