"""Reductions along the leading axis with transcendental arithmetic on every element, at the rows and columns where their geometry changes: one workgroup to a strip
or several, last strips of a few columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 33, 65, 143, 144, 256, 257, 1025, 4096])
@pytest.mark.parametrize("cols", [17, 63, 64, 100, 900, 901, 1028, 4000, 8191])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_sums_by_columns(gpu, D, rng, rows, cols, dtype):
    x = rng.randn(rows, cols).astype(dtype)
    X, wide = D.Array.from_numpy(x), x.astype(np.float64)
    # a term is a few roundings off (4 for one function, 10 for a product of two), their sum in any order at most `rows` more of the sum of magnitudes
    eps = np.finfo(dtype).eps
    for got, terms, own in ((D.op.sum(D.op.exp(X), [0]), np.exp(wide), 4), (D.op.sum(X * D.op.tanh(X), [0]), wide * np.tanh(wide), 10),
                            (D.op.sum(D.op.sigmoid(X) * D.op.tanh(X), [0]), np.tanh(wide) / (1.0 + np.exp(-wide)), 10)):
        assert (np.abs(got.numpy() - terms.sum(0)) <= (rows + own) * eps * np.abs(terms).sum(0)).all()
