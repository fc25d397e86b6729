"""Reductions whose workgroups meet: at the counts of workgroups, strips and rows where the way they meet changes.

Operands are small whole numbers, so that every order of summation gives the same result and it is compared exactly; each case runs twice, the second
time on the counters that the first has set back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def whole(rng, shape, dtype):
    return rng.randint(-8, 9, shape).astype(dtype)


@pytest.mark.parametrize("blocks", [1, 2, 127, 128, 129, 511, 512, 700])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_full_reductions_by_workgroups(gpu, D, rng, blocks, dtype):
    per_block = 256 * 4 * (4 if dtype == np.float64 else 8)
    for n in (blocks * per_block, (blocks - 1) * per_block + 1):
        x = whole(rng, n, dtype)
        X = D.Array.from_numpy(x)
        for _ in range(2):
            assert D.op.sum(X).numpy() == x.sum()
            assert D.op.max(X).numpy() == x.max()
            assert int(D.op.argmax(X).numpy()) == int(x.argmax())


@pytest.mark.parametrize("rows,cols", [(127, 1000), (128, 1000), (129, 1000), (1023, 1000), (1024, 1000), (1025, 1000), (2047, 520), (1023, 16384), (1024, 16384), (1025, 16384),
                                       (1009, 20), (4113, 20)])
def test_totals_beside_a_row_kernel_by_workgroups(gpu, D, rng, rows, cols):
    x = whole(rng, (rows, cols), np.float32)
    X = D.Array.from_numpy(x)
    for _ in range(2):
        top = D.op.max(X, [1], True)
        lower, per_row, total = X - top, D.op.sum(X, [1]), D.op.sum(top)
        D.eval_together([lower, per_row, total])
        assert np.array_equal(lower.numpy(), x - x.max(1, keepdims=True))
        assert np.array_equal(per_row.numpy(), x.sum(1))
        assert total.numpy() == x.max(1).sum()


# rows: around the 32, 64 and 256 that one workgroup takes alone and whole chunks of 128; columns: part of a vector and of a strip, 15 and 16 strips
# (the last with counters of their own for groups), strips that fill the chip
@pytest.mark.parametrize("rows,cols", [(r, c) for r in (1, 31, 33, 64, 65, 127, 256, 257, 1025, 5003) for c in (3, 17, 64, 129, 1920, 1921, 2047, 16384, 16385) if r * c <= 6000000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_leading_axis_reductions_by_strips(gpu, D, rng, rows, cols, dtype):
    x = whole(rng, (rows, cols), dtype)
    X = D.Array.from_numpy(x)
    for _ in range(2):
        assert np.array_equal(D.op.sum(X, [0]).numpy(), x.sum(0))
        assert np.array_equal(D.op.argmax(X, 0).numpy(), x.argmax(0))  # the first of equal ones
        assert np.array_equal(D.op.max(X, [0]).numpy(), x.max(0))
