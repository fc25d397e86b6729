"""Convolutions of channels-last images and the gradients of their filters as products that read the image window by window."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# images, height, width, channels, filters, window, strides: whole slabs; part of a slab of positions and of a window's row; rows of windows shorter and longer
# than a tile; odd channel counts; one to eight rows to a window; stride past the window; outputs of one row and one column
SHAPES = [(24, 40, 40, 64, 128, (3, 3), (1, 1)), (22, 41, 37, 65, 129, (3, 3), (1, 1)), (40, 57, 43, 33, 100, (5, 3), (2, 1)), (50, 28, 28, 200, 260, (1, 1), (1, 1)),
          (80, 61, 59, 96, 136, (2, 2), (3, 2)), (16, 70, 33, 30, 192, (8, 5), (1, 2)), (1300, 7, 7, 128, 130, (7, 3), (1, 1)), (1500, 3, 20, 48, 200, (3, 5), (1, 1)),
          (2, 128, 130, 72, 72, (4, 7), (1, 1))]


def windows64(x, window, strides):
    v = np.lib.stride_tricks.sliding_window_view(x.astype(np.float64), window, axis=(1, 2))[:, ::strides[0], ::strides[1]]
    v = v.transpose(0, 1, 2, 4, 5, 3)
    return v.shape[:3], v.reshape(int(np.prod(v.shape[:3])), -1)


def whole_or_normal(rng, shape, whole):
    return (rng.randint(-4, 5, shape) if whole else rng.randn(*shape)).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("whole", [True, False])
def test_by_windows(gpu, D, rng, shape, whole):
    n, h, w, c, f, window, strides = shape
    x, k = whole_or_normal(rng, (n, h, w, c), whole), whole_or_normal(rng, (f,) + window + (c,), whole)
    grid, patches = windows64(x, window, strides)
    dy = whole_or_normal(rng, grid + (f,), whole)
    X, K, dY = (D.Array.from_numpy(a) for a in (x, k, dy))
    before = D.jit_stats()["kernels"]
    y, dk = D.op.conv2d(X, K, strides[0], strides[1], "valid", "NHWC").numpy(), D.op.conv2d_backward_filters(X, dY, strides[0], strides[1], k.shape, "valid", "NHWC").numpy()
    assert D.jit_stats()["kernels"] == before  # no generated kernel has padded an image or formed patches
    for got, left, right in ((y.reshape(-1, f), patches, k.reshape(f, -1).T.astype(np.float64)), (dk.reshape(f, -1), dy.reshape(-1, f).T.astype(np.float64), patches)):
        want = left @ right
        if whole:
            assert np.array_equal(got, want)  # sums of whole numbers below 2^24
        else:
            # products of pieces leave out at most 2^-24 of a product; sums are kept in 32 bits, in order over at most sqrt(terms) steps of 32
            bound = 2.0 ** -24 * (4 + np.sqrt(left.shape[1] / 32.0)) * np.sqrt((left ** 2).sum(1))[:, None] * np.sqrt((right ** 2).sum(0))[None, :]
            assert (np.abs(got - want) <= bound).all()
            assert np.linalg.norm(got - want) <= 4e-7 * np.linalg.norm(want)


def test_views_and_values_that_are_not_finite(gpu, D, rng):
    x, k = rng.randn(28, 44, 40, 40).astype(np.float32), rng.randn(80, 3, 3, 40).astype(np.float32)
    wide = np.zeros((28, 44, 40, 41), np.float32)
    wide[..., 1:] = x
    dy = rng.randn(28, 42, 38, 80).astype(np.float32)
    X, dY = D.Array.from_numpy(wide)[:, :, :, 1:], D.Array.from_numpy(dy)
    grid, patches = windows64(x, (3, 3), (1, 1))
    y = D.op.conv2d(X, D.Array.from_numpy(k), 1, 1, "valid", "NHWC").numpy().reshape(-1, 80)
    np.testing.assert_allclose(y, patches @ k.reshape(80, -1).T.astype(np.float64), rtol=0, atol=2e-4)
    x[3, 20, 20, 7] = np.inf
    dy[5, 0, 0, 3] = np.nan
    with np.errstate(invalid="ignore"):
        _, patches = windows64(x, (3, 3), (1, 1))
        want_y, want_k = patches @ k.reshape(80, -1).T.astype(np.float64), dy.reshape(-1, 80).T.astype(np.float64) @ patches
    got_y = D.op.conv2d(D.Array.from_numpy(x), D.Array.from_numpy(k), 1, 1, "valid", "NHWC").numpy().reshape(-1, 80)
    got_k = D.op.conv2d_backward_filters(D.Array.from_numpy(x), D.Array.from_numpy(dy), 1, 1, k.shape, "valid", "NHWC").numpy().reshape(80, -1)
    for got, want in ((got_y, want_y), (got_k, want_k)):
        finite = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), finite)
        np.testing.assert_allclose(got[finite], want[finite], rtol=0, atol=1e-3)


def test_a_recording_reads_what_its_operands_hold(gpu, D, rng):
    shape = (24, 40, 40, 64)
    x, k = rng.randint(-4, 5, shape).astype(np.float32), rng.randint(-4, 5, (128, 3, 3, 64)).astype(np.float32)
    X, K = D.Array.from_numpy(x), D.Array.from_numpy(k)
    with D.Recording() as recording:
        y = D.op.conv2d(X, K, 1, 1, "valid", "NHWC").eval()
    for graph in (False, True):
        if graph:
            recording.make_graph()
        for _ in range(3):
            x = rng.randint(-4, 5, shape).astype(np.float32)
            X.assign(D.Array.from_numpy(x))
            recording.replay(1)
            assert np.array_equal(y.numpy().reshape(-1, 128), windows64(x, (3, 3), (1, 1))[1] @ k.reshape(128, -1).T.astype(np.float64))


# 64 filters: more than 1e9 operations, but a size that the products by windows do not take
def test_a_size_that_is_not_taken_has_its_image_copied_once(gpu, D, rng):
    n, h, w, c, f = 28, 44, 40, 40, 64
    wide = rng.randint(-4, 5, (n, h, w, c + 1)).astype(np.float32)
    x, k = np.ascontiguousarray(wide[..., 1:]), rng.randint(-4, 5, (f, 3, 3, c)).astype(np.float32)
    dy = rng.randint(-4, 5, (n, h - 2, w - 2, f)).astype(np.float32)
    for gradient in (0, 1):
        assert gpu.dali_hip_conv2d_nhwc_supported(gradient, n, h, w, c, f, 3, 3, 1, 1) == 0 and gpu.dali_hip_conv2d_nhwc_supported(gradient, n, h, w, c, 2 * f, 3, 3, 1, 1) == 1
    K, dY = D.Array.from_numpy(k), D.Array.from_numpy(dy)
    _, patches = windows64(x, (3, 3), (1, 1))
    launches = []
    for X in (D.Array.from_numpy(x), D.Array.from_numpy(wide)[:, :, :, 1:]):
        with D.Recording() as forward:
            y = D.op.conv2d(X, K, 1, 1, "valid", "NHWC").eval()
        with D.Recording() as backward:
            dk = D.op.conv2d_backward_filters(X, dY, 1, 1, k.shape, "valid", "NHWC").eval()
        launches.append((forward.launches, backward.launches))
        assert np.array_equal(y.numpy().reshape(-1, f), patches @ k.reshape(f, -1).T)
        assert np.array_equal(dk.numpy().reshape(f, -1), dy.reshape(-1, f).T @ patches)
    assert launches[1] == (launches[0][0] + 1, launches[0][1] + 1), launches
