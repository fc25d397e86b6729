"""The native part of the scripting mirror: operands of every kind on either side of an operator, attributes, errors and lifetimes (no device needed)."""
import ctypes
import gc
import sys
import sysconfig
import threading

import numpy as np
import pytest


@pytest.mark.parametrize("other", [2, True, -3.5, 10 ** 12, np.int32(4), np.int64(4), np.float32(1.5), np.float64(1.5)])
def test_numbers_on_either_side(D, other):
    x = D.Array.from_numpy(np.arange(6, dtype=np.float32).reshape(2, 3))
    for node in (x + other, other + x, x - other, other - x, x * other, other * x, x / other, other / x, D.op.pow(x, other)):
        assert isinstance(node, D.Array) and node.shape == (2, 3) and node.dtype == D.DTYPE_FLOAT and not node.is_buffer()
    # the literal has the type that as_array gives it
    scalar = D.array.as_array(other)
    assert (x + other).dtype == (x + scalar).dtype
    assert (D.Array.from_numpy(np.arange(3, dtype=np.int32)) + other).dtype == (D.Array.from_numpy(np.arange(3, dtype=np.int32)) + scalar).dtype


def test_arrays_of_numpy_on_either_side(D):
    x, n = D.Array.from_numpy(np.ones((2, 3), np.float32)), np.ones((2, 3), np.float32)
    for node in (x + n, n + x, x * n, n * x, n - x, n / x):
        assert isinstance(node, D.Array) and node.shape == (2, 3)
    with pytest.raises(TypeError):
        x + "text"
    with pytest.raises(TypeError):
        x + np.ones(3, np.int64)


def test_attributes_and_axes(D):
    x = D.Array.empty((4, 5, 6), D.DTYPE_DOUBLE)
    assert (x.shape, x.ndim, x.dtype, x.strides, x.offset) == ((4, 5, 6), 3, D.DTYPE_DOUBLE, (30, 6, 1), 0)
    assert x[1:, 2].shape == (3, 6) and x[1:, 2].offset == 42
    assert x.T.shape == (6, 5, 4) and x.transpose(0, 2, 1).strides == (30, 1, 6) and x.transpose([1, 0, 2]).shape == (5, 4, 6)
    assert D.Array.empty(()).shape == () and (-x).shape == x.shape
    for axes in ([1], (1,), 1, [np.int64(1)], iter([1])):
        assert D.op.sum(x, axes).shape == (4, 6)
    assert D.op.sum(x).shape == () and D.op.sum(x, axes=[2], keepdims=True).shape == (4, 5, 1) and x.max([-1]).shape == (4, 5)
    assert D.op.argmax(x, axis=1).dtype == D.DTYPE_INT32 and D.op.softmax(x=x, axis=-1).shape == x.shape and D.op.add(a=x, b=1).shape == x.shape
    assert D.op.dot(D.Array.empty((2, 3)), D.Array.empty((3, 4))).shape == (2, 4)


def test_errors_say_what_failed(D):
    x = D.Array.empty((2, 3))
    for what, call in (("add", lambda: x + D.Array.empty((4, 5))), ("sum", lambda: D.op.sum(x, [7])), ("transpose", lambda: x.transpose(0, 0, 0)),
                       ("dot", lambda: D.op.dot(x, D.Array.empty((7, 8)))), ("arg maximum", lambda: D.op.argmax(x, 5))):
        with pytest.raises(D.DaliError, match="^%s failed: " % what):
            call()
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        D.op.softmax(x, "rows")
    with pytest.raises((TypeError, ValueError)):
        D.op.sum(x, ["rows"])


def test_operands_live_as_long_as_what_is_built_on_them(D):
    x = D.Array.empty((2, 3))
    before = sys.getrefcount(x)
    nodes = [x * 2.0 + np.ones((2, 3), np.float32) for _ in range(100)]
    assert sys.getrefcount(x) == before  # a node holds the native array, not the handle
    y = D.op.tanh(x)
    del x
    gc.collect()
    assert (y + 1).shape == (2, 3) and nodes[-1].shape == (2, 3)
    assert isinstance(y._h, int) and y._h != (y + 0)._h


def test_threads_build_nodes(D):
    failures = []

    def work(k):
        try:
            for i in range(200):
                x = D.Array.empty((k + 2, i + 3))
                e = D.op.sigmoid(x) * 2.0 + x - 0.5 * D.op.square(x)
                assert e.shape == (k + 2, i + 3) and D.op.sum(e, [0]).shape == (i + 3,)
        except Exception as error:  # noqa: B902
            failures.append(error)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.parametrize("what", ["buffer", "node that holds the last reference to one"])
def test_the_release_of_a_buffer_lets_other_threads_run(D, what):
    x = D.Array.from_numpy(np.ones(1 << 26, np.float32))  # 256 MiB on the host: giving them back takes milliseconds
    if what != "buffer":
        x = x * 2.0
    go, ran = threading.Event(), []

    def other():
        go.wait()
        ran.append(True)
    thread = threading.Thread(target=other)
    thread.start()
    interval = sys.getswitchinterval()
    sys.setswitchinterval(60.0)  # nobody is made to give up the interpreter lock
    try:
        go.set()
        del x
        seen = bool(ran)
    finally:
        sys.setswitchinterval(interval)
        thread.join()
    assert seen


def test_the_handle_can_be_taken_over(D):
    x = D.Array.from_numpy(np.arange(6, dtype=np.float32))
    handle, x._h = x._h, None
    assert x._h is None
    y = D.Array(handle)
    del x  # released nothing
    assert y.shape == (6,) and np.array_equal(y.numpy(), np.arange(6, dtype=np.float32))
    with pytest.raises(TypeError):
        y._h = "text"
    assert y._h == handle


def test_axes_that_change_their_list_when_they_are_read(D):
    x, axes = D.Array.empty((4, 5, 6)), []

    class Axis(object):
        def __int__(self):
            axes.clear()
            return 0

        __index__ = __int__
    axes.extend([Axis(), 1, 2])
    assert D.op.sum(x, axes).shape == ()  # the three that were given
    axes.extend([Axis(), 2, 1])
    assert x.transpose(axes).shape == (4, 6, 5)


def test_the_extension_is_named_for_this_interpreter(D):
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert D._native._bind.__file__.endswith("_bind" + suffix) and suffix != ".so"
