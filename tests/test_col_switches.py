"""Reductions along the leading axis under the switches that set their geometry (each in a process of its own: a switch is read once)."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(code, **switches):
    env = dict(os.environ, PYTHONPATH=ROOT, **switches)
    out = subprocess.run([sys.executable, "-c", "import numpy as np\nimport dali_amd as D\nop = D.op\n" + code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         timeout=100)
    assert out.returncode == 0, out.stdout[-2000:]
    return out.stdout


def source(what, **switches):
    text = run("D.generate_only([%s])\nprint(D.last_source())" % what, **switches)
    return text[text.rindex('extern "C" __global__'):]


@pytest.mark.parametrize("groups", [0, 1, 2, 4, 16, 3])
@pytest.mark.parametrize("what", ["op.sum(D.Array.empty((5003, 3001)), [0])", "op.argmax(D.Array.empty((5003, 3001), D.DTYPE_DOUBLE), 0)"])
def test_the_fold_takes_every_column_of_a_strip(D, groups, what):
    body = source(what, DALI_HIP_COL_RG=str(groups))
    count, threads, vec = (int(re.search(r"\b%s = (\d+)" % name, body).group(1)) for name in ("NWAVE", "TPP", "VEC"))
    assert count * threads == 256 and (count == groups or groups in (0, 3))  # (three do not divide the threads: as if unset)
    loop = re.search(r"for \(int c = threadIdx\.x; c < TPP \* VEC; c \+= (\d+)\)", body)
    columns = [c for t in range(256) for c in range(t, threads * vec, int(loop.group(1)) if loop else 1024)]
    assert count == 1 or sorted(columns) == list(range(threads * vec))


@pytest.mark.parametrize("strips", range(1, 17))
def test_strips_draw_from_counters_of_their_own(D, strips):
    text = run("D.generate_only([op.sum(D.Array.empty((5003, 300)), [0])])\nprint(D.last_source())")
    body = text[text.rindex('extern "C" __global__'):]
    grouped = re.search(r"const bool grouped = (.*);", body).group(1).replace("&&", "and").replace("gridDim.x", "strips").replace("gridDim.y", "blocks")
    words = int(re.search(r"grouped \? blockIdx\.x \* \((\d+)u \* 64u\)", body).group(1)) * 64
    line, below, above = (int(v) for v in re.search(r"groups = n < (\d+) \? (\d+) : (\d+);", text).groups())
    for blocks in (2, 127, 128, 1023, 1024, 1025, 4096, 65535):
        if eval(grouped, {"strips": strips, "blocks": blocks}):
            groups = below if blocks < line else above
            assert (1 + groups) * 64 <= words and strips * words <= 16384, (strips, blocks)


WHOLE = """
rng = np.random.RandomState(7)
for rows, cols in ((1025, 3001), (64, 2048), (5003, 300), (33, 17), (3, 4100)):
    for dtype in (np.float32, np.float64, np.int32):
        x = rng.randint(-8, 9, (rows, cols)).astype(dtype)  # sums of whole numbers: exact in any order
        X = D.Array.from_numpy(x)
        for _ in range(2):
            assert np.array_equal(op.sum(X, [0]).numpy(), x.sum(0)), (rows, cols, dtype)
            assert np.array_equal(op.max(X, [0]).numpy(), x.max(0)), (rows, cols, dtype)
            assert np.array_equal(op.argmax(X, 0).numpy(), x.argmax(0)), (rows, cols, dtype)
"""


@pytest.mark.gpu
@pytest.mark.parametrize("groups", ["1", "2", "4", "16", "64"])
def test_row_groups(gpu, groups):
    run(WHOLE, DALI_HIP_COL_RG=groups)


@pytest.mark.gpu
def test_more_workgroups_to_a_strip_than_counters_in_its_groups(gpu):
    run("""
x = np.random.RandomState(3).randint(-8, 9, (40000, 300)).astype(np.float32)
X = D.Array.from_numpy(x)
for _ in range(3):
    assert np.array_equal(op.sum(X, [0]).numpy(), x.sum(0)) and np.array_equal(op.argmax(X, 0).numpy(), x.argmax(0))
    assert op.max(op.square(X)).numpy() == 64.0  # draws from the same counters
""", DALI_HIP_COL_MAXY="2048", DALI_HIP_COL_BLOCKS="8192", DALI_HIP_COL_ROWS="8")
