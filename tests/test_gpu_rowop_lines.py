"""rmsnorm and softmax over any number of lines: the values of each line do not
depend on how many there are, next to it or in its block."""
import numpy as np
import pytest

from technograd_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu row op lines: tg_hip_init(0)", flush=True)
    hip.init(0)


def run(op, nrow, cols, x):
    text = "(tgir 1\n  (model ro)\n  (input x (f32 %d %d))\n  (block\n    (%%0 (f32 %d %d) (%s x))\n  )\n  (output %%0))\n" % (
        nrow, cols, nrow, cols, op)
    return hip.Program(text, max_rows=len(x)).batch(x.reshape(len(x), -1))[0].reshape(-1, cols)


@pytest.mark.parametrize("op", ["rmsnorm", "softmax"])
@pytest.mark.parametrize("cols", [32, 33, 500, 4000])
def test_lines_alone_and_together(op, cols):
    print("case row op lines", op, cols, flush=True)
    x = np.random.default_rng(cols).normal(size=(1030, cols)).astype(np.float32)
    x[5, 0] = np.nan
    x[6, cols - 1] = -np.inf
    want = run(op, 1, cols, x)  # 1030 rows of one line, back to back
    if op == "rmsnorm":  # the reference's order: squares added one after another
        s = np.zeros(len(x), np.float32)
        for c in range(cols):
            s = s + x[:, c] * x[:, c]
        inv = np.float32(1) / np.sqrt(s / np.float32(cols) + np.float32(1e-6))
        assert np.array_equal(want.view(np.uint32)[7:], (x * inv[:, None])[7:].view(np.uint32))
    for n in (1, 2, 3, 5, 7, 31, 33, 103):  # counts with every remainder
        got = run(op, 1, cols, x[:n])
        assert np.array_equal(got.view(np.uint32), want[:n].view(np.uint32)), n
    for nrow in (2, 5, 103):  # several lines a row
        got = run(op, nrow, cols, x[:nrow * (1030 // nrow)].reshape(-1, nrow, cols))
        assert np.array_equal(got.view(np.uint32), want[:len(got)].view(np.uint32)), nrow
