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


def softmax64(x):
    """the definition in 64 bits: a NaN anywhere makes its line NaN, an entry of -inf is 0"""
    x = x.astype(np.float64)
    e = np.exp(x - np.fmax.reduce(x, axis=1, keepdims=True))
    return e / e.sum(axis=1, keepdims=True)


@pytest.mark.parametrize("cols", [32, 33, 500, 4000])
def test_softmax_lines_against_64_bits(cols):
    """Each entry within the error of its f32 steps: x - max, exp and the
    division each within a few units of the last place (|x - max| < 16 here, so
    the difference's rounding is at most 16 units of the exponential), and the
    ordered sum of cols terms within cols units."""
    print("case softmax 64", cols, flush=True)
    x = np.random.default_rng([cols, 1]).normal(size=(37, cols)).astype(np.float32)
    x[3, 0] = np.nan
    x[4, cols // 2] = np.nan
    x[5, cols - 1] = -np.inf
    x[6, 0] = -np.inf
    got, want = run("softmax", 1, cols, x).astype(np.float64), softmax64(x)
    assert np.isnan(got[3:5]).all() and np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert (np.abs(got[ok] - want[ok]) <= (cols + 24) * 2.0**-24 * want[ok]).all()
    assert got[5, cols - 1] == 0 and got[6, 0] == 0


@pytest.mark.parametrize("op", ["rmsnorm", "softmax"])
@pytest.mark.parametrize("cols", [32, 64, 500, 4091])
def test_lines_of_rows_apart(op, cols):
    """Rows with another input next to their lines, so that the lines of a
    pass are not back to back: the values of the same lines back to back, any
    number of them a row and in all, blocks that take lines of several rows."""
    print("case row op lines apart", op, cols, flush=True)
    x = np.random.default_rng(cols).normal(size=(2100, cols)).astype(np.float32)
    x[5, 0] = np.nan
    x[6, cols - 1] = -np.inf
    want = run(op, 1, cols, x)
    for nrow in (1, 3, 12, 36, 65):
        text = ("(tgir 1\n  (model ro)\n  (input b (f32 5))\n  (input x (f32 %d %d))\n  (block\n    (%%0 (f32 %d %d) (%s x))\n  )\n  (output %%0))\n"
                % (nrow, cols, nrow, cols, op))
        for n in (1, 2, 2100 // nrow):
            rows = np.concatenate([np.full((n, 5), 1e30, np.float32), x[:n * nrow].reshape(n, -1)], axis=1)
            got = hip.Program(text, max_rows=n).batch(rows)[0].reshape(-1, cols)
            assert np.array_equal(got.view(np.uint32), want[:n * nrow].view(np.uint32)), (nrow, n)
