"""The tiles of quantized products in the reference's order (TG_HIP_EXACT):
every output is the sequential f32 sum, bit for bit, at sizes on both sides of
each tile's edges, both weight widths and both operand layouts."""
import numpy as np
import pytest

from technograd_amd import hip, synth

pytestmark = pytest.mark.gpu

# rows, inputs, channels: the three tile sizes with partial rows, channels and last chunks
SHAPES = [(1, 5, 3), (17, 129, 33), (15, 128, 16), (290, 67, 1021), (256, 64, 1024), (2049, 37, 1025)]
# and a thread per output: fewer terms than are read ahead, as many, one more; a block's last threads
SHAPES += [(1, 1, 1), (300, 7, 5), (129, 8, 2), (40001, 9, 1), (16385, 33, 4), (1031, 24, 127)]


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu exact tiles: tg_hip_init(0)", flush=True)
    hip.init(0)


def pack(codes, bits):
    c = codes.ravel()
    if bits == 8:
        return c
    c = np.concatenate([c, np.zeros(c.size % 2, np.int8)])
    return ((c[0::2] & 15) | ((c[1::2] & 15) << 4)).astype(np.uint8).view(np.int8)


# W @ X, X @ W, and W @ x for a vector x per row
@pytest.mark.parametrize("axis", [0, 1, "vector"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", SHAPES)
def test_sequential_sums(shape, bits, axis):
    print("case", shape, bits, axis, flush=True)
    M, K, C = shape
    rng = np.random.default_rng([M, K, C, bits])
    lim = 7 if bits == 4 else 127
    codes = rng.integers(-lim, lim + 1, (C, K)).astype(np.int8)
    scales = rng.uniform(0.5, 2.0, C).astype(np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[M // 2, K // 2] = np.inf
    x[0, 0] = -0.0
    want = np.zeros((M, C), np.float32)
    with np.errstate(invalid="ignore"):
        for k in range(K):  # the reference's loop: a rounded product, then a rounded add
            want = want + x[:, k, None] * codes[None, :, k].astype(np.float32)
        want = want * scales
    if axis == "vector":
        text = "(tgir 1\n  (model m)\n%s  (input x (f32 %d))\n  (block\n    (%%0 (f32 %d) (matmul W x))\n  )\n  (output %%0))\n" % (
            synth.param_quant("W", codes, scales, bits, 0), K, C)
        got = hip.Program(text, flags=hip.EXACT, max_rows=M).batch(x)[0]
    elif axis == 1:
        got = hip.matmul_q(pack(np.ascontiguousarray(codes.T), bits), bits, scales, x, M, K, C, 1, flags=hip.EXACT)
    else:
        got = hip.matmul_q(pack(codes, bits), bits, scales, np.ascontiguousarray(x.T), C, K, M, 0, flags=hip.EXACT).T
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(np.where(nan, 0, got).view(np.uint32), np.where(nan, 0, want).view(np.uint32))
