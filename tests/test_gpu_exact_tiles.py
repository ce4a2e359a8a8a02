"""The tiles of quantized products in the reference's order (TG_HIP_EXACT):
every output is the sequential f32 sum, bit for bit, at sizes on both sides of
each tile's edges, both weight widths and both operand layouts."""
import numpy as np
import pytest

from technograd_amd import hip

pytestmark = pytest.mark.gpu

# rows, inputs, channels: the three tile sizes with partial rows, channels and last chunks
SHAPES = [(1, 5, 3), (17, 129, 33), (15, 128, 16), (290, 67, 1021), (256, 64, 1024), (2049, 37, 1025)]


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


@pytest.mark.parametrize("axis", [0, 1])
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
    if axis == 1:
        got = hip.matmul_q(pack(np.ascontiguousarray(codes.T), bits), bits, scales, x, M, K, C, 1, flags=hip.EXACT)
    else:
        got = hip.matmul_q(pack(codes, bits), bits, scales, np.ascontiguousarray(x.T), C, K, M, 0, flags=hip.EXACT).T
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(np.where(nan, 0, got).view(np.uint32), np.where(nan, 0, want).view(np.uint32))
