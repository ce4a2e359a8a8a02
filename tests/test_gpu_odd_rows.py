"""Rows of any length and alignment in every digit kernel: the last group of a
row whose inputs do not fill it, with its largest, its outlying and its
non-finite entries there, bit for bit against the path restated on the host."""
import numpy as np
import pytest

from parity import device_path_matmul

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 33), (1, 47), (1, 2917), (1, 8191),             # the fused single-row kernel (int4), digits_k / digits_row_k (int8)
    (3, 35), (203, 1500), (200, 1023), (130, 1041),     # a wave per row
    (5, 2063), (200, 2917), (7, 5001), (3, 9001),       # a block per row
    (513, 37), (700, 1179), (515, 2917), (600, 4095),   # 16 rows per block
]


def pack(codes, bits):
    c = codes.ravel()
    if bits == 8:
        return c
    c = np.concatenate([c, np.zeros(c.size % 2, np.int8)])
    return ((c[0::2] & 15) | ((c[1::2] & 15) << 4)).astype(np.uint8).view(np.int8)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,K", SHAPES)
def test_last_group(M, K, bits):
    from technograd_amd import hip
    print("case odd rows", M, K, bits, flush=True)
    C = 40
    rng = np.random.default_rng([M, K, bits])
    lim = 127 if bits == 8 else 7
    codes = rng.integers(-lim, lim + 1, (K, C)).astype(np.int8)
    codes[K - 1, ::2] = 0
    scales = rng.uniform(0.001, 0.1, C).astype(np.float32)
    last = K - 1 - (K - 1) % 16  # the last group's first input
    kinds = [lambda r: None, lambda r: r.__setitem__(K - 1, 30.0), lambda r: r.__setitem__(K - 1, 1e6), lambda r: r.__setitem__(last, -1e5),
             lambda r: r.__setitem__(K - 1, np.nan), lambda r: r.__setitem__(slice(0, last), 0.0), lambda r: r.__setitem__(last - 1, np.inf)]
    for first in range(len(kinds) if M == 1 else 1):
        x = rng.standard_normal((M, K)).astype(np.float32)
        for m in range(min(M, len(kinds))):
            kinds[(first + m) % len(kinds)](x[m])
        got = hip.matmul_q(pack(codes, bits), bits, scales, x, M, K, C, 1)
        want, _ = device_path_matmul(x, codes, scales)
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(np.where(nan, 0, got).view(np.uint32), np.where(nan, 0, want).astype(np.float32).view(np.uint32))
