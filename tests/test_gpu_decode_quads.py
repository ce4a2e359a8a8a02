"""The decode step's fused norms and silu (four inputs a thread, digits and
class from whole-wave sums) where quads, waves and blocks end: the decoder's
logits against the fixed-length forward's, bit for bit."""
import pytest

from technograd_amd import hip
from test_gpu_decode import check_decode

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu decode quads: tg_hip_init(0)", flush=True)
    hip.init(0)


# model width and MLP width: off quads, off 16-input groups, one wave and one
# input more, the largest width, an MLP row of more than one pass of a block
@pytest.mark.parametrize("D,FF,HD", [(50, 34, 16), (67, 99, 48), (256, 257, 32), (257, 1030, 128), (1023, 61, 256), (4096, 33, 16), (64, 4101, 64)])
def test_widths_equal_fixed_length_forward(D, FF, HD):
    print("case decode quads", D, FF, HD, flush=True)
    check_decode(3, 5, 3, dict(L=2, D=D, NQ=2, NKV=1, HD=HD, FF=FF, V=96))


# prompts of 2048 token rows and more: the many-lines norms, at every padded width, ragged and whole, lines off a block's
@pytest.mark.parametrize("seqs,T0,D,HD", [(33, 63, 64, 64), (33, 63, 100, 128), (41, 50, 256, 48), (33, 63, 509, 256), (33, 63, 1024, 32),
                                          (16, 128, 2047, 64), (16, 129, 2112, 16), (16, 128, 2048, 64), (21, 100, 4040, 48), (16, 128, 4096, 16)])
def test_many_lines_equal_fixed_length_forward(seqs, T0, D, HD):
    print("case many lines", seqs, T0, D, HD, flush=True)
    check_decode(seqs, T0, 2, dict(L=2, D=D, NQ=2, NKV=1, HD=HD, FF=64, V=96))


# the attention's digits for the output projections: sequences off the 32-row blocks, 1 to 8 query heads a KV head (8 of
# 48 do not fit the block's room and take the digit kernel), the largest and smallest heads, a one-token prompt
@pytest.mark.parametrize("seqs,T0,NQ,NKV,HD", [(33, 3, 4, 4, 48), (2, 1, 8, 1, 48), (37, 2, 8, 1, 64), (31, 4, 8, 2, 256), (3, 70, 2, 1, 144)])
def test_attention_digits_equal_fixed_length_forward(seqs, T0, NQ, NKV, HD):
    print("case attention digits", seqs, T0, NQ, NKV, HD, flush=True)
    check_decode(seqs, T0, 3, dict(L=2, D=96, NQ=NQ, NKV=NKV, HD=HD, FF=64, V=96))
