"""The tiled f32 product over every operand layout it has a form for, and a
prompt's attention with its heads in one launch or in several."""
import numpy as np
import pytest

from oracle import oracle as O
from technograd_amd import hip, synth
from test_gpu_decode import check_decode

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu attention tiles: tg_hip_init(0)", flush=True)
    hip.init(0)


# tiles' edges with 16-byte rows (whole quads) and without
@pytest.mark.parametrize("m,k,n", [(64, 16, 64), (132, 100, 68), (65, 33, 67), (1, 31, 4096)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_tile_layouts(m, k, n, ta, tb):
    """A or its transpose times B or its transpose, read in place: the
    reference's order, bit for bit, over several batch rows."""
    print("case tile", m, k, n, ta, tb, flush=True)
    sa, sb = ((k, m) if ta else (m, k)), ((n, k) if tb else (k, n))
    body, a, b, v = "", "a", "b", 0
    if ta:
        body, a, v = body + "    (%%%d (f32 %d %d) (transpose a))\n" % (v, m, k), "%%%d" % v, v + 1
    if tb:
        body, b, v = body + "    (%%%d (f32 %d %d) (transpose b))\n" % (v, k, n), "%%%d" % v, v + 1
    text = "(tgir 1\n  (model t)\n  (input a (f32 %d %d))\n  (input b (f32 %d %d))\n  (block\n%s    (%%%d (f32 %d %d) (matmul %s %s))\n  )\n  (output %%%d))\n" % (
        sa + sb + (body, v, m, n, a, b, v))
    x = np.random.default_rng([m, k, n]).standard_normal((3, m * k + k * n)).astype(np.float32)
    x[1] *= 1e-20
    want, _ = O.Model(text).batch(x)
    got, _ = hip.Program(text, max_rows=4).batch(x)
    assert np.array_equal(np.asarray(got).view(np.uint32), np.asarray(want).view(np.uint32))


# prompts of odd length (no 16-byte rows of scores), just over a tile, and several tiles with 4 heads on 2 KV heads
@pytest.mark.parametrize("seqs,T0", [(3, 65), (2, 131), (2, 196)])
def test_prompt_heads_in_one_launch(seqs, T0):
    print("case heads", seqs, T0, flush=True)
    check_decode(seqs, T0, 2, dict(L=1, D=64, NQ=4, NKV=2, HD=64, FF=96, V=320))


def test_prompt_heads_in_several_launches():
    """Nine prompts of 4088 tokens: the score buffer holds three heads' scores,
    so the four heads run a KV head's pair at a time. Each sequence's logits
    are those of the sequence alone, whose heads run together."""
    print("case head chunks", flush=True)
    T0 = 4088
    text = synth.qwen3_tgir("q", T=8, rope_len=T0 + 1, L=1, D=64, NQ=4, NKV=2, HD=16, FF=96, V=320)
    prog = hip.Program(text, max_rows=1)
    ids = np.random.default_rng(3).integers(0, 320, (9, T0)).astype(np.float32)
    dec = hip.Decoder(prog, 9, T0, T0 + 1)
    _, logits = dec.generate(ids, 1, logits=True)
    dec.close()
    one = hip.Decoder(prog, 1, T0, T0 + 1)
    for s in (0, 8):
        _, want = one.generate(ids[s:s + 1], 1, logits=True)
        assert np.array_equal(logits[0, s].view(np.uint32), want[0, 0].view(np.uint32))
    one.close()
