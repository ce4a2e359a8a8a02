"""All heads' output projections in one product, the heads added in order:
decoded logits against the fixed-length forward bit for bit at head sizes with
one to four 64-input steps, widths off the channel tiles, few rows and many,
and rows off their grid."""
import numpy as np
import pytest

from technograd_amd import hip, synth
from test_gpu_decode import check_decode, fixed_forward

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu heads: tg_hip_init(0)", flush=True)
    hip.init(0)


@pytest.mark.parametrize("seqs,T0,HD,NQ,D,bits", [
    (3, 9, 48, 2, 72, 4),      # one 64-input step, its last 16 padding
    (2, 5, 64, 17, 64, 8),     # more heads than waves
    (3, 4, 48, 65, 40, 4),     # one head more than a step adds at a time
    (2, 3, 64, 144, 32, 8),    # two such groups and a part
    (5, 7, 112, 4, 300, 4),    # channels off the 16- and 256-wide tiles
    (2, 3, 192, 2, 128, 4),    # three steps
    (3, 4, 256, 2, 96, 8),     # four
    (9, 130, 128, 4, 130, 4),  # 1170 prompt rows: the many-row tiles, rows and channels off them
    (11, 99, 64, 2, 260, 8),   # the same at 64 inputs a head
])
def test_heads_equal_fixed_forward(seqs, T0, HD, NQ, D, bits):
    print("case heads", seqs, T0, HD, NQ, D, bits, flush=True)
    check_decode(seqs, T0, 2, dict(L=1, D=D, NQ=NQ, NKV=NQ if NQ % 2 else NQ // 2, HD=HD, FF=96, V=320, bits=bits))


@pytest.mark.parametrize("seqs,T0", [(4, 6), (9, 120)])
def test_heads_rows_off_their_grid(seqs, T0):
    """Values whose lines hold a huge entry, an infinity, a lone outlier or
    only tiny entries: split lines, the reference's loop and results far below
    1, in the step's rows and in a prompt's."""
    print("case heads classes", seqs, T0, flush=True)
    dims = dict(L=1, D=64, NQ=4, NKV=2, HD=64, FF=96, V=320)
    text = synth.qwen3_tgir("q", T=T0, rope_len=T0 + 1, **dims)
    # the values' scales: one column 2^20 times the others, one head's 1e-30, one column beyond 2^100
    def rescale(t, name, f):
        i = t.index("(param %s " % name)
        a = t.index("(scale", i) + 6
        b = t.index(")", a)
        s = np.array(t[a:b].split(), np.float32)
        return t[:a] + "".join(" %.9g" % v for v in f(s)) + t[b:]
    big = np.ones(64, np.float32)
    big[5] = 2.0**20
    models = []
    for f0, f1 in ((lambda s: s * big, lambda s: s * np.float32(1e-36)), (lambda s: s * big, lambda s: np.where(np.arange(64) == 3, np.float32(1e32), s))):
        models.append((f0, f1))
    for f0, f1 in models:
        t = rescale(rescale(text, "Wv_0_0", f0), "Wv_0_1", f1)
        prog = hip.Program(t, max_rows=seqs)
        dec = hip.Decoder(prog, seqs, T0, T0 + 1)
        ids = np.random.default_rng(T0).integers(0, 320, (seqs, T0)).astype(np.float32)
        tokens, logits = dec.generate(ids, 2, logits=True)
        want = prog.batch(ids)[0]
        assert np.array_equal(logits[0].view(np.uint32), want.view(np.uint32))
        t2 = synth.qwen3_tgir("q", T=T0 + 1, **dims)
        t2 = rescale(rescale(t2, "Wv_0_0", f0), "Wv_0_1", f1)
        ids2 = np.concatenate([ids, tokens[:, :1].astype(np.float32)], axis=1)
        want = hip.Program(t2, max_rows=seqs).batch(ids2)[0]
        assert np.array_equal(logits[1].view(np.uint32), want.view(np.uint32))
        dec.close()
