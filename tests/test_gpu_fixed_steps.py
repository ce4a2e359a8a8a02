"""Q16.16 programs too large to compile, run an instruction at a time, against
the row-program interpreter: the same integers, for every kind of instruction,
weights on both sides, rows off the multiples of a wave. That these models do
run so, and not both ways in the interpreter, is test_host_calls.py's."""
import numpy as np
import pytest

from technograd_amd import hip, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    print("gpu fixed steps: tg_hip_init(0)", flush=True)
    hip.init(0)


def quant(name, rows, cols, bits, axis, seed):
    rng = np.random.default_rng(seed)
    lim = 7 if bits == 4 else 127
    n = rows if axis == 0 else cols
    return synth.param_quant(name, rng.integers(-lim, lim + 1, (rows, cols)).astype(np.int8), rng.uniform(0.1, 2.0, n).astype(np.float32) / lim,
                             bits, axis)


def f32(name, *shape, seed=0, scale=0.2):
    return synth.param_f32(name, np.random.default_rng(seed).normal(size=shape) * scale)


def model(params, inputs, body, out):
    return "(tgir 1\n  (model m)\n" + "".join(params) + inputs + "  (block\n" + body + "  )\n  (output %s))\n" % out


# more than 16 K multiply-adds or 1024 values: the compiler refuses them
MODELS = {
    # quantized W @ x chains, the unary fused and not, rmsnorm
    "mlp8": model([quant("W1", 200, 70, 8, 0, 1), quant("W2", 130, 200, 8, 0, 2)], "  (input x (f32 70))\n",
                  "    (%0 (f32 200) (matmul W1 x))\n    (%1 (f32 200) (tanh %0))\n    (%2 (f32 130) (matmul W2 %1))\n"
                  "    (%3 (f32 130) (sigmoid %2))\n    (%4 (f32 130) (mul %2 %3))\n    (%5 (f32 130) (rmsnorm %4))\n", "%5"),
    # x @ W over rows of a matrix, int4, biases and broadcasts, softmax, mean
    "rows4": model([quant("W", 33, 129, 4, 1, 3), f32("b", 129, seed=4), f32("c", 5, 1, seed=5)], "  (input x (f32 5 33))\n",
                   "    (%0 (f32 5 129) (matmul x W))\n    (%1 (f32 5 129) (add %0 b))\n    (%2 (f32 5 129) (mul %1 c))\n"
                   "    (%3 (f32 5 129) (softmax %2))\n    (%4 (f32 129 5) (transpose %3))\n    (%5 (f32 129 129) (matmul %4 %3))\n"
                   "    (%6 (f32) (mean %5))\n    (%7 (f32 5 129) (div %3 %6))\n    (%8 (f32 5 129) (max %7 %2))\n", "%8"),
    # an unquantized param on each side, outer, take, reshape, a sum, saturating values
    "f32": model([f32("A", 90, 40, seed=6, scale=30.0), f32("B", 40, 90, seed=7)], "  (input x (f32 40 4))\n  (input i (f32 3))\n",
                 "    (%0 (f32 90 4) (matmul A x))\n    (%1 (f32 4 40) (transpose x))\n    (%2 (f32 4 90) (matmul %1 B))\n"
                 "    (%3 (f32 90 4) (exp %0))\n    (%4 (f32 3 90) (take %2 i))\n    (%5 (f32 270) (reshape %4))\n    (%6 (f32) (sum %5))\n"
                 "    (%7 (f32 3) (mul i %6))\n    (%8 (f32 3 270) (outer %7 %5))\n    (%9 (f32 90 4) (sub %3 %0))\n"
                 "    (%10 (f32 360) (reshape %9))\n    (%11 (f32 3 360) (outer i %10))\n    (%12 (f32 3 270) (gelu %8))\n"
                 "    (%13 (f32) (sum %11))\n    (%14 (f32 3 270) (add %12 %13))\n", "%14"),
    # groups of row values by row values, ragged; a scan from the last step to the first
    "groups": model([], "  (input a (f32 7 5 33))\n  (input b (f32 7 33 19))\n",
                    "    (%0 (f32 7 5 19) (matmul a b))\n    (%1 (f32 7 19 5) (transpose %0))\n    (%2 (f32 7 5 5) (matmul %0 %1))\n"
                    "    (%3 (f32 7 5 5) (softmax %2))\n    (%4 (f32 7 5 19) (matmul %3 %0))\n", "%4"),
    "reverse": model([f32("h0", 40, seed=8), quant("W", 40, 40, 8, 1, 9)], "  (input x (f32 6 40))\n",
                     "    (scan 6 reverse steps\n      (carry %0 (f32 40) h0)\n      (in %1 (f32 40) x)\n      (body\n"
                     "        (%2 (f32 40) (matmul %0 W))\n        (%3 (f32 40) (add %2 %1))\n        (%4 (f32 40) (tanh %3))\n      )\n"
                     "      (next %0 %4)\n      (emit %5 (f32 6 40) %3)\n    )\n    (%6 (f32 6 40) (softmax %5))\n", "%6"),
}


def check(text, rows, steps=False):
    with pytest.raises(RuntimeError):
        hip.emit_unit(text, hip.FIXED)  # the compiler refuses it
    p = hip.Program(text, flags=hip.FIXED, max_rows=max(rows, 64))
    q = hip.Program(text, flags=hip.FIXED | hip.INTERP, max_rows=max(rows, 64))
    x = np.random.default_rng(rows).normal(size=(rows, p.per)) * 3
    x[0, 0] = 20000.0
    xq = np.round(x * 65536).astype(np.int32)
    got, s0 = p.batch_fixed(xq)
    want, s1 = q.batch_fixed(xq)
    assert np.array_equal(got, want) and np.array_equal(s0, s1)


@pytest.mark.parametrize("rows", [1, 63, 200, 4100])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_steps_equal_interpreter(name, rows):
    print("case fixed steps", name, rows, flush=True)
    check(MODELS[name], rows)


SCAN = synth.ssm_tgir(d_model=16, d_inner=32, n_state=4, dt_rank=4, T=7, blocks=2, classes=3)
G = 65535 + 3  # more groups than a grid has in its third dimension
GROUPS = model([], "  (input a (f32 %d 2 3))\n  (input b (f32 %d 3 1))\n" % (G, G), "    (%%0 (f32 %d 2 1) (matmul a b))\n" % G, "%0")


@pytest.mark.parametrize("rows", [3, 130])
def test_scans_equal_interpreter(rows):
    print("case fixed scan", rows, flush=True)
    check(SCAN, rows)


def test_more_groups_than_a_grid_holds():
    print("case fixed groups", flush=True)
    check(GROUPS, 2)
