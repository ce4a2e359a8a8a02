"""The library's host code around the device (chunks, slots, error paths,
allocations) on a host without one: tests/cpp/fake_device.cpp answers the HIP
calls in host memory and checks every copy against its allocations. Kernels do
nothing there, so these tests look at what is asked of the device, not at
values. Each runs in a process of its own, where the runtime is preloaded."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(not shutil.which("g++") or not os.path.exists(ROCM + "/hip/hip_runtime_api.h"), reason="no g++ or HIP headers")

HEAD = """
import ctypes, gc, os, sys
import numpy as np
sys.path.insert(0, %r)
from technograd_amd import hip, synth
fake = ctypes.CDLL(os.environ["FAKE_DEVICE"])
for f in ("fake_pending", "fake_out_of_range", "fake_launches", "fake_used", "fake_largest"):
    getattr(fake, f).restype = ctypes.c_long
for f in ("fake_fail_launch", "fake_limit"):
    getattr(fake, f).argtypes = [ctypes.c_long]
hip.init(0)
def linear(k, c):
    return synth.linear_tgir("m", synth.rand(1, 0.05, c * k).reshape(c, k), 8)
def pinned(a):
    hb = hip.HostBuffer(max(a.nbytes, 1))
    v = hb.array(a.dtype, a.shape)
    v[:] = a
    return hb, v
""" % ROOT


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_device.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + ROCM, "-o", so, os.path.join(ROOT, "tests", "cpp", "fake_device.cpp")], check=True)

    def go(code):
        env = dict(os.environ, FAKE_DEVICE=so, LD_PRELOAD=":".join(filter(None, (so, os.environ.get("LD_PRELOAD")))))
        r = subprocess.run([sys.executable, "-c", HEAD + code], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    return go


def test_a_chunk_not_down_yet_is_no_error(run):
    """Asking for a chunk that is still on its way leaves "not ready" as the
    runtime's last error, which the launch check of the next pass must not
    report."""
    run("""
prog = hip.Program(linear(64, 40), max_rows=7)
for n in (8, 29, 200):
    y, _ = prog.batch(np.ones((n, 64), np.float32))
    assert fake.fake_out_of_range() == 0 and fake.fake_pending() == 0
""")
@pytest.mark.parametrize("max_rows", [1, 7, 33, 63, 64, 65, 300])
def test_pinned_rows_stay_in_the_slots(run, max_rows):
    """Rows and outputs, pinned or not, travel in chunks no larger than the
    slots, which hold at most max_rows rows."""
    run("""
prog = hip.Program(linear(64, 40), max_rows=%d)
for n in (1, 2, 32, 63, 64, 65, 129, 500):
    (bx, x), (by, y) = pinned(np.ones((n, 64), np.float32)), pinned(np.zeros((n, 40), np.float32))
    for rows, out in ((x, y), (x, np.array(y)), (np.array(x), y), (np.array(x), np.array(y))):
        prog.batch(rows, out)
        assert fake.fake_out_of_range() == 0, n
        assert fake.fake_pending() == 0, n
    bx.free(), by.free()
""" % max_rows)


@pytest.mark.parametrize("pin", [False, True])
def test_nothing_is_in_flight_after_an_error(run, pin):
    """A pass that fails part way through a batch: when the call has returned
    its error, no transfer is left that could write the caller's memory or the
    slots of the next call, and the next call works."""
    run("""
prog = hip.Program(linear(64, 40), max_rows=70)
(bx, x), (by, y) = pinned(np.ones((500, 64), np.float32)), pinned(np.zeros((500, 40), np.float32))
if not %r:
    x, y = np.array(x), np.array(y)
first = fake.fake_launches()
prog.batch(x, y)
for n in range(1, fake.fake_launches() - first + 1):
    fake.fake_fail_launch(n)
    try:
        prog.batch(x, y)
        raise SystemExit("launch %%d of the batch failed without an error" %% n)
    except RuntimeError:
        pass
    assert fake.fake_pending() == 0, n
    prog.batch(x, y)
    assert fake.fake_pending() == 0 and fake.fake_out_of_range() == 0
""" % pin)


def test_programs_share_their_copy_threads(run):
    """Any number of programs that copy pageable rows hold one set of host
    threads, also while several run, and none once they are freed."""
    run("""
import threading
def threads():
    return len(os.listdir("/proc/self/task"))
base = threads()
x = np.ones((9000, 64), np.float32)  # 2.3 MB: copies worth sharing
progs = [hip.Program(linear(64, 64), max_rows=9000) for _ in range(12)]
for p in progs:
    p.batch(x)
assert threads() <= base + 11, (base, threads())
calls = [threading.Thread(target=lambda p=p: [p.batch(x) for _ in range(20)]) for p in progs]
for t in calls:
    t.start()
for t in calls:
    t.join()
assert threads() <= base + 11, (base, threads())
for p in progs[:-1]:
    p.close()
y, _ = progs[-1].batch(x)  # the last one still has them
progs[-1].close()
assert threads() == base, (base, threads())
progs = [hip.Program(linear(64, 64), max_rows=9000) for _ in range(2)]
for p in progs:
    p.batch(x)
    p.close()
assert threads() == base, (base, threads())
""")


def test_an_error_is_reported_once(run):
    """A program or decoder that does not fit the device's memory is refused,
    leaves none of it taken, and the calls after it are not refused for it."""
    run("""
prog = hip.Program(linear(64, 40), max_rows=7)
x = np.ones((20, 64), np.float32)
prog.batch(x)
qwen = hip.Program(synth.qwen3_tgir("q", T=8, rope_len=70, L=1, D=64, NQ=4, NKV=2, HD=64, FF=96, V=320), max_rows=1)
big, used = linear(512, 512), fake.fake_used()
for make in (lambda: hip.Program(big, max_rows=4096), lambda: hip.Decoder(qwen, 4, 64, 70)):
    for left in (4096, 1 << 15, 1 << 17, 300000, 1 << 19, 1 << 20):
        fake.fake_limit(used + left)
        try:
            make()
            raise SystemExit("made in %d bytes" % left)
        except RuntimeError:
            pass
        gc.collect()
        assert fake.fake_used() == used, (left, fake.fake_used() - used)
        prog.batch(x)
    fake.fake_limit(1 << 40)
""")


def test_decoder_needs_no_more_than_one_heads_scores(run):
    """Scores of all heads at once are taken where they fit: with less device
    memory left the decoder keeps fewer heads' and runs the rest of them in
    further launches, down to one head's."""
    run("""
S, T0, NQ = 2, 256, 8
prog = hip.Program(synth.qwen3_tgir("q", T=8, rope_len=T0 + 2, L=1, D=64, NQ=NQ, NKV=2, HD=64, FF=96, V=320), max_rows=1)
base, head = fake.fake_used(), 4 * S * T0 * T0
prompt, tokens = hip.DeviceBuffer(4 * S * T0), hip.DeviceBuffer(8 * S)
def make(left):
    fake.fake_limit(fake.fake_used() + left)
    dec = hip.Decoder(prog, S, T0, T0 + 2)
    used, n = fake.fake_used(), fake.fake_launches()
    dec.generate_device(prompt.ptr, S, T0, 2, tokens.ptr, None)  # (the failed allocations are not its launch error)
    prog.sync()
    assert fake.fake_out_of_range() == 0
    n = fake.fake_launches() - n
    dec.close()
    return used - base, n
base = fake.fake_used()
full, launches = make(1 << 40)
least = full - (NQ - 1) * head
for heads in (1, 2, 3, 4, 7):
    used, n = make(least + (heads - 1) * head)
    assert used <= least + (heads - 1) * head and n > launches, (heads, used, n, launches)
try:
    make(least - 1)
    raise SystemExit("a decoder in less memory than it needs")
except RuntimeError as e:
    assert "out of memory" in str(e)
assert make(1 << 40) == (full, launches)
""")


def test_a_steps_launches_do_not_grow_with_the_heads(run):
    """All heads' output projections of a decoder step are one product,
    however many heads there are."""
    run("""
counts = []
for NQ in (8, 64, 72, 144):
    prog = hip.Program(synth.qwen3_tgir("q", T=8, rope_len=8, L=1, D=32, NQ=NQ, NKV=NQ // 8, HD=48, FF=32, V=96), max_rows=1)
    dec = hip.Decoder(prog, 2, 4, 8)
    prompt = hip.DeviceBuffer(4 * 8)
    n = fake.fake_launches()
    dec.generate_device(prompt.ptr, 2, 4, 1, None, None)
    m = fake.fake_launches()
    dec.generate_device(prompt.ptr, 2, 4, 2, None, None)
    counts.append((m - n, fake.fake_launches() - m))
    dec.close()
assert len(set(counts)) == 1, counts
""")


def test_any_number_of_groups_is_launched(run):
    """A Q16.16 batched product of more groups than a grid has in its third
    dimension."""
    run("""
for G in (65535, 65536, 200000):
    text = ("(tgir 1\\n  (model m)\\n  (input a (f32 %d 2 3))\\n  (input b (f32 %d 3 1))\\n  (block\\n    (%%0 (f32 %d 2 1) (matmul a b))\\n"
            "  )\\n  (output %%0))\\n" % (G, G, G))
    hip.Program(text, flags=hip.FIXED, max_rows=2).batch_fixed(np.ones((2, G * 9), np.int32))
""")


def test_the_fixed_step_models_run_an_instruction_at_a_time(run):
    """Every model of test_gpu_fixed_steps.py takes the executor that the file
    tests, a launch or more per instruction; the interpreter it is compared
    with launches once a pass."""
    run("""
sys.path.insert(0, os.path.join(%r, "tests"))
import test_gpu_fixed_steps as F
for name, text in sorted(F.MODELS.items()) + [("scan", F.SCAN), ("groups", F.GROUPS)]:
    n = []
    for flags in (hip.FIXED, hip.FIXED | hip.INTERP):
        p = hip.Program(text, flags=flags, max_rows=64)
        a = fake.fake_launches()
        p.batch_fixed(np.ones((3, p.per), np.int32))
        n.append(fake.fake_launches() - a)
    assert n[0] >= 3 and n[1] == 1, (name, n)
""" % ROOT)
