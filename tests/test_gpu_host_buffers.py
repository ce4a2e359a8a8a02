"""tg_hip_batch with rows, outputs and steps in pinned memory from
tg_hip_host_alloc (moved over PCIe directly, in smaller chunks) against the
same call on ordinary numpy arrays (copied through the library's staging
slots): the same bits, for a quantized model over several chunks and for a
think model's outputs and steps, with buffers at an offset inside their
allocations."""
import os

import numpy as np
import pytest

from technograd_amd import hip, synth

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


@pytest.fixture(scope="module", autouse=True)
def device():
    print("host buffers: tg_hip_init(0)", flush=True)
    hip.init(0)


def pinned_like(a, offset=64):
    """a copy of a in a HostBuffer, `offset` bytes into the allocation"""
    hb = hip.HostBuffer(a.nbytes + offset)
    v = hb.array(np.uint8, (a.nbytes + offset,))[offset:].view(a.dtype).reshape(a.shape)
    v[:] = a
    return hb, v


@pytest.mark.parametrize("case", ["config2_4096", "latent_f32"])
def test_pinned_buffers_equal_pageable(case):
    print("case host buffers", case, flush=True)
    if case == "config2_4096":
        text = synth.linear_tgir("linear4096", synth.config2_weight(), 4)
        x = synth.normal(2, 1.0, 4096 * 4096).reshape(4096, 4096)
    else:
        with open(os.path.join(GOLDEN, case + ".tgir")) as f:
            text = f.read()
        x = np.load(os.path.join(GOLDEN, case + ".npz"))["x"]
    prog = hip.Program(text, max_rows=len(x))
    want, wsteps = prog.batch(x)
    bx, px = pinned_like(np.ascontiguousarray(x, np.float32))
    by, py = pinned_like(np.zeros_like(want))
    bs, ps = pinned_like(np.zeros_like(wsteps))
    got, gsteps = prog.batch(px, py, ps)
    assert got is py and gsteps is ps
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(gsteps, wsteps)
    # rows pinned, outputs not (and the other way round)
    o1, _ = prog.batch(px)
    o2, _ = prog.batch(x, py, ps)
    assert np.array_equal(o1.view(np.uint32), want.view(np.uint32)) and np.array_equal(o2.view(np.uint32), want.view(np.uint32))
    for b in (bx, by, bs):
        b.free()
    prog.close()


def test_host_free_refuses_foreign_pointers():
    a = np.zeros(16, np.float32)
    assert hip.lib().tg_hip_host_free(a.ctypes.data) == -1
    hb = hip.HostBuffer(64)
    assert hip.lib().tg_hip_host_free(hb.ptr + 16) == -1  # inside, but not the start
    hb.free()


def test_pageable_rows_in_one_chunk_and_many():
    """One, two and several chunks of staged rows, slots refilled, shared
    copies and whole ones: the bits of the same rows on device buffers."""
    W = synth.rand(1, 0.05, 96 * 64).reshape(96, 64)
    text = synth.linear_tgir("chunks", W, 8)
    n = 150001  # 8 MiB chunks of 21845 rows of outputs: seven, the slots used twice
    x = synth.rand(3, 1.0, n * 64).reshape(n, 64)
    prog = hip.Program(text, max_rows=n)
    dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(n * 96 * 4)
    prog.batch_device(dx.ptr, n, dy.ptr)
    prog.sync()
    want = dy.to_array(np.float32, (n, 96))
    for rows in (1, 21845, 21846, n):
        print("case host chunks", rows, flush=True)
        got, steps = prog.batch(x[:rows])
        assert np.array_equal(got.view(np.uint32), want[:rows].view(np.uint32)) and not steps.any()
    prog.close()


@pytest.mark.parametrize("max_rows", [1, 7, 33])
def test_pinned_rows_in_passes_of_a_small_program(max_rows):
    """Pinned rows and outputs through a program of few rows a pass: passes of
    at most that many, the bits of the same rows one pass at a time."""
    print("case small pinned", max_rows, flush=True)
    text = synth.linear_tgir("small", synth.rand(1, 0.05, 40 * 64).reshape(40, 64), 8)
    n = 2 * max_rows + 65
    x = synth.rand(4, 1.0, n * 64).reshape(n, 64).astype(np.float32)
    prog = hip.Program(text, max_rows=max_rows)
    want = np.concatenate([prog.batch(x[a:a + max_rows])[0] for a in range(0, n, max_rows)])
    bx, px = pinned_like(x)
    by, py = pinned_like(np.zeros((n, 40), np.float32))
    got, _ = prog.batch(px, py)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    for b in (bx, by):
        b.free()
    prog.close()
