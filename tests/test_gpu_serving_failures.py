"""Serving requests that fail: a destination that its allocation cuts short is
refused by the copy into it, and the engine and its other requests go on."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd import workloads as W
from fastnoise2_amd.serve import ServeEngine, SERVE_PLAIN, SERVE_BATCHED, SERVE_GRAPH, SERVE_PERSISTENT
from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

MODES = [SERVE_BATCHED, SERVE_GRAPH, SERVE_PLAIN, SERVE_PERSISTENT]


class Slice:
    """`count` floats from float `at` of a DeviceArray or PinnedArray (or of what follows it)."""

    def __init__(self, whole, at, count):
        self.count, self.ptr = count, whole.ptr + 4 * at


def engine(mode, capacity=1 << 16):
    eng = ServeEngine(hbm_budget_bytes=1 << 30, max_batch_points=capacity, mode=mode)
    return eng, eng.add_tree(W.fbm_simplex_2d().encode())


def spec(n):
    return fn.grid_spec(2, [3.0, -7.0], [n, 1], seed=2)


def alone(n):
    return fn.Node.from_encoded(W.fbm_simplex_2d().encode()).gen_uniform_grid_2d(3.0, -7.0, n, 1, seed=2)


@pytest.mark.parametrize("jit", [fn.JIT_OFF, fn.JIT_SYNC])
@pytest.mark.parametrize("mode", MODES)
def test_a_failed_request_does_not_fail_the_next(gpu, mode, jit):
    # a few floats too many, which still lie on the allocation's last page
    old = fn.set_jit_mode(jit)
    try:
        eng, tid = engine(mode)
        pinned = fn.PinnedArray(1000)
        want, mm = alone(1000)
        for at, n in ((0, 1001), (990, 11)):
            rid = eng.submit(tid, spec(n), out=Slice(pinned, at, n))
            with pytest.raises(RuntimeError):
                eng.wait(rid)
            got, got_mm, _ = eng.wait(eng.submit(tid, spec(1000)))
            assert_bitexact(got, want, "after the refusal")
            assert got_mm == mm
        eng.close()
    finally:
        fn.set_jit_mode(old)


@pytest.mark.parametrize("mode", MODES)
def test_device_destinations_beyond_their_allocation_are_refused(gpu, mode):
    # the batch's kernels write device destinations themselves, these not
    eng, tid = engine(mode)
    whole = fn.DeviceArray.from_host(np.full(1000, -777.0, np.float32))
    for at, n in ((0, 1001), (990, 11), (999, 2)):
        rid = eng.submit(tid, spec(n), out=Slice(whole, at, n))
        with pytest.raises(RuntimeError):
            eng.wait(rid)
        assert (whole.to_host() == -777.0).all()
    # up to the allocation's last float
    got_mm = eng.wait(eng.submit(tid, spec(1000), out=Slice(whole, 0, 1000)))[1]
    want, mm = alone(1000)
    assert_bitexact(whole.to_host(), want, "after the refusals")
    assert got_mm == mm
    eng.close()


def test_a_failed_batch_has_ended_when_its_requests_return(gpu):
    # full batches keep the slots busy while a large request into device
    # memory and one that is refused queue up behind them and share a batch
    # (tried again should the dispatcher have taken the first alone)
    n = 1 << 22
    grid = [fn.grid_spec(3, [3.0, -7.0, 1.0], [128, 128, z], seed=2) for z in (n >> 14, n >> 15)]
    enc = W.serving_tree().encode()
    old = fn.set_jit_mode(fn.JIT_OFF)
    try:
        eng = ServeEngine(hbm_budget_bytes=1 << 30, max_batch_points=n, mode=SERVE_BATCHED)
        tid = eng.add_tree(enc)
        want, _ = fn.Node.from_encoded(enc).gen_uniform_grid_3d(3.0, -7.0, 1.0, 128, 128, n >> 15, seed=2)
        short, busy = fn.PinnedArray(1000), [fn.DeviceArray(n) for _ in range(12)]
        eng.wait(eng.submit(tid, grid[0], out=busy[0]))   # tunes the tree
        eng.wait(eng.submit(tid, spec(1000)))
        for _ in range(5):
            whole = fn.DeviceArray.from_host(np.zeros(n // 2, np.float32))
            first = [eng.submit(tid, grid[0], out=b) for b in busy]
            good, bad = eng.submit(tid, grid[1], out=whole), eng.submit(tid, spec(1001), out=Slice(short, 0, 1001))
            with pytest.raises(RuntimeError):
                eng.wait(bad)
            got = whole.to_host()
            try:
                eng.wait(good)
            except RuntimeError:
                break
            finally:
                for rid in first:
                    eng.wait(rid)
        else:
            pytest.fail("the two requests never shared a batch")
        assert_bitexact(got, want, "the batch's other request")
        eng.close()
    finally:
        fn.set_jit_mode(old)


@pytest.mark.parametrize("device_outputs", [False, True])
def test_a_replay_that_stops_waits_for_what_it_submitted(gpu, device_outputs):
    # its output buffers are freed when it returns
    eng, tid = engine(SERVE_BATCHED)
    specs = [spec(1 << 16)] * 40
    with pytest.raises(RuntimeError, match="unknown tree id"):
        eng.replay([tid] * 39 + [tid + 1], specs, None, 64, device_outputs=device_outputs)
    assert eng.stats()["completed"] == 39
    eng.close()
