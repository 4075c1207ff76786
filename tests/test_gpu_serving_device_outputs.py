"""Serving requests whose destinations are device memory: the batch's kernels
write them in place, so neighbouring destinations inside one allocation, at
any float offset, must each hold their own request and nothing else."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd import workloads as W
from fastnoise2_amd.serve import ServeEngine, SERVE_PLAIN, SERVE_BATCHED, SERVE_GRAPH, SERVE_PERSISTENT
from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


class Slice:
    """`count` floats from float `at` of a DeviceArray."""

    def __init__(self, whole, at, count):
        self.count, self.ptr = count, whole.ptr + 4 * at


@pytest.mark.parametrize("mode", [SERVE_BATCHED, SERVE_GRAPH, SERVE_PLAIN, SERVE_PERSISTENT])
def test_device_slices_hold_their_request_alone(gpu, mode):
    node = fn.Node.from_encoded(W.fbm_simplex_2d().encode())
    eng = ServeEngine(hbm_budget_bytes=1 << 30, max_batch_points=1 << 16, mode=mode)
    tid = eng.add_tree(W.fbm_simplex_2d().encode())
    # below, at and above a block; one request beyond the slot's capacity, which runs in parts
    sizes = [(1, 1), (63, 1), (16, 16), (257, 1), (33, 31), (300, 301), (128, 128), (5, 3)]
    guard = -777.0
    gaps = [1, 3, 2, 1, 5, 1, 7, 1]
    total = sum(x * y + g for (x, y), g in zip(sizes, gaps)) + 1
    whole = fn.DeviceArray.from_host(np.full(total, guard, np.float32))
    at, ids, places = 0, [], []
    for k, ((x, y), gap) in enumerate(zip(sizes, gaps)):
        at += gap
        places.append(at)
        ids.append(eng.submit(tid, fn.grid_spec(2, [k * 100.0, -7.0], [x, y], seed=k), out=Slice(whole, at, x * y)))
        at += x * y
    ranges = [eng.wait(i)[1] for i in ids]
    got = whole.to_host()
    want = np.full(total, guard, np.float32)
    for k, ((x, y), p) in enumerate(zip(sizes, places)):
        ref, mm = node.gen_uniform_grid_2d(k * 100.0, -7.0, x, y, seed=k)
        want[p:p + x * y] = ref
        assert ranges[k] == mm
    assert_bitexact(got, want, "device slices")
    eng.close()
