"""Cheap programs write four points per lane: grids whose rows end inside a
lane's four points, totals that are no multiple of four, outputs off 16-byte
alignment (which keep one point per lane) and NaN values, and totals at each
change of the launch's run length and block count, against the oracle and the
neighbouring memory."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.tree import NodeSpec as S
import oracle
from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

TREES = {
    "checkerboard": S("Checkerboard", feature_scale=3.0),
    "white": S("White"),
    "constant": S("Constant", value=-2.5),
    "gradient sum": S("Add", lhs=S("Gradient", multiplier_x=0.5, multiplier_y=-0.25), rhs=S("Checkerboard", feature_scale=7.0)),
}
COUNTS = {2: [(1, 1), (3, 1), (4, 5), (5, 7), (64, 3), (1023, 9), (1, 130), (4099, 2100)], 3: [(1, 1, 3), (5, 3, 2), (8, 8, 8), (31, 17, 9)],
          4: [(3, 2, 5, 2), (8, 4, 3, 3)]}


class Slice:
    def __init__(self, whole, at):
        self.ptr = whole.ptr + 4 * at


@pytest.mark.parametrize("name", TREES)
def test_wide_grids_match_oracle(gpu, name):
    old = fn.set_jit_mode(fn.JIT_SYNC)
    try:
        node = fn.Node.from_encoded(TREES[name].encode())
        tree = oracle.Tree(TREES[name].encode())
        for d, counts in COUNTS.items():
            for count in counts:
                for offset in ([-3.0, 2.5, 0.0, 1.0][:d], [float("nan"), 1.0, 2.0, 3.0][:d]):
                    n = int(np.prod(count))
                    want, want_mm = tree.grid(offset, count, seed=11)
                    for at in (4, 5):   # on and off 16-byte alignment
                        whole = fn.DeviceArray.from_host(np.full(n + 12, -777.0, np.float32))
                        mm = node.generate_device(fn.grid_spec(d, offset, count, seed=11), Slice(whole, at).ptr)
                        got = whole.to_host()
                        assert_bitexact(got[at:at + n], want, "%s %s" % (name, count))
                        assert (got[:at] == -777.0).all() and (got[at + n:] == -777.0).all()
                        assert mm == want_mm or not np.isfinite(want).any()
                        node.generate_device(fn.grid_spec(d, offset, count, seed=11), Slice(whole, at).ptr, minmax=False)
                        assert_bitexact(whole.to_host(), got, "without a range")
    finally:
        fn.set_jit_mode(old)


# 2^24 points, the last with runs of four rounds; a row more, runs of two, and
# more blocks than a call with a range has; the same with ragged rows; 2^25 and a tail
LARGE = [(4096, 4096), (4096, 4097), (8191, 2051), (8191, 4099)]


@pytest.mark.parametrize("name", ["white", "gradient sum"])
def test_wide_runs_match_oracle(gpu, name):
    old = fn.set_jit_mode(fn.JIT_SYNC)
    try:
        node = fn.Node.from_encoded(TREES[name].encode())
        tree = oracle.Tree(TREES[name].encode())
        for count in LARGE:
            n = count[0] * count[1]
            want, want_mm = tree.grid([-3.0, 2.5], count, seed=11, lanes=16, threads=8)
            whole = fn.DeviceArray.from_host(np.full(n + 12, -777.0, np.float32))
            for ranged in (True, False):
                mm = node.generate_device(fn.grid_spec(2, [-3.0, 2.5], count, seed=11), Slice(whole, 4).ptr, minmax=ranged)
                got = whole.to_host()
                assert_bitexact(got[4:4 + n], want, "%s %s" % (name, count))
                assert (got[:4] == -777.0).all() and (got[4 + n:] == -777.0).all()
                assert not ranged or mm == want_mm
                assert fn.lib().fn2Memcpy(whole.ptr, np.full(n + 12, -777.0, np.float32).ctypes.data, 4 * (n + 12), 0) == 0
    finally:
        fn.set_jit_mode(old)
