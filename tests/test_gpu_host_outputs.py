"""Host outputs around the sizes where their way back changes (written to
pinned memory by the kernel; copied; staged in chunks), on programs that walk
rows and bricks, against the oracle and the memory around the output."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.tree import NodeSpec as S
import oracle
from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

TREES = {"rows": S("Simplex", feature_scale=20.0), "bricks": S("CellularDistance", feature_scale=20.0, distance_function="Euclidean")}


@pytest.mark.parametrize("jit", [fn.JIT_OFF, fn.JIT_SYNC])
@pytest.mark.parametrize("name", TREES)
def test_outputs_of_every_way_back(gpu, name, jit):
    old = fn.set_jit_mode(jit)
    try:
        node = fn.Node.from_encoded(TREES[name].encode())
        tree = oracle.Tree(TREES[name].encode())
        for count in [(1, 1), (63, 65), (262143, 1), (512, 512), (2097152, 1), (2097153, 1)]:
            n = count[0] * count[1]
            buf = np.full(n + 8, -777.0, np.float32)
            mm = np.zeros(2, np.float32)
            fn.lib().fnGenUniformGrid2D(node.handle, fn._fp(buf[3:]), 5.0, -7.0, count[0], count[1], 1.0, 1.0, 21, fn._fp(mm))
            assert fn.last_error() == ""
            want, want_mm = tree.grid((5.0, -7.0), count, seed=21, lanes=16, threads=8)
            assert_bitexact(buf[3:3 + n], want, "%s %s" % (name, count))
            assert (buf[:3] == -777.0).all() and (buf[3 + n:] == -777.0).all()
            assert tuple(mm) == want_mm
    finally:
        fn.set_jit_mode(old)


def test_staged_positions_and_outputs_share_the_ring(gpu):
    n = 300001
    rng = np.random.default_rng(5)
    xs = [rng.uniform(-500, 500, n).astype(np.float32) for _ in range(3)]
    node = fn.Node.from_encoded(TREES["rows"].encode())
    out = np.empty(n, np.float32)
    mm = np.zeros(2, np.float32)
    for n in (300001, 200000):
        xs, out = [x[:n].copy() for x in xs], out[:n]
        fn.lib().fnGenPositionArray3D(node.handle, fn._fp(out), n, *[fn._fp(x) for x in xs], 0.5, -0.25, 3.0, 9, fn._fp(mm))
        assert fn.last_error() == ""
        want, want_mm = oracle.Tree(TREES["rows"].encode()).positions(xs, offset=(0.5, -0.25, 3.0), seed=9, lanes=16)
        assert_bitexact(out, want, "positions")
        assert tuple(mm) == want_mm
