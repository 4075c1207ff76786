"""The roots of the cellular nodes against IEEE results: the reciprocal root
of every squared length a 3D or 4D jitter vector can have, and the fast
reciprocal root of a distance over whole binades at both ends and through the
range it is taken for; distances outside that range on the nodes themselves."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.tree import NodeSpec as S
import oracle
from conftest import assert_bitexact
from test_gpu_math import binade, cell_lengths, run

pytestmark = pytest.mark.gpu


def inv_sqrt(x):
    return np.float32(1.0) / np.sqrt(x)


@pytest.mark.parametrize("dims", [3, 4])
def test_every_jitter_length(gpu, dims):
    x = cell_lengths(dims)
    got = run(6, x, fn.DeviceArray(x.size), fn.DeviceArray(x.size))
    bad = np.flatnonzero(got.view(np.uint32) != inv_sqrt(x).view(np.uint32))
    assert bad.size == 0, "%d of %d, first at %r" % (bad.size, x.size, float(x[bad[0]]))


@pytest.mark.parametrize("e", [-60, -59, -31, -30, -13, -12, -5, -4, -3, -2, 23, 40, 41, 59, 60])
def test_distance_roots(gpu, e):
    x = binade(e)
    got = run(2, x, fn.DeviceArray(x.size), fn.DeviceArray(x.size))
    assert np.array_equal(got.view(np.uint32), inv_sqrt(x).view(np.uint32))


@pytest.mark.parametrize("jit", [fn.JIT_OFF, fn.JIT_SYNC])
@pytest.mark.parametrize("dims", [2, 3, 4])
def test_distances_beyond_the_fast_range(gpu, dims, jit):
    # no jitter: points on lattice points have distance 0 (whose root is NaN),
    # points next to them tiny ones; huge positions have huge or no distances
    near = np.float32([0, 1e-30, 1e-20, 3e-19, 1e-9, 1e-3, 0.5, 1.0, 1e9, 3e18, 1e20, 3e38, np.inf, np.nan])
    pos = [np.resize(near, 400), np.zeros(400, np.float32), np.resize(np.float32([0, 1e-25, 2]), 400), np.zeros(400, np.float32)][:dims]
    old = fn.set_jit_mode(jit)
    try:
        for tree_jitter in (0.0, 1.0):
            spec = S("CellularDistance", feature_scale=1.0, distance_function="Euclidean", return_type="Index0Add1",
                     distance_index_0=0, distance_index_1=1, grid_jitter=tree_jitter)
            got, _ = fn.Node.from_encoded(spec.encode()).gen_position_array(pos, seed=3)
            want, _ = oracle.Tree(spec.encode()).positions(pos, seed=3)
            assert_bitexact(got, want, "jitter %g" % tree_jitter)
    finally:
        fn.set_jit_mode(old)
