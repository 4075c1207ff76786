"""The LDS tables behind gradient selection and the orthogonal warp matrices
against the oracle, bit for bit: every leaf alone and fused into fractals, and
the simplex-type warps, in 2D, 3D and 4D, on the interpreter, on specialised
kernels and in serving batches that mix programs with different tables, over
enough points to read every entry, with steps of either sign and huge and
non-finite offsets."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.serve import ServeEngine, SERVE_BATCHED, SERVE_PERSISTENT
from fastnoise2_amd.tree import NodeSpec as S
import oracle
from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

LEAVES = ["Perlin", "Value", "Simplex", "SuperSimplex"]
TREES = {leaf: S(leaf, feature_scale=4.0) for leaf in LEAVES}
TREES.update({"FBm " + leaf: S("FractalFBm", source=S(leaf, feature_scale=60.0, seed_offset=3), octaves=4) for leaf in LEAVES})
for w in ("DomainWarpSimplex", "DomainWarpSuperSimplex"):
    for scheme in ("Orthogonal Gradient Matrix", "Gradient Outer Product"):
        TREES["%s %s" % (w, scheme)] = S(w, source=S("Perlin", feature_scale=35.0), warp_amplitude=12.0, feature_scale=5.0,
                                         vectorization_scheme=scheme)
TREES["rotated 2D to 3D"] = S("DomainRotate", source=S("FractalFBm", source=S("Simplex", feature_scale=50.0), octaves=2), yaw=0.7, pitch=0.3)

GRIDS = [   # offset, step; counts by dimensionality below
    ((0.0, 0.0, 0.0, 0.0), (1.0, 1.0, 1.0, 1.0)),
    ((-7.5, 3.25, 100.0, 2.0), (-9.0, 7.0, 13.0, 3.0)),
    ((3.0e7, -2.0e8, 1.0e6, 5.0e7), (16.0, 64.0, 1.0, 32.0)),
    ((1.0e11, 0.0, -3.0e10, 1.0), (1.0e8, 1.0, 1.0e9, 1.0)),
    ((float("inf"), 1.0, 2.0, 3.0), (1.0, 1.0, 1.0, 1.0)),
    ((1.0, float("nan"), 2.0, 3.0), (1.0, 1.0, 1.0, 1.0)),
]
COUNTS = {2: (37, 29), 3: (13, 9, 11), 4: (7, 5, 6, 6)}


@pytest.fixture(params=[fn.JIT_OFF, fn.JIT_SYNC], ids=["interpreter", "specialised"])
def jit(gpu, request):
    old = fn.set_jit_mode(request.param)
    yield request.param
    fn.set_jit_mode(old)


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("name", TREES)
def test_grids_match_oracle(jit, name, dims):
    node = fn.Node.from_encoded(TREES[name].encode())
    tree = oracle.Tree(TREES[name].encode())
    gen = {2: node.gen_uniform_grid_2d, 3: node.gen_uniform_grid_3d, 4: node.gen_uniform_grid_4d}[dims]
    for offset, step in GRIDS:
        got, mm = gen(*offset[:dims], *COUNTS[dims], *step[:dims], seed=-5)
        want, want_mm = tree.grid(offset[:dims], COUNTS[dims], step[:dims], seed=-5)
        assert_bitexact(got, want, "%s at %s" % (name, (offset, step)))
        assert mm == want_mm or not np.isfinite(want).any()


@pytest.mark.parametrize("mode", [SERVE_BATCHED, SERVE_PERSISTENT])
def test_batches_match_oracle(jit, mode):
    # the blocks of a batch fill the tables of their own job's program (the
    # work queue's those of its kernel)
    eng = ServeEngine(hbm_budget_bytes=1 << 30, max_batch_points=1 << 18, mode=mode)
    names = ["Value", "Perlin", "FBm Simplex", "DomainWarpSimplex Gradient Outer Product", "DomainWarpSimplex Orthogonal Gradient Matrix"]
    ids = {}
    for n in names:
        t = eng.add_tree(TREES[n].encode())
        for d in (2, 3, 4):
            ids[n, d] = eng.submit(t, fn.grid_spec(d, [5.0] * d, COUNTS[d], [3.0] * d, seed=9))
    for (n, d), rid in ids.items():
        want, mm = oracle.Tree(TREES[n].encode()).grid([5.0] * d, COUNTS[d], [3.0] * d, seed=9)
        got, got_mm, _ = eng.wait(rid)
        assert_bitexact(got, want, "%s %dD" % (n, d))
        assert got_mm == mm
    eng.close()
