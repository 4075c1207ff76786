"""Face counts of many chunks at once: a poll that finishes more surface
chunks than one launch takes, and chunk sizes around the kernel's tile of
256 voxels, against counts of the same blocks on the host."""
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.serve import ServeEngine, SERVE_BATCHED
from fastnoise2_amd.world import ChunkWorld, CHUNK_SURFACE
from test_gpu_world import TREE, host_summary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size, rng", [(1, 3.0), (6, 24.0), (7, 30.0), (33, 60.0)])
def test_many_surface_chunks_in_one_poll(gpu, size, rng):
    iso, seed = 0.05, 4
    eng = ServeEngine(hbm_budget_bytes=1 << 30, max_batch_points=1 << 20, mode=SERVE_BATCHED)
    world = ChunkWorld(eng, eng.add_tree(TREE.encode()), chunk_size=size, iso_surface=iso, load_range=rng, seed=seed, max_in_flight=700)
    world.update((2.0, 1.0, 3.0))
    got = world.poll(wait_all=True)
    surface = [r for r in got if r["state"] == CHUNK_SURFACE]
    assert len(got) > 30 and surface
    if size in (6, 7):
        assert len(surface) > 64
    node = fn.Node.from_encoded(TREE.encode())
    for r in surface[:3] + surface[60:70] + surface[-3:]:
        state, mm, quads, solid = host_summary(node, (r["x"], r["y"], r["z"]), size, iso, seed)
        assert (r["state"], r["quads"], r["solid_voxels"]) == (state, quads, solid)
    world.close()
    eng.close()
