"""The range of a call is gathered from a pair per block: calls around the
block size and beyond the largest grid, and calls whose blocks hold no number
at all, on the interpreter and on specialised kernels."""
import numpy as np
import pytest

import fastnoise2_amd as fn
from fastnoise2_amd.tree import NodeSpec as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jit", [fn.JIT_OFF, fn.JIT_SYNC])
@pytest.mark.parametrize("n", [1, 64, 255, 256, 257, 5000, 131072, 131073, (1 << 22) + 300])
def test_range_is_that_of_the_values(gpu, n, jit):
    old = fn.set_jit_mode(jit)
    try:
        node = fn.Node.from_encoded(S("Simplex", feature_scale=30.0).encode())
        rng = np.random.default_rng(n)
        x, y = (rng.uniform(-500, 500, n).astype(np.float32) for _ in range(2))
        spans = [(0, 0), (n // 2, n), (0, max(0, n - 1)), (0, n)]   # of NaN positions: none, half, all but one, all
        for lo, hi in spans:
            px = x.copy()
            px[lo:hi] = np.nan
            out, mm = node.gen_position_array([px, y])
            ok = out[~np.isnan(out)]
            assert np.isnan(out[lo:hi]).all()
            assert mm == ((float(ok.min()), float(ok.max())) if ok.size else (float("inf"), float("-inf")))
            dev = fn.DeviceArray(n)
            pos = [fn.DeviceArray.from_host(px), fn.DeviceArray.from_host(y)]
            assert node.generate_device(fn.positions_spec(pos), dev) == mm
    finally:
        fn.set_jit_mode(old)


def test_timed_launches_include_the_reduction(gpu):
    # 512 blocks of 256 points leave their pairs to the host, one more takes a
    # reduction launch, which costs at least a microsecond
    old = fn.set_jit_mode(fn.JIT_SYNC)
    try:
        node = fn.Node.from_encoded(S("Simplex", feature_scale=30.0).encode())
        out = fn.DeviceArray(131073)
        ms = {n: min(node.bench_device(fn.grid_spec(2, [0.0, 0.0], [n, 1]), out, warmup=5, iters=200)[0] for _ in range(5))
              for n in (131072, 131073)}
        assert ms[131073] - ms[131072] > 1.0e-3
    finally:
        fn.set_jit_mode(old)
