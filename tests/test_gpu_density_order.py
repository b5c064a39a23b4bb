"""density_order in the pass that reads it, the walk over the cells: the
waves take each window's particles in order of their previous iteration
counts in place of slot order, and no particle's result changes a bit."""
import numpy as np
import pytest

from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", [
    {"density_flat": 1}, {"density_lanes": 16, "small_n_lanes": 0}, {"density_lanes": 8, "small_n_lanes": 0, "density_flat": 1},
])
def test_walk_order_bits(sph, tables256, impact, over):
    n = 30011  # the last window is ragged
    ic = _stir(impact(n, 14), 3)
    out = {}
    for order in (0, 16, 32, 512):
        ctx = sph.Context(sph.default_params(density_order=order, **over), ic, tables256)
        g = np.random.default_rng(4)
        h0 = ic["h"] * g.uniform(0.7, 1.4, n).astype(np.float32)
        for _ in range(2):  # the second pass in the order of the first one's counts
            ctx.upload("h", h0)
            ctx.sort()
            ctx.density()
        out[order] = {k: ctx.download(k) for k in ("h", "rho", "gradterm", "balsara", "pressure", "nr_iters")}
        ctx.close()
    assert out[0]["nr_iters"].max() > out[0]["nr_iters"].min() + 3
    for order in (16, 32, 512):
        for k in out[0]:
            assert np.array_equal(out[0][k].view(np.int32), out[order][k].view(np.int32)), (order, k)
