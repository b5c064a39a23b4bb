"""Smoothing lengths that fall from above 1 to below it: the scans after the
one at the larger h then sum the members of that scan only (the reference's
neighbour cache), over that scan's box.  Near the fixed point the lists have
the bits of the cell walk (density_flat) there too, for each number of lanes
that they take."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,over", [
    (3000, {}), (3000, {"small_n_lanes": 0}), (70000, {}), (80000, {"sparse": True}),
    (3000, {"max_nr_iterations": 4}), (3000, {"n_neighbours_estim": 64}),
])
def test_falling_below_one_bits(sph, tables256, n, over):
    over = dict(over)
    sparse = over.pop("sparse", False)
    # a mean h of 0.9
    ic = _stir(_ball(n, n, radius=0.9 / (1.2348 * (4.19 / n) ** (1 / 3))), n)
    g = np.random.default_rng(1)
    ic["h"] = g.uniform(0.85, 1.4, n).astype(np.float32)
    active = (g.random(n) < 0.025).astype(np.uint8)
    if sparse:
        over["activity_rule"] = sph.SPH_ACTIVE_README
    over.setdefault("max_nr_iterations", 400)
    out = []
    for flat in (1, 0):
        prm = sph.default_params(density_stop=1, density_eta=2.5e-6, density_flat=flat, **over)
        ctx = sph.Context(prm, ic, tables256)
        if sparse:
            ctx.upload("active", active)
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f) for f in ("h", "rho", "gradterm", "balsara", "pressure", "nr_iters")})
    assert np.mean(out[0]["h"] < 1) > 0.5 or sparse
    for f in out[0]:
        a, b = (o[f].view(np.int32) for o in out)
        assert np.array_equal(a, b), (f, np.mean(a != b))
