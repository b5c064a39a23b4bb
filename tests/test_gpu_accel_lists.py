"""The acceleration pass from pair lists where they can go wrong: fewer
particles than a wave, ragged waves, lists and bins that overflow into the
launch with a wave per particle and beyond it, radii that differ from pair to
pair, grids that the boxes wrap around, long walks of nearly empty cells, and
active particles spread over the whole list.  One thread per particle is the
order of the lists at accel_lanes 0 too, and lane_split keeps the walk: the
same bits.  For 8 and 16 lanes only the order of at most a few hundred terms
differs: each sum is off by 300 * 2^-24 of the sum of their magnitudes at
most, 2e-5, and those are below 5 times the result in the 2-norm."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,over", [
    (1, {}), (7, {}), (9, {}), (129, {}), (5000, {}), (70001, {}),
    (4000, {"cell_width": 0.5}), (4000, {"cell_width": 0.03}),
    (3000, {"cell_power": 4}), (500, {"cell_power": 2}), (200, {"cell_power": 1}),
    (6000, {"clumps": True}), (6000, {"radii": True}), (40000, {"sparse": True}),
])
def test_accel_lists(sph, tables256, n, over):
    over = dict(over)
    clumps, radii, sparse = (over.pop(k, False) for k in ("clumps", "radii", "sparse"))
    ic = _stir(_ball(n, n, radius=3.0 if sparse else 1.0), n)
    g = np.random.default_rng(6)
    if clumps:
        for first, count, at in ((0, 300, 20.3), (300, 1500, 19.7)):
            ic["pos"][first:first + count, :3] = at + 0.02 * g.standard_normal((count, 3))
    if sparse:
        over["activity_rule"] = sph.SPH_ACTIVE_README
    active = (g.random(n) < 0.025).astype(np.uint8) if sparse else np.ones(n, np.uint8)
    out = {}
    for lanes, split in ((0, 1), (0, 0), (8, 0), (16, 0)):
        prm = sph.default_params(accel_lanes=lanes, list_accel_lanes=lanes, lane_split=split, small_n_lanes=0, **over)
        ctx = sph.Context(prm, ic, tables256)
        if sparse:
            ctx.upload("active", active)
        ctx.sort()
        ctx.density()
        if radii:
            h = ctx.download("h")
            h[::50] *= 3
            ctx.upload("h", h)
        # the walk's density sums come in another order: one set of fields for all
        for f in ("h", "rho", "pressure", "soundspeed", "gradterm", "balsara"):
            if (lanes, split) == (0, 1):
                out[f] = ctx.download(f)
            else:
                ctx.upload(f, out[f])
        ctx.acceleration()
        out[lanes, split] = {f: ctx.download(f)[active > 0] for f in ("acc", "du", "dhdt", "next_active")}
    walk = out[0, 1]
    for f in walk:
        assert np.array_equal(walk[f].view(np.int32), out[0, 0][f].view(np.int32)), f
    for lanes in (8, 16):
        for f in ("acc", "du", "dhdt"):
            a, b = walk[f].astype(np.float64), out[lanes, 0][f].astype(np.float64)
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(a), (f, lanes)
        assert np.mean(walk["next_active"] != out[lanes, 0]["next_active"]) <= 1e-3
