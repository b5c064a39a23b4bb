"""The rule that leaves the neighbour lists for the cell walk where the
resolution gives a particle more neighbours than a list holds, and the order
of the sums on either side of it: the acceleration pass has the same bits for
the same fields, with 0, 8 and 16 lanes, over every particle and over a list
of the active ones."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu

FIELDS = ("h", "rho", "pressure", "soundspeed", "gradterm", "balsara")


@pytest.mark.parametrize("stop", [0, 1])
@pytest.mark.parametrize("n,eta,over", [
    (20000, 2.6, {}), (70000, 2.6, {}), (300000, 1.6, {}), (40000, 2.6, {"small_n_lanes": 0}), (40000, 2.6, {"sparse": True}),
])
def test_density_beyond_the_lists_is_the_walk(sph, tables256, n, eta, over, stop):
    over = dict(over)
    sparse = over.pop("sparse", False)
    if sparse:
        over["activity_rule"] = sph.SPH_ACTIVE_README
    if stop:
        over.update(density_stop=1, density_eta=2.5e-6, max_nr_iterations=400)
    ic = _stir(_ball(n, n), n)
    out = []
    for flat in (1, 0):
        ctx = sph.Context(sph.default_params(density_flat=flat, resolution_eta=eta, **over), ic, tables256)
        if sparse:
            ctx.upload("active", (np.random.default_rng(8).random(n) < 0.1).astype(np.uint8))
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f) for f in FIELDS + ("nr_iters",)})
    for f in out[0]:
        assert np.array_equal(out[0][f].view(np.int32), out[1][f].view(np.int32)), f


@pytest.mark.parametrize("lanes", [0, 8, 16])
@pytest.mark.parametrize("n,over", [
    (1, {}), (9, {}), (129, {}), (5000, {}), (70001, {}), (4000, {"cell_width": 0.5}), (4000, {"cell_width": 0.03}),
    (3000, {"cell_power": 4}), (200, {"cell_power": 1}), (6000, {"clumps": True}), (6000, {"radii": True}),
    (40000, {"sparse": True}),
])
def test_acceleration_has_the_walks_bits(sph, tables256, n, over, lanes):
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
    out, fields = [], {}
    for eta in (1.2348, 2.6):  # (the acceleration pass takes no other notice of it)
        prm = sph.default_params(accel_lanes=lanes, list_accel_lanes=lanes, small_n_lanes=0, resolution_eta=eta, **over)
        ctx = sph.Context(prm, ic, tables256)
        if sparse:
            ctx.upload("active", active)
        ctx.sort()
        ctx.density()
        if not fields:
            fields = {f: ctx.download(f) for f in FIELDS}
            if radii:
                fields["h"][::50] *= 3
        for f in FIELDS:
            ctx.upload(f, fields[f])
        ctx.acceleration()
        out.append({f: ctx.download(f)[active > 0] for f in ("acc", "du", "dhdt", "next_active")})
    for f in out[0]:
        assert np.array_equal(out[0][f].view(np.int32), out[1][f].view(np.int32)), f
