"""Particles with thousands of neighbours within 2h, which no list holds: the
default rule's walk by the whole wave against the cell walk (density_flat).
Each scan adds up to 6000 positive terms in another order, rounded by 2^-24
each: 6000 * 2^-24 = 3.6e-4 of rho if every rounding went one way, and a third
of it on h; 5 standard deviations of as many independent ones are 2.3e-5.  A
particle left out is 1 / 6000 of it.  A count may differ where a change of h lies
within that of the stopping rule's bound (1 in 1000).  Particles that reach the
default cap of 50 iterations have not converged: the crowd lies on the edge of
their 2h, each iteration magnifies the rounding of the one before, and the
cell walk with other numbers of lanes differs from itself by 8e-4 and more."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_guess_cap import _constant
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,over", [
    (7000, {}), (7000, {"small_n_lanes": 0}), (7000, {"sparse": True}), (7000, {"guess": 0.3}), (7000, {"guess": -0.2}),
    (7000, {"max_nr_iterations": 1}), (7000, {"max_nr_iterations": 1, "guess": 0.5}), (7000, {"falling": True}),
    (7000, {"fixes": 0x7F}), (7000, {"cell_width": 0.03}), (7000, {"cell_width": 2.0}), (7000, {"cell_power": 3}),
    (7000, {"cell_power": 1}), (70000, {}),
])
def test_crowd(sph, tables256, n, over):
    over = dict(over)
    sparse, falling, guess = (over.pop(k, None) for k in ("sparse", "falling", "guess"))
    ic = _stir(_ball(n, n, radius=6.0 if falling else 1.0), n)
    g = np.random.default_rng(6)
    ic["pos"][:6000, :3] = 20.3 + 0.02 * g.standard_normal((6000, 3))
    if falling:
        ic["h"] = g.uniform(0.9, 1.3, n).astype(np.float32)
    if sparse:
        over["activity_rule"] = sph.SPH_ACTIVE_README
    out = []
    for flat in (1, 0):
        ctx = sph.Context(sph.default_params(density_flat=flat, **over), ic, tables256)
        net = _constant(sph, guess) if guess is not None else None
        ctx.set_learned_guess(net)
        active = np.ones(n, np.uint8)
        if sparse:
            active = (np.random.default_rng(8).random(n) < 0.1).astype(np.uint8)
            ctx.upload("active", active)
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f)[active > 0] for f in ("h", "rho", "nr_iters")})
        ctx.set_learned_guess(None)
        ctx.close()
    walk, lists = out
    same = walk["nr_iters"] == lists["nr_iters"]
    assert np.mean(~same) <= 1e-3
    same &= walk["nr_iters"] < 50
    assert np.mean(same) > 0.99
    for f in ("h", "rho"):
        assert np.all(np.isfinite(lists[f])) and np.max(np.abs(lists[f] / walk[f] - 1)[same]) < 2.3e-5, f
