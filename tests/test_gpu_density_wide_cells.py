"""Cells of several h: most of a particle's neighbours lie in a few cells, and
so in a few of the bins that the lists are dealt to, one of which per lane
may hold more than its rows.  Near the fixed point the lists have the bits of
the cell walk (density_flat) for each number of lanes, where one bin or more
overflow and where none does."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio", [1.5, 2.5, 3, 4, 6])
@pytest.mark.parametrize("n,over", [(20000, {}), (70000, {}), (20000, {"small_n_lanes": 0}), (40000, {"sparse": True})])
def test_wide_cells_bits(sph, tables256, n, over, ratio):
    over = dict(over)
    sparse = over.pop("sparse", False)
    if sparse:
        over["activity_rule"] = sph.SPH_ACTIVE_README
    ic = _stir(_ball(n, n), n)
    out = []
    for flat in (1, 0):
        prm = sph.default_params(density_stop=1, density_eta=2.5e-6, max_nr_iterations=400, density_flat=flat,
                                 cell_width=float(ratio * ic["h"][0]), **over)
        ctx = sph.Context(prm, ic, tables256)
        if sparse:
            ctx.upload("active", (np.random.default_rng(8).random(n) < 0.1).astype(np.uint8))
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f) for f in ("h", "rho", "gradterm", "balsara", "pressure", "nr_iters")})
        ctx.close()
    for f in out[0]:
        a, b = (o[f].view(np.int32) for o in out)
        assert np.array_equal(a, b), (f, np.mean(a != b))
