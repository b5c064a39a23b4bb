"""A learned guess that its first scan rejects where the iteration cap leaves
no scan after it: the second pass then runs over the members of the guess's
scan, whether or not their list fitted.  The lists against the cell walk
(density_flat): the same bits near the fixed point; with the default rule,
whose sums come in another order, up to 400 positive terms are rounded by
2^-24 each (2.4e-5 of rho at most; a member left out is 1 / 400 of it)."""
import numpy as np
import pytest

from oracle import mlp as omlp
from test_gpu_density_lists import _ball
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu

FIELDS = ("h", "rho", "gradterm", "balsara", "nr_iters")


def _constant(sph, d):
    """A network that predicts log(h_guess / h_start) = d for every particle."""
    net = sph.Mlp(seed=1)
    p = np.zeros(sph.MLP_PARAMS, np.float32)
    p[omlp.OFF_B3] = d
    norm = np.zeros(sph.MLP_NORM, np.float32)
    norm[12:24] = norm[25] = 1
    net.set(p, norm)
    return net


@pytest.mark.parametrize("d", [0.5, 0.12, -0.3])
@pytest.mark.parametrize("n,over", [(5000, {}), (70000, {}), (20000, {"small_n_lanes": 0})])
@pytest.mark.parametrize("stop", [0, 1])
def test_rejected_guess_at_the_cap(sph, tables256, n, over, d, stop):
    ic = _stir(_ball(n, n), n)
    net = _constant(sph, d)
    out = []
    for flat in (1, 0):
        prm = sph.default_params(density_stop=stop, density_eta=2.5e-6 if stop else 0.005, max_nr_iterations=1,
                                 density_flat=flat, **over)
        ctx = sph.Context(prm, ic, tables256)
        ctx.set_learned_guess(net)
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f) for f in FIELDS})
        ctx.set_learned_guess(None)
    walk, lists = out
    assert np.array_equal(walk["nr_iters"], lists["nr_iters"])
    for f in FIELDS[:4] if stop else FIELDS[:2]:
        if stop:
            assert np.array_equal(walk[f].view(np.int32), lists[f].view(np.int32)), (f, np.mean(walk[f] != lists[f]))
        else:
            assert np.max(np.abs(walk[f] / lists[f] - 1)) < 1e-4, f
