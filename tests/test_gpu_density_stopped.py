"""Particles that stop before others of their wave: a guess whose list does
not fit takes its first scan from the cells, and is then one scan ahead of the
rest of the wave at the iteration cap.  Near the fixed point its second pass
has the bits of the cell walk (density_flat) all the same."""
import numpy as np
import pytest

from test_gpu_density_lists import _ball
from test_gpu_guess_cap import FIELDS, _constant
from test_gpu_parity import _stir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [2, 3, 5])
@pytest.mark.parametrize("d", [0.12, -0.3])
@pytest.mark.parametrize("n,over", [(5000, {}), (70000, {}), (20000, {"small_n_lanes": 0})])
def test_stopped_ahead_of_the_wave(sph, tables256, n, over, d, cap):
    ic = _stir(_ball(n, n), n)
    net = _constant(sph, d)
    out = []
    for flat in (1, 0):
        prm = sph.default_params(density_stop=1, density_eta=2.5e-6, max_nr_iterations=cap, density_flat=flat, **over)
        ctx = sph.Context(prm, ic, tables256)
        ctx.set_learned_guess(net)
        ctx.sort()
        ctx.density()
        out.append({f: ctx.download(f) for f in FIELDS})
        ctx.set_learned_guess(None)
    for f in FIELDS:
        a, b = (o[f].view(np.int32) for o in out)
        assert np.array_equal(a, b), (f, np.mean(a != b))
