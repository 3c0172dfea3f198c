"""RK4 steps whose stages move the state by less than half a unit in the last place, and whose
whole step moves it by about one: the tendency has to be summed over the stages before it
joins the state, or the state never moves."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
NSTEPS = 64


def combined(d, f):
    return np.stack([d.field_combine_semi_spectral(f[c]) for c in range(3)])


@pytest.mark.parametrize("shape", [(16, 12, 48), (16, 16, 64), (12, 16, 256)])   # quad and wave z kernels
def test_stages_below_the_last_place_add_up(shape):
    from ps3d_amd import gpu as G
    print("small steps", shape, flush=True)
    # no dissipation: the columns do not decay
    kw = dict(BOX, filtering="Hou & Li", nnu=3, prediss=0.0, pretype="vorch")
    w = ics.beltrami_multimode(*shape, seed=3, noise=0.3)
    d = G.Ps3dGpu(G.make_params(*shape, **kw))
    d.set_vorticity(w)
    d.vor2vel()
    d.adapt(0.0)
    d.source()
    s0, tend = combined(d, d.get(G.SVOR)), combined(d, d.get(G.SVORTS))
    d.close()
    with np.errstate(over="ignore"):
        per_dt = np.abs(tend) / np.spacing(np.abs(s0))   # units in the last place per unit of time
    k = [np.minimum(np.arange(n), n - np.arange(n)) <= n // 4 for n in shape[:2]]   # filter: 1
    low = (k[0][:, None] & k[1][None, :])[None, :, :, None]
    dt = 1.4 / np.quantile(per_dt[np.broadcast_to(low, per_dt.shape)], 0.5)
    # a stage adds dt/3 of the tendency at most, 0.47 units; the step 0.8 to 1.4
    sel = low & (per_dt * dt >= 0.8) & (per_dt * dt <= 1.4)
    assert sel.sum() > 500
    d = G.Ps3dGpu(G.make_params(*shape, dt_fixed=dt, **kw))
    d.set_vorticity(w)
    d.advance_n(NSTEPS)
    moved = combined(d, d.get(G.SVOR)) - s0
    d.close()
    share = (moved[sel] * tend[sel]).sum() / (NSTEPS * dt * (tend[sel] ** 2).sum())
    print("share", share, flush=True)
    # rounded to whole units, 0.8 to 1.4 become one: 0.7 to 1.25 of the tendency; lost stages: 0
    assert 0.5 < share < 1.5
