"""RK4 steps made of ps3d_gpu_rk_substep calls with a look at the state in between: reading
svor, or resampling it, leaves the step that is under way as it is."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))


def substeps(G, shape, look, batch):
    """One step in ps3d's order of operators (impl_rk4.f90:76-207); look(d) between them."""
    p = G.make_params(*shape, **BOX, filtering="2/3-rule", nnu=3, prediss=30.0, pretype="vorch")
    w = ics.beltrami_multimode(*shape, seed=3, noise=1e-2)
    vdiss = np.full(shape[:2], 1e-3)
    d = G.Ps3dGpu(p)
    if batch:   # the handle of a batch of one takes the plain calls too
        d.close()
        b = G.Ps3dBatch(p, 1)
        d.h = b.h
    d.set_vorticity(w)
    for stage in range(1, 5):
        d.vor2vel()
        look(d)
        if stage == 1:
            d.adapt(0.0)
        d.source()
        look(d)
        d.rk_substep(stage, 1e-3, vdiss)
        look(d)
    s = d.get(G.SVOR)
    if batch:
        d.h = type(d.h)()
        b.close()
    d.close()
    return s


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("shape", [(24, 16, 32), (16, 12, 64)])   # quad and wave z kernels
def test_reading_svor_between_substeps_leaves_the_step(shape, batch):
    from ps3d_amd import gpu as G
    print("substeps", shape, batch, flush=True)
    plain = substeps(G, shape, lambda d: None, batch)
    assert np.array_equal(substeps(G, shape, lambda d: d.get(G.SVOR), batch), plain)


def test_resampling_svor_between_substeps_leaves_the_step():
    from ps3d_amd import gpu as G
    shape = (24, 16, 32)
    print("substeps resample", flush=True)
    c = G.Ps3dGpu(G.make_params(16, 12, 16, **BOX, filtering="2/3-rule", nnu=3, prediss=30.0, pretype="vorch"))
    plain = substeps(G, shape, lambda d: None, False)
    assert np.array_equal(substeps(G, shape, lambda d: G.resample(c, d), False), plain)
    c.close()
