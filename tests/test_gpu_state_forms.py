"""Handles that a caller has given svor itself (ps3d_gpu_set, the mixed form) step the same
through every entry point that steps them: the batch calls and the ensemble's take a handle
of one instance, which the plain calls take too."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
SHAPE = (16, 12, 64)


def plain_view(G, batch):
    """The plain calls on the handle of a batch of one."""
    d = G.Ps3dGpu.__new__(G.Ps3dGpu)
    d.p, d.h, d.t = batch.p, batch.h, 0.0
    d.nx, d.ny, d.nz = SHAPE
    d.shape = (SHAPE[0], SHAPE[1], SHAPE[2] + 1)
    return d


@pytest.mark.parametrize("how", ["batch", "streams", "graph", "tune"])
def test_a_state_put_into_svor_steps_the_same_through_the_batch_calls(how):
    from ps3d_amd import gpu as G
    print("state form", how, flush=True)
    p = G.make_params(*SHAPE, **BOX, filtering="2/3-rule", nnu=3, prediss=30.0, pretype="vorch")
    w = ics.beltrami_multimode(*SHAPE, seed=3)
    ref = G.Ps3dGpu(p)
    ref.set_vorticity(w)
    s = 0.75 * ref.get(G.SVOR)
    ref.set(G.SVOR, s)
    ref.advance_n(3)
    ens = None if how == "batch" else G.Ps3dEnsemble([p], [1])
    b = G.Ps3dBatch(p, 1) if ens is None else ens.groups[0]
    b.set_vorticity(0, w)
    d = plain_view(G, b)
    d.set(G.SVOR, s)
    if how == "batch":
        b.advance_n(3)
    else:
        if how == "tune":
            ens.tune(steps=1)
        ens.advance(3, graph=how != "streams")
    got = b.get_svor(0)
    d.h = None
    (b if ens is None else ens).close()
    want = ref.get(G.SVOR)
    ref.close()
    assert np.abs(got - want).max() <= 1e-14 * np.abs(want).max()   # batched against single handles
