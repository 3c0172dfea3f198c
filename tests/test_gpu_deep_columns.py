"""The deepest columns (nz = 1024, three levels per thread) against the oracle, operator by
operator and step by step: the z kernels with the most registers, and the only ones of their
family at this depth."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
TOL = 1e-12    # the trajectories' parity tolerance


def close(a, b):
    for c in range(3):
        assert np.abs(a[c] - b[c]).max() <= TOL * np.abs(b).max()


@pytest.mark.parametrize("stepper", ["impl-diff-rk4", "cn2"])
@pytest.mark.parametrize("filtering", ["2/3-rule", "Hou & Li"])
@pytest.mark.parametrize("shape", [(8, 6, 1024), (4, 10, 1024)])
def test_operators_and_steps_match_the_oracle(oracle_mod, shape, filtering, stepper):
    from ps3d_amd import gpu as G
    print("deep columns", shape, filtering, stepper, flush=True)
    kw = dict(BOX, filtering=filtering, stepper=stepper, nnu=3, prediss=30.0, pretype="max-strain",
              f_cor=(0.3, 0.1, 0.7))
    o = oracle_mod.Oracle(oracle_mod.make_params(*shape, **kw))
    d = G.Ps3dGpu(G.make_params(*shape, **kw))
    w = ics.beltrami_multimode(*shape, seed=4, noise=1e-2)
    for s in (o, d):
        s.set_vorticity(w)
        s.vor2vel()
    close(d.get(G.VEL), o.get(oracle_mod.VEL))
    dt = o.adapt(0.0)[0]
    assert abs(d.adapt(0.0)[0] - dt) <= TOL * dt
    for s in (o, d):
        s.source()
    close(d.get(G.SVORTS), o.get(oracle_mod.SVORTS))
    for s in (o, d):
        s.t = s.step(0.0, dt)
    close(d.get(G.SVOR), o.get(oracle_mod.SVOR))
    o.advance_n(2), d.advance_n(2)
    close(d.get(G.SVOR), o.get(oracle_mod.SVOR))
    o.close()
    d.close()
