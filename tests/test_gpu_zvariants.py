"""Every register variant of the wave z kernels on mixed svor (cn2, and RK4 with PS3D_ZFUSE=0)
against the quad kernels: the RK4 steps on combined columns have one wave build, so the
variants differ in these passes only."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))


@pytest.mark.parametrize("nz", [64, 128, 256, 512])
@pytest.mark.parametrize("variant", ["1", "2", "3"])
@pytest.mark.parametrize("stepper", ["cn2", "impl-diff-rk4"])
def test_wave_variants_match_the_quad_kernels(monkeypatch, stepper, variant, nz):
    from ps3d_amd import gpu as G
    print("variants", stepper, variant, nz, flush=True)
    shape = (16, 12, nz)
    w = ics.beltrami_multimode(*shape, seed=5, noise=1e-2)
    monkeypatch.setenv("PS3D_ZFUSE", "0")
    out = []
    for v in ("0", variant):
        monkeypatch.setenv("PS3D_ZWAVE", v)
        d = G.Ps3dGpu(G.make_params(*shape, **BOX, filtering="2/3-rule", stepper=stepper, nnu=3, prediss=30.0,
                                    pretype="vorch"))
        d.set_vorticity(w)
        d.vor2vel()
        dt, _ = d.adapt(0.0)
        d.source()
        d.t = d.step(0.0, dt)
        out.append((d.advance_n(2), d.get(G.SVOR)))
        d.close()
    (ra, sa), (rb, sb) = out
    np.testing.assert_allclose(rb, ra, rtol=1e-12, atol=1e-12 * np.abs(ra).max())   # the trajectories' tolerance
    for c in range(3):
        assert np.abs(sb[c] - sa[c]).max() <= 1e-12 * np.abs(sa[c]).max()
