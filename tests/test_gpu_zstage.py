"""The z passes of the RK4 step on the semi-spectral state (launch_zstage) against the
passes on svor (PS3D_ZFUSE=0, read when a handle is created): every kind of z kernel
(wave depths; quad kernels with compile-time and run-time plans and one to three levels
per thread), both filters, the whole step and the operator-by-operator sequence."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
# shapes: lids next to each other, remainders of 64 levels, every kernel family
SHAPES = [(4, 6, 2), (8, 12, 32), (16, 10, 48), (8, 8, 64), (20, 24, 100), (6, 4, 250), (8, 6, 256), (4, 8, 540),
          (8, 6, 1024)]


def pair(monkeypatch, G, shape, filtering):
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("PS3D_ZFUSE", fuse)
        d = G.Ps3dGpu(G.make_params(*shape, **BOX, filtering=filtering, nnu=3, prediss=30.0, pretype="max-strain",
                                    f_cor=(0.3, 0.1, 0.7)))
        d.set_vorticity(ics.beltrami_multimode(*shape, seed=4, noise=1e-2))
        out.append(d)
    return out


def close(a, b, tol=1e-12):   # the trajectories' parity tolerance
    for c in range(3):
        assert np.abs(a[c] - b[c]).max() <= tol * np.abs(b[c]).max()


@pytest.mark.parametrize("filtering", ["2/3-rule", "Hou & Li"])
@pytest.mark.parametrize("shape", SHAPES)
def test_semi_spectral_steps_match_the_passes_on_svor(monkeypatch, shape, filtering):
    from ps3d_amd import gpu as G
    print("zstage", shape, filtering, flush=True)
    a, b = pair(monkeypatch, G, shape, filtering)
    close(a.get(G.SVOR), b.get(G.SVOR), 2e-14)
    ra, rb = a.advance_n(3), b.advance_n(3)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    close(a.get(G.SVOR), b.get(G.SVOR))
    # vor2vel, adapt, source, step as separate calls
    for d in (a, b):
        d.vor2vel()
        dt, _ = d.adapt(d.t)
        d.source()
        d.t = d.step(d.t, dt)
    assert abs(a.t - b.t) <= 1e-12 * b.t
    close(a.get(G.SVOR), b.get(G.SVOR))
    # a state put there by the caller
    s = b.get(G.SVOR)
    for d in (a, b):
        d.set(G.SVOR, s)
    close(a.get(G.SVOR), s, 2e-14)
    ra, rb = a.advance_n(1), b.advance_n(1)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    close(a.get(G.SVOR), b.get(G.SVOR))
    a.close()
    b.close()


@pytest.mark.parametrize("nz", [30, 40, 60, 80, 100, 120, 160, 200])
def test_depths_with_a_factor_of_5_match_the_oracle(oracle_mod, nz):
    """Both steppers, three steps on the compile-time plans of these depths, to the
    trajectories' parity tolerance."""
    from ps3d_amd import gpu as G
    print("z plan", nz, flush=True)
    shape = (8, 6, nz)
    for stepper in ("impl-diff-rk4", "cn2"):
        kw = dict(BOX, stepper=stepper, filtering="Hou & Li", nnu=3, prediss=30.0, pretype="vorch",
                  length_scale="Kolmogorov")
        o = oracle_mod.Oracle(oracle_mod.make_params(*shape, **kw))
        d = G.Ps3dGpu(G.make_params(*shape, **kw))
        w = ics.beltrami_multimode(*shape, seed=4)
        for s in (o, d):
            s.set_vorticity(w)
        o.advance_n(3), d.advance_n(3)
        close(d.get(G.SVOR), o.get(oracle_mod.SVOR))
        o.close()
        d.close()
