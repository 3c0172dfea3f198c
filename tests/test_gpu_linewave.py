"""The line passes with the lines in a wave's registers (linewave.hip) against the tile
passes (PS3D_LINE_SCHED set, read when a handle is created): every built length along x and
along y, level counts that leave remainders of a wave's and a block's levels, the fused step
and the separate operators (which take physical input along x)."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
SHAPES = [(64, 128, 2), (128, 64, 32), (256, 64, 6), (64, 256, 16), (512, 64, 10), (64, 512, 30), (128, 128, 64)]
# n = A B, every pair of factors along x and along y
SHAPES += [(16, 18, 6), (18, 20, 32), (20, 24, 10), (24, 30, 18), (30, 32, 2), (32, 36, 64), (36, 40, 20), (40, 48, 4),
           (48, 50, 30), (50, 54, 12), (54, 60, 2), (60, 72, 16), (72, 80, 6), (80, 90, 8), (90, 96, 10), (96, 100, 4),
           (100, 108, 2), (108, 120, 6), (120, 144, 4), (144, 150, 2), (150, 160, 12), (160, 162, 2), (162, 180, 4),
           (180, 192, 2), (192, 200, 6), (200, 216, 2), (216, 240, 2), (240, 250, 4), (250, 270, 2), (270, 288, 2),
           (288, 300, 2), (300, 320, 2), (320, 324, 4), (324, 360, 2), (360, 384, 2), (384, 16, 10)]


def pair(monkeypatch, G, shape, **kw):
    out = []
    for tiles in (False, True):
        if tiles:
            monkeypatch.setenv("PS3D_LINE_SCHED", "0,0")
        else:
            monkeypatch.delenv("PS3D_LINE_SCHED", raising=False)
        d = G.Ps3dGpu(G.make_params(*shape, **BOX, nnu=3, prediss=30.0, pretype="vorch", f_cor=(0.2, 0.4, 0.6), **kw))
        d.set_vorticity(ics.beltrami_multimode(*shape, seed=5, noise=1e-2))
        out.append(d)
    return out


def close(a, b, tol):
    assert np.abs(a - b).max() <= tol * np.abs(b).max()


@pytest.mark.parametrize("shape", SHAPES)
def test_wave_line_passes_match_the_tile_passes(monkeypatch, shape):
    from ps3d_amd import gpu as G
    print("linewave", shape, flush=True)
    a, b = pair(monkeypatch, G, shape, filtering="2/3-rule")
    f = np.random.default_rng(3).standard_normal((shape[0], shape[1], shape[2] + 1))
    close(a.fftxyp2s(f), b.fftxyp2s(f), 2e-14)       # the operators' tolerance
    close(a.fftxys2p(f), b.fftxys2p(f), 2e-14)
    # vor2vel, adapt and source by themselves, then the step
    for d in (a, b):
        d.vor2vel()
    close(a.get(G.VEL), b.get(G.VEL), 2e-13)
    close(a.get(G.VOR), b.get(G.VOR), 2e-13)
    (dta, ra), (dtb, rb) = a.adapt(0.0), b.adapt(0.0)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    for d in (a, b):
        d.source()
    close(a.get(G.SVORTS), b.get(G.SVORTS), 1e-12)
    assert abs(a.step(0.0, dta) - b.step(0.0, dtb)) <= 1e-12 * dtb
    # fused steps (the trajectories' parity tolerance)
    ra, rb = a.advance_n(2), b.advance_n(2)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    for c in range(3):
        close(a.get(G.SVOR)[c], b.get(G.SVOR)[c], 1e-12)
    a.close()
    b.close()


def test_wave_line_passes_without_a_band_limit(monkeypatch):
    from ps3d_amd import gpu as G
    a, b = pair(monkeypatch, G, (128, 64, 20), filtering="Hou & Li")
    ra, rb = a.advance_n(3), b.advance_n(3)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    for c in range(3):
        close(a.get(G.SVOR)[c], b.get(G.SVOR)[c], 1e-12)
    a.close()
    b.close()


@pytest.mark.parametrize("shape", [(64, 64, 64), (48, 40, 30)])
def test_line_passes_of_the_other_stepper(monkeypatch, shape):
    """cn2 steps on svor: line passes of both kinds around the z passes of its own."""
    from ps3d_amd import gpu as G
    a, b = pair(monkeypatch, G, shape, filtering="2/3-rule", stepper="cn2")
    ra, rb = a.advance_n(3), b.advance_n(3)
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    for c in range(3):
        close(a.get(G.SVOR)[c], b.get(G.SVOR)[c], 1e-12)
    a.close()
    b.close()
