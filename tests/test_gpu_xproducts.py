"""The x products pass on both sides of the line between its tile and wave kernels
(linewave_xmain), at every length that has both, single and batched, against the tile passes
alone (PS3D_LINE_SCHED set, read when a handle is created)."""
import math

import numpy as np
import pytest

from ps3d_amd import ics

pytestmark = pytest.mark.gpu

BOX = dict(lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi))
# n, then ny and nz of a grid just below and just above the line (200000 points below 96, else
# 450000); above, levels that leave remainders of a wave's
SHAPES = [(32, 48, 128), (32, 48, 144), (48, 32, 128), (48, 64, 72), (64, 48, 64), (64, 64, 54), (96, 48, 96),
          (96, 96, 50), (128, 64, 50), (128, 96, 40), (192, 36, 64), (192, 48, 50), (256, 32, 50), (256, 48, 40),
          (384, 18, 64), (384, 36, 36)]


def points(shape):
    return shape[0] * shape[1] * (shape[2] + 1)


def make(monkeypatch, G, shape, tiles, filtering="2/3-rule"):
    if tiles:
        monkeypatch.setenv("PS3D_LINE_SCHED", "0,0")
    else:
        monkeypatch.delenv("PS3D_LINE_SCHED", raising=False)
    p = G.make_params(*shape, **BOX, filtering=filtering, nnu=3, prediss=30.0, pretype="vorch", f_cor=(0.2, 0.4, 0.6))
    return p


def close(a, b, tol):
    assert np.abs(a - b).max() <= tol * np.abs(b).max()


def test_shapes_lie_on_both_sides():
    for below, above in zip(SHAPES[::2], SHAPES[1::2]):
        assert below[0] == above[0]
        line = 200000 if below[0] < 96 else 450000
        assert points(below) <= line < points(above)


@pytest.mark.parametrize("shape", SHAPES)
def test_products_match_the_tile_pass(monkeypatch, shape):
    from ps3d_amd import gpu as G
    print("xproducts", shape, flush=True)
    w = ics.beltrami_multimode(*shape, seed=5, noise=1e-2)
    out = []
    for tiles in (False, True):
        d = G.Ps3dGpu(make(monkeypatch, G, shape, tiles))
        d.set_vorticity(w)
        d.vor2vel()
        d.adapt(0.0)
        d.source()
        ts = d.get(G.SVORTS)
        rows = d.advance_n(2)      # the adapt stage takes the velocity maxima from the pass
        out.append((ts, rows, d.get(G.SVOR)))
        d.close()
    (ta, ra, sa), (tb, rb, sb) = out
    close(ta, tb, 1e-12)           # the trajectories' parity tolerance
    np.testing.assert_allclose(ra, rb, rtol=1e-12, atol=1e-12 * np.abs(rb).max())
    for c in range(3):
        close(sa[c], sb[c], 1e-12)


def test_a_batch_counts_all_its_instances(monkeypatch):
    """Eight instances of 32^3 take the wave kernel, one the tiles: the same steps."""
    from ps3d_amd import gpu as G
    shape = (32, 32, 32)
    assert points(shape) <= 200000 < 8 * points(shape)
    p = make(monkeypatch, G, shape, False)
    w = [ics.beltrami_multimode(*shape, seed=s, noise=1e-2) for s in range(8)]
    b = G.Ps3dBatch(p, 8)
    for i in range(8):
        b.set_vorticity(i, w[i])
    print("xproducts batch", flush=True)
    rows = b.advance_n(3, series=True)
    for i in (0, 7):
        d = G.Ps3dGpu(p)
        d.set_vorticity(w[i])
        np.testing.assert_allclose(rows[i], d.advance_n(3), rtol=1e-12, atol=1e-12 * np.abs(rows[i]).max())
        close(b.get_svor(i), d.get(G.SVOR), 1e-12)
        d.close()
    b.close()
