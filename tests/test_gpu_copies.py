"""Field copies between host and device: what is put into a field is what comes back, bit for
bit, for fields that fit the first staging buffer (16 MiB with the columns' padding) and for
those that several threads copy in chunks of 4 MiB."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one column pair; just below and just above 16 MiB; chunks that leave a remainder
SHAPES = [(2, 2, 2), (90, 96, 64), (96, 96, 64), (100, 60, 150), (128, 180, 80)]


@pytest.mark.parametrize("shape", SHAPES)
def test_fields_come_back_as_they_were_put(shape):
    from ps3d_amd import gpu as G
    print("copies", shape, flush=True)
    d = G.Ps3dGpu(G.make_params(*shape, lower=(0.0, 0.0, 0.0), extent=(2 * math.pi, 2 * math.pi, math.pi),
                                filtering="2/3-rule", nnu=3, prediss=30.0, pretype="vorch"))
    rng = np.random.default_rng(5)
    for which in (G.SVORTS, G.SVOR):
        f = rng.standard_normal((3,) + d.shape)
        d.set(which, f)
        assert np.array_equal(d.get(which), f)
    # a single volume in and out: the z derivative of a linear column is its slope
    z = np.broadcast_to(np.arange(shape[2] + 1) * 0.5, d.shape)
    assert np.abs(d.central_diffz(z) - 0.5 * shape[2] / math.pi).max() <= 1e-12 * shape[2]
    d.close()
