"""The algorithmic bytes that ps3d_gpu_profile_kernels states per launch, against a count by
hand of the fields each kernel of the step reads and writes, for the three kinds of step: RK4
on the wave line passes, RK4 on tiles, cn2 (host code only, over the stand-in for the HIP
runtime of test_copy_host.py)."""
import pytest

from .test_copy_host import run  # noqa: F401  (fixture)

BODY = """
import numpy as np
p = G.make_params(64, 64, 64, extent=(1.0, 1.0, 1.0), filtering="2/3-rule", stepper=%r)
d = G.Ps3dGpu(p)
d.set(G.SVOR, np.zeros((3,) + d.shape))
ms, n, b = np.zeros(10), np.zeros(10, np.int32), np.zeros(10)
ptr = lambda x: x.ctypes.data_as(C.c_void_p)
assert G.lib().ps3d_gpu_profile_kernels(d.h, 1, ptr(ms), ptr(n), ptr(b)) == 0
b /= 8.0 * 64 * 64 * 65
ZINV, YINV, XMAIN, YFWD, ZTEND, YADAPT, XADAPT, REDUCE, MEAN, ZSTAGE = range(10)
want = %s
for k, v in want.items():
    assert abs(b[k] - v) < 1e-9, (k, b[k], v)
assert {k: int(n[k]) for k in range(10) if n[k]} == %s
"""
# the 2/3 rule of 64 points passes the indices up to 21: 43 slots of 64
X, XY = "43 / 64", "(43 / 64) ** 2"
# xi, eta, zeta -> u, v, w and the projected vorticity, no midpoints; y inverse of the six and
# the derivatives of three; omega, three y derivatives, and u, w for their x derivatives
WAVES = {"ZINV": "9", "YINV": "12", "XMAIN": "6 + 3 * " + X, "YFWD": "3 * %s + 3 * %s" % (X, XY),
         "ZTEND": "6 + 6 * " + XY, "YADAPT": "15", "XADAPT": "8",
         "ZSTAGE": "9 + %s * (6 + 9 + 9) / 3" % XY}
# tiles: the midpoints of omega are three more fields from the z to the x pass
TILES = dict(WAVES, ZINV="12", YADAPT="21", XADAPT="11")
# mixed svor, every column: (3 + 6, and at the adapt stage 2 + 3 more); 3 + 3 + ... of r, q, p
CN2 = {"ZINV": "(14 + 9 + 9) / 3", "YINV": "12", "XMAIN": "9", "YFWD": "6", "ZTEND": "10", "YADAPT": "21", "XADAPT": "11"}


def literal(d):
    return "{%s}" % ", ".join("%s: %s" % kv for kv in d.items())


@pytest.mark.parametrize("stepper, tiles, want", [("impl-diff-rk4", False, WAVES), ("impl-diff-rk4", True, TILES),
                                                  ("cn2", False, CN2)])
def test_bytes_are_those_of_the_fields(run, stepper, tiles, want):  # noqa: F811
    rk4 = "{ZINV: 1, YINV: 3, XMAIN: 4, YFWD: 4, ZTEND: 1, YADAPT: 1, XADAPT: 1, REDUCE: 2, ZSTAGE: 3}"
    cn2 = "{ZINV: 3, YINV: 2, XMAIN: 3, YFWD: 3, ZTEND: 3, YADAPT: 1, XADAPT: 1, REDUCE: 2, MEAN: 3}"
    run(BODY % (stepper, literal(want), cn2 if stepper == "cn2" else rk4), **({"PS3D_LINE_SCHED": "0,0"} if tiles else {}))
