"""The ensemble tuner times only what changes a step (host code, over the stand-in for the HIP
runtime of test_copy_host.py, which counts kernel launches)."""
import pytest

from .test_copy_host import run  # noqa: F401  (fixture)

BODY = """
n, count, stepper = %r
p = G.make_params(n, n, n, extent=(1.0, 1.0, 1.0), filtering="2/3-rule", stepper=stepper)
e = G.Ps3dEnsemble([p], [count])
for b in range(count):
    e.groups[0].set_vorticity(b, np.zeros((3,) + e.groups[0].shape))
def launches(f):
    before = stub.stub_launches()
    f()
    return stub.stub_launches() - before
step = launches(lambda: e.groups[0].advance_n(1))
before = e.line_choices(), e.fft_schedules()
got = launches(lambda: e.tune(steps=1))
assert got == 2 * %d * step, (got, step)     # a warm-up and a timed step per candidate
if %r:
    assert (e.line_choices(), e.fft_schedules()) == before
assert e.tune(steps=1)[0] in (1, 2, 4, 8, 101) + ((100, 102) if stepper == "cn2" else ())
for code in (100, 101, 102) if n %% 64 == 0 else (1,):      # all stay selectable
    e.set_choice(0, code)
"""


@pytest.mark.parametrize("case, candidates, none_on_tiles", [
    ((32, 8, "impl-diff-rk4"), 4, True),        # 1, 2, 4, 8 quads a block
    ((64, 2, "impl-diff-rk4"), 1 + 3, True),    # waves; 1, 2, 4 quads
    # one 32^3: its x products are on tiles, three block sizes
    ((32, 1, "impl-diff-rk4"), 4 + 3, False),
    # cn2: three wave builds, three quad shapes; x products on waves, the adapt stage's two
    # passes on tiles, three block sizes each
    ((64, 2, "cn2"), 6 + 6, False)])
def test_candidates_differ(run, case, candidates, none_on_tiles):  # noqa: F811
    run(BODY % (case, candidates, none_on_tiles))
