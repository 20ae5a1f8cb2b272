"""ptf_step_record where the spacing of the records meets the ends of its type and where the
clock's step counter is negative: which steps are recorded and how many steps are taken are
whole numbers, compared with the records' definition (every step whose new clock.step is a
multiple of `every`); the state equals that of the same steps taken without records.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows._lib import call

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion


def _problem(dev, nd):
    flow = [ptf.OneDAdvectingFlow, ptf.TwoDAdvectingFlow][nd - 1]()
    p = TAD.Problem(dev, flow, nx=16, κ=1e-2, dt=0.01, **({"ny": 16} if nd == 2 else {}))
    TAD.set_c_(p, np.random.default_rng(1).standard_normal((16,) * nd))
    return p


@pytest.mark.parametrize("nd", [1, 2])
@pytest.mark.parametrize("first,nsteps,every", [(0, 3, 2 ** 63 - 1), (5, 7, 2 ** 63 - 1), (5, 7, 2 ** 62 + 1),
                                                (-5, 7, 2 ** 63 - 1), (-7, 12, 3), (-6, 6, 3), (4, 300, 299)])
def test_spacing_of_the_records(dev, nd, first, nsteps, every):
    print(f"record {nd}D first={first} nsteps={nsteps} every={every}", flush=True)
    a, b = _problem(dev, nd), _problem(dev, nd)
    for p in (a, b):
        call("ptf_set_clock", p._h, 0.0, first)
        p._sync_clock()
    rec = ptf.record_(a, nsteps, every, concentration=False)
    want = [s for s in range(first + 1, first + nsteps + 1) if s % every == 0]
    assert list(rec["step"]) == want and len(rec["mass"]) == len(want)
    ptf.stepforward_(b, nsteps)
    assert a.clock.step == b.clock.step == first + nsteps
    assert np.array_equal(a.sol, b.sol)
