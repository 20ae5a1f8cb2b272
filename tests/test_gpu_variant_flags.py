"""A selected variant is the one that is reported: radix, width and flags of every slot, and of FP32
column lines of 64 threads along the bricked axis, whose only form is the workgroup one, with and
without the flag for it (the same kernel, so the same bits).
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows._lib import PTFError

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion


@pytest.mark.parametrize("n", [(128, 256), (64, 512), (96, 192), (32, 64), (64, 64, 64), (50, 54)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_selected_is_reported(dev, n, T):
    flow = [ptf.TwoDAdvectingFlow, ptf.ThreeDAdvectingFlow][len(n) - 2]()
    p = TAD.Problem(dev, flow, κ=1e-3, dt=1e-3, T=T, **dict(zip(("nx", "ny", "nz"), n)))
    took = 0
    for i in range(len(p.slots())):
        for R in (16, 8, 4, 12, 6, 10, 5):
            for W in (8, 4, 1):
                for flags in [(False, False, False), (True, False, False), (False, True, False), (False, False, True),
                              (True, False, True), (False, True, True)]:
                    before = p.get_variant(i)
                    try:
                        p.set_variant(i, R, W, *flags)
                    except PTFError:
                        assert p.get_variant(i) == before
                        continue
                    assert p.get_variant(i) == (R, W, *flags)
                    assert (" wg " in p.slots()[i]) == flags[2]
                    took += 1
    assert took > 0


def test_the_only_form_takes_the_flag(dev):
    c0 = np.random.default_rng(3).standard_normal((256, 128))
    sols = []
    for wg in (False, True):
        p = TAD.Problem(dev, ptf.TwoDAdvectingFlow(u=lambda x, y: np.sin(y) + 0 * x, v=lambda x, y: np.cos(x) + 0 * y),
                        nx=128, ny=256, κ=1e-3, dt=1e-3, T=np.float32)
        for i, s in enumerate(p.slots()):
            if "stage_inverse" in s:
                p.set_variant(i, 4, 2, wg=wg)
        TAD.set_c_(p, c0)
        ptf.stepforward_(p, 3)
        sols.append(p.sol.copy())
    assert np.array_equal(*sols)
