"""Advection rows side by side in groups that are no whole wavefronts (lines 2^a 3^b 5^c): one
step against the FP64 oracle, with the last block of rows partly empty, rows of odd half length
and three inputs as well as two.  Bars as for the other step tests: FP64 relative L2 <= 1e-12,
mixed form <= 1e-5.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows._lib import PTFError

from test_gpu_mixed_radix import _problem
from test_gpu_step import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,n", [(2, (50, 20)), (2, (200, 18)), (2, (216, 50)), (2, (250, 36)), (2, (500, 54)),
                                    (2, (864, 20)), (2, (1152, 100)), (2, (2000, 12)), (3, (100, 20, 18)),
                                    (3, (72, 18, 50))])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_padded_groups_vs_oracle(dev, ndim, n, T):
    p, o = _problem(dev, ndim, n, T, "RK4")
    sol0 = o.sol.copy()
    o.stepforward(1)
    rows = [i for i, s in enumerate(p.slots()) if "x_advect" in s]
    R = 5 if (n[0] // 2) % 2 and n[0] % 5 == 0 else (6 if n[0] % 3 == 0 else 10)
    ran = 0
    for W in (1, 2, 4, 8, 16):
        try:
            for i in rows:
                p.set_variant(i, R, W, par=True)
        except PTFError:
            continue
        print(f"row groups n={n} {T.__name__} R={R} W={W}", flush=True)
        p.sol = sol0
        ptf.stepforward_(p, 1)
        assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)
        ran += 1
    assert ran >= 1
