"""Whole-run kernel of 1D problems at the lengths where its elements change hands between the
transforming lanes and the rest of the block: half lines shorter than a wavefront, just over one,
of 64 and 128 transforming lanes, several elements a lane, and the first that keep one layout.

Bars as for the other step tests: FP64 relative L2 <= 1e-12 against the FP64 oracle, mixed form
<= 1e-5.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from oracle import tad as O

from test_gpu_line import _numbers
from test_gpu_step import _device_problem, _rand_setup, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 64, 72, 100, 144, 256, 384, 400, 768, 1000, 1280, 1536, 1600, 2000, 2048, 2560])
@pytest.mark.parametrize("T,stepper", [(np.float64, "FilteredRK4"), (np.float64, "ETDRK4"), (np.float32, "RK4"),
                                       (np.float32, "FilteredETDRK4")])
def test_run_vs_oracle(dev, n, T, stepper):
    print(f"line n={n} {T.__name__} {stepper}", flush=True)
    g, flows, c0 = _rand_setup(1, (n,), seed=9)
    dt, kappa = _numbers(n)
    p = _device_problem(dev, 1, (n,), flows, T, stepper, dt, kappa)
    o = O.Problem(g, flows, kappa=kappa, dt=dt, stepper=stepper)
    o.set_c(c0)
    p.sol = o.sol
    o.stepforward(6)
    ptf.stepforward_(p, 5)
    ptf.stepforward_(p, 1)
    assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)
