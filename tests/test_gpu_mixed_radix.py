"""Register layouts of lines that are no powers of two: the narrow one (3, 5, 6 or 10 elements
a thread, composite radices 6 and 10) and the wide one (12 or 20), at the widths compiled for
each, on grids whose last blocks are partly empty.  Whole steps against the FP64 oracle; bars as for the other step tests: FP64 relative L2 <= 1e-12,
mixed form <= 1e-5.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from oracle import tad as O
from passivetracerflows._lib import PTFError

from test_gpu_step import _device_problem, _rand_setup, rel

pytestmark = pytest.mark.gpu

# odd half lengths, one wavefront and several, the longest; bricked and plain last axes
SHAPES = [(2, (24, 18)), (2, (50, 20)), (2, (54, 36)), (2, (100, 96)), (2, (250, 48)),
          (2, (400, 216)), (2, (432, 100)), (2, (1536, 24)), (2, (24, 1600)), (2, (32, 2000)),
          (2, (3456, 8)), (2, (16, 1728)), (2, (640, 768)),
          (3, (24, 20, 12)), (3, (40, 48, 80)), (3, (96, 36, 96)), (3, (32, 50, 144)), (3, (54, 16, 200))]


def _problem(dev, ndim, n, T, stepper):
    g, flows, c0 = _rand_setup(ndim, n, seed=11 + ndim)
    dt = min(0.01, 1.0 / max(n))
    kappa = min(1e-2, 0.5 / (dt * sum((k // 2) ** 2 for k in n)))
    p = _device_problem(dev, ndim, n, flows, T, stepper, dt, kappa)
    o = O.Problem(g, flows, kappa=kappa, eta=p.params.η, iota=p.params.ι, dt=dt, stepper=stepper)
    o.set_c(c0)
    p.sol = o.sol
    return p, o


def _elements(n):
    """(wide, narrow) elements a thread of a line of n points."""
    wide = 1
    for q in (3, 5):
        wide *= q if n % q == 0 else 1
    two = n & -n
    return wide * min(two, 4), wide * min(two, 2)


@pytest.mark.parametrize("ndim,n", SHAPES)
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_default_layouts_vs_oracle(dev, ndim, n, T):
    for stepper in ("RK4", "ETDRK4"):
        print(f"mixed radix ndim={ndim} n={n} {stepper} {T.__name__}", flush=True)
        p, o = _problem(dev, ndim, n, T, stepper)
        o.stepforward(3)
        ptf.stepforward_(p, 3)
        assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)


@pytest.mark.parametrize("ndim,n", [(2, (100, 96)), (2, (400, 216)), (3, (96, 40, 144)), (3, (36, 80, 192))])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_every_layout_and_width_vs_oracle(dev, ndim, n, T):
    """Each compiled layout, width and mapping of every kernel of the step, in turn."""
    p, o = _problem(dev, ndim, n, T, "RK4")
    sol0 = o.sol.copy()
    o.stepforward(1)
    ran = 0
    for R in sorted({e for k in n for m in (k, k // 2) if m & (m - 1) for e in _elements(m)}):
        for W in (1, 2, 4, 8, 16, 32):
            for par in (False, True):
                took = 0
                for i in range(len(p.slots())):
                    try:
                        p.set_variant(i, R, W, par=par)
                        took += 1
                    except PTFError:
                        pass
                if not took:
                    continue
                print(f"mixed radix n={n} {T.__name__} R={R} W={W} par={par}: {took} slots", flush=True)
                p.sol = sol0
                ptf.stepforward_(p, 1)
                assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)
                ran += 1
    assert ran >= 4
