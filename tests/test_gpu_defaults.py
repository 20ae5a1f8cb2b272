"""Default kernel variants (the ones a problem starts with) at the edges of the rule that
picks them: the smallest and longest lines, oblong grids, few and many lines, each stepper
family, single problems and batches.  Bars as for the other step tests: FP64 relative L2
<= 1e-12 against the FP64 oracle, mixed form <= 1e-5.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from oracle import tad as O

from test_gpu_step import _device_problem, _rand_setup, rel

pytestmark = pytest.mark.gpu

SHAPES = [(1, (16,), "RK4"), (1, (4096,), "RK4"),
          (2, (16, 8), "RK4"), (2, (16, 2048), "RK4"), (2, (4096, 16), "ETDRK4"),
          (2, (2048, 512), "RK4"), (2, (1024, 64), "ETDRK4"), (2, (64, 1024), "RK4"),
          (2, (128, 128), "FilteredRK4"), (2, (256, 256), "RK4"), (2, (1024, 1024), "RK4"),
          (3, (16, 8, 8), "RK4"), (3, (32, 32, 32), "ETDRK4"), (3, (64, 128, 32), "RK4"),
          (3, (128, 128, 128), "RK4"), (3, (16, 64, 512), "RK4"), (3, (512, 16, 64), "RK4")]


@pytest.mark.parametrize("ndim,n,stepper", SHAPES)
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_default_variants_vs_oracle(dev, ndim, n, stepper, T):
    print(f"defaults ndim={ndim} n={n} {stepper} {T.__name__}", flush=True)
    g, flows, c0 = _rand_setup(ndim, n, seed=7 + ndim)
    kmax2 = sum((k // 2) ** 2 for k in n)
    dt = min(0.01, 1.0 / max(n))
    kappa = min(1e-2, 0.5 / (dt * kmax2))
    p = _device_problem(dev, ndim, n, flows, T, stepper, dt, kappa)
    L = O.linear_operator(g, kappa, p.params.η, p.params.ι)
    o = O.Problem(g, flows, kappa=kappa, eta=p.params.η, iota=p.params.ι, dt=dt, stepper=stepper)
    assert np.array_equal(o.L, L)
    o.set_c(c0)
    p.sol = o.sol
    o.stepforward(3)
    ptf.stepforward_(p, 3)
    assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)


@pytest.mark.parametrize("n,count", [(128, 2), (128, 40), (256, 70), (512, 34), (1024, 3)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_default_variants_of_batches(dev, n, count, precision):
    """Batches from a few members to more than a streaming launch's worth: first and last
    member against the oracle."""
    print(f"defaults batch {count}x{n}^2 {precision}", flush=True)
    g, flows, c0 = _rand_setup(2, (n, n), seed=3)
    dt = 1.0 / n
    kappa = min(1e-2, 0.5 / (dt * 0.5 * n * n))
    e = ptf.Ensemble([dict(n=n, kappa=kappa * (1 + i / count)) for i in range(count)], dt, precision=precision)
    for i in range(count):
        e.set_flow(i, flows[0], flows[1])
        e.set_c(i, c0)
    e.step(3)
    for i in (0, count - 1):
        o = O.Problem(g, flows, kappa=kappa * (1 + i / count), dt=dt)
        o.set_c(c0)
        o.stepforward(3)
        assert rel(e.get_sol(i), o.sol) <= (1e-12 if precision == "fp64" else 1e-5)
