"""Whole-run kernel of 1D problems (line_run_kernel) at the edges of its launch: the shortest
and longest lines, lines of one wavefront and of several, mixed-radix lengths (an odd half
length among them), every stepper, runs longer than one launch, and the stage kernels that a
caller selects instead.  Bars as for the other step tests: FP64 relative L2 <= 1e-12 against
the FP64 oracle, mixed form <= 1e-5.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from oracle import tad as O

from test_gpu_step import _device_problem, _rand_setup, rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion

SIZES = [16, 24, 36, 50, 54, 96, 128, 200, 512, 640, 1024, 3456, 4000, 4096]


def _numbers(n):
    dt = min(0.01, 1.0 / n)
    return dt, min(1e-2, 0.5 / (dt * (n // 2) ** 2))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("stepper", ["RK4", "ETDRK4", "FilteredRK4", "FilteredETDRK4"])
def test_run_vs_oracle(dev, n, T, stepper):
    print(f"line n={n} {T.__name__} {stepper}", flush=True)
    g, flows, c0 = _rand_setup(1, (n,), seed=5)
    dt, kappa = _numbers(n)
    p = _device_problem(dev, 1, (n,), flows, T, stepper, dt, kappa)
    o = O.Problem(g, flows, kappa=kappa, dt=dt, stepper=stepper)
    o.set_c(c0)
    p.sol = o.sol
    o.stepforward(7)
    ptf.stepforward_(p, 3)
    ptf.stepforward_(p, 4)
    assert p.clock.step == 7 and abs(p.clock.t - o.clock.t) < 1e-14
    assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)


@pytest.mark.parametrize("stepper", ["RK4", "ETDRK4"])
def test_long_run_records_and_stage_kernels(dev, stepper):
    """More steps than one launch takes; recorded diagnostics in between; the same run by the
    stage kernels (selected by a caller) to rounding."""
    g, flows, c0 = _rand_setup(1, (128,), seed=6)
    dt, kappa = _numbers(128)
    a, b = (_device_problem(dev, 1, (128,), flows, np.float64, stepper, dt, kappa) for _ in range(2))
    R, W, occ3, par, wg = b.get_variant(0)
    b.set_variant(0, R, W, occ3=occ3, par=par, wg=wg)
    for p in (a, b):
        TAD.set_c_(p, c0)
    ra = ptf.record_(a, 600, 250)
    rb = ptf.record_(b, 600, 250)
    assert list(ra["step"]) == [250, 500] and a.clock.step == 600
    assert rel(a.sol, b.sol) <= 1e-12 and rel(ra["c"], rb["c"]) <= 1e-12
    o = O.Problem(g, flows, kappa=kappa, dt=dt, stepper=stepper)
    o.set_c(c0)
    o.stepforward(600)
    assert rel(a.sol, o.sol) <= 1e-12


def test_time_varying_flow(dev):
    """A flow that changes every step (uploaded, and synthesised on the GPU)."""
    g, _, c0 = _rand_setup(1, (64,), seed=8)
    x = g.x
    host = TAD.Problem(dev, ptf.OneDAdvectingFlow(u=lambda x, t: np.cos(3 * t) * np.sin(x), steadyflow=False),
                       nx=64, κ=1e-2, dt=0.01)
    term = ptf.flows.FlowTerm(0, 1.0, fx="sin", kx=1.0, time="cos", omega=3.0)
    gpu = TAD.Problem(dev, ptf.flows.AnalyticAdvectingFlow(1, [term]), nx=64, κ=1e-2, dt=0.01)
    o = O.Problem(g, lambda t: (np.cos(3 * t) * np.sin(x),), kappa=1e-2, dt=0.01)
    o.set_c(c0)
    o.stepforward(20)
    for p in (host, gpu):
        TAD.set_c_(p, c0)
        ptf.stepforward_(p, 20)
        assert rel(p.sol, o.sol) <= 1e-12
