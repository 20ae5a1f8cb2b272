"""What a 1D problem steps with: the whole-run kernel unless a caller selects a stage kernel, and
again after a selection with the run flag; the same with a tuning cache, tuned or loaded; and the
profiled step.  The kernels are deterministic, so states taken by the same kernel are compared
bit for bit; the stage kernels against the whole-run kernel at the bar of the other step tests
(FP64 relative L2 <= 1e-12, mixed form <= 1e-5).
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows._lib import PTFError

from test_gpu_step import _device_problem, _rand_setup, rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion


def _stepped(p, c0, n=20):
    TAD.set_c_(p, c0)
    ptf.stepforward_(p, n)
    return p.sol.copy()


def _make(dev, T, stepper="RK4", n=128):
    g, flows, c0 = _rand_setup(1, (n,), seed=6)
    return _device_problem(dev, 1, (n,), flows, T, stepper, 1.0 / n, 1e-4), c0


@pytest.mark.parametrize("T,stepper", [(np.float64, "RK4"), (np.float64, "FilteredETDRK4"), (np.float32, "RK4"),
                                       (np.float32, "ETDRK4")])
def test_selection_and_profile(dev, T, stepper):
    print(f"1D selection {T.__name__} {stepper}", flush=True)
    p, c0 = _make(dev, T, stepper)
    ns = len(p.slots())
    assert all(p.whole_run(i) for i in range(ns)) and all(" run " in s for s in p.slots())
    run = _stepped(p, c0)
    TAD.set_c_(p, c0)
    ms = p.step_profiled(20)
    assert len(ms) == ns and ms[0] > 0 and ms[1:] == [0.0] * (ns - 1)
    assert np.array_equal(p.sol, run)
    p.autotune()                                   # nothing to choose, nothing changed
    assert p.whole_run(0) and np.array_equal(_stepped(p, c0), run)
    v = p.get_variant(1)
    p.set_variant(1, *v)                           # the stage kernels
    assert not any(p.whole_run(i) for i in range(ns)) and not any(" run " in s for s in p.slots())
    stages = _stepped(p, c0)
    assert rel(stages, run) <= (1e-12 if T == np.float64 else 1e-5)
    TAD.set_c_(p, c0)
    assert min(p.step_profiled(20)) > 0 and np.array_equal(p.sol, stages)
    p.set_variant(3, *p.get_variant(3), run=True)  # the whole-run kernel again
    assert all(p.whole_run(i) for i in range(ns)) and np.array_equal(_stepped(p, c0), run)


@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_tuning_cache_runs_the_same_kernel(dev, tmp_path, T):
    path = str(tmp_path / "tuning.json")
    ref, c0 = _make(dev, T)
    want = _stepped(ref, c0)
    for how in ("tuned", "cache"):
        p, _ = _make(dev, T)
        assert p.autotune(cache=path) == how
        assert p.whole_run(0) and np.array_equal(_stepped(p, c0), want)


def test_profiled_steps_of_an_analytic_flow(dev):
    term = ptf.flows.FlowTerm(0, 1.0, fx="sin", kx=1.0, time="cos", omega=3.0)
    c0 = np.random.default_rng(2).standard_normal(64)
    a, b = (TAD.Problem(dev, ptf.flows.AnalyticAdvectingFlow(1, [term]), nx=64, κ=1e-2, dt=0.01) for _ in range(2))
    for p in (a, b):
        TAD.set_c_(p, c0)
    ptf.stepforward_(a, 7)
    ms = b.step_profiled(7)
    assert a.clock.t == b.clock.t and np.array_equal(a.sol, b.sol)
    assert ms[0] > 0 and ms[1] > 0 and ms[2:] == [0.0] * (len(ms) - 2)


def test_run_flag_where_no_run_kernel_is(dev):
    p = TAD.Problem(dev, ptf.TwoDAdvectingFlow(), nx=16, κ=1e-2, dt=0.01)
    with pytest.raises(PTFError):
        p.set_variant(0, *p.get_variant(0), run=True)


def test_members_have_no_run_kernel(dev):
    e = ptf.Ensemble([dict(n=16, kappa=1e-3)] * 2, 0.01)
    assert not any(e.whole_run(i) for i in range(len(e.slots())))
