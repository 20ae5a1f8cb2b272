"""Kernels whose work is dealt out by rows: the analytic flow synthesis (every layout, numbers of
terms around the four read together) and dealias! (batches, axes shorter than a wavefront).

Bars: a synthesised flow against the same flow evaluated by numpy: the nonlinear term agrees to
1e-12 (FP64) and 1e-5 (mixed form); dealias! is exact.
"""
import numpy as np
import pytest

import passivetracerflows as ptf
from oracle import tad as O
from passivetracerflows import flows as F

from test_gpu_flows import _c0, evaluate
from test_gpu_step import rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion


@pytest.mark.parametrize("n", [(36,), (40, 50), (24, 72), (500, 64), (16, 20, 12), (40, 36, 96), (128, 24, 64)])
@pytest.mark.parametrize("terms", [1, 4, 5, 16])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_analytic_synthesis(dev, n, terms, T):
    print(f"analytic n={n} terms={terms} {T.__name__}", flush=True)
    nd = len(n)
    rng = np.random.default_rng(terms)
    pick = lambda: ["1", "sin", "cos"][rng.integers(3)]
    ts = [F.FlowTerm(i % nd, rng.uniform(0.2, 1), fx=pick(), fy=pick(), fz=pick(), kx=1.0, ky=2.0, kz=1.0,
                     px=rng.uniform(), py=rng.uniform(), pz=rng.uniform(), time="cos", omega=3.0, tphase=0.2)
          for i in range(terms)]
    flow = F.AnalyticAdvectingFlow(nd, ts)
    g = O.Grid(nd, n[0], **dict(zip(("ny", "nz"), n[1:])))
    p = TAD.Problem(dev, flow, κ=1e-3, dt=1e-3, T=T, **dict(zip(("nx", "ny", "nz"), n)))
    o = O.Problem(g, lambda t: evaluate(flow, g, t), kappa=1e-3, dt=1e-3)
    c0 = _c0(g, 4)
    o.set_c(c0)
    TAD.set_c_(p, c0)
    o.stepforward(3)
    ptf.stepforward_(p, 3)
    assert rel(p.sol, o.sol) <= (1e-12 if T == np.float64 else 1e-5)


@pytest.mark.parametrize("n,layers", [((64, 48), 5), ((16, 20), 3), ((500, 36), 1), ((24, 32), 257)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_dealias_layers(dev, n, layers, T):
    print(f"dealias n={n} layers={layers} {T.__name__}", flush=True)
    grid = ptf.FourierFlows.TwoDGrid(dev, nx=n[0], ny=n[1], T=T)
    plan = ptf.FourierFlows.RFFTPlan(grid, nlayers=layers)
    g = O.Grid(2, n[0], ny=n[1])
    shape = ((layers,) if layers > 1 else ()) + (n[1], n[0] // 2 + 1)
    rng = np.random.default_rng(1)
    fh = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(
        np.complex128 if T == np.float64 else np.complex64)
    d = ptf.FourierFlows.DeviceArray.from_host(fh)
    ptf.dealias_(d, grid, plan)
    got = d.to_host()
    for k in range(layers):
        a, b = (got[k], fh[k]) if layers > 1 else (got, fh)
        assert np.array_equal(a, O.dealias(g, b))
