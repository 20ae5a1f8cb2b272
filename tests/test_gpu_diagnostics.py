"""Mass and variance (block sums with compensation) from one block's worth of elements to more
than the blocks of a launch, against long-double sums of the state on the host.  The compensated
FP64 sums are good to a few units of the last place of the result: 1e-14 relative.
"""
import numpy as np
import pytest

import passivetracerflows as ptf

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion


def _exact(sol, shape):
    w = np.full(sol.shape[-1], 2.0, np.longdouble)
    w[0] = w[-1] = 1
    s = sol.astype(np.clongdouble)
    n = np.longdouble(np.prod(shape))
    tot = (w * (s.real ** 2 + s.imag ** 2)).sum() - (s.flat[0].real ** 2 + s.flat[0].imag ** 2)
    return float(s.flat[0].real), float(tot / (n * n))


@pytest.mark.parametrize("n", [(16,), (2048,), (16, 8), (64, 64), (100, 36), (256, 256), (2048, 1024), (16, 8, 8),
                               (128, 64, 128)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_mass_and_variance(dev, n, T):
    print(f"diagnostics {n} {T.__name__}", flush=True)
    rng = np.random.default_rng(4)
    flow = [ptf.OneDAdvectingFlow, ptf.TwoDAdvectingFlow, ptf.ThreeDAdvectingFlow][len(n) - 1]()
    p = TAD.Problem(dev, flow, κ=1e-3, dt=1e-3, T=T, **dict(zip(("nx", "ny", "nz"), n)))
    p.sol = rng.standard_normal(p.grid.spec_shape) + 1j * rng.standard_normal(p.grid.spec_shape)
    mass, var = _exact(p.sol, n)
    assert TAD.mass(p) == mass
    assert abs(TAD.variance(p) - var) <= 1e-14 * var
    rec = ptf.record_(p, 2, 1, concentration=False)
    mass, var = _exact(p.sol, n)
    assert rec["mass"][1] == mass == TAD.mass(p) and rec["variance"][1] == TAD.variance(p)
    assert abs(rec["variance"][1] - var) <= 1e-14 * var
