"""Fields read back through pinned slots (ptf_updatevars, ptf_get_sol, ptf_ensemble_get_c): one
slot, several, more chunks than slots, and the sizes from which helper threads copy, with
bricked and plain layouts and a ragged last chunk.

Bars: set_c! then updatevars! is one forward and one inverse transform: relative error at most
20 eps of the working precision (log2 of 3e6 points is 22, and the error of a transform pair
grows with its square root); spectra against numpy likewise.  A misplaced value is an error of
order one.
"""
import numpy as np
import pytest

import passivetracerflows as ptf

from test_gpu_step import rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion

# 8 bytes a point (FP64): 512 KB is one slot; 8 MB starts the helper threads; 18 MB and the
# spectrum of it are more than 8 slots of 2 MB
SIZES = [(16,), (256, 256), (288, 256), (250, 500), (1024, 1024), (1152, 2000), (24, 20, 50), (144, 144, 144)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_field_and_spectrum(dev, n, T):
    print(f"read back n={n} {T.__name__}", flush=True)
    nd = len(n)
    flow = [ptf.OneDAdvectingFlow(), ptf.TwoDAdvectingFlow(), ptf.ThreeDAdvectingFlow()][nd - 1]
    kw = dict(zip(("nx", "ny", "nz"), n))
    p = TAD.Problem(dev, flow, κ=1e-3, dt=1e-3, T=T, **kw)
    c = np.random.default_rng(3).standard_normal(tuple(reversed(n)))
    TAD.set_c_(p, c)
    bar = 20 * np.finfo(T).eps
    for _ in range(2):     # the second time through slots that are there
        TAD.updatevars_(p)
        assert rel(p.vars.c, c) <= bar
        assert rel(p.sol, np.fft.rfftn(c)) <= bar
    assert np.abs(p.vars.c - c).max() <= 100 * bar


def test_problems_read_back_at_once(dev):
    """Two problems of different sizes, each read back by a thread of its own."""
    import threading
    out = {}

    def work(n):
        p = TAD.Problem(dev, ptf.TwoDAdvectingFlow(), nx=n, κ=1e-3, dt=1e-3)
        c = np.random.default_rng(n).standard_normal((n, n))
        TAD.set_c_(p, c)
        worst = 0.0
        for _ in range(5):
            TAD.updatevars_(p)
            worst = max(worst, rel(p.vars.c, c))
        out[n] = worst

    threads = [threading.Thread(target=work, args=(n,)) for n in (128, 1024)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sorted(out) == [128, 1024] and max(out.values()) <= 20 * np.finfo(np.float64).eps
