"""Transforms at the lines of the rule that gives a plan its default kernels: rows of 2048 and 4096
points (one, few, and enough to stream), columns of 256 points that stream and that do not.  Against
numpy in FP64; bars as for the other transforms: 1e-14 in FP64 and 1e-6 in FP32, relative L2.
"""
import numpy as np
import pytest

import passivetracerflows as ptf

from test_gpu_step import rel

pytestmark = pytest.mark.gpu
FF = ptf.FourierFlows


@pytest.mark.parametrize("n,layers", [((4096,), 1), ((2048,), 1), ((4096, 16), 1), ((2048, 64), 31), ((2048, 64), 33),
                                      ((4096, 1024), 1), ((2048, 2048), 1), ((256, 256, 256), 1), ((256, 16, 256), 1)])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_both_directions(dev, n, layers, T):
    print(f"plan {n} x{layers} {T.__name__}", flush=True)
    grid = [FF.OneDGrid, FF.TwoDGrid, FF.ThreeDGrid][len(n) - 1](dev, T=T, **dict(zip(("nx", "ny", "nz"), n)))
    plan = FF.RFFTPlan(grid, nlayers=layers)
    shape = ((layers,) if layers > 1 else ()) + tuple(reversed(n))
    a = np.random.default_rng(2).standard_normal(shape).astype(T)
    f = FF.DeviceArray.from_host(a)
    fh = FF.DeviceArray(shape[:-1] + (n[0] // 2 + 1,), np.complex128 if T == np.float64 else np.complex64)
    ptf.mul_(fh, plan, f)
    axes = tuple(range(len(shape) - len(n), len(shape)))
    bar = 1e-14 if T == np.float64 else 1e-6
    assert rel(fh.to_host(), np.fft.rfftn(a.astype(np.float64), axes=axes)) <= bar
    ptf.ldiv_(f, plan, fh)
    assert rel(f.to_host(), a) <= bar
