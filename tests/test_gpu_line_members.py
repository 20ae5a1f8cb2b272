"""Groups of 1D members, which the C interface of the ensemble takes: every member steps as a problem
of its own does (the same whole-run kernel, so the same bits), with graphs, without, by the stage
kernels when a caller selects them (to rounding: FP64 1e-12, mixed 1e-5), and its diagnostics are the
problem's.
"""
import ctypes as C

import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows import _lib
from passivetracerflows._lib import call, dptr

from test_gpu_step import rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion
N, DT = [128, 128, 50, 128], 2e-3


def _desc(n, kappa, T, stepper):
    d = _lib.ptf_desc()
    d.ndim = 1
    d.precision = _lib.PTF_FP64 if T == np.float64 else _lib.PTF_MIXED
    d.n[0], d.n[1], d.n[2] = n, 1, 1
    d.L[0], d.L[1], d.L[2] = 2 * np.pi, 1.0, 1.0
    d.kappa = d.eta = d.iota = kappa
    d.stepper = _lib.STEPPERS[stepper.upper()]
    d.dt = DT
    d.flow_kind = _lib.PTF_FLOW_STEADY
    return d


@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("stepper", ["RK4", "ETDRK4"])
def test_members_step_as_problems(dev, T, stepper):
    rng = np.random.default_rng(5)
    kappa = [1e-3 * (i + 1) for i in range(len(N))]
    u = [1 + 0.3 * np.sin(np.arange(n) * 2 * np.pi / n + i) for i, n in enumerate(N)]
    c0 = [rng.standard_normal(n) for n in N]
    want = []
    for i, n in enumerate(N):
        p = TAD.Problem(dev, ptf.OneDAdvectingFlow(u=lambda x, i=i: u[i]), nx=n, κ=kappa[i], dt=DT, T=T, stepper=stepper)
        TAD.set_c_(p, c0[i])
        ptf.stepforward_(p, 37)
        want.append((p.sol.copy(), TAD.mass(p), TAD.variance(p)))
    descs = (_lib.ptf_desc * len(N))(*[_desc(n, k, T, stepper) for n, k in zip(N, kappa)])
    for graph, stages in [(1, False), (0, False), (1, True)]:
        h = C.c_void_p()
        call("ptf_ensemble_create", descs, len(N), C.byref(h))
        h = h.value
        for i in range(len(N)):
            call("ptf_ensemble_set_flow", h, i, dptr(np.ascontiguousarray(u[i])), None)
            call("ptf_ensemble_set_c", h, i, dptr(c0[i]))
        if stages:
            ns = C.c_int32()
            call("ptf_ensemble_num_slots", h, C.byref(ns))
            for s in range(ns.value):
                R, W, f = C.c_int32(), C.c_int32(), C.c_int32()
                call("ptf_ensemble_get_variant", h, s, C.byref(R), C.byref(W), C.byref(f))
                if f.value & 8:          # the first of a group turns its run kernel off
                    call("ptf_ensemble_set_variant", h, s, R.value, W.value, f.value & ~8)
        call("ptf_ensemble_step", h, 37, graph)
        for i, n in enumerate(N):
            sol = np.zeros(n // 2 + 1, np.complex128)
            call("ptf_ensemble_get_sol", h, i, dptr(sol.view(np.float64)))
            if stages:
                assert rel(sol, want[i][0]) <= (1e-12 if T == np.float64 else 1e-5)
                continue
            m, v = C.c_double(), C.c_double()
            call("ptf_ensemble_diagnostics", h, i, C.byref(m), C.byref(v))
            assert np.array_equal(sol, want[i][0]) and (m.value, v.value) == want[i][1:]
        call("ptf_ensemble_destroy", h)
