"""FP64 RK4 steps add to the state once a step.  Adding the first three stages' part and then the
last one's rounds the state twice, which shows as a larger error.

Bar: the error of the device's steps against the same steps in extended precision, over several
random fields, at most the mean of what the two ways give in numpy FP64 on these fields (ratio about
sqrt(2) where the rounding of the state is all there is).  All modes are excited alike, so that the
error does not hang on a few of them, and the time step is small: the errors of the transforms, which are
not the same here and there, enter with it.
"""
import numpy as np
import pytest
import scipy.fft as sf

import passivetracerflows as ptf

TAD = ptf.TracerAdvectionDiffusion
NX, NY, STEPS, SEEDS = 200, 108, 60, 3
LD = np.longdouble


def _axis(n):
    return (-LD(np.pi) + np.arange(n) * (LD(2 * np.pi) / n)).astype(np.float64)


def _inputs(seed):
    rng = np.random.default_rng([seed, 41])
    x, y = _axis(NX)[None, :], _axis(NY)[:, None]
    U, k = rng.uniform(0.5, 1.5), float(rng.integers(1, 4))
    u, v = -U * np.sin(k * x) * np.cos(k * y), U * np.cos(k * x) * np.sin(k * y)
    c = rng.standard_normal((NY, NX))     # all modes alike: the error does not hang on a few of them
    dt = 0.02 / (1.5 * (NX // 2 + NY // 2))     # the transforms' errors enter with dt: keep them small
    return u, v, c, dt, 0.02 / (dt * ((NX // 2) ** 2 + (NY // 2) ** 2))


def _c2r(ch):
    ch = sf.ifft(ch, axis=0)
    ch[:, 0] = ch[:, 0].real
    ch[:, -1] = ch[:, -1].real
    return sf.irfft(ch, n=NX, axis=1)


def _r2c(c):
    return sf.fft(sf.rfft(c, axis=1), axis=0)


def _steps(seed, T, roundings):
    """The state after the steps, computed in T (float64 or longdouble)."""
    u, v, c, dt, kappa = _inputs(seed)
    u, v, c = (a.astype(T) for a in (u, v, c))
    dt, kappa = T(dt), T(kappa)
    kx, ky = np.arange(NX // 2 + 1.0).astype(T)[None, :], np.fft.fftfreq(NY, 1.0 / NY).astype(T)[:, None]
    I = (1j * np.ones(1, T))[0]
    L = -kappa * kx ** 2 - kappa * ky ** 2
    sol = _r2c(c)

    def N(x):
        return _r2c(-u * _c2r(I * kx * x) - v * _c2r(I * ky * x))
    for _ in range(STEPS):
        r1 = N(sol) + L * sol
        r2 = N(sol + dt / 2 * r1) + L * (sol + dt / 2 * r1)
        x3 = sol + dt / 2 * r2
        r3 = N(x3) + L * x3
        x4 = sol + dt * r3
        s = (r1 / 6 + r2 / 3) + r3 / 3 + L / 6 * x4
        n4 = N(x4) / 6
        sol = sol + dt * (s + n4) if roundings == 1 else (sol + dt * s) + dt * n4
    return sol


def _errors(states):
    """Mean over the seeds of the relative L2 error of the fields of the states."""
    out = []
    for seed, sol in enumerate(states):
        want = _c2r(_steps(seed, LD, 1))
        got = _c2r(np.asarray(sol).astype(np.clongdouble))
        out.append(float(np.sqrt(((got - want) ** 2).sum() / (want ** 2).sum())))
    return np.mean(out)


def test_the_two_ways_differ():
    one, two = (_errors(_steps(s, np.float64, r) for s in range(2)) for r in (1, 2))
    assert 1e-17 < one < two < 1e-15


@pytest.mark.gpu
def test_one_rounding_of_the_state(dev):
    one, two = (_errors(_steps(s, np.float64, r) for s in range(SEEDS)) for r in (1, 2))

    def run(seed):
        u, v, c, dt, kappa = _inputs(seed)
        p = TAD.Problem(dev, ptf.TwoDAdvectingFlow(u=lambda x, y: u, v=lambda x, y: v), nx=NX, ny=NY, κ=kappa, dt=dt)
        TAD.set_c_(p, c)
        ptf.stepforward_(p, STEPS)
        return p.sol.copy()
    got = _errors(run(s) for s in range(SEEDS))
    print(f"one rounding {one:.3e}, two {two:.3e}, here {got:.3e}", flush=True)
    assert got <= 0.5 * (one + two)
