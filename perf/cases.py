"""The work that programs have this framework do, as cases whose time can be measured.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call (a
problem on the GPU with its flow and initial field, an ensemble, a transform plan with its
device arrays), ``run`` is one pass: advance the problem a number of steps and read the field
back, as a program does between two outputs.  Kernel variants are the ones the library picks by
itself: most programs do not call the autotuner.

The library runs in a process of its own.  It is built against one HIP runtime and refuses to
start where another framework (torch) has brought a different one into the process, so a program
that uses it does not load torch first.  ``prepare`` and ``run`` therefore talk to a helper
process (this file, started with ``serve``) that has only the library and numpy; the fields that
a pass returns are read back into memory that both processes map.

Fields are numpy arrays, x fastest.  FP32 problems ("f32": the mixed form) return FP32 fields.
"""
import json
import math
import mmap
import os
import subprocess
import sys
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TWO_PI = 2 * math.pi

# line lengths with a compiled transform that the drawn cases use: powers of two and 2^a m
POW2 = [16, 32, 64, 128, 256, 512, 1024, 2048]
RAGGED = [24, 36, 40, 48, 72, 80, 96, 100, 108, 144, 160, 192, 200, 216, 250, 288, 320, 384, 400,
          432, 500, 576, 640, 768, 800, 864, 1000, 1152, 1280, 1536, 1600, 1728, 2000]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _step(name, ndim, n, T, stepper, flow, nsteps, record=0):
    n = list(n) + [1] * (3 - len(n))
    if record:
        nsteps -= nsteps % record        # every pass makes the same number of records
    c = dict(kind="step", ndim=ndim, nx=n[0], ny=n[1], nz=n[2], T=T, stepper=stepper, flow=flow,
             nsteps=nsteps, record=record)
    return dict(c, name=name) if name else c


def _ensemble(name, counts, T, stepper, nsteps):
    c = dict(kind="ensemble", counts=",".join(f"{k}x{n}" for n, k in counts), T=T, stepper=stepper,
             nsteps=nsteps)
    return dict(c, name=name) if name else c


def _transform(name, nx, ny, nlayers, T, rounds):
    c = dict(kind="transform", nx=nx, ny=ny, nlayers=nlayers, T=T, rounds=rounds)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest problem: diffusion of a 1D Gaussian, mass and variance followed (a
        # script that plots them against the closed form)
        _step("diffusion1d_128_f64", 1, (128,), "f64", "RK4", "steady", 200, record=20),
        # a 1D advection-diffusion line at high resolution, exponential stepper
        _step("advect1d_1024_f32", 1, (1024,), "f32", "ETDRK4", "steady", 200),
        # a small 2D cellular-flow study with mass and variance followed
        _step("cellular2d_128_f64", 2, (128, 128), "f64", "RK4", "steady", 100, record=10),
        # the usual 2D size, FP32
        _step("cellular2d_256_f32", 2, (256, 256), "f32", "RK4", "steady", 160),
        # a 2D channel-shaped grid whose sides are no powers of two, filtered stepper
        _step("channel2d_400x216_f64", 2, (400, 216), "f64", "FilteredRK4", "steady", 80),
        # turbulent stirring by an unsteady random-phase flow at production resolution
        _step("turbulent2d_2048_f64", 2, (2048, 2048), "f64", "ETDRK4", "spectral", 24),
        # the same at exploratory resolution in FP32
        _step("turbulent2d_1024_f32", 2, (1024, 1024), "f32", "ETDRK4", "spectral", 60),
        # 3D chaotic advection by the ABC flow: the largest work
        _step("abc3d_256_f64", 3, (256, 256, 256), "f64", "RK4", "steady", 40),
        # the same at exploratory resolution in FP32
        _step("abc3d_128_f32", 3, (128, 128, 128), "f32", "RK4", "steady", 80),
        # a 3D box with sides that are no powers of two in an oscillating flow (evaluated on
        # the GPU at every step's clock)
        _step("tidal3d_96x80x144_f64", 3, (96, 80, 144), "f64", "RK4", "analytic", 40),
        # a parameter sweep: many cellular-flow members of four sizes advanced together
        _ensemble("ensemble512_f32", [(64, 273), (128, 137), (256, 68), (512, 34)], "f32", "RK4", 128),
        # a program's own pseudospectral loop over a layered field with the transform plan
        _transform("layers_256x256x8_f32", 256, 256, 8, "f32", 40),
    ]


def draw(rng):
    """One more case of the ranges above: grids from tens of points to 2048 a side, powers of
    two and not, both types, the steppers and the flows; the steps follow from the size so
    that a pass stays within the cost of the largest listed case."""
    def log_pick(sizes, lo, hi):
        ok = [s for s in sizes if lo <= s <= hi]
        t = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(ok, key=lambda s: abs(math.log(s / t)) + 0.02 * rng.random())

    def side(lo, hi):
        return log_pick(POW2 if rng.random() < 0.5 else RAGGED, lo, hi)

    def steps(points, lo, hi):
        work = 10 ** rng.uniform(6.5, 8.0)
        return int(min(hi, max(lo, work / points)))

    T = rng.choice(["f64", "f32"])
    family = rng.choice(["1d", "2d", "2d", "turb", "3d", "3d", "ensemble", "transform"])
    if family == "1d":
        nx = side(32, 2000)
        return _step(None, 1, (nx,), T, rng.choice(["RK4", "ETDRK4", "FilteredRK4"]), "steady",
                     rng.randrange(40, 320), record=rng.choice([0, 10, 25]) if T == "f64" else 0)
    if family == "2d":
        nx, ny = side(48, 1024), side(48, 1024)
        return _step(None, 2, (nx, ny), T, rng.choice(["RK4", "RK4", "ETDRK4", "FilteredETDRK4"]),
                     rng.choice(["steady", "steady", "analytic"]), steps(nx * ny, 10, 200),
                     record=rng.choice([0, 0, 10]) if T == "f64" else 0)
    if family == "turb":
        n = side(256, 2000)
        return _step(None, 2, (n, n), T, "ETDRK4", "spectral", steps(n * n, 8, 120))
    if family == "3d":
        nx, ny, nz = side(32, 216), side(32, 216), side(32, 216)
        return _step(None, 3, (nx, ny, nz), T, rng.choice(["RK4", "RK4", "ETDRK4"]),
                     rng.choice(["steady", "steady", "analytic"]), steps(nx * ny * nz, 8, 80))
    if family == "ensemble":
        sizes = rng.sample([32, 64, 96, 128, 192, 256], rng.choice([1, 2, 3]))
        counts = [(n, rng.randrange(2, max(3, min(160, 600000 // (n * n))))) for n in sorted(sizes)]
        points = sum(k * n * n for n, k in counts)
        return _ensemble(None, counts, T, rng.choice(["RK4", "RK4", "ETDRK4"]), steps(points, 20, 128))
    nx, ny = side(64, 1024), side(64, 1024)
    layers = rng.randrange(1, max(2, min(24, 2000000 // (nx * ny))))
    return _transform(None, nx, ny, layers, T, rng.randrange(10, 60))


# ---------------------------------------------------------------------------
# inputs: made from the case and the seed alone
# ---------------------------------------------------------------------------
def _dims(case):
    return [case["nx"], case["ny"], case["nz"]][: case.get("ndim", 2)]


def _points(n):
    start, step = np.longdouble(-TWO_PI / 2), np.longdouble(TWO_PI / n)
    return (start + np.arange(n, dtype=np.longdouble) * step).astype(np.float64)


def _axes(dims):
    """Coordinates shaped to broadcast over (z, y, x) fields."""
    nd = len(dims)
    return [_points(n).reshape([-1 if nd - 1 - a == i else 1 for i in range(nd)]) for a, n in enumerate(dims)]


def _blob(xs, centre, width):
    out = 1.0
    for x, c in zip(xs, centre):
        d = (x - c + math.pi) % TWO_PI - math.pi
        out = out * np.exp(-d * d / (2 * width * width))
    return out


def _initial(case, rng, dims):
    """A tracer field of unit size: a Gaussian patch on a background with large-scale waves."""
    xs = _axes(dims)
    c = 1.0 + _blob(xs, rng.uniform(-1, 1, len(dims)), rng.uniform(0.4, 0.6))
    for _ in range(3):
        wave = rng.uniform(0.1, 0.3)
        for x, k in zip(xs, rng.integers(1, 5, len(dims))):
            wave = wave * np.cos(k * x + rng.uniform(0, TWO_PI))
        c = c + wave
    if case.get("flow") == "spectral":
        c = c + 0.01 * rng.standard_normal(c.shape)
    return np.array(np.broadcast_to(c, tuple(reversed(dims))))


def _flow_numbers(case, rng):
    """The numbers of the case's flow."""
    if case["ndim"] == 3:
        f = dict(A=rng.uniform(0.5, 1), B=rng.uniform(0.5, 1), C=rng.uniform(0.5, 1))
    else:
        f = dict(U=rng.uniform(0.5, 1.5), k=int(rng.integers(1, 4)))
    if case["flow"] == "analytic":
        f.update(omega=rng.uniform(1, 6), tphase=rng.uniform(0, TWO_PI))
    return {k: float(v) for k, v in f.items()}


def _velocity(case, f, xs):
    """The steady part of the flow on the grid (functions of broadcastable coordinates)."""
    if case["ndim"] == 1:
        return [f["U"] * np.sin(f["k"] * xs[0]) + 0.25]
    if case["ndim"] == 2:
        x, y = xs
        return [-f["U"] * np.sin(f["k"] * x) * np.cos(f["k"] * y), f["U"] * np.cos(f["k"] * x) * np.sin(f["k"] * y)]
    x, y, z = xs
    return [f["A"] * np.sin(z) + f["C"] * np.cos(y), f["B"] * np.sin(x) + f["A"] * np.cos(z),
            f["C"] * np.sin(y) + f["B"] * np.cos(x)]


def _spectral_flow(n, rng, kpeak=8.0):
    """Half spectrum of a random-phase streamfunction (energy k^3 exp(-(k/kpeak)^2)) with unit
    rms velocity, and the frequencies |k|^(1/2) its phases turn at."""
    kx = np.arange(n // 2 + 1, dtype=np.float64)[None, :]
    ky = np.fft.fftfreq(n, 1.0 / n)[:, None]
    K = np.sqrt(kx * kx + ky * ky)
    low = K < 8 * kpeak                      # the rest is below 1e-27 of the peak
    amp = np.where(low & (K > 0), np.exp(-0.5 * (K / kpeak) ** 2), 0.0)
    theta = np.zeros_like(K)
    theta[low] = rng.uniform(0.0, TWO_PI, int(low.sum()))
    psih = amp * np.exp(1j * theta)
    col = psih[1:n // 2, 0]                  # a real psi: the kx = 0 column is Hermitian
    psih[n - 1:n // 2:-1, 0] = np.conj(col)
    psih[n // 2, 0] = 0
    weight = np.where((kx == 0) | (kx == n // 2), 1.0, 2.0)
    rms = math.sqrt(float((weight * K * K * np.abs(psih) ** 2).sum())) / (n * n)
    return psih / rms, np.sqrt(K)


def _numbers(case, rng):
    """Time step and diffusivities: the step resolves the advection of the largest wavenumber,
    ETDRK4 problems take fourth-order hyperdiffusion, the others plain diffusion."""
    dims = _dims(case)
    kmax = [n // 2 for n in dims]
    dt = 0.6 / (1.5 * sum(kmax))
    if case["stepper"].endswith("ETDRK4") and case["ndim"] == 2 and case["flow"] != "analytic":
        return dict(dt=dt, kappa=0.0, kappah=1e12 / float(max(kmax)) ** 8, nkappah=4)
    kappa = min(2e-3, 0.5 / (dt * sum(k * k for k in kmax)))
    return dict(dt=dt, kappa=kappa * rng.uniform(0.5, 1.0), kappah=0.0, nkappah=0)


def _inputs(case, seed):
    """Everything a pass of a stepping case depends on, as plain numbers and arrays."""
    rng = np.random.default_rng([seed, 17])
    d = dict(_numbers(case, rng))
    dims = _dims(case)
    if case["flow"] == "spectral":
        d["psih0"], d["omega"] = _spectral_flow(dims[0], rng)
    else:
        d["f"] = _flow_numbers(case, rng)
    d["c0"] = _initial(case, rng, dims)
    return d


def _counts(case):
    return [(int(n), int(k)) for k, n in (s.split("x") for s in case["counts"].split(","))]


def _members(case, seed):
    """Per size: (n, kappa, u, v, c0) with the members along the first axis.  One time step for
    all, which the largest grid resolves."""
    rng = np.random.default_rng([seed, 23])
    counts = _counts(case)
    nmax = max(n for n, _ in counts)
    dt = 0.6 / (1.5 * nmax)
    out = []
    for n, k in counts:
        x = _points(n)
        kappa = np.minimum(np.exp(rng.uniform(math.log(5e-4), math.log(5e-3), k)), 0.5 / (dt * 0.5 * n * n))
        wave, U = rng.integers(1, 5, k).astype(np.float64), rng.uniform(0.5, 1.5, k)
        s, c = np.sin(wave[:, None] * x), np.cos(wave[:, None] * x)
        u = -(U[:, None] * c)[:, :, None] * s[:, None, :]
        v = (U[:, None] * s)[:, :, None] * c[:, None, :]
        cen, wid = rng.uniform(-math.pi, math.pi, (k, 2)), rng.uniform(0.3, 0.5, k)
        g = [np.exp(-((x - cen[:, a, None] + math.pi) % TWO_PI - math.pi) ** 2 / (2 * wid[:, None] ** 2)) for a in (0, 1)]
        out.append((n, kappa, u, v, 1.0 + g[1][:, :, None] * g[0][:, None, :]))
    return dt, out


def _field(case, seed):
    """The layered real field that a transform case starts from."""
    rng = np.random.default_rng([seed, 29])
    dt = np.float64 if case["T"] == "f64" else np.float32
    out = np.empty((case["nlayers"], case["ny"], case["nx"]), dt)
    for a in out:
        a[...] = _initial({}, rng, [case["nx"], case["ny"]])
        a += 0.1 * rng.standard_normal(a.shape)
    return out


def _outputs(case):
    """(name, shape, dtype) of what a pass returns."""
    real = "float64" if case["T"] == "f64" else "float32"
    if case["kind"] == "step":
        o = [("c", list(reversed(_dims(case))), real)]
        if case["record"]:
            n = case["nsteps"] // case["record"]
            o += [("mass", [n], "float64"), ("variance", [n], "float64")]
        return o
    if case["kind"] == "ensemble":
        return [(f"c{n}", [k, n, n], real) for n, k in _counts(case)]
    lead = [case["nlayers"]] if case["nlayers"] > 1 else []
    return [("f", lead + [case["ny"], case["nx"]], real),
            ("fh", lead + [case["ny"], case["nx"] // 2 + 1], "complex128" if case["T"] == "f64" else "complex64")]


def _nbytes(shape, dtype):
    return int(np.prod(shape)) * np.dtype(dtype).itemsize


def _mapped(case, buf):
    """The case's output arrays over a shared buffer (each at a 4 KiB boundary)."""
    out, at = {}, 0
    for name, shape, dtype in _outputs(case):
        out[name] = np.frombuffer(buf, dtype=dtype, count=int(np.prod(shape)), offset=at).reshape(shape)
        at += -(-_nbytes(shape, dtype) // 4096) * 4096
    return out


def _mapped_bytes(case):
    return sum(-(-_nbytes(s, d) // 4096) * 4096 for _, s, d in _outputs(case))


# ---------------------------------------------------------------------------
# the helper process: the program that uses the library
# ---------------------------------------------------------------------------
def _make_step(ptf, case, seed, out):
    from passivetracerflows._lib import call, dptr
    TAD = ptf.TracerAdvectionDiffusion
    d = _inputs(case, seed)
    kw = dict(nx=case["nx"], κ=d["kappa"], dt=d["dt"], stepper=case["stepper"],
              T=np.float64 if case["T"] == "f64" else np.float32)
    if case["ndim"] >= 2:
        kw["ny"] = case["ny"]
    if case["ndim"] == 3:
        kw["nz"] = case["nz"]
    if case["ndim"] == 2:
        kw.update(κh=d["kappah"], nκh=d["nkappah"])
    if case["flow"] == "spectral":
        flow = ptf.SpectralStreamfunctionFlow(d["psih0"], d["omega"])
    elif case["flow"] == "analytic":
        f = d["f"]
        osc = dict(time="cos", omega=f["omega"], tphase=f["tphase"])
        flow = (ptf.flows.abc_flow(f["A"], f["B"], f["C"], **osc) if case["ndim"] == 3 else
                ptf.flows.cellular_flow(f["U"], f["k"], **osc))
    else:
        vel = _velocity(case, d["f"], _axes(_dims(case)))
        fns = [lambda *a, v=v: v for v in vel]
        flow = [ptf.OneDAdvectingFlow, ptf.TwoDAdvectingFlow, ptf.ThreeDAdvectingFlow][case["ndim"] - 1](*fns)
    prob = TAD.Problem(ptf.ROCm(0), flow, **kw)
    call("ptf_set_c", prob._h, dptr(d["c0"]))
    c = out["c"] if out["c"].dtype == np.float64 else np.empty(out["c"].shape)

    def go():
        if case["record"]:
            r = ptf.record_(prob, case["nsteps"], case["record"], concentration=False)
            out["mass"][...], out["variance"][...] = r["mass"], r["variance"]
        else:
            ptf.stepforward_(prob, case["nsteps"])
        call("ptf_updatevars", prob._h, dptr(c))     # updatevars! into the program's own array
        if c is not out["c"]:
            out["c"][...] = c
    return go


def _make_ensemble(ptf, case, seed, out):
    from passivetracerflows._lib import call, dptr
    ptf.ROCm(0)
    dt, groups = _members(case, seed)
    members = [dict(n=n, kappa=float(k)) for n, kappa, *_ in groups for k in kappa]
    ens = ptf.Ensemble(members, dt, precision="mixed" if case["T"] == "f32" else "fp64", stepper=case["stepper"])
    i, to = 0, []
    for n, kappa, u, v, c0 in groups:
        o = out[f"c{n}"]
        for b in range(len(kappa)):
            ens.set_flow(i, u[b], v[b])
            ens.set_c(i, c0[b])
            to.append((i, o[b], o[b] if o.dtype == np.float64 else np.empty((n, n))))
            i += 1

    def go():
        ens.step(case["nsteps"])
        for m, o, c in to:
            call("ptf_ensemble_get_c", ens._h, m, dptr(c))
            if c is not o:
                o[...] = c
    return go


def _make_transform(ptf, case, seed, out):
    from passivetracerflows._lib import call
    FF = ptf.FourierFlows
    grid = FF.TwoDGrid(ptf.ROCm(0), nx=case["nx"], ny=case["ny"], T=np.float64 if case["T"] == "f64" else np.float32)
    plan = FF.RFFTPlan(grid, nlayers=case["nlayers"])
    a = _field(case, seed)
    f = FF.DeviceArray.from_host(a if case["nlayers"] > 1 else a[0])
    fh = FF.DeviceArray(out["fh"].shape, out["fh"].dtype)

    def go():
        for _ in range(case["rounds"]):
            ptf.mul_(fh, plan, f)
            ptf.dealias_(fh, grid, plan)
            ptf.ldiv_(f, plan, fh)
        for name, x in (("f", f), ("fh", fh)):
            call("ptf_device_synchronize")
            call("ptf_buffer_download", out[name].ctypes.data, x.ptr, x.nbytes)
    return go


def _serve():
    answers = os.fdopen(os.dup(1), "wb", buffering=0)
    os.dup2(2, 1)                        # whatever else is printed goes to stderr
    sys.path[:0] = [ROOT, os.path.join(ROOT, "passivetracerflows.jl_amd")]
    make = dict(step=_make_step, ensemble=_make_ensemble, transform=_make_transform)
    states = {}
    for line in sys.stdin.buffer:
        try:
            do, _, rest = line.decode().rstrip("\n").partition(" ")
            if do == "run":
                states[int(rest)][0]()
            elif do == "drop":
                states.pop(int(rest), None)
                continue
            else:
                import passivetracerflows as ptf
                d = json.loads(rest)
                with open(d["file"], "r+b") as f:
                    buf = mmap.mmap(f.fileno(), 0)
                out = _mapped(d["case"], buf)
                for a in out.values():
                    a.fill(0)
                go = make[d["case"]["kind"]](ptf, d["case"], d["seed"], out)
                ptf._lib.call("ptf_device_synchronize")
                states[d["id"]] = (go, buf)
            answers.write(b"ok\n")
        except Exception as e:
            answers.write((f"{type(e).__name__}: {e}".replace("\n", " ") + "\n").encode())
    os._exit(0)


class _Helper:
    one = None

    def __init__(self):
        self.p = subprocess.Popen([sys.executable, "-u", os.path.abspath(__file__), "serve"], cwd=ROOT,
                                  stdin=subprocess.PIPE, stdout=subprocess.PIPE, bufsize=0)
        self.answers = os.fdopen(os.dup(self.p.stdout.fileno()), "rb")
        self.count = 0

    def tell(self, line):
        os.write(self.p.stdin.fileno(), line)

    def ask(self, line):
        self.tell(line)
        got = self.answers.readline()
        if got != b"ok\n":
            raise RuntimeError(got.decode().strip() or f"the helper process ended ({self.p.poll()})")


class _State:
    def __init__(self, case, seed):
        if _Helper.one is None:
            _Helper.one = _Helper()
        self.helper = h = _Helper.one
        h.count += 1
        self.id = h.count
        with tempfile.NamedTemporaryFile(dir="/dev/shm" if os.path.isdir("/dev/shm") else None) as f:
            f.truncate(_mapped_bytes(case))
            self.out = _mapped(case, mmap.mmap(f.fileno(), 0))
            h.ask(b"make " + json.dumps(dict(id=self.id, case=case, seed=seed, file=f.name)).encode() + b"\n")
        self.line = b"run %d\n" % self.id

    def __del__(self):
        try:
            self.helper.tell(b"drop %d\n" % self.id)
        except Exception:
            pass


def prepare(case, seed):
    return _State(case, int(seed))


def run(state):
    state.helper.ask(state.line)
    return state.out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every step reads the state and the flow and writes the state once (the flow of
    a spectral problem is read as its spectrum); the pass writes the field it returns.  Flops:
    the real transforms of four stages (2.5 N log2 N each: one inverse per dimension, one
    forward) and about 10 operations a point and dimension beside them."""
    r = 8 if case["T"] == "f64" else 4

    def stepping(dims, nsteps, members=1, spectral=False):
        nd, N = len(dims), math.prod(dims)
        S = (dims[0] // 2 + 1) * math.prod(dims[1:])
        flow = S * 24 if spectral else N * nd * r
        one = 4 * ((nd + 1) * 2.5 * N * math.log2(N) + 10 * nd * N)
        return members * (nsteps * (2 * S * 2 * r + flow) + N * r), members * nsteps * one

    if case["kind"] == "step":
        if case["flow"] == "analytic":   # evaluated from small tables
            b, f = stepping(_dims(case), case["nsteps"])
            b -= case["nsteps"] * math.prod(_dims(case)) * case["ndim"] * r
        else:
            b, f = stepping(_dims(case), case["nsteps"], spectral=case["flow"] == "spectral")
        return {"bytes": b, "flops": f}
    if case["kind"] == "ensemble":
        w = [stepping([n, n], case["nsteps"], k) for n, k in _counts(case)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    N = case["nx"] * case["ny"]
    S = (case["nx"] // 2 + 1) * case["ny"]
    R = case["nlayers"] * case["rounds"]
    # forward: field in, spectrum out; inverse: spectrum in, field out
    return {"bytes": R * 2 * (N * r + S * 2 * r), "flops": R * 2 * 2.5 * N * math.log2(N)}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------
def exact(case, seed):
    import torch
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if case["kind"] == "transform":
        f = torch.from_numpy(_field(case, int(seed)).astype(np.float64)).to(dev)
        for _ in range(case["rounds"]):
            fh = _dealiased(torch, case, f)
            f = _c2r(torch, fh, [case["ny"], case["nx"]])
        if case["nlayers"] == 1:
            f, fh = f[0], fh[0]
        return {"f": f.cpu().numpy(), "fh": fh.cpu().numpy()}
    if case["kind"] == "ensemble":
        dt, groups = _members(case, int(seed))
        out = {}
        for n, kappa, u, v, c0 in groups:
            k = torch.from_numpy(kappa).to(dev)[:, None, None]
            vel = [torch.from_numpy(a).to(dev) for a in (u, v)]
            kx, ky = _wavenumbers(torch, [n, n], dev)
            L = -k * kx ** 2 - k * ky ** 2
            c, _ = _advance(torch, torch.from_numpy(c0).to(dev), lambda t: vel, L, dt, case["stepper"], case["nsteps"], 0)
            out[f"c{n}"] = c.cpu().numpy()
        return out
    dims = _dims(case)
    d = _inputs(case, int(seed))
    ks = _wavenumbers(torch, dims, dev)
    L = sum(-d["kappa"] * k ** 2 for k in ks)
    if d["nkappah"]:
        L = L - d["kappah"] * sum(k ** 2 for k in ks) ** d["nkappah"]
    if case["flow"] == "spectral":
        psih, om = torch.from_numpy(d["psih0"]).to(dev)[None], torch.from_numpy(d["omega"]).to(dev)[None]

        def vel(t):
            p = psih * torch.exp(-1j * om * t)
            return [_c2r(torch, -1j * ks[1] * p, [dims[1], dims[0]]), _c2r(torch, 1j * ks[0] * p, [dims[1], dims[0]])]
    else:
        steady = [torch.from_numpy(np.array(np.broadcast_to(a, d["c0"].shape)))[None].to(dev)
                  for a in _velocity(case, d["f"], _axes(dims))]

        def vel(t):
            if case["flow"] == "steady":
                return steady
            a = math.cos(d["f"]["omega"] * t + d["f"]["tphase"])
            return [a * s for s in steady]
    c, rec = _advance(torch, torch.from_numpy(d["c0"]).to(dev)[None], vel, L, d["dt"], case["stepper"],
                      case["nsteps"], case["record"])
    out = {"c": c[0].cpu().numpy()}
    if case["record"]:
        out["mass"], out["variance"] = (np.array(r) for r in zip(*rec))
    return out


def _wavenumbers(torch, dims, dev):
    """kr, l, m shaped to broadcast over (members, z, y, x) half spectra."""
    nd = len(dims)
    out = []
    for a, n in enumerate(dims):
        k = np.arange(n // 2 + 1.0) if a == 0 else np.fft.fftfreq(n, 1.0 / n)
        out.append(torch.from_numpy(k).to(dev).reshape([1] + [-1 if nd - 1 - a == i else 1 for i in range(nd)]))
    return out


def _c2r(torch, ch, shape):
    """Inverse real transform: complex inverses along z and y, then along x with the real parts
    of the first and last wavenumbers."""
    nd = len(shape)
    if nd > 1:
        ch = torch.fft.ifftn(ch, dim=list(range(-nd, -1)))
    else:
        ch = ch.clone()
    for k in (0, -1):
        ch[..., k] = ch[..., k].real + 0j
    return torch.fft.irfft(ch, n=shape[-1], dim=-1)


def _r2c(torch, c, nd):
    ch = torch.fft.rfft(c, dim=-1)
    return torch.fft.fftn(ch, dim=list(range(-nd, -1))) if nd > 1 else ch


def _dealiased(torch, case, f):
    """Spectrum of the field with the aliased third of the wavenumbers removed."""
    fh = _r2c(torch, f, 2)
    lo = [math.floor((1 - 1 / 3) / 2 * n) for n in (case["nx"], case["ny"])]
    hi = math.ceil((1 + 1 / 3) / 2 * case["ny"])
    fh[..., lo[0]:] = 0
    fh[..., lo[1]:hi, :] = 0
    return fh


def _advance(torch, c, vel, L, dt, stepper, nsteps, record):
    nd, shape = c.dim() - 1, list(c.shape[1:])
    dims = shape[::-1]
    ks = _wavenumbers(torch, dims, c.device)
    sol = _r2c(torch, c, nd)

    def N(x):
        g = 0
        for k, w in zip(ks, flow):
            g = g - w * _c2r(torch, 1j * k * x, shape)
        return _r2c(torch, g, nd)

    filt = None
    if stepper.startswith("Filtered"):
        K = torch.sqrt(sum((2 * k / n) ** 2 for k, n in zip(ks, dims)))
        decay = -math.log(1e-15) / (1 - 0.65) ** 4
        filt = torch.where(K < 0.65, torch.ones_like(K), torch.exp(-decay * (K - 0.65) ** 4))
    etd = stepper.endswith("ETDRK4")
    if etd:
        E, E2 = torch.exp(dt * L), torch.exp(dt * L / 2)
        zeta, alpha, beta, gamma = 0, 0, 0, 0
        for j in range(32):              # contour means around each dt L
            z = dt * L + complex(math.cos(TWO_PI * (j + 0.5) / 32), math.sin(TWO_PI * (j + 0.5) / 32))
            ez = torch.exp(z)
            zeta = zeta + ((torch.exp(z / 2) - 1) / z).real
            alpha = alpha + ((-4 - z + ez * (4 - 3 * z + z ** 2)) / z ** 3).real
            beta = beta + ((2 + z + ez * (-2 + z)) / z ** 3).real
            gamma = gamma + ((-4 - 3 * z - z ** 2 + ez * (4 - z)) / z ** 3).real
        zeta, alpha, beta, gamma = (dt / 32 * q for q in (zeta, alpha, beta, gamma))
    t, rec = 0.0, []
    for i in range(nsteps):
        flow = vel(t)
        if etd:
            n1 = N(sol)
            s1 = E2 * sol + zeta * n1
            n2 = N(s1)
            n3 = N(E2 * sol + zeta * n2)
            n4 = N(E2 * s1 + zeta * (2 * n3 - n1))
            sol = E * sol + alpha * n1 + 2 * beta * (n2 + n3) + gamma * n4
        else:
            r1 = N(sol) + L * sol
            x = sol + dt / 2 * r1
            r2 = N(x) + L * x
            x = sol + dt / 2 * r2
            r3 = N(x) + L * x
            x = sol + dt * r3
            r4 = N(x) + L * x
            sol = sol + dt * (r1 / 6 + r2 / 3 + r3 / 3 + r4 / 6)
        if filt is not None:
            sol = filt * sol
        t += dt
        if record and (i + 1) % record == 0:
            x = _c2r(torch, sol, shape)
            rec.append((float(x.sum()), float(((x - x.mean()) ** 2).mean())))
    return _c2r(torch, sol, shape), rec


if __name__ == "__main__" and sys.argv[1:] == ["serve"]:
    _serve()
