"""Host memory that reading fields back keeps: the pinned slots belong to the process, so many
problems read once each, one after another or by several threads at once, map no more than the few
sets that the library holds (16 MiB each), not a set a problem.

Bar: growth of the process's readable mappings over the read-backs at most 16 MiB for each thread
and 64 MiB for everything else (stacks and heaps of the threads).  With slots for each of 24 problems
it would be 192 MiB.
"""
import threading

import numpy as np
import pytest

import passivetracerflows as ptf
from passivetracerflows._lib import call, dptr

from test_gpu_step import rel

pytestmark = pytest.mark.gpu
TAD = ptf.TracerAdvectionDiffusion
N = 1024


def _mapped():
    """Bytes of the process's mappings that can be read."""
    total = 0
    with open("/proc/self/maps") as f:
        for line in f:
            span, mode = line.split()[:2]
            if mode[0] == "r":
                a, b = (int(x, 16) for x in span.split("-"))
                total += b - a
    return total


def _problems(dev, count):
    out = []
    for i in range(count):
        p = TAD.Problem(dev, ptf.TwoDAdvectingFlow(), nx=N, κ=1e-3, dt=1e-3)
        c = np.random.default_rng(i).standard_normal((N, N))
        call("ptf_set_c", p._h, dptr(c))
        out.append((p, c, np.zeros((N, N))))
    call("ptf_device_synchronize")
    return out


@pytest.mark.parametrize("threads", [1, 4])
def test_reading_many_problems_once(dev, threads):
    probs = _problems(dev, 24)
    before = _mapped()

    def read(mine):
        for p, _, out in mine:
            call("ptf_updatevars", p._h, dptr(out))
    th = [threading.Thread(target=read, args=(probs[k::threads],)) for k in range(threads)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    grown = _mapped() - before
    print(f"{threads} threads: mapped memory grew by {grown / 2**20:.1f} MiB", flush=True)
    for _, c, out in probs:
        assert rel(out, c) <= 20 * np.finfo(np.float64).eps
    assert grown <= (64 + 16 * threads) << 20
