"""Persistent kernel-variant choices (the autotuner's output, reused across processes).

The autotuner (``ptf_autotune``) times every compiled variant of every launch slot on the
problem's own buffers and keeps the fastest.  Its choice varies a little from run to run
where two variants are within noise of each other, so a benchmark that is profiled in a
second process would otherwise time one variant and profile another.  A cache file maps a
problem key (shape, precision, stepper, flow kind) to the per-slot (radix, width,
3-waves/SIMD, input-parallel, workgroup-lines) choice; applying it needs no timing.
Entries written before the workgroup-lines flag existed (five fields) read it as off.
"""
from __future__ import annotations

import json
import os


def _base(name: str) -> str:
    return name.split(" [")[0]


def load(path):
    if path and os.path.exists(path):
        with open(path) as f:
            return json.load(f)
    return {}


def store(path, data):
    tmp = path + ".tmp"
    with open(tmp, "w") as f:
        json.dump(data, f, indent=1, sort_keys=True)
        f.write("\n")
    os.replace(tmp, path)


def apply_or_tune(obj, key, path, tune=None):
    """Apply the cached variants of ``key`` to ``obj`` (a Problem or an Ensemble: slots(),
    set_variant(i, R, W, occ3, par, wg), get_variant(i), whole_run(i)); if there is no matching
    entry, run the autotuner (``tune``, default the object's own) and store its choice.  Slots that
    the whole-run kernel of a 1D problem stands in for keep it: the autotuner has no choice to make
    there, and selecting a stage kernel would switch it off.  Returns "cache" or "tuned"."""
    data = load(path)
    names = [_base(n) for n in obj.slots()]
    entry = data.get(key)
    whole_run = getattr(obj, "whole_run", lambda i: False)
    if entry and [e[0] for e in entry] == names:
        for i, e in enumerate(entry):
            R, W, occ3, par = e[1:5]
            wg = e[5] if len(e) > 5 else False
            if int(R) == 0 or whole_run(i):
                continue   # a fixed-shape kernel (whole-member step, 1D run): nothing to select
            obj.set_variant(i, int(R), int(W), occ3=bool(occ3), par=bool(par), wg=bool(wg))
        return "cache"
    (tune or obj.autotune)()
    data[key] = [[names[i], *obj.get_variant(i)] for i in range(len(names))]
    store(path, data)
    return "tuned"
