"""bench.py's byte model of the fused stage kernels against the fields that the device code loads
and stores (csrc/ptf_device.hpp: rk4_load, rk4_finish_L, etd_load, etd_finish), counted here from
what each stage needs: FP64 RK4 13 state fields a step, the mixed form 15; ETDRK4 12 (mixed 18) and
10 coefficient arrays.  Each fused stage kernel also moves its input and two outputs (3 fields).
"""
import pytest

import bench

# (loads, stores) of state fields by stage; the mixed form's low parts in the second list
RK4 = [("sol", "acc"), ("sol acc", "x3 acc"), ("x3 sol acc", "acc"), ("sol acc", "sol")]
RK4_LO = [("", ""), ("", ""), ("", ""), ("lo", "lo")]
ETD = [("sol", "sol1 n1"), ("sol", "n2"), ("sol sol1 n1 n2", "acc"), ("acc", "sol")]
ETD_LO = [("lo", ""), ("lo", ""), ("lo", "acclo"), ("acclo", "lo")]
COEFFS = ["E2 zeta", "E2 zeta", "E2 zeta E alpha beta", "gamma"]


def _fields(*pairs):
    return sum(len(a.split()) + len(b.split()) for a, b in pairs)


@pytest.mark.parametrize("cb", [16, 8])
@pytest.mark.parametrize("stepper,hi,lo", [("RK4", RK4, RK4_LO), ("FilteredRK4", RK4, RK4_LO),
                                           ("ETDRK4", ETD, ETD_LO)])
def test_each_stage(cb, stepper, hi, lo):
    nS, nR = 1000, 2000
    total = 0
    for s in range(4):
        want = (_fields(hi[s]) + (_fields(lo[s]) if cb == 8 else 0) + 3) * nS * cb
        if stepper == "ETDRK4":
            want += len(COEFFS[s].split()) * nS * 8
        got = bench.moved_bytes(f"stage{s + 1}_y_forward_stage_inverse [x]", nS, nR, cb, cb // 2, s, stepper)
        assert got == want, (stepper, s)
        total += got
    S = nS * cb
    assert total == {("RK4", 16): 25 * S, ("RK4", 8): 27 * S, ("FilteredRK4", 16): 25 * S, ("FilteredRK4", 8): 27 * S,
                     ("ETDRK4", 16): 24 * S + 10 * nS * 8, ("ETDRK4", 8): 30 * S + 10 * nS * 8}[stepper, cb]


def test_other_launches_as_the_pass_model():
    for name in ("stage1_x_advect [row_advect3 N=256 R=4 W=8 f64]", "stage2_y_forward [x]", "flow_y_synthesis [x]",
                 "stage3_y_forward_stage [x]"):
        assert bench.moved_bytes(name, 1000, 2000, 16, 8, 2) == bench.kernel_bytes(name, 1000, 2000, 16, 8, 2)


def test_a_measurement_belongs_to_the_code(tmp_path, monkeypatch):
    """The hash follows the code of the kernels, not their comments."""
    a = bench.kernel_source_hash()
    csrc = tmp_path / "passivetracerflows.jl_amd" / "csrc"
    csrc.mkdir(parents=True)
    import os
    real = os.path.join(bench.ROOT, "passivetracerflows.jl_amd", "csrc")
    text = {}
    for f in ("ptf_device.hpp", "ptf_kernels.hpp"):
        with open(os.path.join(real, f)) as src:
            text[f] = src.read()
        (csrc / f).write_text("// another comment\n" + text[f])
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.kernel_source_hash() == a
    (csrc / "ptf_device.hpp").write_text(text["ptf_device.hpp"] + "\nconstexpr int more = 1;\n")
    assert bench.kernel_source_hash() != a
