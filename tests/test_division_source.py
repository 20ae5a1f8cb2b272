"""div_by of csrc/ptf_device.hpp itself, compiled for the host: its source text with the fused
multiply-add of the C library and, for the last instruction, what that instruction does (v_div_fixup:
quotient, denominator, numerator -> the quotient's magnitude with the sign of a division, and the
division's results for NaN, infinities and zeros).

Against true division: equal wherever the quotient is a normal number, for zeros of both signs,
infinities and NaN; within one unit of the last place where it is subnormal (ties there go with the
rounding of 1/D, which is as close to the quotient as the even neighbour).
"""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(os.path.dirname(HERE), "passivetracerflows.jl_amd", "csrc", "ptf_device.hpp")

PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#define __device__
#define __forceinline__ inline
template <typename T>
static T fixup(T q, T d, T n) {
  const T sign = std::signbit(d) != std::signbit(n) ? (T)-1 : (T)1;
  if (std::isnan(n) || std::isnan(d) || (n == 0 && d == 0) || (std::isinf(n) && std::isinf(d))) return (T)NAN;
  if (d == 0 || std::isinf(n)) return sign * (T)INFINITY;
  if (std::isinf(d) || n == 0) return sign * (T)0;
  return sign * std::fabs(q);
}
static double __builtin_amdgcn_div_fixup(double q, double d, double n) { return fixup(q, d, n); }
static float __builtin_amdgcn_div_fixupf(float q, float d, float n) { return fixup(q, d, n); }
%s
template <typename T, int D>
static void run(const char* in, const char* out) {
  FILE* f = std::fopen(in, "rb");
  FILE* o = std::fopen(out, "wb");
  T x;
  while (std::fread(&x, sizeof(T), 1, f) == 1) {
    const T y = div_by<D>(x);
    std::fwrite(&y, sizeof(T), 1, o);
  }
  std::fclose(f);
  std::fclose(o);
}
int main(int, char** v) {
  const bool dbl = std::strcmp(v[1], "float64") == 0;
  const int D = std::atoi(v[2]);
  if (dbl && D == 3) run<double, 3>(v[3], v[4]);
  else if (dbl && D == 6) run<double, 6>(v[3], v[4]);
  else if (D == 3) run<float, 3>(v[3], v[4]);
  else if (D == 6) run<float, 6>(v[3], v[4]);
  else return 1;
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    with open(SOURCE) as f:
        text = f.read()
    fns = re.findall(r"template <int D>\n__device__ __forceinline__ (?:double|float) div_by\(.*?\n}\n", text, re.S)
    assert len(fns) == 2
    d = tmp_path_factory.mktemp("div")
    src, exe = str(d / "div.cpp"), str(d / "div")
    with open(src, "w") as f:
        f.write(PROGRAM % "\n".join(fns))
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-ffp-contract=off", src, "-o", exe])
    return exe


def _run(program, tmp_path, T, D, x):
    a, b = str(tmp_path / "in"), str(tmp_path / "out")
    x.tofile(a)
    subprocess.check_call([program, np.dtype(T).name, str(D), a, b])
    return np.fromfile(b, T)


@pytest.mark.parametrize("D", [3, 6])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_is_division(program, tmp_path, T, D):
    rng = np.random.default_rng(D)
    info = np.finfo(T)
    lo, hi = np.log2(float(info.tiny)) + 4, np.log2(float(info.max)) - 1
    x = np.concatenate([
        rng.choice([-1.0, 1.0], 200000) * rng.uniform(1, 2, 200000) * 2.0 ** np.floor(rng.uniform(lo, hi, 200000)),
        np.arange(-3000, 3000), [info.max, -info.max, 0.0, -0.0, np.inf, -np.inf, np.nan]]).astype(T)
    with np.errstate(all="ignore"):
        x = np.concatenate([x, np.nextafter(x, T(0)), np.nextafter(x, T(np.inf))])
        want = x / T(D)
    got = _run(program, tmp_path, T, D, x)
    normal = ~((want != 0) & (np.abs(want) < info.tiny))
    bits = np.int64 if T == np.float64 else np.int32
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    ok = normal & ~nan
    assert np.array_equal(got[ok].view(bits), want[ok].view(bits))      # signs of zeros included


@pytest.mark.parametrize("D", [3, 6])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_subnormal_quotients(program, tmp_path, T, D):
    rng = np.random.default_rng(10 + D)
    unit = np.nextafter(T(0), T(1))
    k = np.concatenate([np.arange(1, 5000), rng.integers(1, 2 ** 21, 50000)])
    x = (k * np.float64(unit)).astype(T) if T == np.float32 else k.astype(T) * unit
    got = _run(program, tmp_path, T, D, x)
    units = np.round(got / unit).astype(np.int64)
    assert np.abs(2 * D * units - 2 * k).max() <= D      # within half a unit of k / D
