// The compiled whole-run kernels of 1D problems (ptf_line.hpp).  Compiled once per (precision,
// stepper family) with -DPTF_T=<double|float> -DPTF_TNAME=<f64|f32> -DPTF_ETD=<0|1>; exports
//   const void* ptf_line_<TNAME>_<ETD>(int nx, int* threads)
#include "ptf_line.hpp"

using namespace ptf;

namespace {
template <int NX>
const void* entry(int* threads) {
  constexpr int M = NX / 2, R = line_run_e(M);
  if constexpr (R > 0) {
    *threads = line_run_threads(M, R);
    return reinterpret_cast<const void*>(&line_run_kernel<PTF_T, NX, R, PTF_ETD != 0>);
  } else {
    return nullptr;
  }
}
template <int... NX>
const void* pick(int nx, int* threads) {
  const void* p = nullptr;
  ((nx == NX ? (p = entry<NX>(threads), true) : false) || ...);
  return p;
}
}  // namespace

#define PTF_JOIN3_(a, b, c) a##_##b##_##c
#define PTF_JOIN3(a, b, c) PTF_JOIN3_(a, b, c)

extern "C" const void* PTF_JOIN3(ptf_line, PTF_TNAME, PTF_ETD)(int nx, int* threads) {
  return pick<16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 24, 36, 40, 48, 50, 54, 72, 80, 96, 100, 108, 144,
              160, 192, 200, 216, 250, 288, 320, 384, 400, 432, 500, 576, 640, 768, 800, 864, 1000, 1152, 1280,
              1536, 1600, 1728, 2000, 2304, 2560, 3072, 3200, 3456, 4000>(nx, threads);
}
