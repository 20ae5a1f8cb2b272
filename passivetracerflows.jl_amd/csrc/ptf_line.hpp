// Whole-run kernel for 1D problems.
//
// A 1D problem is one line: nothing but its own few KB is touched in a step, so a step is bound
// by the latency of the stage kernels' memory round trips and launches (128 points FP64:
// 23.6 us a step, four launches of one 64-lane block).  Here one workgroup advances a line by
// `nsteps` whole steps in one launch: the state, the stage inputs, the operators and the flow
// stay in registers, each thread holding elements j + q P (q < R) of the half-length line and
// lane 0 the Nyquist element as well; LDS holds only the exchanges and the twiddle table.
// Transforms of up to 64 lanes (lines of 512 points at radix 4) order their exchanges within one
// wavefront, without workgroup barriers.  Radix 4 (6, 10, 3, 5 for the lengths that are no
// powers of two): few elements per lane, since the time of a step is the instructions that one
// wavefront issues one after the other (1024 points FP32 ETDRK4 in one wavefront of radix 8:
// 17.5 us a step against 11).  Half of them are outside the transforms: the operators, the real
// pre- and post-processing.  Where the transforms take up to 128 lanes those go to up to four
// wavefronts, an element or two a lane, for two more exchanges a stage: 6.5 -> 4.6 us a step at
// 128 points FP64 (4.3 with div_by), 25 -> 12.6 (12.2) at 1000, 12 -> 10.8 at 1024 FP32 ETDRK4.
//
// Per stage (calcN! S:695-710 for a steady 1D flow, then the stage update):
//   N = R2C(-u C2R(i kr x))
#pragma once
#include "ptf_kernels.hpp"

namespace ptf {

template <typename T>
struct LineArgs {
  StageArgs<T> st;         // state, operators, stepper
  const T* flow;           // physical u, members back to back
  const cpx<T>* tw;        // exp(-2 pi i m / nx), m < nx
  long long pmstride;      // physical values per member
  double kscale_x;
  double scale;            // C2R scale 1 / nx
  int nsteps;
};

// One skew entry every 8 elements: a pass writes at the strides of its radix and reads at
// stride 1, and both spread over the banks (as the column stage kernels' layout).
struct LayLine {
  __device__ __forceinline__ int idx(int, int i) const { return i + (i >> 3); }
  __device__ __forceinline__ int idx_split(int, int i0, int off) const { return i0 + (i0 >> 3) + off + (off >> 3); }
};

// Elements per thread of a half-length line of M points; 0 where none is compiled.
constexpr int line_run_e(int M) {
  if (M < 8) return 0;
  if ((M & (M - 1)) == 0) return M <= 2048 ? 4 : 0;
  const int e3 = M % 2 == 0 ? 6 : 3, e5 = M % 2 == 0 ? 10 : 5;
  if (M % 3 == 0 && M % 5 != 0 && fft_ok(M, e3) && M / e3 <= 512) return e3;
  if (M % 5 == 0 && M % 3 != 0 && fft_ok(M, e5) && M / e5 <= 512) return e5;
  return 0;
}

// Lines whose transforms leave SIMDs of the CU idle (up to 64 threads, or 128) spread over up to
// four wavefronts outside the transforms: see the kernel's header.
constexpr bool line_run_spread(int M, int R) { return M / R <= 64 || M / R == 128; }
constexpr int line_run_threads(int M, int R) {
  return !line_run_spread(M, R) ? M / R : (M >= 256 ? 256 : (M + 63) / 64 * 64);
}

template <typename T, int NX, int R, bool ETD>
__global__ __attribute__((amdgpu_flat_work_group_size(1, line_run_threads(NX / 2, R)),
                          amdgpu_waves_per_eu(1, (line_run_threads(NX / 2, R) + 255) / 256)))
void line_run_kernel(LineArgs<T> a) {
  constexpr int M = NX / 2;
  constexpr int P = M / R;
  constexpr bool kSpread = line_run_spread(M, R);
  constexpr int TP = line_run_threads(M, R);   // threads of the block
  constexpr int EP = kSpread ? (M + TP - 1) / TP : R;   // elements of a thread outside the transforms
  constexpr bool kWave = TP <= 64;       // the exchanges of the block
  constexpr bool kWaveFft = P <= 64;     // ... and of a transform
  constexpr bool kMixed = sizeof(T) == 4;
  const LayLine lay{};
  __shared__ cpx<T> lds[M + 1 + (M >> 3)];
  __shared__ cpx<T> twl[NX];
  const int j = threadIdx.x;
  const int member = blockIdx.x;
  for (int i = j; i < NX; i += TP) twl[i] = a.tw[i];
  __syncthreads();
  const long long ubase = (long long)member * a.st.mstride;
  const OpParams opm = a.st.op[member];
  const T dt = (T)a.st.dt, h2 = (T)(a.st.dt / 2);
  const T sc = (T)a.scale;
  const bool nyq = j == 0;   // lane 0 also holds element M, at index EP
  // Wavenumber index of register e, and whether this lane holds it (lanes without an element
  // compute on zeros, with the indices of element M - 1 or M).
  auto kof = [&](int e) { return e == EP ? M : (kSpread && j + e * TP >= M ? M - 1 : j + e * TP); };
  auto holds = [&](int e) { return e == EP ? nyq : (!kSpread || j + e * TP < M); };
  const bool tf = !kSpread || j < P;   // lanes that transform
  const int wv = __builtin_amdgcn_readfirstlane(j / 64);

  cpx<T> s[EP + 1], lo[kMixed ? EP + 1 : 1], u[R], w[kSpread ? EP : 1];
  T L[ETD ? 1 : EP + 1];
  double E[ETD ? EP + 1 : 1], E2[ETD ? EP + 1 : 1], ze[ETD ? EP + 1 : 1], al[ETD ? EP + 1 : 1], be[ETD ? EP + 1 : 1],
      ga[ETD ? EP + 1 : 1];
  double fil[EP + 1];
  const cpx<T>* up = reinterpret_cast<const cpx<T>*>(a.flow + (long long)member * a.pmstride);
#pragma unroll
  for (int q = 0; q < R; ++q) u[q] = up[tf ? j + q * P : 0];
  if constexpr (kSpread) {
#pragma unroll
    for (int e = 0; e < EP; ++e) w[e] = twl[kof(e)];
  }
#pragma unroll
  for (int e = 0; e <= EP; ++e) {
    const int k = kof(e);
    const bool have = holds(e);
    s[e] = {(T)0, (T)0};
    if (have) s[e] = a.st.sol[ubase + k];
    if constexpr (kMixed) {
      lo[e] = {(T)0, (T)0};
      if (have) lo[e] = a.st.sol_lo[ubase + k];
    }
    if constexpr (ETD) {
      E[e] = a.st.E[ubase + k];
      E2[e] = a.st.E2[ubase + k];
      ze[e] = a.st.zeta[ubase + k];
      al[e] = a.st.alpha[ubase + k];
      be[e] = a.st.beta[ubase + k];
      ga[e] = a.st.gam[ubase + k];
    } else {
      L[e] = (T)linear_op(a.st.g, opm, a.st.nkappah, k, 0, 0);
    }
    fil[e] = a.st.filtered ? filter_value(a.st.g, a.st.f_order, a.st.f_innerK, a.st.f_decay, k, 0, 0) : 1.0;
  }

  // N = R2C(-u C2R(i kr x)) of the stage input x
  auto calcN = [&](const cpx<T>(&x)[EP + 1], cpx<T>(&N)[EP + 1]) {
    if constexpr (kSpread) {
      cpx<T> z[EP], f[R];
      lds_sync(kWave);
#pragma unroll
      for (int e = 0; e < EP; ++e) {
        z[e] = times_ik(x[e], (T)(kof(e) * a.kscale_x));
        if (holds(e)) lds[lay.idx(0, kof(e))] = z[e];
      }
      if (nyq) lds[lay.idx(0, M)] = times_ik(x[EP], (T)(M * a.kscale_x));
      lds_sync(kWave);
#pragma unroll
      for (int e = 0; e < EP; ++e) z[e] = c2r_pre(z[e], lds[lay.idx(0, M - kof(e))], w[e], sc, kof(e) == 0);
      lds_sync(kWave);
#pragma unroll
      for (int e = 0; e < EP; ++e)
        if (holds(e)) lds[lay.idx(0, kof(e))] = z[e];
      lds_sync(kWave);
      auto transforms = [&]() {
#pragma unroll
        for (int q = 0; q < R; ++q) f[q] = lds[lay.idx(0, j + q * P)];
        line_fft<T, M, R, +1, LayLine>(f, lds, lay, 0, j, twl, 2, kWaveFft);
#pragma unroll
        for (int q = 0; q < R; ++q) f[q] = {-u[q].re * f[q].re, -u[q].im * f[q].im};
        line_fft<T, M, R, -1, LayLine>(f, lds, lay, 0, j, twl, 2, kWaveFft);
        lds_sync(kWaveFft);
#pragma unroll
        for (int q = 0; q < R; ++q) lds[lay.idx(0, j + q * P)] = f[q];
      };
      if constexpr (kWaveFft) {
        if (tf) transforms();
      } else {
        // whole wavefronts transform; the others match their barriers
        static_assert(P % 64 == 0, "whole wavefronts");
        if (wv < P / 64) {
          transforms();
        } else {
          for (int i = 0; i < 2 * fft_barriers(M, R) + 1; ++i) __syncthreads();
        }
      }
      lds_sync(kWave);
#pragma unroll
      for (int e = 0; e < EP; ++e) {
        const int k = kof(e);
        const cpx<T> Z = lds[lay.idx(0, k)], Zm = lds[lay.idx(0, k == 0 ? 0 : M - k)];
        N[e] = k == 0 ? cpx<T>{Z.re + Z.im, (T)0} : r2c_post(Z, Zm, w[e]);
        if (e == 0) N[EP] = nyq ? cpx<T>{Z.re - Z.im, (T)0} : cpx<T>{(T)0, (T)0};
      }
      return;
    } else {
    cpx<T> z[R];
    lds_sync(kWave);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int k = j + q * P;
      z[q] = times_ik(x[q], (T)(k * a.kscale_x));
      lds[lay.idx(0, k)] = z[q];
    }
    if (nyq) lds[lay.idx(0, M)] = times_ik(x[EP], (T)(M * a.kscale_x));
    lds_sync(kWave);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int k = j + q * P;
      z[q] = c2r_pre(z[q], lds[lay.idx(0, M - k)], twl[k], sc, k == 0);
    }
    line_fft<T, M, R, +1, LayLine>(z, lds, lay, 0, j, twl, 2, kWave);
#pragma unroll
    for (int q = 0; q < R; ++q) z[q] = {-u[q].re * z[q].re, -u[q].im * z[q].im};
    line_fft<T, M, R, -1, LayLine>(z, lds, lay, 0, j, twl, 2, kWave);
    lds_sync(kWave);
#pragma unroll
    for (int q = 0; q < R; ++q) lds[lay.idx(0, j + q * P)] = z[q];
    lds_sync(kWave);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int k = j + q * P;
      // lane 0's partner of k = 0 is not used
      const cpx<T> Zm = lds[lay.idx(0, k == 0 ? 0 : M - k)];
      N[q] = k == 0 ? cpx<T>{z[q].re + z[q].im, (T)0} : r2c_post(z[q], Zm, twl[k]);
    }
    N[EP] = nyq ? cpx<T>{z[0].re - z[0].im, (T)0} : cpx<T>{(T)0, (T)0};
    }
  };

#pragma unroll 1
  for (int step = 0; step < a.nsteps; ++step) {
    cpx<T> x[EP + 1], N[EP + 1];
#pragma unroll
    for (int e = 0; e <= EP; ++e) x[e] = s[e];
    if constexpr (!ETD) {
      // as rk4_load / rk4_finish, the operands in registers: sp is the FP64 form's sol after
      // the third stage; x_4 stays at hand, so its linear part joins in the fourth
      cpx<T> ac[EP + 1], sp[kMixed ? 1 : EP + 1];
#pragma unroll 1
      for (int stage = 0; stage < 4; ++stage) {
        calcN(x, N);
        switch (stage) {
          case 0:
#pragma unroll
            for (int e = 0; e <= EP; ++e) {
              const cpx<T> rhs = {N[e].re + L[e] * x[e].re, N[e].im + L[e] * x[e].im};
              ac[e] = rhs;
              x[e] = {s[e].re + h2 * rhs.re, s[e].im + h2 * rhs.im};
            }
            break;
          case 1:
#pragma unroll
            for (int e = 0; e <= EP; ++e) {
              const cpx<T> rhs = {N[e].re + L[e] * x[e].re, N[e].im + L[e] * x[e].im};
              ac[e] = {div_by<6>(ac[e].re) + div_by<3>(rhs.re), div_by<6>(ac[e].im) + div_by<3>(rhs.im)};
              x[e] = {s[e].re + h2 * rhs.re, s[e].im + h2 * rhs.im};
            }
            break;
          case 2:
#pragma unroll
            for (int e = 0; e <= EP; ++e) {
              const cpx<T> rhs = {N[e].re + L[e] * x[e].re, N[e].im + L[e] * x[e].im};
              x[e] = {s[e].re + dt * rhs.re, s[e].im + dt * rhs.im};
              ac[e] = {ac[e].re + div_by<3>(rhs.re), ac[e].im + div_by<3>(rhs.im)};
              if constexpr (!kMixed) sp[e] = {s[e].re + dt * ac[e].re, s[e].im + dt * ac[e].im};
            }
            break;
          default:
#pragma unroll
            for (int e = 0; e <= EP; ++e) {
              const cpx<T> rhs = {N[e].re + L[e] * x[e].re, N[e].im + L[e] * x[e].im};
              if constexpr (!kMixed) {
                s[e] = {sp[e].re + dt * div_by<6>(rhs.re), sp[e].im + dt * div_by<6>(rhs.im)};
                if (a.st.filtered) s[e] = {(T)fil[e] * s[e].re, (T)fil[e] * s[e].im};
              } else {
                const cpx<T> tot = {ac[e].re + div_by<6>(rhs.re), ac[e].im + div_by<6>(rhs.im)};
                T hr, lr, hi, li;
                comp_add(s[e].re, lo[e].re, dt * tot.re, hr, lr);
                comp_add(s[e].im, lo[e].im, dt * tot.im, hi, li);
                if (a.st.filtered) {
                  const double xr = ((double)hr + (double)lr) * fil[e], xi = ((double)hi + (double)li) * fil[e];
                  hr = (T)xr;
                  hi = (T)xi;
                  lr = (T)(xr - (double)hr);
                  li = (T)(xi - (double)hi);
                }
                s[e] = {hr, hi};
                lo[e] = {lr, li};
              }
            }
        }
      }
    } else {
      // as etd_load / etd_finish; pr, pi: the partial update between the last two stages
      cpx<T> n1[EP + 1], n2[EP + 1], s1[EP + 1];
      double pr[EP + 1], pi[EP + 1];
      auto state = [&](int e, double& re, double& im) {
        re = (double)s[e].re;
        im = (double)s[e].im;
        if constexpr (kMixed) {
          re += (double)lo[e].re;
          im += (double)lo[e].im;
        }
      };
#pragma unroll 1
      for (int stage = 0; stage < 4; ++stage) {
        calcN(x, N);
#pragma unroll
        for (int e = 0; e <= EP; ++e) {
          const double nre = (double)N[e].re, nim = (double)N[e].im;
          if (stage <= 1) {
            double sr, si;
            state(e, sr, si);
            x[e] = {(T)(E2[e] * sr + ze[e] * nre), (T)(E2[e] * si + ze[e] * nim)};
            if (stage == 0) {
              n1[e] = N[e];
              s1[e] = x[e];
            } else {
              n2[e] = N[e];
            }
          } else if (stage == 2) {
            double sr, si;
            state(e, sr, si);
            x[e] = {(T)(E2[e] * (double)s1[e].re + ze[e] * (2.0 * nre - (double)n1[e].re)),
                    (T)(E2[e] * (double)s1[e].im + ze[e] * (2.0 * nim - (double)n1[e].im))};
            const double b2 = 2.0 * be[e];
            pr[e] = E[e] * sr + al[e] * (double)n1[e].re + b2 * ((double)n2[e].re + nre);
            pi[e] = E[e] * si + al[e] * (double)n1[e].im + b2 * ((double)n2[e].im + nim);
          } else {
            const double sr = (pr[e] + ga[e] * nre) * fil[e], si = (pi[e] + ga[e] * nim) * fil[e];
            s[e] = {(T)sr, (T)si};
            if constexpr (kMixed) lo[e] = {(T)(sr - (double)s[e].re), (T)(si - (double)s[e].im)};
          }
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e <= EP; ++e) {
    if (holds(e)) {
      a.st.sol[ubase + kof(e)] = s[e];
      if constexpr (kMixed) a.st.sol_lo[ubase + kof(e)] = lo[e];
    }
  }
}

// The compiled kernel for nx points (null when there is none); threads = its workgroup size.
const void* line_kernel(bool dbl, bool etd, int nx, int* threads);

}  // namespace ptf
