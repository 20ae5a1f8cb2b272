// Setup, conversion and diagnostic kernels of libptf_hip (host runtime only).
#pragma once
#include "ptf_kernels.hpp"

namespace ptf {

// --------------------------------------------------------------------------
// setup, conversion and diagnostic kernels
// --------------------------------------------------------------------------

// ETDRK4 coefficients ([FF] getetdcoeffs(dt, L; ncirc=32, rcirc=1), getexpLs): FP64
__global__ void etd_coeff_kernel(const double* __restrict__ L, long long n, double dt, int ncirc,
                                 double rcirc, double* E, double* E2, double* zeta, double* alpha,
                                 double* beta, double* gam) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double zr = dt * L[i];
  double sz = 0, sa = 0, sb = 0, sg = 0;  // real parts of the contour sums
  for (int jj = 0; jj < ncirc; ++jj) {
    double sn, cs;
    sincospi(2.0 * (jj + 0.5) / ncirc, &sn, &cs);
    // z = zr + rcirc e^{i theta}
    const double xr = zr + rcirc * cs, xi = rcirc * sn;
    // e^z, e^{z/2}
    const double ea = exp(xr);
    double s1, c1;
    sincos(xi, &s1, &c1);
    const double ezr = ea * c1, ezi = ea * s1;
    const double eh = exp(xr / 2);
    double s2, c2;
    sincos(xi / 2, &s2, &c2);
    const double ehr = eh * c2, ehi = eh * s2;
    // 1/z, 1/z^3
    const double den = xr * xr + xi * xi;
    const double izr = xr / den, izi = -xi / den;
    const double z2r = xr * xr - xi * xi, z2i = 2 * xr * xi;
    const double iz2r = izr * izr - izi * izi, iz2i = 2 * izr * izi;
    const double iz3r = iz2r * izr - iz2i * izi, iz3i = iz2r * izi + iz2i * izr;
    // zeta: (e^{z/2} - 1)/z
    {
      const double nr = ehr - 1, ni = ehi;
      sz += nr * izr - ni * izi;
    }
    // alpha: (-4 - z + e^z (4 - 3z + z^2))/z^3
    {
      const double pr = 4 - 3 * xr + z2r, pi = -3 * xi + z2i;
      const double nr = -4 - xr + (ezr * pr - ezi * pi);
      const double ni = -xi + (ezr * pi + ezi * pr);
      sa += nr * iz3r - ni * iz3i;
    }
    // beta: (2 + z + e^z (-2 + z))/z^3
    {
      const double pr = -2 + xr, pi = xi;
      const double nr = 2 + xr + (ezr * pr - ezi * pi);
      const double ni = xi + (ezr * pi + ezi * pr);
      sb += nr * iz3r - ni * iz3i;
    }
    // Gamma: (-4 - 3z - z^2 + e^z (4 - z))/z^3
    {
      const double pr = 4 - xr, pi = -xi;
      const double nr = -4 - 3 * xr - z2r + (ezr * pr - ezi * pi);
      const double ni = -3 * xi - z2i + (ezr * pi + ezi * pr);
      sg += nr * iz3r - ni * iz3i;
    }
  }
  zeta[i] = dt * (sz / ncirc);
  alpha[i] = dt * (sa / ncirc);
  beta[i] = dt * (sb / ncirc);
  gam[i] = dt * (sg / ncirc);
  E[i] = exp(dt * L[i]);
  E2[i] = exp(dt * L[i] / 2);
}

template <typename TO, typename TI>
__global__ void convert_kernel(TO* __restrict__ out, const TI* __restrict__ in, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (TO)in[i];
}

template <typename T>
__global__ void copy_kernel(T* __restrict__ out, const T* __restrict__ in, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i];
}

// (sum, comp) += x with Neumaier compensation
__device__ __forceinline__ void neumaier_add(double& sum, double& comp, double x) {
  const double t = sum + x;
  comp += (fabs(sum) >= fabs(x)) ? (sum - t) + x : (x - t) + sum;
  sum = t;
}

// Compensated sum over the block's 256 threads of their (sum, comp) pairs, in thread 0.
__device__ __forceinline__ void block_sum_256(double& sum, double& comp) {
  __shared__ double ssum[256];
  __shared__ double scomp[256];
  const int t = threadIdx.x;
  ssum[t] = sum;
  scomp[t] = comp;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) {
      double a = ssum[t], c = scomp[t] + scomp[t + off];
      neumaier_add(a, c, ssum[t + off]);
      ssum[t] = a;
      scomp[t] = c;
    }
    __syncthreads();
  }
  sum = ssum[0];
  comp = scomp[0];
}

// Neumaier-compensated FP64 partial sums of w_k |sol_k|^2 (Hermitian weights
// 1 at kx = 0 and nx/2, 2 elsewhere), one (sum, compensation) pair per block of 256;
// the field may be in the brick layout (kx of element i is (i >> lb) mod nxh).
template <typename T>
__global__ void variance_partial_kernel(const cpx<T>* __restrict__ sol, const cpx<T>* __restrict__ sol_lo,
                                        long long n, int nxh, int lb, double* __restrict__ partial) {
  double sum = 0.0, comp = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int kx = (int)((i >> lb) % nxh);   // brick layout: 2^lb planes innermost
    const double w = (kx == 0 || kx == nxh - 1) ? 1.0 : 2.0;
    // the mixed form's compensated state is sol + sol_lo, summed in FP64
    const cpx<T> v = sol[i];
    double vr = (double)v.re, vi = (double)v.im;
    if (sol_lo) {
      vr += (double)sol_lo[i].re;
      vi += (double)sol_lo[i].im;
    }
    neumaier_add(sum, comp, w * (vr * vr + vi * vi));
  }
  block_sum_256(sum, comp);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = sum;
    partial[2 * blockIdx.x + 1] = comp;
  }
}

// Element (row r, entry k) of a field in the working layout: rows are the (y, z)
// lines of x (r = y + ny z); with the last axis in bricks of 2^lb planes the rows
// are regrouped so that 2^lb consecutive planes sit innermost.
__device__ __forceinline__ long long work_index(long long r, long long k, long long rowlen, int lb,
                                                int ndim, int ny) {
  if (lb == 0) return r * rowlen + k;
  const long long B = 1ll << lb, mask = B - 1;
  const long long mid = ndim == 3 ? ny : 1;
  const long long l = r / mid, m = r % mid;
  const long long b = ((l >> lb) * mid + m) * B + (l & mask);
  return ((b >> lb) * rowlen + k) * B + (b & mask);
}

// Public FP64 layout (rows x rowlen entries of w doubles, x fastest) -> working
// layout in T; with dst_lo the FP64 value is split into hi + lo (compensated state).
template <typename T>
__global__ void layout_in_kernel(const double* __restrict__ src, T* __restrict__ dst,
                                 T* __restrict__ dst_lo, long long rows, int rowlen, int w, int lb,
                                 int ndim, int ny) {
  const long long n = rows * rowlen * w;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int e = (int)(i % w);
    const long long q = i / w;
    const long long k = q % rowlen, r = q / rowlen;
    const long long d = work_index(r, k, rowlen, lb, ndim, ny) * w + e;
    const double x = src[i];
    const T hi = (T)x;
    dst[d] = hi;
    if (dst_lo) dst_lo[d] = (T)(x - (double)hi);
  }
}

// Values [first, last) of the public layout from the working layout (T, plus the low part
// when src_lo), value i at dst[i - first].  OT is the type that crosses to the host: T where T
// holds the whole value.  dst is pinned host memory: the stores go over the bus, contiguous.
template <typename T, typename OT>
__global__ void layout_out_kernel(const T* __restrict__ src, const T* __restrict__ src_lo,
                                  OT* __restrict__ dst, long long first, long long last, int rowlen,
                                  int w, int lb, int ndim, int ny) {
  for (long long i = first + (long long)blockIdx.x * blockDim.x + threadIdx.x; i < last;
       i += (long long)gridDim.x * blockDim.x) {
    const int e = (int)(i % w);
    const long long q = i / w;
    const long long k = q % rowlen, r = q / rowlen;
    const long long d = work_index(r, k, rowlen, lb, ndim, ny) * w + e;
    OT x = (OT)src[d];
    if (src_lo) x += (OT)src_lo[d];
    dst[i - first] = x;
  }
}

// Analytic separable flow at one time: out[c] at physical point (ix, iy, iz) is
// sum over the terms k of component c of ((amp[k] tx[k][ix]) ty[k][iy]) tz[k][iz]
// (amp already holds amp * T(omega t + phase)).  Values are stored in the
// library's physical layout: x-pairs, with the last axis in bricks of 2^lb rows.
//
// Bound by its stores: a flow that depends on time is written before every step.  A block
// writes 256 consecutive x-pairs of one brick row (group: 2^lb rows that share their middle
// index), so its indices come from one division a block and the stores of a wavefront are
// contiguous.
constexpr int kMaxFlowTerms = 16;
template <typename T>
struct AnalyticArgs {
  int nterms;
  int comp[kMaxFlowTerms];
  double amp[kMaxFlowTerms];
  const double* tx;   // [nterms][nx]
  const double* ty;   // [nterms][ny]
  const double* tz;   // [nterms][nz]
  T* out[3];
  int ndim, nx, ny, nz, lb;
  int parts;          // blocks' worth of pairs in a group
  unsigned tiles;     // groups * parts
};

template <typename T>
__global__ void analytic_flow_kernel(AnalyticArgs<T> a) {
  const unsigned mask = (1u << a.lb) - 1;
  const unsigned mid = a.ndim == 3 ? (unsigned)a.ny : 1u;
  const unsigned len = ((unsigned)a.nx / 2) << a.lb;   // pairs of a group
  for (unsigned tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    const unsigned group = tile / (unsigned)a.parts, part = tile % (unsigned)a.parts;
    const unsigned t = part * 256u + threadIdx.x;
    if (t >= len) continue;
    const unsigned last = ((group / mid) << a.lb) + (t & mask);   // index along the last axis
    const int ix = 2 * (int)(t >> a.lb);
    const int iy = a.ndim == 3 ? (int)(group % mid) : (int)last;
    cpx<double> v[3] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
    // four terms at a time, so that their table reads are in flight together
    for (int k0 = 0; k0 < a.nterms; k0 += 4) {
      cpx<double> x[4];
      double y[4], z[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = k0 + i < a.nterms ? k0 + i : a.nterms - 1;
        const double* tx = a.tx + (long long)k * a.nx + ix;
        x[i] = {tx[0], tx[1]};
        y[i] = a.ndim >= 2 ? a.ty[(long long)k * a.ny + iy] : 0.0;
        z[i] = a.ndim == 3 ? a.tz[(long long)k * a.nz + last] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (k0 + i >= a.nterms) break;
        const double amp = a.amp[k0 + i];
        x[i] = {amp * x[i].re, amp * x[i].im};
        if (a.ndim >= 2) x[i] = {x[i].re * y[i], x[i].im * y[i]};
        if (a.ndim == 3) x[i] = {x[i].re * z[i], x[i].im * z[i]};
        const int c = a.comp[k0 + i];
        if (c == 0) v[0] = v[0] + x[i];
        else if (c == 1) v[1] = v[1] + x[i];
        else v[2] = v[2] + x[i];
      }
    }
    const long long o = (long long)group * len + t;
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (c < a.ndim) reinterpret_cast<cpx<T>*>(a.out[c])[o] = {(T)v[c].re, (T)v[c].im};
  }
}

// dealias!: zero the spectral elements whose kr index lies in [rlo, nxh) or whose
// y (z) index lies in [ylo, yhi) ([zlo, zhi)); plain (unbricked) half-spectrum
// layout (nx/2+1, ny, nz, batch), x fastest.  A wavefront clears a row, so that the row's
// place is found once and kept elements are not visited.
template <typename T>
__global__ void dealias_kernel(cpx<T>* __restrict__ f, unsigned rows, int nxh, int ny, int nz,
                               int rlo, int ylo, int yhi, int zlo, int zhi) {
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  for (unsigned r = blockIdx.x * 4u + wave; r < rows; r += gridDim.x * 4u) {
    const int iy = (int)(r % (unsigned)ny);
    const int iz = (int)((r / (unsigned)ny) % (unsigned)nz);
    const bool all = (iy >= ylo && iy < yhi) || (iz >= zlo && iz < zhi);
    cpx<T>* row = f + (long long)r * nxh;
    for (int k = (all ? 0 : rlo) + lane; k < nxh; k += 64) row[k] = cpx<T>{(T)0, (T)0};
  }
}

// Mass and variance record from the partial sums of variance_partial_kernel:
// rec[0] = Re sol[0] (mass = sum of c; sol + sol_lo in the mixed form), rec[1] = variance.
// One block of 256 threads: each sums its share of the partials with compensation, then the
// block its threads'.  What bounds it is the chain of dependent FP64 adds: 100 steps of 2D
// 128^2 FP64 with 10 records took 6.04 ms with one thread adding the 2048 values in turn,
// four steps' worth a record, and take 4.40 ms this way.
template <typename T>
__global__ void diag_record_kernel(const cpx<T>* __restrict__ sol, const cpx<T>* __restrict__ sol_lo,
                                   const double* __restrict__ partial, int npartial, double npoints,
                                   double* __restrict__ rec) {
  double sum = 0.0, comp = 0.0;
  for (int i = threadIdx.x; i < npartial; i += 256) {
    neumaier_add(sum, comp, partial[2 * i]);
    comp += partial[2 * i + 1];
  }
  block_sum_256(sum, comp);
  if (threadIdx.x != 0) return;
  double s0re = (double)sol[0].re, s0im = (double)sol[0].im;
  if (sol_lo) {
    s0re += (double)sol_lo[0].re;
    s0im += (double)sol_lo[0].im;
  }
  const double dc = s0re * s0re + s0im * s0im;
  rec[0] = s0re;
  rec[1] = ((sum - dc) + comp) / (npoints * npoints);
}

}  // namespace ptf
