// Running single-bin DFTs of the electric field (FieldMonitor.update,
// field_monitors.py:59-102): acc[c][f][n] += E_c[n] * phase[f] for every cell
// n and component c, with phase[f] = exp(-2 pi i f t) supplied by the caller,
// as numpy evaluates it: complex64 (P = float) when t is an FP32 scalar,
// complex128 (P = double) otherwise. The product E * phase is numpy's complex
// multiply of (E + 0i)(re + i im) = (E re - 0 im, E im + 0 re) in the promoted
// type (FP32 for FP32 E with a complex64 phase, FP64 otherwise), then added to
// the complex128 accumulator.
#pragma once
#include "fit_common.h"

#include <type_traits>

namespace wf {

template <typename S, typename P>
__global__ void __launch_bounds__(256)
k_monitor(const S *__restrict__ E, int64_t N, const P *__restrict__ phase, int nf,
          double *__restrict__ acc) {
  using R = typename std::conditional<sizeof(S) == 4 && sizeof(P) == 4, float, double>::type;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * N) return;
  const int c = (int)(t / N);
  const int64_t n = t - (int64_t)c * N;
  const R e = (R)E[t];
  for (int f = 0; f < nf; ++f) {
    double *a = acc + 2 * (((int64_t)c * nf + f) * N + n);
    const R re = (R)phase[2 * f], im = (R)phase[2 * f + 1];
    const R pr = e * re - R(0) * im;
    const R pi = e * im + R(0) * re;
    a[0] = a[0] + (double)pr;
    a[1] = a[1] + (double)pi;
  }
}

// The same for the E of nk <= MON_STEPS steps in turn: each accumulator crosses
// memory once for all of them (16 bytes read and written per component,
// frequency and cell, against 4 or 8 for a step's E), the sum in the same order.
// Bound by those bytes: 96x96x160 FP32, 2 frequencies, 59 us for 8 steps at 7.2 TB/s
// (the accumulators stay in the last cache), 46 us for one step before.
constexpr int MON_STEPS = 8;
template <typename S>
struct MonFields {
  const S *e[MON_STEPS];
};

template <typename S, typename P>
__global__ void __launch_bounds__(256)
k_monitor_steps(MonFields<S> E, int nk, int64_t N, const P *__restrict__ phase, int nf,
                double *__restrict__ acc) {
  using R = typename std::conditional<sizeof(S) == 4 && sizeof(P) == 4, float, double>::type;
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int c = blockIdx.y;
  R e[MON_STEPS];
#pragma unroll
  for (int k = 0; k < MON_STEPS; ++k) e[k] = k < nk ? (R)E.e[k][c * N + n] : R(0);
  for (int f = 0; f < nf; ++f) {
    double2 *a = reinterpret_cast<double2 *>(acc) + (((int64_t)c * nf + f) * N + n);
    double2 s = *a;
#pragma unroll
    for (int k = 0; k < MON_STEPS; ++k) {
      if (k >= nk) break;
      const R re = (R)phase[2 * ((int64_t)k * nf + f)], im = (R)phase[2 * ((int64_t)k * nf + f) + 1];
      const R pr = e[k] * re - R(0) * im;
      const R pi = e[k] * im + R(0) * re;
      s.x = s.x + (double)pr;
      s.y = s.y + (double)pi;
    }
    *a = s;
  }
}

}  // namespace wf
