// Weight codes of the two-step kernel: per cell a row of a table that holds the
// products of metric, material and dt which the kernel otherwise forms at every
// cell and step.
//
// On uniform spacing (FP32: the spacings of np.linspace, equal after rounding)
// the metric takes one value for the inner cells of an axis and others at its
// first and last cell, where masks and boundary copies act: 27 classes. A cell's
// weights then follow from its class and its material code; the distinct rows
// that occur are few (4 to 60), and 255 fit a byte.
#pragma once
#include "fit_common.h"

namespace wf {

// values of a row: 12 weights, ieps, sigma, 2 unused (80 bytes: 16-byte reads,
// and rows spread over the LDS banks)
constexpr int WC_ROW = 20;

__device__ __forceinline__ int wc_class(int i, int n) { return i == 0 ? 0 : i == n - 1 ? 2 : 1; }
// a cell of class c; an axis of two cells has no inner one
__device__ __forceinline__ int wc_cell(int c, int n) { return c == 0 ? 0 : c == 2 ? n - 1 : 1; }

template <typename S>
struct Metric2d {
  const S *iAx, *iAy, *iAz, *itAx, *itAy, *itAz;
  __device__ explicit Metric2d(const GridDev &g, const S *t) {
    const int64_t yz = (int64_t)g.Ny * g.Nz, xz = (int64_t)g.Nx * g.Nz, xy = (int64_t)g.Nx * g.Ny;
    iAx = t; iAy = t + yz; iAz = t + yz + xz;
    itAx = t + yz + xz + xy; itAy = itAx + yz; itAz = itAy + xz;
  }
};

// rows[key] of every class and material, with the roundings of h_row and e_sum
template <typename S>
__global__ void __launch_bounds__(256)
k_weight_rows(GridDev g, MetricDev<S> m, const S *__restrict__ mat, int nmat,
              const S *__restrict__ metric2d, S dt, S *__restrict__ rows, int *__restrict__ used) {
  const int key = blockIdx.x * 256 + threadIdx.x;
  if (key == 0) used[27 * nmat] = 0;
  if (key >= 27 * nmat) return;
  used[key] = 0;
  const int cls = key / nmat, cz = cls / 9, cy = cls / 3 % 3, cx = cls % 3;
  const int i = wc_cell(cx, g.Nx), j = wc_cell(cy, g.Ny), k = wc_cell(cz, g.Nz);
  const S *t = mat + 9 * (key - cls * nmat);
  const Metric2d<S> d(g, metric2d);
  const int64_t jk = j + (int64_t)g.Ny * k, ik = i + (int64_t)g.Nx * k, ij = i + (int64_t)g.Nx * j;
  const S a0 = (S)(d.iAx[jk] * t[0]), a1 = (S)(d.iAy[ik] * t[1]), a2 = (S)(d.iAz[ij] * t[2]);
  const S b0 = (S)(t[3] * d.itAx[jk]), b1 = (S)(t[4] * d.itAy[ik]), b2 = (S)(t[5] * d.itAz[ij]);
  S *o = rows + (int64_t)key * WC_ROW;
  o[0] = dt * (S)(a0 * m.Ly[j]); o[1] = dt * (S)(a0 * m.Lz[k]);
  o[2] = dt * (S)(a1 * m.Lx[i]); o[3] = dt * (S)(a1 * m.Lz[k]);
  o[4] = dt * (S)(a2 * m.Lx[i]); o[5] = dt * (S)(a2 * m.Ly[j]);
  o[6] = b0 * m.tLy[j]; o[7] = b0 * m.tLz[k];
  o[8] = b1 * m.tLx[i]; o[9] = b1 * m.tLz[k];
  o[10] = b2 * m.tLx[i]; o[11] = b2 * m.tLy[j];
  for (int c = 0; c < 6; ++c) o[12 + c] = t[3 + c];
  o[18] = o[19] = S(0);
}

// used[key] = 1 where a cell has it, and used[27 nmat] = 1 if a metric value
// differs from that of its class (`used` zeroed by k_weight_rows before)
template <typename S>
__global__ void __launch_bounds__(256)
k_weight_scan(GridDev g, MetricDev<S> m, const uint8_t *__restrict__ code, int nmat,
              const S *__restrict__ metric2d, int *__restrict__ used) {
  extern __shared__ int s_used[];  // [27 nmat + 1]
  const int nk = 27 * nmat;
  for (int t = threadIdx.x; t <= nk; t += 256) s_used[t] = 0;
  __syncthreads();
  const Metric2d<S> d(g, metric2d);
  const int lane = threadIdx.x & 63;
  // one row of cells per wave
  const int64_t nrows = (int64_t)g.Ny * g.Nz;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < nrows;
       row += (int64_t)gridDim.x * 4) {
    const int k = (int)(row / g.Ny), j = (int)(row - (int64_t)k * g.Ny);
    const int cy = wc_class(j, g.Ny), cz = wc_class(k, g.Nz);
    const int J = wc_cell(cy, g.Ny), K = wc_cell(cz, g.Nz);
    bool bad = false;
    if (lane == 0) {
      const int64_t a = j + (int64_t)g.Ny * k, b = J + (int64_t)g.Ny * K;
      bad = d.iAx[a] != d.iAx[b] || d.itAx[a] != d.itAx[b];
      if (k == 0) bad = bad || m.Ly[j] != m.Ly[J] || m.tLy[j] != m.tLy[J];
      if (j == 0) bad = bad || m.Lz[k] != m.Lz[K] || m.tLz[k] != m.tLz[K];
    }
    for (int i = lane; i < g.Nx; i += 64) {
      const int cx = wc_class(i, g.Nx), I = wc_cell(cx, g.Nx);
      const int cd = code[row * g.Nx + i];
      if (cd < nmat) s_used[(cx + 3 * (cy + 3 * cz)) * nmat + cd] = 1;
      else bad = true;
      if (j == 0) {
        const int64_t a = i + (int64_t)g.Nx * k, b = I + (int64_t)g.Nx * K;
        bad = bad || d.iAy[a] != d.iAy[b] || d.itAy[a] != d.itAy[b];
      }
      if (k == 0) {
        const int64_t a = i + (int64_t)g.Nx * j, b = I + (int64_t)g.Nx * J;
        bad = bad || d.iAz[a] != d.iAz[b] || d.itAz[a] != d.itAz[b];
      }
      if (row == 0) bad = bad || m.Lx[i] != m.Lx[I] || m.tLx[i] != m.tLx[I];
    }
    if (bad) s_used[nk] = 1;
  }
  __syncthreads();
  for (int t = threadIdx.x; t <= nk; t += 256)
    if (s_used[t]) used[t] = 1;
}

// wcode[n] = map[class * nmat + code[n]], one row of cells per wave
static __global__ void __launch_bounds__(256)
k_weight_codes(GridDev g, const uint8_t *__restrict__ code, int nmat,
               const uint8_t *__restrict__ map, uint8_t *__restrict__ wcode) {
  const int64_t nrows = (int64_t)g.Ny * g.Nz;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < nrows;
       row += (int64_t)gridDim.x * 4) {
    const int k = (int)(row / g.Ny), j = (int)(row - (int64_t)k * g.Ny);
    const uint8_t *mp = map + 3 * (wc_class(j, g.Ny) + 3 * wc_class(k, g.Nz)) * nmat;
    for (int i = threadIdx.x & 63; i < g.Nx; i += 64) {
      const int64_t n = row * g.Nx + i;
      wcode[n] = mp[wc_class(i, g.Nx) * nmat + code[n]];
    }
  }
}

}  // namespace wf
