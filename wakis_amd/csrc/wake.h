// Wake potential and impedance kernels (FP64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wf {

// WakeSolver.calc_long_WP_3d (wakeSolver.py:485-537). For one s sample the
// captured lines are walked in order carrying the running value (WP is zeroed
// once, then WP += sum_k Ez*dz and WP /= q*1e12 per line), accumulating over k
// in increasing order: the exact operation sequence of the reference's loop.
//   forward (CM false, wakeSolver.py:520-533): row k of the line,
//     ts = (z[k] + s)/v - zref_v - t0 + ti, weight dz[k], zref_v = zmin/v;
//   counter-moving (CM true, wakeSolver.py:503-517): row nz-1-k,
//     ts = (z[nz-1-k] - s)/(-v) - zref_v - t0 + ti, weight (-dz[k]),
//     zref_v = zmax/(-v).
// it = trunc(ts/dt) is kept when it < nt; a negative it indexes from the end
// of the reference's Ezt, which has ncols columns of which the first nt hold
// samples (the others are zero). A term that is not kept is added as +0, which
// leaves the sum as it is.
//
// What bounds it: the chain of nlines * nz additions per s, and the gather (for
// one s every k reads another row of the capture). A workgroup takes WP_NS
// samples: its first wave only adds, the others form the products of the next
// WP_KC rows in LDS meanwhile, so the chain never waits for memory, and few
// samples per workgroup spread the gather over the CUs (the lane-per-sample
// form had 1 to 30 workgroups, each waiting for its loads row by row). The
// columns hold for every line and are formed once (two FP64 divisions each)
// where LDS has room for them (wp_keep_columns). us, lane per sample -> this: 9 lines of 128 rows, 2,062
// samples, FP64 443 -> 39; 9 x 300 rows, 8,000 samples, FP64 1,115 -> 94; 9 x 462
// rows, 3,622 samples, FP32 2,506 -> 174.
constexpr int WP_NS = 16, WP_KC = 128, WP_THREADS = 320;
// rows of columns that LDS holds beside the two product buffers
constexpr int WP_COLS_MAX = 1800;
// Whether a launch keeps them: for several lines, and unless they hold a CU to one
// workgroup (past 768 rows) where the launch has more. us, kept / formed on each
// line, FP64, dz = 1.75 v dt: 9 lines of 1,000 rows, 2,000 samples 296 / 464, 20,000
// 1,841 / 1,128, 130,000 11,674 / 6,026; of 300 rows, 20,000 264 / 345; one line of
// 500 rows, 130,000 samples 585 / 360, of 1,000 rows 1,730 / 686.
inline bool wp_keep_columns(int nlines, int nz, int64_t ns, int64_t nt, int ncu) {
  constexpr int64_t LDS_CU = 163840, prod = 2 * WP_KC * WP_NS * (int64_t)sizeof(double);
  if (nlines < 2 || nz > WP_COLS_MAX || nt >= (int64_t)1 << 31) return false;
  const int64_t per_cu = LDS_CU / (prod + (int64_t)nz * WP_NS * (int64_t)sizeof(int));
  return per_cu > 1 || (ns + WP_NS - 1) / WP_NS <= ncu;
}

template <typename S, bool CM>
__global__ void __launch_bounds__(WP_THREADS)
k_wake_wp(const S *__restrict__ cap, int nlines, int64_t cap_samples, int Nz, int k0, int nz,
          const double *__restrict__ z, const double *__restrict__ dz,
          const double *__restrict__ s, int64_t ns, double v, double zref_v, double t0,
          double ti, double dt, int64_t nt, int64_t ncols, double qe12, bool kept,
          double *__restrict__ WP3d) {
  __shared__ double prod[2][WP_KC * WP_NS];
  extern __shared__ int wp_cols[];  // [nz][WP_NS] if kept
  const int sub = (int)threadIdx.x & (WP_NS - 1);
  const int64_t n = (int64_t)blockIdx.x * WP_NS + sub;
  const double sn = s[n < ns ? n : ns - 1];
  const double nv = -v;
  // the column of Ezt that row k of a line reads for this s, -1: none
  const auto column = [&](int k) -> int64_t {
    const int kr = CM ? nz - 1 - k : k;
    double ts = CM ? (z[kr] - sn) / nv : (z[kr] + sn) / v;
    ts = ts - zref_v;
    ts = ts - t0;
    ts = ts + ti;
    const int64_t it = (int64_t)(ts / dt);
    const int64_t col = it < 0 ? it + ncols : it;  // python negative index
    return (it < nt && col >= 0 && col < nt) ? col : -1;
  };
  if (kept) {
    for (int k = (int)threadIdx.x / WP_NS; k < nz; k += WP_THREADS / WP_NS)
      wp_cols[k * WP_NS + sub] = (int)column(k);
    __syncthreads();
  }
  const int nch = (nz + WP_KC - 1) / WP_KC;  // chunks of rows per line
  const int total = nlines * nch;
  constexpr int ROWS = (WP_THREADS - 64) / WP_NS;  // rows the producing waves take at once
  const bool adds = threadIdx.x < 64;
  const int row = ((int)threadIdx.x - 64) / WP_NS;
  const auto produce = [&](int g) {
    const int l = g / nch, kb = (g - l * nch) * WP_KC;
    const S *line = cap + (int64_t)l * cap_samples * Nz + k0;
    double *out = prod[g & 1];
#pragma unroll
    for (int i = 0; i < WP_KC / ROWS; ++i) {
      const int kk = row + i * ROWS, k = kb + kk;
      if (k < nz) {
        const int64_t col = kept ? (int64_t)wp_cols[k * WP_NS + sub] : column(k);
        double e = 0.0;
        if (col >= 0) e = (double)line[col * Nz + (CM ? nz - 1 - k : k)];
        out[kk * WP_NS + sub] = col >= 0 ? e * (CM ? -dz[k] : dz[k]) : 0.0;
      }
    }
  };
  if (!adds && total > 0) produce(0);
  __syncthreads();
  double acc = 0.0;
  for (int g = 0; g < total; ++g) {
    if (adds) {
      const int l = g / nch, kb = (g - l * nch) * WP_KC;
      const int m = min(WP_KC, nz - kb);
      const double *in = prod[g & 1] + sub;
      if (m == WP_KC) {
#pragma unroll 16
        for (int i = 0; i < WP_KC; ++i) acc = acc + in[i * WP_NS];
      } else {
        for (int i = 0; i < m; ++i) acc = acc + in[i * WP_NS];
      }
      if (kb + WP_KC >= nz) {
        acc = acc / qe12;
        if (threadIdx.x < WP_NS && n < ns) WP3d[(int64_t)l * ns + n] = acc;
      }
    } else if (g + 1 < total) {
      produce(g + 1);
    }
    __syncthreads();
  }
  if (total == 0 && threadIdx.x < WP_NS && n < ns)  // no rows kept: every line is 0 / q
    for (int l = 0; l < nlines; ++l) WP3d[(int64_t)l * ns + n] = 0.0 / qe12;
}

// numpy's float64 add-reduce of a contiguous block of at most 8192 values:
// fewer than 8 -> sequential; up to 128 -> 8 interleaved accumulators combined
// ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)) then the tail; otherwise split at
// n2 = n/2 - (n/2 % 8) and add the two halves.
//
// One wave sums a block: 8 lanes hold the accumulators of a leaf, 8 leaves at a
// time, and the leaf sums meet in `val` (128 values) along the tree. Called by
// every wave of a workgroup with the same n (the barriers are the workgroup's).
// A node of the tree is named by its path from the root, one bit per split.
struct NpNode {
  int lo, len;
  bool leaf_above;  // a leaf was met before the path's end
};
__device__ __forceinline__ NpNode np_node(int n, int path, int depth) {
  NpNode x{0, n, false};
  for (int d = depth - 1; d >= 0; --d) {
    if (x.len <= 128) {
      // below a leaf only the path of zeros names the leaf itself
      x.leaf_above = x.leaf_above || (path & ((2 << d) - 1)) != 0;
      return x;
    }
    int n2 = x.len / 2;
    n2 -= n2 % 8;
    if ((path >> d) & 1) {
      x.lo += n2;
      x.len -= n2;
    } else {
      x.len = n2;
    }
  }
  return x;
}

__device__ inline double np_pairwise_wave(const double *__restrict__ a, int n, double *val) {
  const int lane = (int)threadIdx.x & 63, sub = lane & 7;
  int depth = 0;  // splits on the path of right halves, the longest ones
  for (int len = n; len > 128; ++depth) {
    int n2 = len / 2;
    n2 -= n2 % 8;
    len -= n2;
  }
  for (int base = 0; base < (1 << depth); base += 8) {
    const int slot = base + (lane >> 3);
    const NpNode x = np_node(n, slot, depth);
    const bool ok = slot < (1 << depth) && !x.leaf_above;
    const double *p = a + x.lo;
    double r = 0.0;
    if (ok && x.len >= 8) {
      const int m = x.len - x.len % 8;
      r = p[sub];
      double w[15];
#pragma unroll
      for (int i = 0; i < 15; ++i) w[i] = 8 * (i + 1) < m ? p[8 * (i + 1) + sub] : 0.0;
#pragma unroll
      for (int i = 0; i < 15; ++i)
        if (8 * (i + 1) < m) r = r + w[i];
    }
    r = r + __shfl_xor(r, 1);
    r = r + __shfl_xor(r, 2);
    r = r + __shfl_xor(r, 4);
    if (ok && sub == 0) {
      if (x.len < 8) {
        r = 0.0;
        for (int i = 0; i < x.len; ++i) r = r + p[i];
      } else {
        for (int i = x.len - x.len % 8; i < x.len; ++i) r = r + p[i];
      }
      val[slot] = r;
    }
  }
  __syncthreads();
  for (int d = depth - 1; d >= 0; --d) {  // nodes after d splits, the two halves of each
    const int sh = depth - d;
    if (lane < (1 << d)) {
      const NpNode x = np_node(n, lane, d);
      if (!x.leaf_above && x.len > 128)
        val[lane << sh] = val[lane << sh] + val[(lane << sh) | (1 << (sh - 1))];
    }
    __syncthreads();
  }
  const double r = val[0];
  __syncthreads();
  return r;
}

// WakeSolver.calc_trans_WP (wakeSolver.py:583-612) on a 3x3 window (i-major):
// the prefix sums of four lines up to every s, each summed as numpy does. A
// workgroup takes one s, a wave each line. Bound by the additions, which the
// tree of the pairwise sum spreads over 64 lanes (a thread per s had chains of
// ns additions): 385 -> 10 us at 2,062 samples, 1,495 -> 80 us at 8,000.
static __global__ void __launch_bounds__(256)
k_wake_trans(const double *__restrict__ WP3d, int64_t ns, double ds, double dxsum,
             double dysum, double *__restrict__ WPx, double *__restrict__ WPy) {
  __shared__ double val[4][128], sums[4];
  const int64_t n = blockIdx.x;
  const int w = (int)threadIdx.x >> 6;
  const int line = w == 0 ? 7 : w == 1 ? 1 : w == 2 ? 5 : 3;
  const double *a = WP3d + line * ns;
  double res = 0.0;
  for (int64_t lo = 0; lo < n; lo += 8192) {
    const int m = (int)((n - lo) < 8192 ? (n - lo) : 8192);
    res = res + np_pairwise_wave(a + lo, m, val[w]);
  }
  if ((threadIdx.x & 63) == 0) sums[w] = res * ds;
  __syncthreads();
  if (threadIdx.x == 0) {
    WPx[n] = (-(sums[0] - sums[1])) / dxsum;
    WPy[n] = (-(sums[2] - sums[3])) / dysum;
  }
}

// Neumaier compensated accumulation.
struct Comp {
  double s, c;
  __device__ void add(double x) {
    const double t = s + x;
    if (fabs(s) >= fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
  }
};

// One workgroup per bin and NS signals: X[f] = sum_n x[n] exp(-2 pi i f n / N).
// Bound by the FP64 operations of sincospi, which the signals of a call share;
// the phase f n mod N is carried from sample to sample (no division), and the
// threads' sums meet in a tree. Three signals and then two of 2,062 samples took
// 61 us a launch, now 17 and 14; of 8,000 samples 109, now 53 and 40.
template <int NS>
__global__ void __launch_bounds__(256)
k_dft(const double *__restrict__ x, int64_t len, int64_t N, int64_t nbins,
      double *__restrict__ out) {
  const int64_t f = blockIdx.x;
  Comp re[NS], im[NS];
#pragma unroll
  for (int g = 0; g < NS; ++g) re[g] = im[g] = Comp{0.0, 0.0};
  int64_t ph = (f * (int64_t)threadIdx.x) % N;  // exact phase reduction
  const int64_t step = (f * (int64_t)blockDim.x) % N;
  for (int64_t n = threadIdx.x; n < len; n += blockDim.x) {
    double sn, cs;
    sincospi(-2.0 * (double)ph / (double)N, &sn, &cs);
#pragma unroll
    for (int g = 0; g < NS; ++g) {
      const double v = x[g * len + n];
      re[g].add(v * cs);
      im[g].add(v * sn);
    }
    ph += step;
    if (ph >= N) ph -= N;
  }
  __shared__ double part[4][2 * NS][2];
#pragma unroll
  for (int g = 0; g < 2 * NS; ++g) {
    Comp c = g < NS ? re[g] : im[g - NS];
    for (int o = 32; o > 0; o >>= 1) {
      const double ps = __shfl_xor(c.s, o), pc = __shfl_xor(c.c, o);
      c.add(ps);
      c.c += pc;
    }
    if ((threadIdx.x & 63) == 0) {
      part[threadIdx.x >> 6][g][0] = c.s;
      part[threadIdx.x >> 6][g][1] = c.c;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2 * NS) {
    const int g = threadIdx.x;
    Comp c{0.0, 0.0};
    for (int w = 0; w < 4; ++w) {
      c.add(part[w][g][0]);
      c.c += part[w][g][1];
    }
    const int sig = g < NS ? g : g - NS;
    out[((int64_t)sig * nbins + f) * 2 + (g < NS ? 0 : 1)] = c.s + c.c;
  }
}

}  // namespace wf
