// Two leapfrog steps per launch (k_fused4_t2): tile shapes and the launcher,
// included by the FP32 and FP64 translation units.
#pragma once
#include "lib_fused.h"
#include "step_fused_t2.h"

#include <cmath>

#pragma GCC visibility push(hidden)
namespace wff {

template <typename S>
using T2Fn = void (*)(wf::GridDev, wf::MetricDev<S>, const S *, const S *, S *, S *, S *,
                      wf::Coefs<S>, S, wf::T2Aux, const S *, const S *, S *);

template <typename S>
T2Fn<S> pick_t2(bool cond, bool desc, bool rag, bool wc) {
#define WF_T2(CO, DE)                                                                          \
  do {                                                                                         \
    if constexpr (sizeof(S) == 4)                                                              \
      if (wc)                                                                                  \
        return rag ? &wf::k_fused4_t2<S, CO, DE, true, true>                                   \
                   : &wf::k_fused4_t2<S, CO, DE, false, true>;                                 \
    return rag ? &wf::k_fused4_t2<S, CO, DE, true, false>                                      \
               : &wf::k_fused4_t2<S, CO, DE, false, false>;                                    \
  } while (0)
  if (cond) {
    if (desc) WF_T2(true, true);
    WF_T2(true, false);
  }
  if (desc) WF_T2(false, true);
  WF_T2(false, false);
#undef WF_T2
}

template <typename S>
using T2MonFn = void (*)(wf::GridDev, wf::MetricDev<S>, const S *, const S *, S *, S *, S *,
                         wf::Coefs<S>, S, wf::T2Aux, const S *, const S *, S *, S *);

template <typename S>
T2MonFn<S> pick_t2_mon(bool cond, bool desc, bool rag, bool wc) {
#define WF_T2(CO, DE)                                                                          \
  do {                                                                                         \
    if constexpr (sizeof(S) == 4)                                                              \
      if (wc)                                                                                  \
        return rag ? &wf::k_fused4_t2_mon<S, CO, DE, true, true>                               \
                   : &wf::k_fused4_t2_mon<S, CO, DE, false, true>;                             \
    return rag ? &wf::k_fused4_t2_mon<S, CO, DE, true, false>                                  \
               : &wf::k_fused4_t2_mon<S, CO, DE, false, false>;                                \
  } while (0)
  if (cond) {
    if (desc) WF_T2(true, true);
    WF_T2(true, false);
  }
  if (desc) WF_T2(false, true);
  WF_T2(false, false);
#undef WF_T2
}

// A tile shape of the two-step kernel and the z chunk of a launch.
struct T2Shape {
  bool ok = false;
  int ntx, T, OW, Q, QS, l0, ln, KZ;
  size_t lds;  // dynamic
};

constexpr size_t T2_LDS_CU = 163840;  // LDS of a CU: one workgroup on it
// static LDS of the kernel: E0 and E1 in three blocks per cell of a lane, H1 and
// H2 in two and one block more
template <typename S>
constexpr size_t t2_static_lds() {
  constexpr size_t V = 16 / sizeof(S);
  using C = wf::T2Slots;
  return sizeof(S) * (3 * V * (C::E0 + C::E1) + (2 * V + 1) * (C::H1 + C::H2));
}

// The shape with the least time by a model of the busiest CU: rounds of
// workgroups times planes marched (a chunk of KZ planes marches KZ + 3) times
// the time of a plane. Fitted to 9 to 120 shapes of each of 17 grids from
// 32x32x64 to 333x300x100 (FP32, FP64, with and without conduction): the shape
// it picks is within 2% of the best measured one on average, 9% at most.
// `others`: workgroups of other grids on the machine beside these.
template <typename S>
T2Shape t2_shape(const wf::GridDev &g, int nmat, bool wc, int ncu, int want_rows, int want_kz,
                 int others = 0) {
  constexpr int V = 16 / (int)sizeof(S);
  using C = wf::T2Slots;
  T2Shape out;
  double best = 1e300;
  for (int ntx = 1; ntx <= 64; ++ntx) {
    T2Shape s;
    s.ok = true;
    s.ntx = ntx;
    s.OW = V * ((g.Nx + V * ntx - 1) / (V * ntx));
    if (ntx > 1 && (s.OW < 4 * V || (int64_t)s.OW * (ntx - 1) >= g.Nx)) break;
    s.ln = s.OW / V;
    if (ntx == 1 && s.ln % 64 == 0) {
      s.l0 = 0; s.Q = s.ln; s.QS = s.Q + 1;
    } else {
      s.l0 = 1; s.Q = s.ln + (ntx == 1 ? 1 : 2); s.QS = s.Q;
    }
    const int Q = s.Q, QS = s.QS;
    int tmax = std::min(std::min(wf::T2_NT / Q - 4, (C::E0 - 1) / QS - 4),
                        std::min(std::min((C::H1 - 1) / QS - 3, (C::E1 - 1) / QS - 2),
                                 (C::H2 - 1) / QS - 1));
    if (want_rows) tmax = std::min(tmax, want_rows);
    if (tmax < 1) continue;
    const int nty0 = (g.Ny + tmax - 1) / tmax;
    for (int nty = nty0, last = 0; nty <= std::min(g.Ny, 4 * nty0); ++nty) {
      s.T = (g.Ny + nty - 1) / nty;
      if (s.T == last) continue;
      last = s.T;
      const int64_t tiles = (int64_t)ntx * ((g.Ny + s.T - 1) / s.T);
      for (int r = 1; r <= 8; ++r) {
        const int64_t ntz = std::max<int64_t>(1, (int64_t)r * ncu / tiles);
        s.KZ = want_kz ? std::min(want_kz, g.Nz) : (int)std::max<int64_t>(1, (g.Nz + ntz - 1) / ntz);
        // the planes whose scalars (four a plane) fit beside the rest
        const int64_t room = ((int64_t)T2_LDS_CU - (int64_t)t2_static_lds<S>()) / (int64_t)sizeof(S);
        const int64_t kz_max = (room - wf::t2_dyn_values(V, Q, s.T, 0, nmat, wc)) / 4;
        if (kz_max < 1) continue;
        s.KZ = (int)std::min<int64_t>(s.KZ, kz_max);
        s.lds = (size_t)wf::t2_dyn_values(V, Q, s.T, s.KZ, nmat, wc) * sizeof(S);
        const int64_t wgs = tiles * ((g.Nz + s.KZ - 1) / s.KZ);
        const int64_t rounds = (wgs + ncu - 1) / ncu;
        // us of a plane: the instructions of the four updates (whole waves of
        // rows in each), the bytes they move (in 128-byte lines), or at least
        // the chain of its three phases
        const double w = (4 * s.T + 6) * Q / 64.0 + (Q % 64 ? 4 : 0);
        const double lines = std::ceil(s.ln / 8.0) + (ntx > 1 || g.Nx * sizeof(S) % 128 ? 1 : 0);
        const double bytes = 6 * ((s.T + 3.5) * lines * 128 + s.T * s.ln * 16.0);
        const double busy = (double)std::min<int64_t>(wgs, ncu) + others;
        const double plane = std::max(std::max(0.12 * w, bytes * busy / 6.5e6), 3.0);
        const double t = (double)rounds * (s.KZ + 3) * plane;
        if (t < best * 0.999) { best = t; out = s; }
      }
    }
  }
  return out;
}

// whether pairs of steps run on weight codes: FP32 with a table of them
inline bool t2_weights(const wf_handle *h, const wf_step_args *a) {
  return h->dtype == WF_F32 && a->wcode && a->wtab && a->nw > 0;
}

inline void t2_aux(const T2Shape &sh, const wf::GridDev &g, const wf_step_args *a, wf::T2Aux &x) {
  // FP32 stores streamed past the caches where tiles write whole 128-byte lines and
  // E and H with their spare buffers about fill the 256 MB of last-level cache. ms a
  // pass, streamed against not: 256x256x512 597 / 620, 160x160x200 39.5 / 40.2, but
  // 128x128x160 21.1 / 18.7, 96x96x160 with a monitor 24.7 / 23.6, and on part lines
  // 300x220x180 71.6 / 67.1, 200x200x400 with conduction 153.6 / 151.2. FP64 always:
  // 160x160x200 82.2 / 84.3, 48x48x128 19.7 / 20.9.
  x.stream = g.Nx % 32 == 0 && (sh.ntx == 1 || sh.OW % 32 == 0) && 48.0 * (double)g.N > 200e6;
  x.ixs = a->ixs;
  x.iys = a->iys;
  x.cap_ix0 = a->cap_ix0; x.cap_iy0 = a->cap_iy0; x.cap_nx = a->cap_nx; x.cap_ny = a->cap_ny;
  x.cap_samples = a->cap_samples;
  x.ntx = sh.ntx; x.T = sh.T; x.OW = sh.OW; x.Q = sh.Q; x.QS = sh.QS;
  x.l0 = sh.l0; x.ln = sh.ln; x.KZ = sh.KZ;
  x.nty = (g.Ny + sh.T - 1) / sh.T;
  x.ntz = (g.Nz + sh.KZ - 1) / sh.KZ;
}

template <typename S>
int launch_t2(wf_handle *h, wf_step_args *a, const wf::MetricDev<S> &m, hipStream_t st,
              bool end_paired) {
  const wf::GridDev &g = h->g;
  constexpr int V = 16 / (int)sizeof(S);
  const bool wc = t2_weights(h, a);
  const int nrows = wc ? a->nw : a->nmat;
  const T2Shape sh =
      t2_shape<S>(g, nrows, wc, h->ncu, a->two_step > 1 ? a->two_step : 0, a->kz);
  if (!sh.ok) {  // one step per launch
    wf_step_args b = *a;
    b.two_step = 0;
    const int rc = sizeof(S) == 4 ? step_fused_f32(h, &b, st) : step_fused_f64(h, &b, st);
    a->result_swapped = b.result_swapped;
    return rc;
  }
  wf::T2Aux x{};
  t2_aux(sh, g, a, x);
  const bool rag = g.Nx % V != 0, cond = a->conductive != 0, desc = g.m1desc != 0;
  const T2Fn<S> kern = pick_t2<S>(cond, desc, rag, wc);
  const int threads = ((sh.T + 4) * sh.Q + 63) / 64 * 64;
  const int64_t nb = (int64_t)x.ntx * x.nty * x.ntz;
  if (nb > 2147483647LL) return fail(WF_ERANGE, "wf_step: grid too large for the fused path");
  wf::Coefs<S> cf;
  cf.a = (const S *)a->a; cf.b = (const S *)a->b;
  cf.ieps = (const S *)a->ieps; cf.sigma = (const S *)a->sigma;
  cf.code = (const uint8_t *)(wc ? a->wcode : a->code);
  cf.mat = (const S *)(wc ? a->wtab : a->mat); cf.nmat = nrows;
  {
    const S *t = (const S *)a->metric2d;
    const int64_t yz = (int64_t)g.Ny * g.Nz, xz = (int64_t)g.Nx * g.Nz, xy = (int64_t)g.Nx * g.Ny;
    cf.iAx = t; cf.iAy = t + yz; cf.iAz = t + yz + xz;
    cf.itAx = t + yz + xz + xy; cf.itAy = cf.itAx + yz; cf.itAz = cf.itAy + xz;
  }
  const S dt = (S)a->dt;
  S *Ebuf[2] = {(S *)a->E, (S *)a->E2};
  S *Hbuf[2] = {(S *)a->H, (S *)a->H2};
  const S *table = (const S *)a->beam_table;
  // steps taken in pairs; the rest one at a time (an odd step, or the last one
  // or two when the spare buffers have to hold the fields one step back)
  const int paired = end_paired ? a->nsteps / 2 * 2 : (a->nsteps - 1) / 2 * 2;
  int cur = 0, s = 0;
  // with a field monitor, the E of up to mon_slots + 1 steps in turn (a first
  // step's and all but the last second step's in the work array), then one pass
  // over the accumulators
  if (a->mon_acc) {
    const T2MonFn<S> mkern = pick_t2_mon<S>(cond, desc, rag, wc);
    const int per = std::min(wf::MON_STEPS, a->mon_slots + 1) / 2;  // pairs per pass
    const auto slot = [&](int i) { return (S *)a->mon_work + (int64_t)i * 3 * g.N; };
    while (s < paired) {
      const int np = std::min(per, (paired - s) / 2);
      wf::MonFields<S> f{};
      const S *e = Ebuf[cur];
      for (int p = 0; p < np; ++p, s += 2) {
        S *e1 = slot(2 * p), *e2 = p + 1 < np ? slot(2 * p + 1) : Ebuf[(cur + np) & 1];
        const S *row1 = table + (a->beam_row0 + s) * g.Nz;
        x.cap_sample = a->cap_sample0 + s;
        x.skip_j = 1;  // J = sigma E is stored by the single steps at the end
        hipLaunchKernelGGL(mkern, dim3((unsigned)nb), dim3(threads), sh.lds, st, g, m, e,
                           Hbuf[(cur + p) & 1], e2, Hbuf[(cur + p + 1) & 1], (S *)a->J, cf, dt, x,
                           row1, row1 + g.Nz, (S *)a->capture, e1);
        WF_LAUNCH_CHECK();
        f.e[2 * p] = e1;
        f.e[2 * p + 1] = e = e2;
      }
      monitor_steps<S>(h, a, f, s - 2 * np, 2 * np, st);
      WF_LAUNCH_CHECK();
      cur = (cur + np) & 1;
    }
  }
  for (; s < paired; s += 2) {
    const S *row1 = table ? table + (a->beam_row0 + s) * g.Nz : nullptr;
    const S *row2 = table ? table + (a->beam_row0 + s + 1) * g.Nz : nullptr;
    x.cap_sample = a->cap_sample0 + s;
    x.skip_j = (s + 2 < a->nsteps) ? 1 : 0;  // J = sigma E stored by the last launch
    hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(threads), sh.lds, st, g, m, Ebuf[cur],
                       Hbuf[cur], Ebuf[1 - cur], Hbuf[1 - cur], (S *)a->J, cf, dt, x, row1, row2,
                       (S *)a->capture);
    WF_LAUNCH_CHECK();
    cur = 1 - cur;
  }
  if (s < a->nsteps) {  // the remaining single steps on the current buffers
    wf_step_args b = *a;
    b.two_step = 0;
    b.nsteps = a->nsteps - s;
    b.beam_row0 = a->beam_row0 + s;
    b.cap_sample0 = a->cap_sample0 + s;
    b.mon_row0 = a->mon_row0 + s;
    if (cur) {
      b.E = a->E2; b.E2 = a->E;
      b.H = a->H2; b.H2 = a->H;
    }
    const int rc = sizeof(S) == 4 ? step_fused_f32(h, &b, st) : step_fused_f64(h, &b, st);
    if (rc != WF_OK) return rc;
    if (b.result_swapped) cur = 1 - cur;
  }
  a->result_swapped = cur;
  a->two_step_used = end_paired ? 1 : 2;
  return WF_OK;
}

}  // namespace wff
#pragma GCC visibility pop
