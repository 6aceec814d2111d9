// Batches: pairs of steps over many grids in one launch (k_fused4_t2_batch).
#include "lib_fused_t2.h"

#pragma GCC visibility push(hidden)
namespace {

template <typename S>
int build(const wf::BatchDesc<S> *bd, wf_handle *const *hs, const wf_step_args *as, int n,
          batch_t2 *t) {
  std::vector<wf::T2Batch<S>> d(n);
  const int ncu = hs[0]->ncu;
  double cells = 0;
  for (int i = 0; i < n; ++i) cells += (double)hs[i]->g.N;
  int64_t tiles = 0;
  t->wc = 1;
  for (int i = 0; i < n; ++i)
    if (!wff::t2_weights(hs[i], &as[i])) t->wc = 0;
  for (int i = 0; i < n; ++i) {
    const wf::GridDev &g = hs[i]->g;
    // the grid's share of the CUs
    const int share = std::max(1, (int)std::lround(BATCH_T2_LOAD * ncu * (double)g.N / cells));
    const wff::T2Shape sh = wff::t2_shape<S>(g, t->wc ? as[i].nw : as[i].nmat, t->wc != 0,
                                             std::min(share, ncu), 0, 0,
                                             std::max(0, ncu - share));
    if (!sh.ok || !wf::t2_in_reach(g.N, sizeof(S))) return 0;
    d[i].b = bd[i];
    if (t->wc) {
      wf::Coefs<S> &cf = d[i].b.cf;
      cf.code = (const uint8_t *)as[i].wcode;
      cf.mat = (const S *)as[i].wtab;
      cf.nmat = as[i].nw;
    }
    wff::t2_aux(sh, g, &as[i], d[i].x);
    d[i].tile0 = (int)tiles;
    tiles += (int64_t)d[i].x.ntx * d[i].x.nty * d[i].x.ntz;
    t->lds = std::max(t->lds, sh.lds);
    t->threads = std::max(t->threads, ((sh.T + 4) * sh.Q + 63) / 64 * 64);
    if (g.Nx % (16 / (int)sizeof(S))) t->rag = 1;
  }
  if (tiles > 2147483647LL) return 0;
  t->ntiles = (int)tiles;
  WF_HIP(hipMalloc(&t->desc_dev, sizeof(wf::T2Batch<S>) * n));
  WF_HIP(hipMemcpy(t->desc_dev, d.data(), sizeof(wf::T2Batch<S>) * n, hipMemcpyHostToDevice));
  return 1;
}

template <typename S>
void launch(const batch_t2 *t, int n, int cond, int desc, int s, int step0, int end, int flip,
            hipStream_t st) {
#define WF_BT2(CO, DE, RA, WC)                                                                   \
  hipLaunchKernelGGL((wf::k_fused4_t2_batch<S, CO, DE, RA, WC>), dim3((unsigned)t->ntiles),      \
                     dim3(t->threads), t->lds, st, (const wf::T2Batch<S> *)t->desc_dev, n,       \
                     t->ntiles, s, step0, end, flip)
#define WF_BT2R(CO, DE)                                                                          \
  do {                                                                                           \
    if constexpr (sizeof(S) == 4) {                                                              \
      if (t->wc) {                                                                               \
        if (t->rag) WF_BT2(CO, DE, true, true);                                                  \
        else WF_BT2(CO, DE, false, true);                                                        \
        break;                                                                                   \
      }                                                                                          \
    }                                                                                            \
    if (t->rag) WF_BT2(CO, DE, true, false);                                                     \
    else WF_BT2(CO, DE, false, false);                                                           \
  } while (0)
  if (cond) {
    if (desc) WF_BT2R(true, true);
    else WF_BT2R(true, false);
  } else {
    if (desc) WF_BT2R(false, true);
    else WF_BT2R(false, false);
  }
#undef WF_BT2R
#undef WF_BT2
}

}  // namespace

int batch_t2_build(int dtype, const void *bd, wf_handle *const *hs, const wf_step_args *as, int n,
                   batch_t2 *t) {
  return dtype == WF_F64 ? build((const wf::BatchDesc<double> *)bd, hs, as, n, t)
                         : build((const wf::BatchDesc<float> *)bd, hs, as, n, t);
}

int batch_t2_launch(int dtype, const batch_t2 *t, int n, int cond, int desc, int s, int step0,
                    int end, int flip, hipStream_t st) {
  if (dtype == WF_F64) launch<double>(t, n, cond, desc, s, step0, end, flip, st);
  else launch<float>(t, n, cond, desc, s, step0, end, flip, st);
  WF_LAUNCH_CHECK();
  return WF_OK;
}

#pragma GCC visibility pop
