// Two leapfrog steps per launch (k_fused4_t2): the applicability rule and the
// FP64 launcher.
#include "lib_fused_t2.h"

#pragma GCC visibility push(hidden)

// 0: one step per launch; 1: pairs of steps, the call may end with a pair;
// 2: pairs of steps, the call ends with a single step
int fused_t2_applies(const wf_handle *h, const wf_step_args *a) {
  const wf::GridDev &g = h->g;
  const bool lut = a->code && a->mat && a->nmat > 0 && a->metric2d;
  const bool box = a->box_hi[0] > a->box_lo[0] && a->box_hi[1] > a->box_lo[1] &&
                   a->box_hi[2] > a->box_lo[2];
  // the wakefield step: a beam line fed from the beam table (with conduction,
  // J = sigma E elsewhere)
  const bool jok = a->beam_table && (a->conductive ? a->jmode == WF_J_FULL
                                                   : a->jmode == WF_J_LINE);
  const int elem = h->dtype == WF_F64 ? 8 : 4, vn = 16 / elem;  // cells per lane
  if (a->two_step == 0 || !lut || !a->zero_masked || a->code_escape || a->compute_f64 || !jok ||
      !wf::t2_in_reach(g.N, elem) || a->variant != 0 ||
      a->full_rows > 0 || (a->cells_per_lane != 0 && a->cells_per_lane != vn) || box ||
      a->traj_E || (a->mon_acc && (!a->mon_work || a->mon_slots < 1)) || a->nsteps < 2)
    return 0;
  // Pairs are the faster launches at every size measured (us per step, one step
  // per launch against pairs: 32x32x64 FP32 16.0 / 7.5, 48x48x128 FP64 17.2 /
  // 8.6, 91x75x161 FP32 35.0 / 12.4, 160x160x200 FP64 267 / 58, 300x220x180
  // FP32 270 / 66). Where a call always ended with a single step, so that
  // the spare buffers hold the fields one step back, it still does: rows that
  // are no whole number of lanes or longer than 256 cells, runs with a field
  // monitor and, by default (1), grids under 2^20 cells and FP64 rows under 224 cells.
  const bool big = a->two_step != 1 ||
                   (g.N >= (int64_t)1 << 20 && (h->dtype == WF_F32 || g.Nx >= 224));
  if (big && g.Nx <= 256 && g.Nx % vn == 0 && !a->mon_acc) return 1;
  return a->nsteps >= 3 ? 2 : 0;
}

int step_fused_t2_f64(wf_handle *h, wf_step_args *a, hipStream_t st, bool end_paired) {
  return wff::launch_t2<double>(h, a, h->md, st, end_paired);
}

#pragma GCC visibility pop
