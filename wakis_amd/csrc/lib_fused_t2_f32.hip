// Two leapfrog steps per launch with FP32 storage.
#include "lib_fused_t2.h"

#pragma GCC visibility push(hidden)
int step_fused_t2_f32(wf_handle *h, wf_step_args *a, hipStream_t st, bool end_paired) {
  return wff::launch_t2<float>(h, a, h->mf, st, end_paired);
}
#pragma GCC visibility pop
