// hd_probe.hip -- C entries for the tests (not in include/): which kernel a
// size takes, and kernels that a call reaches only under conditions that a
// test cannot bring about.
#include "hd_handles.h"

extern "C" {

// 1: the potential solves of these x cells run on strips
int hd_probe_vp_strips(int degree, int n0, int n1)
{
  const int n[3] = {n0, n1, 0};
  return hd::vp_poisson2d_supported(2, degree + 1, (long long)n0 * n1) &&
         hd::vp_strips_supported(2, degree + 1, n);
}

} // extern "C"
