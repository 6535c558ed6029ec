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

// 1: an apply or stage on a periodic deformed mesh takes the factorised form;
// x_cells and v_cells: of the two spaces
int hd_probe_curved(int dim_x, int dim_v, int degree, long long x_cells,
                    long long v_cells, int precision, int stage)
{
  return hd::curved_supported(dim_x, dim_v, degree + 1, x_cells, v_cells) &&
         hd::curved_faster(dim_x, dim_v, degree + 1, x_cells * v_cells,
                           precision == HD_FP64, stage != 0);
}

// The potential solver of a Vlasov-Poisson operator on one workgroup, or on
// strips with `comm` as their inboxes (hd_probe_strips_bytes of device memory,
// reset once): the residual image of phi where res_image is given, else a
// solve from phi, with a guess as x values or (guess_image) as an image.
// Pointers are the device's; the null stream.
long long hd_probe_strips_bytes(hd_advection *op)
{
  return (long long)hd::vp_strips_bytes(op->mf->nd, op->xdev.n);
}

int hd_probe_strips_reset(hd_advection *op, void *comm)
{
  return (int)hd::vp_strips_reset(comm, op->mf->nd, op->xdev.n);
}

int hd_probe_poisson(hd_advection *op, void *comm, const double *rho,
                     double *phi, double *efield, const double *guess,
                     const float *guess_image, const double *guess_scale,
                     float *res_image, double *res_scale, double *phi_copy,
                     double rel_tol, int max_it, long long *stats)
{
  hd::ResidualImage residual;
  residual.image = res_image;
  residual.scale = res_scale;
  residual.phi_copy = phi_copy;
  hd::GuessImage image;
  image.image = guess_image;
  image.scale = guess_scale;
  return (int)hd::vp_poisson(op->xdev, op->mf->nd, rho, phi, guess, efield,
                             op->work, rel_tol, max_it, stats, nullptr,
                             op->ptab, res_image ? &residual : nullptr, false,
                             comm, image);
}

} // extern "C"
