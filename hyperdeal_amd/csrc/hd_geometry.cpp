// hd_geometry.cpp -- host-side geometry of a deformed phase-space mesh (see
// hd_geometry.h).
#include "hd_geometry.h"
#include "hd_tables.h"

#include <algorithm>
#include <cmath>

namespace hd
{
namespace
{
constexpr double kPi = 3.14159265358979323846;

// closed-form inverse of a 1x1, 2x2 or 3x3 matrix; returns the determinant
double invert_small(int dim, const double J[3][3], double Ji[3][3])
{
  if (dim == 1)
    {
      Ji[0][0] = 1.0 / J[0][0];
      return J[0][0];
    }
  if (dim == 2)
    {
      const double det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
      Ji[0][0] = J[1][1] / det;
      Ji[0][1] = -J[0][1] / det;
      Ji[1][0] = -J[1][0] / det;
      Ji[1][1] = J[0][0] / det;
      return det;
    }
  const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
  Ji[0][0] = c00 / det;
  Ji[1][0] = c01 / det;
  Ji[2][0] = c02 / det;
  Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) / det;
  Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) / det;
  Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) / det;
  Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) / det;
  Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) / det;
  Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / det;
  return det;
}

void cell_index(const SpaceMap &m, long long c, int *idx)
{
  for (int d = 0; d < m.dim; ++d)
    {
      idx[d] = (int)(c % m.n[d]);
      c /= m.n[d];
    }
}
} // namespace

void space_map(const SpaceMap &m, double *x)
{
  double s = m.delta;
  for (int j = 0; j < m.dim; ++j)
    s *= std::sin(m.freq * kPi * (x[j] - m.lo[j]) / (m.hi[j] - m.lo[j]));
  for (int j = 0; j < m.dim; ++j)
    x[j] += s;
}

void space_jacobian(const SpaceMap &m, const int *idx, const double *xi,
                    double Ji[3][3], double &det)
{
  double sn[3], cs[3];
  for (int j = 0; j < m.dim; ++j)
    {
      const double xh = m.lo[j] + (idx[j] + xi[j]) * m.h[j];
      const double arg = m.freq * kPi * (xh - m.lo[j]) / (m.hi[j] - m.lo[j]);
      sn[j] = std::sin(arg);
      cs[j] = std::cos(arg);
    }
  // x_i = x^_i + s(x^) for every i: d x_i / d x^_j = delta_ij + ds/dx^_j,
  // and d x^_j / d xi_j = h_j
  double J[3][3] = {};
  for (int j = 0; j < m.dim; ++j)
    {
      double ds = m.delta * m.freq * kPi / (m.hi[j] - m.lo[j]) * cs[j];
      for (int k = 0; k < m.dim; ++k)
        if (k != j)
          ds *= sn[k];
      for (int i = 0; i < m.dim; ++i)
        J[i][j] = ((i == j ? 1.0 : 0.0) + ds) * m.h[j];
    }
  det = invert_small(m.dim, J, Ji);
}

void space_tables(const SpaceMap &m, int nq, const double *xq,
                  const double *wq, const double *a, std::vector<double> &cell,
                  std::vector<double> &face)
{
  const int dim = m.dim;
  int npt = 1, nfpt = 1;
  for (int d = 0; d < dim; ++d)
    npt *= nq;
  for (int d = 1; d < dim; ++d)
    nfpt *= nq;
  const long long nc = m.n_cells();
  const int per = a ? dim + 1 : 1;
  cell.assign((size_t)nc * npt * per, 0.0);
  face.assign(a ? (size_t)nc * 2 * dim * nfpt : 0, 0.0);
  for (long long c = 0; c < nc; ++c)
    {
      int idx[3] = {0, 0, 0};
      cell_index(m, c, idx);
      for (int q = 0; q < npt; ++q)
        {
          double xi[3] = {0, 0, 0}, w = 1.0;
          int r = q;
          for (int j = 0; j < dim; ++j)
            {
              xi[j] = xq[r % nq];
              w *= wq[r % nq];
              r /= nq;
            }
          double Ji[3][3], det;
          space_jacobian(m, idx, xi, Ji, det);
          double *out = &cell[((size_t)c * npt + q) * per];
          if (a)
            for (int d = 0; d < dim; ++d)
              {
                double v = 0.0;
                for (int i = 0; i < dim; ++i)
                  v += Ji[d][i] * a[i];
                out[d] = v;
              }
          out[per - 1] = std::fabs(det) * w;
        }
      if (!a)
        continue;
      for (int d = 0; d < dim; ++d)
        for (int s = 0; s < 2; ++s)
          for (int p = 0; p < nfpt; ++p)
            {
              double xi[3] = {0, 0, 0}, w = 1.0;
              int r = p;
              for (int j = 0; j < dim; ++j)
                {
                  if (j == d)
                    {
                      xi[j] = s;
                      continue;
                    }
                  xi[j] = xq[r % nq];
                  w *= wq[r % nq];
                  r /= nq;
                }
              double Ji[3][3], det;
              space_jacobian(m, idx, xi, Ji, det);
              double v = 0.0;
              for (int i = 0; i < dim; ++i)
                v += Ji[d][i] * a[i];
              face[(((size_t)c * 2 * dim) + 2 * d + s) * nfpt + p] =
                (s ? 1.0 : -1.0) * v * std::fabs(det) * w;
            }
    }
}

void curved_space_operator(const SpaceMap &m, const Tables1D &t, double skew,
                           const std::vector<double> &cell,
                           const std::vector<double> &face, CurvedHost &out)
{
  const int dim = m.dim, nd = t.nd, nq = t.nq;
  int n = 1, np = 1, nf = 1, npf = 1;
  for (int d = 0; d < dim; ++d)
    {
      n *= nd;
      np *= nq;
      if (d > 0)
        {
          nf *= nd;
          npf *= nq;
        }
    }
  const int sides = 2 * dim, nb = sides * nf;
  out.cells = m.n_cells();
  out.K.assign((size_t)out.cells * n * n, 0.0);
  out.B.assign((size_t)out.cells * n * nb, 0.0);
  // tensor products of the 1D tables: nodes -> points of the cell and of a
  // face, points -> nodes
  auto tensor = [](const std::vector<double> &A, int rows, int cols, int k) {
    int R = 1, C = 1;
    std::vector<double> r(1, 1.0);
    for (int d = 0; d < k; ++d)
      {
        // direction d is slower than the ones before it
        std::vector<double> s((size_t)R * rows * C * cols);
        for (int i = 0; i < rows; ++i)
          for (int a = 0; a < R; ++a)
            for (int j = 0; j < cols; ++j)
              for (int b = 0; b < C; ++b)
                s[((size_t)(i * R + a)) * (C * cols) + j * C + b] =
                  A[i * cols + j] * r[(size_t)a * C + b];
        r.swap(s);
        R *= rows;
        C *= cols;
      }
    return r;
  };
  const std::vector<double> V = tensor(t.S, nq, nd, dim);
  const std::vector<double> Vf = tensor(t.S, nq, nd, dim - 1);
  const std::vector<double> P = tensor(t.Sinv, nd, nq, dim);
  int sd[3] = {1, nq, nq * nq};
  std::vector<double> X((size_t)np * np), XV((size_t)np * n);
  std::vector<double> L((size_t)np * nb);
  for (long long c = 0; c < out.cells; ++c)
    {
      const double *ca = &cell[(size_t)c * np * (dim + 1)];
      const double *fa = &face[(size_t)c * sides * npf];
      std::fill(X.begin(), X.end(), 0.0);
      std::fill(L.begin(), L.end(), 0.0);
      for (int d = 0; d < dim; ++d)
        {
          // cell term along the lines of direction d
          for (int q = 0; q < np; ++q)
            {
              const int iq = q / sd[d] % nq, base = q - iq * sd[d];
              for (int p = 0; p < nq; ++p)
                {
                  const int r = base + p * sd[d];
                  const double cq = ca[(size_t)q * (dim + 1) + d] *
                                    ca[(size_t)q * (dim + 1) + dim];
                  const double cr = ca[(size_t)r * (dim + 1) + d] *
                                    ca[(size_t)r * (dim + 1) + dim];
                  X[(size_t)q * np + r] +=
                    (1.0 - skew) * t.Dq[p * nq + iq] * cr -
                    skew * t.Dq[iq * nq + p] * cq;
                }
            }
          // faces: the own trace where the flow goes out, the neighbour's
          // values where it comes in
          for (int side = 0; side < 2; ++side)
            for (int p = 0; p < npf; ++p)
              {
                const double an = fa[(size_t)(2 * d + side) * npf + p];
                const double own = (an > 0.0 ? an : 0.0) - skew * an;
                const double in = an < 0.0 ? an : 0.0;
                const int base = p % sd[d] + (p / sd[d]) * sd[d] * nq;
                for (int i = 0; i < nq; ++i)
                  {
                    const double Fi = t.F[side * nq + i];
                    const size_t row = (size_t)(base + i * sd[d]);
                    for (int j = 0; j < nq; ++j)
                      X[row * np + base + j * sd[d]] -=
                        Fi * own * t.F[side * nq + j];
                    for (int b = 0; b < nf; ++b)
                      L[row * nb + (2 * d + side) * nf + b] -=
                        Fi * in * Vf[(size_t)p * nf + b];
                  }
              }
        }
      // inverse mass matrix: divide by JxW, then the projection
      for (int q = 0; q < np; ++q)
        {
          const double s = 1.0 / ca[(size_t)q * (dim + 1) + dim];
          double *row = &XV[(size_t)q * n];
          std::fill(row, row + n, 0.0);
          for (int r = 0; r < np; ++r)
            {
              // the lines through q only
              const double x = X[(size_t)q * np + r] * s;
              if (x != 0.0)
                for (int j = 0; j < n; ++j)
                  row[j] += x * V[(size_t)r * n + j];
            }
          for (int b = 0; b < nb; ++b)
            L[(size_t)q * nb + b] *= s;
        }
      double *K = &out.K[(size_t)c * n * n], *B = &out.B[(size_t)c * n * nb];
      for (int i = 0; i < n; ++i)
        for (int q = 0; q < np; ++q)
          {
            const double w = P[(size_t)i * np + q];
            for (int j = 0; j < n; ++j)
              K[(size_t)i * n + j] += w * XV[(size_t)q * n + j];
            for (int b = 0; b < nb; ++b)
              B[(size_t)i * nb + b] += w * L[(size_t)q * nb + b];
          }
    }
}

double space_max_speed(const SpaceMap &m, int nq, const double *xq,
                       const double *a)
{
  int npt = 1;
  for (int d = 0; d < m.dim; ++d)
    npt *= nq;
  double vmax = 0.0;
  const long long nc = m.n_cells();
  for (long long c = 0; c < nc; ++c)
    {
      int idx[3] = {0, 0, 0};
      cell_index(m, c, idx);
      for (int q = 0; q < npt; ++q)
        {
          double xi[3] = {0, 0, 0};
          int r = q;
          for (int j = 0; j < m.dim; ++j)
            {
              xi[j] = xq[r % nq];
              r /= nq;
            }
          double Ji[3][3], det;
          space_jacobian(m, idx, xi, Ji, det);
          for (int j = 0; j < m.dim; ++j)
            {
              double v = 0.0;
              for (int i = 0; i < m.dim; ++i)
                v += Ji[i][j] * a[i];
              vmax = std::fmax(vmax, std::fabs(v));
            }
        }
    }
  return vmax;
}
} // namespace hd
