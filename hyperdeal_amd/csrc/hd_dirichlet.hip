// hd_dirichlet.hip -- Dirichlet boundaries for the collapsed kernels: the
// boundary correction of a collapsed apply or LSRK stage (gfx950).
//
// The collapsed kernels read the inflow face of every cell from its
// neighbour, across the box edge as if the mesh were periodic.  At a
// Dirichlet boundary the reference (advection_operation.h:484-520, ECL;
// 1005-1100, FCL) uses the exterior value u+ = -u- + 2 g at the face
// quadrature points (u+ = -u- for homogeneous data).  With full upwinding an
// outflow face does not see u+, so only the inflow faces differ from the
// periodic operator, and the difference is linear: for a cell on the inflow
// boundary of direction d (side +1: inflow from the left, the cell's first
// layer; side -1: the last layer)
//   K(p) += b_d[p_d] ( -u(p_d = own inflow node, p_t) + 2 G(p_t)
//                      - u_wrap(p_d = its outflow node, p_t) )
// where u_wrap is the periodic image the kernel read, b_d the collapsed
// face column and G = (x)_{t != d} Sinv_t g(q_t): the face integral of g
// against the tangential basis, after the tangential inverse mass matrix
// (Sinv = (S^T W S)^-1 S^T W; S^-1 for n_points = k+1, I for collocation).
//
// The boundary functions are products of 1D functions (Landau: a sum of two),
// and so is their projection: G(p_t) = sum_c f_d(x_d) prod_t h_t(p_t), h_t =
// Sinv_t f_t(q_t), D n_points evaluations per cell instead of
// n_points^(D-1) of all D factors and D - 1 contractions.
//
// One block per cell on an inflow boundary (one to four waves, as many as a
// face has nodes), one launch for all directions: a cell belongs to the first
// of its boundary directions, and its block adds the corrections of all of
// them in order, so corner cells are never updated by two blocks at once.
// A thread per face node walks its line along d: with a thread per node of the
// cell instead the same stage takes 354 us (3+3, k = 3: the step 11.3 ->
// 12.7 ms), as every thread then repeats the data's products and the face
// loads.  What is left is memory: the input's two face layers and a
// read-modify-write of every line of the cell per direction.  2+2, k = 3, 24^4
// cells, FP64 stage with all four directions: 4 x 64 us with one launch per
// direction and the data evaluated point by point -> 193 us (137 us for a
// stage that leaves the solution).
// The correction reads only the input vector (not dst / ti_out / sol, which
// the kernel before it wrote), so it runs after the collapsed kernel:
// sol += b_dt C and ti_out += a_dt C in a stage.
#include "hd_device.h"

#include <algorithm>

namespace hd
{
namespace dirichlet
{
constexpr int kBlock = 256;
// Inhomogeneous data on more face points (3+3 with 7 or 8 points per direction)
// is refused: no other kernel here takes those sizes, and none is tested there.
constexpr int kMaxFacePoints = 7776;

__host__ __device__ inline long long ipow_ll(int b, int e)
{
  long long r = 1;
  for (int i = 0; i < e; ++i)
    r *= b;
  return r;
}

// the directions with an inflow boundary, in order; blocks start[k] ..
// start[k + 1] - 1 own the cells on boundary k that lie on no earlier one
struct Layers
{
  int n;
  int d[kMaxDim], side[kMaxDim]; // side +1: the first layer, -1: the last
  long long start[kMaxDim + 1];
};

// the boundary function is terms() products of factor(): the factor of
// direction d at x (the functions of eval_function, hd_functions.h)
__device__ inline int terms(int id) { return id == 5 ? 2 : 1; }
__device__ inline double factor(int id, const double *prm, int dim_x, int d,
                                int term, double x, double t)
{
  const double pi = 3.14159265358979323846;
  switch (id)
    {
      case 1:
        {
          const double y = 2.0 * pi * (x - t * prm[d]);
          return d == 0 ? sin(y) : cos(y);
        }
      case 2:
        return 1.0;
      case 3:
        return d == 0 ? sin(x * pi) : cos(x * pi);
      case 4:
        return sin(2.0 * pi * (x - t * prm[d]));
      case 5:
        {
          // (1 + eps prod_{d < np} cos(k x_d)) times the Maxwellian
          double r = d >= dim_x ? exp(-0.5 * x * x) / sqrt(2.0 * pi) : 1.0;
          if (term == 1)
            r *= (d == 0 ? prm[0] : 1.0) *
                 (d < (int)prm[2] ? cos(prm[1] * x) : 1.0);
          return r;
        }
      default:
        return 0.0;
    }
}

// MODE 0: apply; 1: stage; 2: stage without ti_out; 3: stage that leaves sol
template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void correct_kernel(
  const T *__restrict__ src, T *dst, const T *__restrict__ coef, MeshDev mesh,
  QuadDev q, StageDev stage, Layers ly, int D, int N, int NQ, int dim_x,
  double time)
{
  // 1D factors: at the quadrature points, at the cell's edge on boundary k,
  // and projected on the nodes
  __shared__ double fq[2][kMaxDim][8], fe[2][kMaxDim], h[2][kMaxDim][8];
  const int tid = threadIdx.x, nthr = blockDim.x;
  // the cell: coordinates from the index among its boundary's own cells
  int k0 = 0;
  while (k0 + 1 < ly.n && blockIdx.x >= ly.start[k0 + 1])
    ++k0;
  int c[kMaxDim];
  unsigned rem = (unsigned)(blockIdx.x - ly.start[k0]);
  long long cell = 0;
  for (int j = 0; j < D; ++j)
    {
      int own = -1; // j is boundary `own`
      for (int k = 0; k < ly.n; ++k)
        own = ly.d[k] == j ? k : own;
      const int n = mesh.n[j];
      if (own == k0)
        c[j] = ly.side[k0] > 0 ? 0 : n - 1;
      else
        {
          // not on an earlier boundary
          const bool off = own >= 0 && own < k0;
          const unsigned m = off ? n - 1 : n;
          c[j] = (int)(rem % m) + (off && ly.side[own] > 0 ? 1 : 0);
          rem /= m;
        }
      cell += (long long)c[j] * mesh.stride[j];
    }

  const int nterm = q.bc_inhomogeneous ? terms(q.bc_function) : 0;
  if (q.bc_inhomogeneous)
    {
      // (NQ + 1 places per direction: the points, then the edge)
      for (int i = tid; i < nterm * D * (NQ + 1); i += nthr)
        {
          const int e = i % (NQ + 1), j = i / (NQ + 1) % D;
          const int term = i / ((NQ + 1) * D);
          int side = 0;
          for (int k = 0; k < ly.n; ++k)
            side = ly.d[k] == j ? ly.side[k] : side;
          const double local = e < NQ ? q.qp[e] : (side > 0 ? 0.0 : 1.0);
          const double v =
            factor(q.bc_function, q.bc_params, dim_x, j, term,
                   mesh.lo[j] + (c[j] + local) * mesh.h[j], time);
          if (e < NQ)
            fq[term][j][e] = v;
          else
            fe[term][j] = v;
        }
      __syncthreads();
      for (int i = tid; i < nterm * D * N; i += nthr)
        {
          const int p = i % N, j = i / N % D, term = i / (N * D);
          double s = 0.0;
          for (int e = 0; e < NQ; ++e)
            s += q.Sinv[p * NQ + e] * fq[term][j][e];
          h[term][j][p] = s;
        }
      __syncthreads();
    }

  const int face_nodes = (int)ipow_ll(N, D - 1);
  const long long cell_dofs = ipow_ll(N, D);
  const int per = N * N + N;
  for (int k = k0; k < ly.n; ++k)
    {
      const int d = ly.d[k], side = ly.side[k];
      if (c[d] != (side > 0 ? 0 : mesh.n[d] - 1))
        continue; // uniform for the block
      if (k > k0)
        __syncthreads(); // the previous direction's updates are done
      const long long wrap =
        cell +
        (side > 0 ? 1 : -1) * (long long)(mesh.n[d] - 1) * mesh.stride[d];
      const int sd = (int)ipow_ll(N, d); // node stride of direction d
      const int own_node = side > 0 ? 0 : N - 1;
      const int wrap_node = side > 0 ? N - 1 : 0;
      const T *bcol = coef + d * per + N * N;
      for (int f = tid; f < face_nodes; f += nthr)
        {
          // node index of face point f (tangential coordinates, first
          // fastest) and the data there
          int base = 0, m = 1, r = f;
          double g0 = nterm > 0 ? fe[0][d] : 0.0;
          double g1 = nterm > 1 ? fe[1][d] : 0.0;
          for (int j = 0; j < D; ++j)
            {
              if (j != d)
                {
                  const int p = r % N;
                  base += p * m;
                  r /= N;
                  if (nterm > 0)
                    g0 *= h[0][j][p];
                  if (nterm > 1)
                    g1 *= h[1][j][p];
                }
              m *= N;
            }
          const double own =
            (double)src[cell * cell_dofs + base + own_node * sd];
          const double wr =
            (double)src[wrap * cell_dofs + base + wrap_node * sd];
          const double diff = 2.0 * (g0 + g1) - own - wr;
          for (int pd = 0; pd < N; ++pd)
            {
              const long long idx = cell * cell_dofs + base + pd * sd;
              const double corr = (double)bcol[pd] * diff;
              if (MODE == 0)
                dst[idx] = (T)((double)dst[idx] + corr);
              else
                {
                  if (MODE != 3)
                    stage.sol[idx] += stage.b_dt * corr;
                  if (MODE == 1 || MODE == 3)
                    {
                      T *ti = static_cast<T *>(stage.ti_out);
                      ti[idx] = (T)((double)ti[idx] + stage.a_dt * corr);
                    }
                }
            }
        }
    }
}

template <typename T>
hipError_t correct(int D, int N, int NQ, int mode, const T *src, T *dst,
                   const T *coef, const MeshDev &mesh, const InflowDev &inflow,
                   const QuadDev &q, const StageDev &stage, double time,
                   int dim_x, hipStream_t stream)
{
  Layers ly{};
  for (int d = 0; d < D; ++d)
    {
      if (q.periodic[d] || inflow.side[d] == 0)
        continue;
      // cells on this boundary and on none before it
      long long cells = 1;
      for (int j = 0; j < D; ++j)
        {
          bool earlier = false;
          for (int k = 0; k < ly.n; ++k)
            earlier = earlier || ly.d[k] == j;
          if (j != d)
            cells *= earlier ? mesh.n[j] - 1 : mesh.n[j];
        }
      ly.d[ly.n] = d;
      ly.side[ly.n] = inflow.side[d];
      ly.start[ly.n + 1] = ly.start[ly.n] + cells;
      ++ly.n;
    }
  if (ly.n == 0)
    return hipSuccess;
  const long long face_nodes = ipow_ll(N, D - 1);
  const int threads =
    (int)std::min<long long>(kBlock, (face_nodes + 63) / 64 * 64);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)ly.start[ly.n]), dim3(threads),
                       0, stream, src, dst, coef, mesh, q, stage, ly, D, N,
                       NQ, dim_x, time);
    return hipGetLastError();
  };
  if (mode == 0)
    return go(correct_kernel<T, 0>);
  if (stage.keep != kSolUpdate)
    return go(correct_kernel<T, 3>);
  return stage.ti_out ? go(correct_kernel<T, 1>) : go(correct_kernel<T, 2>);
}
} // namespace dirichlet

bool dirichlet_collapsed_supported(int D, int NQ, bool inhomogeneous)
{
  return D >= 2 && D <= kMaxDim && NQ <= 8 &&
         (!inhomogeneous ||
          dirichlet::ipow_ll(NQ, D - 1) <= dirichlet::kMaxFacePoints);
}

hipError_t dirichlet_correct_f64(int D, int N, int NQ, int mode,
                                 const double *src, double *dst,
                                 const double *coef, const MeshDev &mesh,
                                 const InflowDev &inflow, const QuadDev &q,
                                 const StageDev &stage, double time,
                                 int dim_x, hipStream_t stream)
{
  return dirichlet::correct<double>(D, N, NQ, mode, src, dst, coef, mesh,
                                    inflow, q, stage, time, dim_x, stream);
}

hipError_t dirichlet_correct_f32(int D, int N, int NQ, int mode,
                                 const float *src, float *dst,
                                 const float *coef, const MeshDev &mesh,
                                 const InflowDev &inflow, const QuadDev &q,
                                 const StageDev &stage, double time,
                                 int dim_x, hipStream_t stream)
{
  return dirichlet::correct<float>(D, N, NQ, mode, src, dst, coef, mesh,
                                   inflow, q, stage, time, dim_x, stream);
}
} // namespace hd
