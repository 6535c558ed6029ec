// hd_curved.hip -- constant-velocity advection apply and LSRK stage on
// periodic deformed meshes, gfx950: the exact factorisation of the quadrature
// operator over the two spaces, as matrix-core products.
//
// The phase-space Jacobian is block diagonal, so every factor of the
// quadrature algorithm (operators/advection/advection_operation.h:221-566) is
// an x factor times a v factor, and the v factors of an x-direction term
// cancel against the inverse mass matrix (S^-1 S = I along v, JxW_v / JxW_v):
//
//   dst(x, v) = sum_x' Kx[x][x'] u(x', v) + sum_f Bx[x][f] u_nb,f(v)
//             + sum_v' Kv[v][v'] u(x, v') + sum_g Bv[v][g] u_nb,g(x)
//
// with one small dense matrix per x cell (Kx, and Bx over the nodes of its
// 2 dim_x neighbours' faces) and one per v cell, built once per operator on
// the host (curved_space_operator).  All x cells of a v cell share Kv, all v
// cells of an x cell share Kx.
//
// Measured (2+2, k = 3, 24^4 cells, 85M values): FP64 apply 3213 -> 434 us
// (3.1 TB/s of its 16 bytes per value), FP32 2250 -> 200 us, against the
// quadrature kernel; k = 4, 20^4 cells 4.1 -> 1.0 ms.
//
// Work decomposition.  A wave owns kXB consecutive x cells (their Kx sits in
// registers) and walks a chunk of v cells.  A cell's values are the matrix
// u[x node][v node]: the x term is Kx u (u as the B operand), the v term
// u Kv^T (u as the A operand), both accumulated in the same 16 x 16 result
// tiles, so no layout change and no LDS is needed; the two operand forms of u
// are two loads of the same lines.  Where the x nodes fill whole tiles (k = 3
// in 2D) the slots of a tile are permuted so that a lane holds four
// contiguous values of u and of the result.
//
// What bounds it: memory (16 or 8 bytes per value and the faces); the
// products are 2 (nodes + face nodes) multiply-adds per value and space at
// the matrix rate, 0.14 ms of FP64 at 2+2, k = 3, 24^4 cells.  Faces through
// which nothing flows in have zero columns and are skipped (a bit per step
// and cell).
#include "hd_device.h"
#include "hd_geometry.h"

#include <algorithm>
#include <cstring>
#include <vector>

namespace hd
{
namespace curved
{
constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

template <class T>
struct Frag;
template <>
struct Frag<double>
{
  typedef double V4 __attribute__((ext_vector_type(4)));
  static __device__ inline V4 mfma(double a, double b, V4 c)
  {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Frag<float>
{
  typedef float V4 __attribute__((ext_vector_type(4)));
  static __device__ inline V4 mfma(float a, float b, V4 c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// One space: n nodes, nf face nodes per face, T tiles of 16 nodes, SN steps
// of four nodes, SF steps of four face nodes (the faces' nodes packed).
template <int N, int DIM>
struct Space
{
  static constexpr int n = ipow(N, DIM);
  static constexpr int nf = ipow(N, DIM - 1);
  static constexpr int faces = 2 * DIM * nf;
  static constexpr int T = (n + 15) / 16;
  static constexpr int SN = (n + 3) / 4;
  static constexpr int SF = (faces + 3) / 4;
  static constexpr int S = SN + SF;
  static constexpr bool kVec = n % 16 == 0;
};

// node of product slot (step s, lane group g): whole tiles are permuted so
// that a lane's four steps are four contiguous nodes
template <int N, int DIM>
__host__ __device__ constexpr int slot_node(int s, int g)
{
  return Space<N, DIM>::kVec ? 16 * (s / 4) + 4 * g + s % 4 : 4 * s + g;
}

// The result tile of a 16x16x4 product: register r of lane group g is row
// 4 r + g (FP64) or 4 g + r (FP32).  The x node in row i of a tile:
// permuted in FP64 where x fills whole tiles, so that registers 0..3 are
// contiguous nodes.
template <class T, bool VEC>
__host__ __device__ constexpr int row_node(int i)
{
  return sizeof(T) == 8 && VEC ? 4 * (i % 4) + i / 4 : i;
}
template <class T>
__host__ __device__ constexpr int result_row(int r, int g)
{
  return sizeof(T) == 8 ? 4 * r + g : 4 * g + r;
}

// the face and node of packed face slot q: the in-cell index of the
// neighbour's node on that face (side 0: the left neighbour's last layer)
template <int N, int DIM>
__host__ __device__ inline int face_node(int side, int node)
{
  const int d = side / 2;
  const int sd = ipow(N, d);
  const int lo = node % sd, hi = node / sd;
  return lo + (side % 2 == 0 ? N - 1 : 0) * sd + hi * sd * N;
}

struct Args
{
  const void *xtab, *vtab;       // [cell][step][tile][lane]
  const unsigned *xmask, *vmask; // per cell: the face steps with inflow
  int nxc, nvc;                  // cells per space
  int nx[3], nv[3];              // cells per direction
  int chunk;                     // v cells per unit
  int xgroups;                   // units per v chunk
  long long units;
};

// the neighbour's lexicographic id within one space across `side`, wrapped
template <int DIM>
__device__ inline int neighbour(int c, const int *n, int side)
{
  int st = 1;
  for (int d = 0; d < side / 2; ++d)
    st *= n[d];
  const int nd = n[side / 2];
  const int i = c / st % nd;
  if (side % 2 == 0)
    return i == 0 ? c + (nd - 1) * st : c - st;
  return i == nd - 1 ? c - (nd - 1) * st : c + st;
}

template <class T>
struct alignas(16) Quad16
{
  T v[16 / sizeof(T)];
};

template <int N, int DX, int DV, class T, int MODE, int XB>
__global__ __launch_bounds__(kBlock) void curved_kernel(
  const T *__restrict__ src, T *__restrict__ dst, Args a, StageDev stage)
{
  using X = Space<N, DX>;
  using V = Space<N, DV>;
  using V4 = typename Frag<T>::V4;
  constexpr int nx = X::n, nv = V::n, CELL = nx * nv;
  constexpr bool VEC = X::kVec;

  // every XCD walks a contiguous range of units
  const long long per = (a.units + 7) / 8;
  const long long unit = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || unit >= a.units)
    return;
  const int xg = (int)(unit % a.xgroups);
  const int v0 = (int)(unit / a.xgroups) * a.chunk;
  const int v1 = min(v0 + a.chunk, a.nvc);
  const int lane = threadIdx.x % 64, j = lane % 16, g = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int x0 = (xg * kWaves + wave) * XB;
  if (x0 >= a.nxc)
    return;

  // this wave's x cells: coefficients, face addresses relative to the cell
  T kx[XB][X::S][X::T];
  int fxo[XB][X::SF];
  unsigned xm[XB];
#pragma unroll
  for (int b = 0; b < XB; ++b)
    {
      const int xc = min(x0 + b, a.nxc - 1);
      const T *t = static_cast<const T *>(a.xtab) +
                   (size_t)xc * (X::S * X::T * 64) + lane;
#pragma unroll
      for (int s = 0; s < X::S; ++s)
#pragma unroll
        for (int r = 0; r < X::T; ++r)
          kx[b][s][r] = t[(s * X::T + r) * 64];
      xm[b] = a.xmask[xc];
#pragma unroll
      for (int s = 0; s < X::SF; ++s)
        {
          const int q = min(4 * s + g, X::faces - 1);
          const int side = q / X::nf;
          fxo[b][s] = (neighbour<DX>(xc, a.nx, side) - xc) * CELL +
                      face_node<N, DX>(side, q % X::nf);
        }
    }
  // v node of this lane's column per tile (clamped: columns beyond the last
  // node are not stored), x node of this lane's row
  int vcol[V::T], xrow[X::T];
#pragma unroll
  for (int c = 0; c < V::T; ++c)
    vcol[c] = min(16 * c + j, nv - 1) * nx;
#pragma unroll
  for (int r = 0; r < X::T; ++r)
    xrow[r] = min(16 * r + row_node<T, VEC>(j), nx - 1);

  for (int vc = v0; vc < v1; ++vc)
    {
      T kv[V::S][V::T];
      const T *t = static_cast<const T *>(a.vtab) +
                   (size_t)vc * (V::S * V::T * 64) + lane;
#pragma unroll
      for (int s = 0; s < V::S; ++s)
#pragma unroll
        for (int c = 0; c < V::T; ++c)
          kv[s][c] = t[(s * V::T + c) * 64];
      const unsigned vm = a.vmask[vc];
      int vnb[2 * DV];
#pragma unroll
      for (int s = 0; s < 2 * DV; ++s)
        vnb[s] = neighbour<DV>(vc, a.nv, s);
      // operand forms and inflow faces of the wave's cells, all in flight
      // before the first product; slots beyond the last node are zero
      T uxb[XB][X::SN][V::T], uvb[XB][V::SN][X::T];
      T fxb[XB][X::SF][V::T], fvb[XB][V::SF][X::T];
#pragma unroll
      for (int b = 0; b < XB; ++b)
        {
          const int xc = min(x0 + b, a.nxc - 1);
          const T *u = src + ((long long)vc * a.nxc + xc) * CELL;
          if constexpr (VEC)
            {
              constexpr int W = 16 / sizeof(T);
#pragma unroll
              for (int c = 0; c < V::T; ++c)
#pragma unroll
                for (int k = 0; k < X::SN; k += W)
                  {
                    const Quad16<T> w = *reinterpret_cast<const Quad16<T> *>(
                      u + vcol[c] + slot_node<N, DX>(k, g));
#pragma unroll
                    for (int e = 0; e < W; ++e)
                      uxb[b][k + e][c] = w.v[e];
                  }
            }
          else
            {
#pragma unroll
              for (int s = 0; s < X::SN; ++s)
                {
                  const int x = slot_node<N, DX>(s, g);
#pragma unroll
                  for (int c = 0; c < V::T; ++c)
                    {
                      const T w = u[vcol[c] + min(x, nx - 1)];
                      uxb[b][s][c] = x < nx ? w : T(0);
                    }
                }
            }
#pragma unroll
          for (int s = 0; s < V::SN; ++s)
            {
              const int v = slot_node<N, DV>(s, g);
#pragma unroll
              for (int r = 0; r < X::T; ++r)
                {
                  const T w = u[xrow[r] + min(v, nv - 1) * nx];
                  uvb[b][s][r] = v < nv ? w : T(0);
                }
            }
          // the faces with inflow
#pragma unroll
          for (int s = 0; s < X::SF; ++s)
            if (xm[b] >> s & 1u)
              {
#pragma unroll
                for (int c = 0; c < V::T; ++c)
                  {
                    const T w = u[fxo[b][s] + vcol[c]];
                    fxb[b][s][c] = 4 * s + g < X::faces ? w : T(0);
                  }
              }
#pragma unroll
          for (int s = 0; s < V::SF; ++s)
            if (vm >> s & 1u)
              {
                const int q = min(4 * s + g, V::faces - 1);
                const int side = q / V::nf;
                int nb = vnb[0];
#pragma unroll
                for (int e = 1; e < 2 * DV; ++e)
                  nb = side == e ? vnb[e] : nb;
                const T *f = src + ((long long)nb * a.nxc + xc) * CELL +
                             face_node<N, DV>(side, q % V::nf) * nx;
#pragma unroll
                for (int r = 0; r < X::T; ++r)
                  {
                    const T w = f[xrow[r]];
                    fvb[b][s][r] = 4 * s + g < V::faces ? w : T(0);
                  }
              }
        }
#pragma unroll
      for (int b = 0; b < XB; ++b)
        {
          const int xc = min(x0 + b, a.nxc - 1);
          V4 acc[X::T][V::T];
#pragma unroll
          for (int r = 0; r < X::T; ++r)
#pragma unroll
            for (int c = 0; c < V::T; ++c)
              acc[r][c] = V4{0, 0, 0, 0};
#pragma unroll
          for (int s = 0; s < X::SN; ++s)
#pragma unroll
            for (int r = 0; r < X::T; ++r)
#pragma unroll
              for (int c = 0; c < V::T; ++c)
                acc[r][c] = Frag<T>::mfma(kx[b][s][r], uxb[b][s][c], acc[r][c]);
#pragma unroll
          for (int s = 0; s < V::SN; ++s)
#pragma unroll
            for (int r = 0; r < X::T; ++r)
#pragma unroll
              for (int c = 0; c < V::T; ++c)
                acc[r][c] = Frag<T>::mfma(uvb[b][s][r], kv[s][c], acc[r][c]);
#pragma unroll
          for (int s = 0; s < X::SF; ++s)
            if (xm[b] >> s & 1u)
              {
#pragma unroll
                for (int r = 0; r < X::T; ++r)
#pragma unroll
                  for (int c = 0; c < V::T; ++c)
                    acc[r][c] =
                      Frag<T>::mfma(kx[b][X::SN + s][r], fxb[b][s][c], acc[r][c]);
              }
#pragma unroll
          for (int s = 0; s < V::SF; ++s)
            if (vm >> s & 1u)
              {
#pragma unroll
                for (int r = 0; r < X::T; ++r)
#pragma unroll
                  for (int c = 0; c < V::T; ++c)
                    acc[r][c] =
                      Frag<T>::mfma(fvb[b][s][r], kv[V::SN + s][c], acc[r][c]);
              }
          if (x0 + b >= a.nxc)
            continue;
          const long long g0 = ((long long)vc * a.nxc + xc) * CELL;
#pragma unroll
          for (int c = 0; c < V::T; ++c)
            {
              if (16 * c + j >= nv)
                continue;
#pragma unroll
              for (int r = 0; r < X::T; ++r)
                {
                  // whole tiles: registers 0..3 are contiguous x nodes
                  double so[4];
                  long long at[4];
                  bool in[4];
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    {
                      const int x =
                        16 * r + row_node<T, VEC>(result_row<T>(e, g));
                      in[e] = x < nx;
                      at[e] = g0 + vcol[c] + x;
                    }
                  if constexpr (MODE == 0)
                    {
                      if constexpr (VEC)
                        {
                          constexpr int W = 16 / sizeof(T);
#pragma unroll
                          for (int k = 0; k < 4; k += W)
                            {
                              typedef T VW
                                __attribute__((ext_vector_type(W)));
                              VW w;
#pragma unroll
                              for (int e = 0; e < W; ++e)
                                w[e] = acc[r][c][k + e];
                              __builtin_nontemporal_store(
                                w, reinterpret_cast<VW *>(dst + at[k]));
                            }
                        }
                      else
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                          if (in[e])
                            dst[at[e]] = acc[r][c][e];
                    }
                  else
                    {
                      // (FP64: the input's own values where the solution
                      // is the input, or is recovered from it)
                      const bool input =
                        sizeof(T) == 8 && stage.keep == kSolInput;
#pragma unroll
                      for (int e = 0; e < 4; ++e)
                        if (in[e])
                          so[e] = input ? (double)src[at[e]]
                                        : stage.sol[at[e]];
                      if (sizeof(T) == 8 && stage.recover != 0.0)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                          if (in[e])
                            so[e] = stage_solution(stage, so[e],
                                                   (double)src[at[e]]);
                      if (sizeof(T) == 4 || stage.keep == kSolUpdate)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                          if (in[e])
                            stage.sol[at[e]] =
                              so[e] + stage.b_dt * (double)acc[r][c][e];
                      if (stage.ti_out)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                          if (in[e])
                            static_cast<T *>(stage.ti_out)[at[e]] =
                              (T)(so[e] + stage.a_dt * (double)acc[r][c][e]);
                    }
                }
            }
        }
    }
}

// x cells per wave: they share the v coefficients' loads and find each
// other's x faces in L1.  At 2+2, k = 3, 24^4 cells (FP64 / FP32 apply):
// one 490 / 223, two 457 / 208, three 434 / 200 us, four leave two waves per
// SIMD and measured 451 / 219.  Padded tiles (k = 2: two, 264 us, three
// 275) and several tiles per space (k = 4: one, 998 us) hold fewer.
template <int N, int DX, int DV>
constexpr int kXB = Space<N, DX>::T * Space<N, DV>::T > 1 ? 1
                    : Space<N, DX>::kVec                  ? 3
                                                          : 2;

template <int N, int DX, int DV, class T>
hipError_t launch(int mode, const T *src, T *dst, const CurvedDev &cv,
                  const MeshDev &mesh, const StageDev &stage,
                  hipStream_t stream)
{
  constexpr int XB = kXB<N, DX, DV>;
  Args a{};
  a.xtab = sizeof(T) == 8 ? (const void *)cv.xtab64 : (const void *)cv.xtab32;
  a.vtab = sizeof(T) == 8 ? (const void *)cv.vtab64 : (const void *)cv.vtab32;
  a.xmask = cv.xmask;
  a.vmask = cv.vmask;
  a.nxc = a.nvc = 1;
  for (int d = 0; d < 3; ++d)
    {
      a.nx[d] = d < DX ? mesh.n[d] : 1;
      a.nv[d] = d < DV ? mesh.n[DX + d] : 1;
      a.nxc *= a.nx[d];
      a.nvc *= a.nv[d];
    }
  a.xgroups = (a.nxc + kWaves * XB - 1) / (kWaves * XB);
  // v cells per unit: enough that the x coefficients are loaded seldom, few
  // enough for several rounds of blocks on 256 compute units
  a.chunk = (int)std::clamp<long long>((long long)a.xgroups * a.nvc / 4096, 1,
                                       8);
  a.units = (long long)a.xgroups * ((a.nvc + a.chunk - 1) / a.chunk);
  const dim3 grid(8u * (unsigned)((a.units + 7) / 8));
  if (mode == 0)
    hipLaunchKernelGGL((curved_kernel<N, DX, DV, T, 0, XB>), grid,
                       dim3(kBlock), 0, stream, src, dst, a, stage);
  else
    hipLaunchKernelGGL((curved_kernel<N, DX, DV, T, 1, XB>), grid,
                       dim3(kBlock), 0, stream, src, dst, a, stage);
  return hipGetLastError();
}

// the dense per-cell matrices in the order the kernel's lanes read them, and
// the face-step masks
template <int N, int DIM, class T, bool XROWS>
void pack(const std::vector<double> &K, const std::vector<double> &B,
          long long cells, std::vector<T> &tab, std::vector<unsigned> &mask)
{
  using S = Space<N, DIM>;
  constexpr int kSelf = S::SN * S::T * 64, kAll = S::S * S::T * 64;
  // where each entry of a cell's table comes from (K, then B; -1: padding)
  std::vector<int> from(kAll, -1);
  for (int s = 0; s < S::S; ++s)
    for (int r = 0; r < S::T; ++r)
      for (int l = 0; l < 64; ++l)
        {
          const int j = l % 16, g = l / 16;
          const int row = 16 * r + (XROWS ? row_node<T, S::kVec>(j) : j);
          const int col =
            s < S::SN ? slot_node<N, DIM>(s, g) : 4 * (s - S::SN) + g;
          const int cols = s < S::SN ? S::n : S::faces;
          if (row < S::n && col < cols)
            from[(s * S::T + r) * 64 + l] = row * cols + col;
        }
  tab.resize((size_t)cells * kAll);
  mask.assign((size_t)cells, 0u);
  for (long long c = 0; c < cells; ++c)
    {
      T *t = &tab[(size_t)c * kAll];
      const double *k = &K[(size_t)c * S::n * S::n];
      const double *f = &B[(size_t)c * S::n * S::faces];
      for (int e = 0; e < kSelf; ++e)
        t[e] = from[e] < 0 ? T(0) : (T)k[from[e]];
      for (int s = 0; s < S::SF; ++s)
        {
          bool any = false;
          for (int e = kSelf + s * S::T * 64; e < kSelf + (s + 1) * S::T * 64;
               ++e)
            {
              const double v = from[e] < 0 ? 0.0 : f[from[e]];
              any = any || v != 0.0;
              t[e] = (T)v;
            }
          mask[c] |= any ? 1u << s : 0u;
        }
    }
}

template <class T>
hipError_t upload(const std::vector<T> &v, T **dev)
{
  hipError_t e = hipMalloc(reinterpret_cast<void **>(dev),
                           v.size() * sizeof(T));
  if (e == hipSuccess)
    e = hipMemcpy(*dev, v.data(), v.size() * sizeof(T),
                  hipMemcpyHostToDevice);
  return e;
}

template <int N, int DIM, bool XROWS>
hipError_t create_space(const std::vector<double> &K,
                        const std::vector<double> &B, long long cells,
                        double **tab64, float **tab32, unsigned **mask)
{
  std::vector<double> t64;
  std::vector<float> t32;
  std::vector<unsigned> m;
  pack<N, DIM, float, XROWS>(K, B, cells, t32, m);
  pack<N, DIM, double, XROWS>(K, B, cells, t64, m);
  hipError_t e = upload(t64, tab64);
  if (e == hipSuccess)
    e = upload(t32, tab32);
  if (e == hipSuccess)
    e = upload(m, mask);
  return e;
}

template <bool XROWS>
hipError_t create_space_dispatch(int N, int dim, const std::vector<double> &K,
                                 const std::vector<double> &B,
                                 long long cells, double **tab64,
                                 float **tab32, unsigned **mask)
{
#define HD_CV(NN, DD)                                                        \
  if (N == NN && dim == DD)                                                  \
    return create_space<NN, DD, XROWS>(K, B, cells, tab64, tab32, mask);
  HD_CV(2, 1) HD_CV(3, 1) HD_CV(4, 1) HD_CV(5, 1)
  HD_CV(2, 2) HD_CV(3, 2) HD_CV(4, 2) HD_CV(5, 2)
#undef HD_CV
  return hipErrorInvalidValue;
}

template <class T>
hipError_t dispatch(int dx, int dv, int N, int mode, const T *src, T *dst,
                    const CurvedDev &cv, const MeshDev &mesh,
                    const StageDev &stage, hipStream_t stream)
{
#define HD_CV(NN, A, B)                                                      \
  if (N == NN && dx == A && dv == B)                                         \
    return launch<NN, A, B, T>(mode, src, dst, cv, mesh, stage, stream);
  HD_CV(2, 1, 1) HD_CV(3, 1, 1) HD_CV(4, 1, 1) HD_CV(5, 1, 1)
  HD_CV(2, 2, 1) HD_CV(3, 2, 1) HD_CV(4, 2, 1) HD_CV(5, 2, 1)
  HD_CV(2, 1, 2) HD_CV(3, 1, 2) HD_CV(4, 1, 2) HD_CV(5, 1, 2)
  HD_CV(2, 2, 2) HD_CV(3, 2, 2) HD_CV(4, 2, 2) HD_CV(5, 2, 2)
#undef HD_CV
  return hipErrorInvalidValue;
}
} // namespace curved

// Degrees 1..4 in one and two dimensions per space: beyond that the padded
// products outweigh what the quadrature kernel spends.  The tables of a space
// stay within 64 MB per precision (16,384 cells at k = 3 in 2D), so that
// they are small beside the vectors and cheap to build.
bool curved_supported(int dim_x, int dim_v, int N, long long n_x_cells,
                      long long n_v_cells)
{
  if (dim_x > 2 || dim_v > 2 || N < 2 || N > 5)
    return false;
  for (int s = 0; s < 2; ++s)
    {
      const int dim = s ? dim_v : dim_x;
      const long long n = ipow(N, dim), f = 2 * dim * ipow(N, dim - 1);
      const long long bytes =
        ((n + 3) / 4 + (f + 3) / 4) * ((n + 15) / 16) * 64 * 8;
      if (bytes * (s ? n_v_cells : n_x_cells) > (64LL << 20))
        return false;
    }
  return true;
}

// Where this form is faster than the quadrature kernel.  Up to 50,000 cells it
// always is: the other one is bound by latency there (1+1, k = 1 apply 18 us
// from the smallest to 220^2 cells, here 8 to 17).  Above, tiles of 16 x 16
// that a cell of 2 x 2 values leaves empty cost more than the other kernel's
// passes, and a stage's accesses, element by element where nodes do not fill a
// tile, cost more than its arithmetic saves.  us for this form and the other,
// 1+1 FP64 steps: k = 1 270^2 cells 121 and 114, k = 2 800^2 956 and 952, k = 4
// 500^2 671 and 792, 1100^2 3837 and 3673; FP32 steps: k = 2 270^2 146 and 173,
// 330^2 210 and 182, k = 3 270^2 174 and 177, 420^2 440 and 324, k = 4 500^2
// 690 and 704, 800^2 1635 and 1602; FP32 apply k = 2 800^2 122 and 125, 1100^2
// 226 and 217.  k = 1 FP32 steps: 2+1 40^3 166 and 245, 50^3 302 and 286; 1+2
// 100^3 1505 and 1518, 140^3 4551 and 4096.  All else: faster throughout.
bool curved_faster(int dim_x, int dim_v, int N, long long cells, bool fp64,
                   bool stage)
{
  if (cells <= 50000)
    return true;
  if (dim_x + dim_v == 2)
    {
      if (N == 2)
        return false;
      if (!stage)
        return fp64 || N > 3 || cells <= 600000;
      if (fp64)
        return N == 4 || cells <= 500000;
      return cells <= (N == 5 ? 250000 : 75000);
    }
  if (dim_x + dim_v == 3 && N == 2 && stage && !fp64)
    return cells <= (dim_x == 1 ? 1000000 : 100000);
  return true;
}

hipError_t curved_create(int dim_x, int dim_v, int N, const CurvedHost &x,
                         const CurvedHost &v, CurvedDev *out)
{
  hipError_t e = curved::create_space_dispatch<true>(
    N, dim_x, x.K, x.B, x.cells, &out->xtab64, &out->xtab32, &out->xmask);
  if (e == hipSuccess)
    e = curved::create_space_dispatch<false>(N, dim_v, v.K, v.B, v.cells,
                                             &out->vtab64, &out->vtab32,
                                             &out->vmask);
  if (e != hipSuccess)
    curved_destroy(*out);
  return e;
}

void curved_destroy(CurvedDev &c)
{
  for (void *p : {(void *)c.xtab64, (void *)c.vtab64, (void *)c.xtab32,
                  (void *)c.vtab32, (void *)c.xmask, (void *)c.vmask})
    if (p)
      (void)hipFree(p);
  c = CurvedDev{};
}

hipError_t curved_apply_f64(int dim_x, int dim_v, int N, int mode,
                            const double *src, double *dst,
                            const CurvedDev &cv, const MeshDev &mesh,
                            const StageDev &stage, hipStream_t stream)
{
  return curved::dispatch<double>(dim_x, dim_v, N, mode, src, dst, cv, mesh,
                                  stage, stream);
}

hipError_t curved_apply_f32(int dim_x, int dim_v, int N, int mode,
                            const float *src, float *dst, const CurvedDev &cv,
                            const MeshDev &mesh, const StageDev &stage,
                            hipStream_t stream)
{
  return curved::dispatch<float>(dim_x, dim_v, N, mode, src, dst, cv, mesh,
                                 stage, stream);
}
} // namespace hd
