// hd_cres.hip -- the collapsed apply and LSRK stage of 3+3 cells that do not
// fit LDS (k = 4, 5: 5^6 and 6^6 values), in one pass (gfx950).
//
// The collapsed operator (see hd_collapsed.hip) is a sum of 1D operators, one
// per direction.  A block works on one cell at a time (k = 5 in FP64: two
// blocks share a cell, every other output plane each; few cells: a block per
// plane); the cell's result
// lives in the block's registers and the input streams through LDS one chunk
// of fixed i5 (N^5 values) at a time:
//   - thread t owns the chunk's values e = t + m BLOCK and the results
//     (e, i5) of the block's planes: loading its values it adds
//     A5[i5][j] u(e) to all of them and writes the values into U (LDS);
//   - directions 0 to 4, one per phase: a thread reads its lines from U and
//     adds the line's sums to R (LDS);
//   - the owners add R to plane j of their results.
// The inflow faces of d < 5 go from L2 / HBM into registers of the threads
// that use them, one phase ahead; that of direction 5 enters as one more
// input plane.
//
// What bounds it: the fabric.  Every value is read once and written once,
// plus one cell's worth of faces (24 bytes per value for the FP64 apply, 12
// for FP32; the second block's reads of a cell hit the XCD's L2); beside it
// 16 LDS accesses and 42 multiply-adds per value.  Measured, 6^6 cells: k = 5
// FP64 apply 20.9 -> 12.1 ms (the two-pass split form moved 48 bytes per
// value), FP32 11.1 -> 6.6 ms (lines read by every point they pass, 30 LDS
// accesses), k = 4 FP64 8.6 -> 4.3, FP32 4.5 -> 2.2 ms.  N x N tiles of two
// directions per phase instead of lines (14 LDS accesses, three phases) need
// 40 more registers: FP32 7.4 ms, FP64 spills (13.5 to 60 ms).
//
// Blocks of an XCD take consecutive cells in step, so that the faces across
// x0 and x1, whose values are spread over every line of the neighbour, hit
// its L2.
#include "hd_device.h"

#include <algorithm>
#include <type_traits>

namespace hd
{
namespace cres
{
template <class T>
using cptr = const __attribute__((address_space(4))) T *;
template <class T>
using gptr = __attribute__((address_space(1))) T *;

// orders LDS accesses without draining the loads in flight
__device__ inline void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  __builtin_amdgcn_sched_barrier(0);
}

// HALVES blocks share a cell, BLOCK threads, WAVES per SIMD (the register
// budget 512 / WAVES).  Measured, 6^6 cells, apply: k = 5 FP64 two blocks of
// 1024 threads 12.1, 768 12.5, 512 13.4 ms, one block (192 registers of
// results) spills, 26 ms; FP32 one block of 1024 threads 6.6, 768 7.1, 512
// 7.5, two blocks of 512 6.9 ms; k = 4 FP64 256 threads 4.3, 512 4.7, FP32
// 256 threads 2.24, 512 2.43 ms (two or three blocks per CU overlap their
// phases)
template <int N, class T>
struct Geo;
template <>
struct Geo<6, double>
{
  static constexpr int HALVES = 2, BLOCK = 1024, WAVES = 4;
};
template <>
struct Geo<6, float>
{
  static constexpr int HALVES = 1, BLOCK = 1024, WAVES = 4;
};
template <>
struct Geo<5, double>
{
  static constexpr int HALVES = 1, BLOCK = 256, WAVES = 2;
};
template <>
struct Geo<5, float>
{
  static constexpr int HALVES = 1, BLOCK = 256, WAVES = 3;
};

template <int N, class T, int MODE, int HALVES>
__global__ __launch_bounds__((Geo<N, T>::BLOCK), (Geo<N, T>::WAVES)) void
  cres_kernel(const T *__restrict__ src_, T *__restrict__ dst_,
              const T *__restrict__ coef, MeshDev mesh, InflowDev inflow,
              StageDev stage)
{
  using G = Geo<N, T>;
  constexpr int BLOCK = G::BLOCK;
  constexpr int NN = N * N, P = NN * NN, CH = P * N;
  constexpr long long CELL = (long long)CH * N;
  constexpr int M = (CH + BLOCK - 1) / BLOCK;   // owned values per chunk
  constexpr int KL = (P + BLOCK - 1) / BLOCK;   // lines per thread
  __shared__ __align__(16) T U[CH], R[CH];

  const gptr<const T> src = (gptr<const T>)src_;
  const gptr<T> dst = (gptr<T>)dst_;
  const gptr<double> sol = (gptr<double>)stage.sol;
  const gptr<T> ti_out = (gptr<T>)static_cast<T *>(stage.ti_out);
  cptr<T> cc = (cptr<T>)coef;
  constexpr int DC = NN + N; // coefficients per direction: A_d, b_d
  int fnode[6];
#pragma unroll
  for (int d = 0; d < 6; ++d)
    fnode[d] = inflow.side[d] < 0 ? 0 : N - 1;

  // consecutive cells per XCD (blocks are dispatched round-robin over them);
  // HALVES blocks share a cell: block h keeps the planes i5 = h, h + HALVES,
  // .. and takes the other planes of the input for direction 5 only, from
  // the L2 that the other blocks' loads have filled (step is a multiple of
  // HALVES, so h is the block's own)
  constexpr int NPL = (N + HALVES - 1) / HALVES;
  static_assert(N % HALVES == 0, "planes per block");
  const long long per = (mesh.n_cells + 7) / 8 * HALVES;
  const long long u_end =
    min(mesh.n_cells * HALVES, (long long)(blockIdx.x % 8 + 1) * per);
  const int step = gridDim.x / 8;
  long long unit = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (unit >= u_end)
    return; // uniform for the block, before any barrier
  const int h = (int)(unit % HALVES);

  // the lane index, made opaque per phase: addresses derived from it are
  // recomputed instead of held in registers across the chunk loop
  auto lane = [&]() {
    unsigned t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  auto values = [&](gptr<const T> from, T *v) {
    const unsigned t = lane();
#pragma unroll
    for (int m = 0; m < M; ++m)
      {
        // (uniform base, 32-bit lane offset)
        const gptr<const T> base = from + m * BLOCK;
        const unsigned e =
          m + 1 < M ? t : min(t, (unsigned)(CH - 1 - m * BLOCK));
        v[m] = base[e];
      }
  };

  typedef T Planes __attribute__((ext_vector_type(NPL)));
  Planes acc[M];
  T pu[M]; // the next chunk's own values
  values(src + unit / HALVES * CELL, pu);
  for (; unit < u_end; unit += step)
    {
      const long long cell = unit / HALVES;
      long long nb[6];
#pragma unroll
      for (int d = 0; d < 6; ++d)
        nb[d] = inflow_neighbour(mesh, cell, d, inflow.side[d]);
      {
        // the inflow face across direction 5: one more input plane
        const cptr<T> b5 = cc + 5 * DC + NN;
        const unsigned t = lane();
        const gptr<const T> s5 = src + nb[5] * CELL + (long long)CH * fnode[5];
#pragma unroll
        for (int m0 = 0; m0 < M; m0 += 4)
          {
            // four values in flight at a time (registers)
            T f5[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (m0 + e < M)
                {
                  constexpr int last = CH - 1 - (M - 1) * BLOCK;
                  const gptr<const T> base = s5 + (m0 + e) * BLOCK;
                  f5[e] =
                    base[m0 + e + 1 < M ? t : min(t, (unsigned)last)];
                }
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (m0 + e < M)
#pragma unroll
                for (int i = 0; i < NPL; ++i)
                  acc[m0 + e < M ? m0 + e : M - 1][i] =
                    b5[h + HALVES * i] * f5[e];
          }
      }
      for (int j = 0; j < N; ++j)
        {
          asm volatile("" : "+s"(cc));
          // the inflow values of this thread's lines along d, and the lines:
          // sums into R (d = 0) or added
          auto line_faces = [&](auto dc, T *f) {
            constexpr int d = decltype(dc)::value, sd = ipow(N, d);
            const unsigned t = lane();
            const gptr<const T> s =
              src + nb[d] * CELL + (long long)CH * j + fnode[d] * sd;
#pragma unroll
            for (int k = 0; k < KL; ++k)
              {
                const unsigned l = min(t + k * BLOCK, (unsigned)(P - 1));
                f[k] = s[l % sd + l / sd * (unsigned)(sd * N)];
              }
          };
          auto lines = [&](auto dc, const T *f) {
            constexpr int d = decltype(dc)::value, sd = ipow(N, d);
            const unsigned t = lane();
            const cptr<T> A = cc + d * DC, bv = A + NN;
#pragma unroll
            for (int k = 0; k < KL; ++k)
              {
                const unsigned l = t + k * BLOCK;
                if (P % BLOCK != 0 && k + 1 == KL && l >= P)
                  continue;
                const unsigned base = l % sd + l / sd * (unsigned)(sd * N);
                T u[N];
#pragma unroll
                for (int i = 0; i < N; ++i)
                  u[i] = U[base + i * sd];
#pragma unroll
                for (int i = 0; i < N; ++i)
                  {
                    T s = bv[i] * f[k];
#pragma unroll
                    for (int q = 0; q < N; ++q)
                      s += A[i * N + q] * u[q];
                    T *r = &R[base + i * sd];
                    *r = d == 0 ? s : *r + s;
                  }
              }
          };
          using D0 = std::integral_constant<int, 0>;
          using D1 = std::integral_constant<int, 1>;
          using D2 = std::integral_constant<int, 2>;
          using D3 = std::integral_constant<int, 3>;
          using D4 = std::integral_constant<int, 4>;

          // 1) own values: direction 5, and into U
          const bool mine = HALVES == 1 || j % HALVES == h;
          T f0[KL], f1[KL];
          if (mine)
            line_faces(D0(), f0);
          {
            const unsigned t = lane();
            const cptr<T> A5 = cc + 5 * DC + j + h * N;
#pragma unroll
            for (int m = 0; m < M; ++m)
              {
#pragma unroll
                for (int i = 0; i < NPL; ++i)
                  acc[m][i] += A5[i * HALVES * N] * pu[m];
                if (mine &&
                    (CH % BLOCK == 0 || m + 1 < M || t + m * BLOCK < CH))
                  U[t + m * BLOCK] = pu[m];
              }
          }
          // the next chunk: of this cell, or the next cell's first
          const long long nc =
            j + 1 < N ? cell
                      : (unit + step < u_end ? (unit + step) / HALVES : cell);
          const gptr<const T> next =
            src + nc * CELL + (long long)CH * (j + 1 < N ? j + 1 : 0);
          if (!mine)
            {
              values(next, pu);
              continue;
            }
          lds_barrier();
          values(next, pu);
          // 2) the lines of directions 0 to 3, the faces one ahead
          line_faces(D1(), f1);
          lines(D0(), f0);
          lds_barrier();
          line_faces(D2(), f0);
          lines(D1(), f1);
          lds_barrier();
          line_faces(D3(), f1);
          lines(D2(), f0);
          lds_barrier();
          line_faces(D4(), f0);
          lines(D3(), f1);
          lds_barrier();
          lines(D4(), f0);
          lds_barrier();
          // 3) the chunk's sums into plane j (the next chunk's U may be
          // written meanwhile: nobody reads U before the next barrier)
          {
            const unsigned t = lane();
            // (j is uniform: plane j of a register vector is one indexed
            // access; a switch over j kept two copies of every result)
#pragma unroll
            for (int m = 0; m < M; ++m)
              if (CH % BLOCK == 0 || m + 1 < M || t + m * BLOCK < CH)
                acc[m][j / HALVES] += R[t + m * BLOCK];
          }
        }
      // the results (e, i5): coalesced, not read again by this kernel
      const unsigned t = lane();
#pragma unroll
      for (int m = 0; m < M; ++m)
        {
          if (!(CH % BLOCK == 0 || m + 1 < M || t + m * BLOCK < CH))
            continue;
          constexpr bool kReadsSol = MODE != 0 && MODE != 3;
          constexpr bool kOwn = MODE == 3 || MODE == 5 || MODE == 6;
          double so[kReadsSol ? NPL : 1], own[kOwn ? NPL : 1];
#pragma unroll
          for (int i = 0; i < NPL; ++i)
            {
              const long long g = cell * CELL + m * BLOCK +
                                  (long long)CH * (h + HALVES * i);
              if constexpr (kReadsSol)
                so[i] = (sol + g)[t];
              if constexpr (kOwn)
                own[i] = (double)(src + g)[t];
            }
#pragma unroll
          for (int i = 0; i < NPL; ++i)
            {
              const long long g = cell * CELL + m * BLOCK +
                                  (long long)CH * (h + HALVES * i);
              const T k = acc[m][i];
              if constexpr (MODE == 0)
                __builtin_nontemporal_store(k, &(dst + g)[t]);
              else
                {
                  double s;
                  if constexpr (MODE == 3)
                    s = own[i];
                  else if constexpr (MODE == 5 || MODE == 6)
                    s = so[i] + stage.recover * (own[i] - so[i]);
                  else
                    s = so[i];
                  if constexpr (kReadsSol && MODE != 4)
                    __builtin_nontemporal_store(s + stage.b_dt * (double)k,
                                                &(sol + g)[t]);
                  if constexpr (MODE != 2 && MODE != 6)
                    __builtin_nontemporal_store(
                      (T)(s + stage.a_dt * (double)k), &(ti_out + g)[t]);
                }
            }
        }
    }
}

template <int N, class T>
hipError_t launch(int mode, const T *src, T *dst, const T *coef,
                  const MeshDev &mesh, const InflowDev &inflow,
                  const StageDev &stage, hipStream_t stream)
{
  using G = Geo<N, T>;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                            dev) != hipSuccess ||
      cus < 8)
    cus = 256;
  // as many persistent blocks as are resident, a multiple of the XCDs
  auto resident = [&](auto kernel) {
    int bpc = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, kernel, G::BLOCK,
                                                     0) != hipSuccess ||
        bpc < 1)
      bpc = 1;
    return (long long)cus * bpc;
  };
  auto start = [&](auto kernel, int halves, long long blocks) {
    const long long most = (mesh.n_cells + 7) / 8 * 8 * halves;
    const unsigned grid = (unsigned)std::min<long long>(
      most, blocks / (8 * halves) * (8 * halves));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(G::BLOCK), 0, stream, src,
                       dst, coef, mesh, inflow, stage);
    return hipGetLastError();
  };
  // Few cells: a block per output plane, as long as all are resident at once
  // (a cell's N chunks one after the other are what a small mesh waits for).
  // us for an apply, the two-pass split form, a cell per block (k = 5 FP64: two
  // blocks) and a plane per block: k = 4 FP64 1 cell 17, 32, 12, 96 cells 28,
  // 33, 16; k = 4 FP32 1 cell -, 24, 9.5; k = 5 FP64 1 cell 25, 31, 19, 16 cells
  // 28, 32, 20; k = 5 FP32 1 cell -, 36, 13.  With more cells than that a plane
  // per block reads every input value N times from L2.
  auto go = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
    const auto planes = cres_kernel<N, T, MODE, N>;
    const long long blocks = resident(planes);
    if (mesh.n_cells * N <= blocks)
      return start(planes, N, blocks);
    const auto cells = cres_kernel<N, T, MODE, G::HALVES>;
    return start(cells, G::HALVES, resident(cells));
  };
  using std::integral_constant;
  if (mode == 0)
    return go(integral_constant<int, 0>());
  if constexpr (sizeof(T) == 8)
    {
      if (stage.keep == kSolInput)
        return go(integral_constant<int, 3>());
      if (stage.keep == kSolKeep)
        return go(integral_constant<int, 4>());
      if (stage.recover != 0.0)
        return stage.ti_out ? go(integral_constant<int, 5>())
                            : go(integral_constant<int, 6>());
    }
  return stage.ti_out ? go(integral_constant<int, 1>())
                      : go(integral_constant<int, 2>());
}
} // namespace cres

bool collapsed_cres_supported(int D, int N)
{
  return D == 6 && (N == 5 || N == 6);
}

hipError_t collapsed_cres_f64(int N, int mode, const double *src, double *dst,
                              const double *coef, const MeshDev &mesh,
                              const InflowDev &inflow, const StageDev &stage,
                              hipStream_t stream)
{
  return N == 5 ? cres::launch<5>(mode, src, dst, coef, mesh, inflow, stage,
                                  stream)
                : cres::launch<6>(mode, src, dst, coef, mesh, inflow, stage,
                                  stream);
}

hipError_t collapsed_cres_f32(int N, int mode, const float *src, float *dst,
                              const float *coef, const MeshDev &mesh,
                              const InflowDev &inflow, const StageDev &stage,
                              hipStream_t stream)
{
  return N == 5 ? cres::launch<5>(mode, src, dst, coef, mesh, inflow, stage,
                                  stream)
                : cres::launch<6>(mode, src, dst, coef, mesh, inflow, stage,
                                  stream);
}
} // namespace hd
