// hd_vpcg.hip -- the periodic 2D potential solve on several compute units,
// gfx950: the same system, start, stopping rule and outputs as the
// one-workgroup solver (poisson2d_kernel in hd_vlasov.hip), with the x mesh
// cut into strips of cell rows, one workgroup each.
//
// What bounds a solve is the latency of an iteration: on one workgroup a
// matrix-vector product of 32^2 cells at k = 3 is 2,100 vector instructions
// per wave on four SIMDs, 11 us per iteration.  Spread over 32 workgroups
// the product takes about 0.3 us and an iteration is one exchange between
// workgroups.  Conjugate gradients in the form of Chronopoulos and Gear (1989)
// needs a single reduction per iteration: with r known everywhere it is
// needed, w = A r, the sums (r, r) and (w, r) and the rows of w that the
// neighbouring strips need travel together, and every workgroup updates its
// own rows of p, s, x, r and its copy of the neighbours' rows of s and r by
// the same recurrences.
//
// A has the constants as its null space.  CG cannot lower the mean that
// rounding leaves in r, and once r is no larger than that, steps along the
// constants (den near 0) make r grow without bound: at 4 x 96 cells, k = 3
// and a tolerance of 1e-13, below the 2e-11 that b - A x reaches in 64 bits,
// solves ended at 1e-5.  So r's mean is removed every kProject iterations;
// b - A x then stays where it is for any tolerance.
//
// The exchange.  Every value has a slot of its own in the receiving
// workgroup's inbox (relaxed agent-scope 8-byte atomics, which the level-2
// caches of the XCDs do not hold back); an empty slot holds kEmpty, a NaN
// that no result is (a result with its bits is replaced by another NaN).  The
// receiver polls the slot, takes the value and empties the slot, so no flag
// and no fence is needed.  Slots alternate between two sets: a set is
// written again two exchanges later, after the writer has received values
// that the reader sent after it emptied the set (the reader waits for its
// stores and passes a workgroup barrier before it sends).  A poll is bounded:
// a workgroup that waits too long (others not scheduled) leaves and marks
// the launch, whose work the small kernel launched behind this one then does
// on its own; without the mark it returns at once.
//
// Measured (MI355X, k = 3, field updates of 393 iterations): 11.0 -> 3.1 us per
// iteration at 32^2 x cells, 4.1 us before the sums went through lane
// permutations and the stores that empty slots overlapped the product; the
// check of an exact start 94 -> 12 us.
#include "hd_device.h"

#include <algorithm>
#include <type_traits>

namespace hd
{
namespace vpcg
{
constexpr int kThreads = 512;
constexpr int kMaxStrips = 32;
constexpr int kSums = 8; // most sums of one exchange
constexpr unsigned long long kEmpty = ~0ull;
constexpr int kMaxPolls = 1 << 18; // about 0.2 s, once per exchange
// iterations between removals of r's mean (one more exchange; restated on the
// CPU, every iteration to every 64th end at the same residuals.  As a third sum
// of every 16th exchange it cost every iteration 8 %, 3.13 -> 3.38 us at 32^2
// cells)
constexpr int kProject = 64;

template <class T>
using cptr = const __attribute__((address_space(4))) T *;

struct Strips
{
  int count, rows;            // strips, rows per strip (the last may be less)
  unsigned long long *row_in; // [2][strip][2][n0 NN]
  unsigned long long *sum_in; // [2][strip][strip][kSums]
  int *mark;                  // 1: a workgroup gave up
};

__device__ inline void send(unsigned long long *slot, double v)
{
  unsigned long long b = __double_as_longlong(v);
  if (b == kEmpty)
    b = 0x7ff8000000000000ull;
  __hip_atomic_store(slot, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline bool receive(unsigned long long *slot, double &v)
{
  unsigned long long b = kEmpty;
  for (int i = 0; i < kMaxPolls; ++i)
    {
      b = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (b != kEmpty)
        break;
    }
  v = __longlong_as_double(b);
  __hip_atomic_store(slot, kEmpty, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  return b != kEmpty;
}

// Orders the workgroup's LDS accesses; the stores that empty slots may be in
// flight across it.
__device__ inline void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int ctrl>
__device__ inline double dpp_add(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, ctrl, 0xf, 0xf, true);
  const int hi =
    __builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, 0xf, 0xf, true);
  return v + __longlong_as_double(((long long)hi << 32) |
                                  (unsigned long long)(unsigned)lo);
}
// the sum over each row of 16 lanes, in every lane of the row (in-register
// lane permutations: a shuffle through LDS takes ten times their latency)
__device__ inline double row_sum(double v)
{
  v = dpp_add<0xb1>(v);  // lanes 1 0 3 2
  v = dpp_add<0x4e>(v);  // lanes 2 3 0 1
  v = dpp_add<0x141>(v); // half row mirrored
  return dpp_add<0x140>(v); // row mirrored
}
__device__ inline double lane_value(double v, int lane)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) |
                              (unsigned long long)(unsigned)lo);
}

// NPT nodes per thread: thread t < T owns the strip's nodes t + k T (T a
// multiple of the nodes per cell, so that a thread's nodes have one place in
// their cells)
template <int N, int NPT>
__global__ __launch_bounds__(kThreads) void strip_kernel(
  XDev xd, const double *__restrict__ tab, const double *__restrict__ rho,
  double *__restrict__ phi, const double *__restrict__ guess,
  double *__restrict__ efield, Strips st, double rel_tol, int max_it,
  long long *__restrict__ stats, int guess_alone,
  float *__restrict__ res_image, double *__restrict__ res_scale,
  double *__restrict__ phi_copy, GuessImage guess_image)
{
  constexpr int NN = N * N, T = kThreads / NN * NN;
  extern __shared__ double sm[];
  const int n0 = xd.n[0], n1 = xd.n[1], W = n0 * NN; // values per row
  const int sb = blockIdx.x, t = threadIdx.x;
  const int y0 = sb * st.rows, nr = min(st.rows, n1 - y0);
  const int n_own = nr * W;
  const int below = (sb + st.count - 1) % st.count, above = (sb + 1) % st.count;
  double *rL = sm;                   // rows y0 - 1 .. y0 + nr, W values each
  double *z0 = rL + (st.rows + 2) * W, *z1 = z0 + st.rows * W;
  double *red = z1 + st.rows * W;    // wave sums: 8 x kSums
  double *got = red + 8 * kSums;     // the sums over all strips
  __shared__ int lost;
  if (t == 0)
    lost = 0;
  // another workgroup has given up: the kernel behind does the work
  if (*st.mark != 0)
    return;
  // a chain of latencies: its waves go first where a compute unit also works
  // on something else (training beside the solve: 3.7 us per iteration)
  __builtin_amdgcn_s_setprio(3);

  const int node = t % NN, ix = node % N, iy = node / N;
  bool own[NPT], halo[NPT];
  int q[NPT]; // the strip's node, also the node of a halo row
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    {
      q[k] = t + k * T;
      own[k] = t < T && q[k] < n_own;
      halo[k] = t < T && q[k] < W;
      if (!own[k])
        q[k] = t < T && halo[k] ? q[k] : node;
    }
  // this thread's rows of the 1D operators
  double L0[3][N], L1[3][N], M0[N], M1[N], m0 = 0.0, m1 = 0.0;
#pragma unroll
  for (int j = 0; j < N; ++j)
    {
#pragma unroll
      for (int k = 0; k < 3; ++k)
        {
          L0[k][j] = tab[k * NN + ix * N + j];
          L1[k][j] = tab[(3 + k) * NN + iy * N + j];
        }
      M0[j] = tab[6 * NN + ix * N + j];
      M1[j] = tab[7 * NN + iy * N + j];
      m0 += M0[j];
      m1 += M1[j];
    }

  int epoch = 0;
  // sums over all strips of v[0 .. ns), and (rows) the neighbours' adjacent
  // rows of x into h (below, above); false: another workgroup is lost
  auto exchange = [&](auto ns_c, double *v, bool rows, const double *x,
                      double (*h)[NPT]) -> bool {
    constexpr int ns = decltype(ns_c)::value;
    const int par = epoch & 1;
    ++epoch;
    // the slots that the last exchange emptied are empty before anything
    // else is sent: every thread's stores are complete
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (rows)
      {
        // my first row is the row above the strip below, my last one the
        // row below the strip above
#pragma unroll
        for (int k = 0; k < NPT; ++k)
          if (own[k])
            {
              if (q[k] < W)
                send(st.row_in + ((par * st.count + below) * 2 + 1) * W + q[k],
                     x[k]);
              if (q[k] >= n_own - W)
                send(st.row_in + ((par * st.count + above) * 2 + 0) * W +
                       (q[k] - (n_own - W)),
                     x[k]);
            }
      }
#pragma unroll
    for (int s = 0; s < ns; ++s)
      {
        const double a = row_sum(v[s]);
        v[s] = (lane_value(a, 0) + lane_value(a, 16)) +
               (lane_value(a, 32) + lane_value(a, 48));
        if ((t & 63) == 0)
          red[(t >> 6) * kSums + s] = v[s];
      }
    lds_barrier();
    // thread (strip, sum): this strip's sum to that strip's inbox, and that
    // strip's sum from the own inbox
    bool fine = true;
    const int peer = t % kMaxStrips, s = t / kMaxStrips;
    const bool sums_here = s < ns && peer < st.count;
    if (sums_here)
      {
        double a = 0.0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w)
          a += red[w * kSums + s];
        send(st.sum_in + ((par * st.count + peer) * st.count + sb) * kSums + s,
             a);
      }
    if (rows)
      {
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int k = 0; k < NPT; ++k)
            if (halo[k])
              fine = fine && receive(st.row_in +
                                       ((par * st.count + sb) * 2 + d) * W +
                                       q[k],
                                     h[d][k]);
      }
    double a = 0.0;
    if (sums_here)
      fine = fine &&
             receive(st.sum_in +
                       ((par * st.count + sb) * st.count + peer) * kSums + s,
                     a);
    // half a wave holds a sum's terms, one per strip
    if (t < (ns + 1) / 2 * 64)
      {
        a = row_sum(a);
        const double lo = lane_value(a, 0) + lane_value(a, 16);
        const double hi = lane_value(a, 32) + lane_value(a, 48);
        if (t % kMaxStrips == 0)
          got[s] = t % 64 == 0 ? lo : hi;
      }
    if (!fine)
      lost = 1;
    lds_barrier();
#pragma unroll
    for (int e = 0; e < ns; ++e)
      v[e] = got[e];
    const bool go = lost == 0;
    lds_barrier(); // red, got and lost may be written again
    return go;
  };
  auto give_up = [&]() {
    if (t == 0)
      __hip_atomic_store(st.mark, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  };
  // own rows and halo rows of x(row, value) into rL
  auto load_rows = [&](auto x) {
    for (int e = t; e < (nr + 2) * W; e += kThreads)
      {
        int y = y0 - 1 + e / W;
        y = y < 0 ? y + n1 : (y >= n1 ? y - n1 : y);
        rL[e] = x(y, e % W);
      }
  };
  // the guess; from an image: scale times the mean of the pixels that lie at
  // the node (two on a cell face, four in a corner)
  auto guess_at = [&](int y, int e) -> double {
    if (!guess_image.image)
      return guess[(long long)y * W + e];
    const int c = e / NN, gx = e % N, gy = e % NN / N;
    const int PX = n0 * N, PY = n1 * N, X = c * N + gx, Y = y * N + gy;
    const int x2 = gx == 0       ? (X == 0 ? PX - 1 : X - 1)
                   : gx == N - 1 ? (X == PX - 1 ? 0 : X + 1)
                                 : X;
    const int y2 = gy == 0       ? (Y == 0 ? PY - 1 : Y - 1)
                   : gy == N - 1 ? (Y == PY - 1 ? 0 : Y + 1)
                                 : Y;
    const float *im = guess_image.image;
    double a = (double)im[(long long)Y * PX + X];
    int n = 1;
    if (x2 != X)
      {
        a += (double)im[(long long)Y * PX + x2];
        ++n;
      }
    if (y2 != Y)
      {
        a += (double)im[(long long)y2 * PX + X];
        ++n;
        if (x2 != X)
          {
            a += (double)im[(long long)y2 * PX + x2];
            ++n;
          }
      }
    return *guess_image.scale * a / n;
  };
  // y = A r on the own nodes; r in rL (complete before: a barrier)
  auto product = [&](double *y) {
#pragma unroll
    for (int k = 0; k < NPT; ++k)
      if (own[k])
        {
          const int c = q[k] / NN, row = c / n0, cx = c - row * n0;
          const double *line = rL + (row + 1) * W + iy * N;
          const int xn[3] = {cx == 0 ? n0 - 1 : cx - 1, cx,
                             cx == n0 - 1 ? 0 : cx + 1};
          double a = 0.0, b = 0.0;
#pragma unroll
          for (int e = 0; e < 3; ++e)
#pragma unroll
            for (int j = 0; j < N; ++j)
              {
                a += L0[e][j] * line[xn[e] * NN + j];
                b += L1[e][j] * rL[(row + e) * W + cx * NN + ix + N * j];
              }
          z0[q[k]] = a;
          z1[q[k]] = b;
        }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < NPT; ++k)
      {
        y[k] = 0.0;
        if (own[k])
          {
            const int c = q[k] - node;
#pragma unroll
            for (int j = 0; j < N; ++j)
              y[k] += M1[j] * z0[c + ix + N * j] + M0[j] * z1[c + j + N * iy];
          }
      }
  };
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  using S6 = std::integral_constant<int, 6>;
  const double nx = (double)xd.n_cells * NN;

  // b = -(M_0 (x) M_1)(rho - mean rho), then b -= mean b (its sum from the
  // column sums of the symmetric mass matrices)
  double sums[kSums] = {};
  double b[NPT], x[NPT], r[NPT], w[NPT], p[NPT], s[NPT], h[2][NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      {
        const long long i = (long long)y0 * W + q[k];
        b[k] = rho[i];
        sums[0] += b[k];
        sums[1] += m0 * m1 * b[k];
        if (guess)
          sums[2] += guess_at(y0 + q[k] / W, q[k] % W);
      }
  if (!exchange(S3(), sums, false, b, h))
    return give_up();
  const double mean_rho = sums[0] / nx;
  double msum = 0.0;
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j)
      {
        double a = 0.0, c = 0.0;
        for (int e = 0; e < N; ++e)
          {
            a += tab[6 * NN + i * N + e];
            c += tab[7 * NN + j * N + e];
          }
        msum += a * c;
      }
  const double mean_b =
    -(sums[1] - mean_rho * msum * (double)xd.n_cells) / nx;
  const double mean_g = sums[2] / nx;
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      z0[q[k]] = b[k] - mean_rho;
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      {
        double a = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j)
          a += M0[j] * z0[q[k] - node + j + N * iy];
        z1[q[k]] = a;
      }
  load_rows([&](int y, int e) { return phi[(long long)y * W + e]; });
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    {
      b[k] = 0.0;
      if (own[k])
        {
          double a = 0.0;
#pragma unroll
          for (int j = 0; j < N; ++j)
            a += M1[j] * z1[q[k] - node + ix + N * j];
          b[k] = -a - mean_b;
        }
    }
  lds_barrier(); // z1 is free

  // the start: phi, or its combination with the guess
  double y[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    x[k] = own[k] ? rL[W + q[k]] : 0.0;
  product(y);
  double alpha0 = 1.0, beta0 = 0.0, rr_warm = -1.0;
  if (guess)
    {
      double g[NPT], ag[NPT];
      lds_barrier(); // every thread has read rL and z
      load_rows([&](int y, int e) { return guess_at(y, e) - mean_g; });
      lds_barrier();
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        g[k] = own[k] ? rL[W + q[k]] : 0.0;
      product(ag);
      double d[kSums] = {};
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        if (own[k])
          {
            d[0] += x[k] * y[k];
            d[1] += x[k] * ag[k];
            d[2] += g[k] * ag[k];
            d[3] += x[k] * b[k];
            d[4] += g[k] * b[k];
            d[5] += (b[k] - y[k]) * (b[k] - y[k]);
          }
      if (!exchange(S6(), d, false, b, h))
        return give_up();
      rr_warm = d[5];
      if (guess_alone)
        {
          // an exact guess: the start is the guess itself (a combination
          // with a previous phi that is nearly parallel to it would be an
          // ill-conditioned 2 x 2 system)
          alpha0 = 0.0;
          beta0 = 1.0;
        }
      else
        {
          const double det = d[0] * d[2] - d[1] * d[1];
          if (d[0] > 0.0 && d[2] > 0.0 && det > 1e-12 * d[0] * d[2])
            {
              alpha0 = (d[3] * d[2] - d[4] * d[1]) / det;
              beta0 = (d[0] * d[4] - d[1] * d[3]) / det;
            }
          else if (!(d[0] > 0.0) && d[2] > 0.0)
            {
              alpha0 = 0.0;
              beta0 = d[4] / d[2];
            }
          if (!isfinite(alpha0) || !isfinite(beta0))
            {
              alpha0 = 1.0;
              beta0 = 0.0;
            }
        }
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        {
          // (a guess that is left out may hold NaN)
          x[k] = beta0 == 0.0 ? alpha0 * x[k] : alpha0 * x[k] + beta0 * g[k];
          y[k] = beta0 == 0.0 ? alpha0 * y[k] : alpha0 * y[k] + beta0 * ag[k];
        }
    }
  if (res_image)
    {
      // the residual of the start only (no solve), r = b - A phi, as the
      // image (r - mean r) / rms(r - mean r) of the x nodes (row = x1 node,
      // x0 node fastest) and its scale rms, and a copy of phi
      if (phi_copy)
#pragma unroll
        for (int k = 0; k < NPT; ++k)
          if (own[k])
            phi_copy[(long long)y0 * W + q[k]] = x[k];
      double v[kSums] = {};
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        {
          r[k] = own[k] ? b[k] - y[k] : 0.0;
          v[0] += r[k];
          v[1] += r[k] * r[k];
        }
      if (!exchange(S2(), v, false, r, h))
        return give_up();
      // (b and A phi have no mean: the square of r's is rounding beside the
      // mean square)
      const double mean = v[0] / nx;
      const double rms = sqrt(fmax(v[1] / nx - mean * mean, 0.0));
      const double inv = rms > 0.0 ? 1.0 / rms : 0.0;
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        if (own[k])
          {
            const int c = q[k] / NN, row = c / n0, cx = c - row * n0;
            res_image[((long long)(y0 + row) * N + iy) * (n0 * N) + cx * N +
                      ix] = (float)((r[k] - mean) * inv);
          }
      if (sb == 0 && t == 0)
        *res_scale = rms;
      return;
    }
  sums[0] = sums[1] = 0.0;
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    {
      r[k] = own[k] ? b[k] - y[k] : 0.0;
      sums[0] += r[k] * r[k];
      sums[1] += b[k] * b[k];
    }
  if (!exchange(S2(), sums, true, r, h))
    return give_up();
  double rr = sums[0];
  const double bb = sums[1], rr_start = rr;
  const double stop = rel_tol * sqrt(bb);
  // r and its copies of the neighbours' rows into rL
  double sh[2][NPT];
  auto store_r = [&]() {
#pragma unroll
    for (int k = 0; k < NPT; ++k)
      if (own[k])
        rL[W + q[k]] = r[k];
  };
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    {
      p[k] = s[k] = sh[0][k] = sh[1][k] = 0.0;
      if (halo[k])
        {
          rL[q[k]] = h[0][k];
          rL[(nr + 1) * W + q[k]] = h[1][k];
        }
    }
  store_r();
  int it = 0;
  if (sqrt(rr) > stop && max_it > 0)
    {
      lds_barrier();
      product(w);
      double v[kSums] = {};
#pragma unroll
      for (int k = 0; k < NPT; ++k)
        v[0] += w[k] * r[k];
      if (!exchange(S1(), v, true, w, h))
        return give_up();
      double wr = v[0], alpha = 0.0, beta = 0.0;
      bool go = true;
      while (go && sqrt(rr) > stop && it < max_it)
        {
          const int until = min(max_it, it + kProject);
          while (sqrt(rr) > stop && it < until)
            {
              const double den = it == 0 ? wr : wr - beta * rr / alpha;
              go = den > 0.0;
              if (!go)
                break; // r is rounding
              alpha = rr / den;
#pragma unroll
              for (int k = 0; k < NPT; ++k)
                {
                  p[k] = r[k] + beta * p[k];
                  s[k] = w[k] + beta * s[k];
                  x[k] += alpha * p[k];
                  r[k] -= alpha * s[k];
                  if (halo[k])
                    {
                      sh[0][k] = h[0][k] + beta * sh[0][k];
                      sh[1][k] = h[1][k] + beta * sh[1][k];
                      rL[q[k]] -= alpha * sh[0][k];
                      rL[(nr + 1) * W + q[k]] -= alpha * sh[1][k];
                    }
                }
              store_r();
              lds_barrier();
              product(w);
              v[0] = v[1] = 0.0;
#pragma unroll
              for (int k = 0; k < NPT; ++k)
                if (own[k])
                  {
                    v[0] += r[k] * r[k];
                    v[1] += w[k] * r[k];
                  }
              if (!exchange(S2(), v, true, w, h))
                return give_up();
              beta = v[0] / rr;
              rr = v[0];
              wr = v[1];
              ++it;
            }
          if (!go || it < until || it == max_it)
            break;
          // r's mean, in the own rows and the copies of the neighbours' (w
          // and (w, r) do not change: A 1 = 0)
          v[0] = 0.0;
#pragma unroll
          for (int k = 0; k < NPT; ++k)
            v[0] += r[k];
          if (!exchange(S1(), v, false, r, h))
            return give_up();
          const double mean = v[0] / nx;
#pragma unroll
          for (int k = 0; k < NPT; ++k)
            {
              r[k] -= own[k] ? mean : 0.0;
              if (halo[k])
                {
                  rL[q[k]] -= mean;
                  rL[(nr + 1) * W + q[k]] -= mean;
                }
            }
        }
    }

  // phi, and grad phi at the quadrature points
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      {
        phi[(long long)y0 * W + q[k]] = x[k];
        rL[W + q[k]] = x[k];
      }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      {
        double a = 0.0, c = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j)
          {
            const double v = rL[W + q[k] - node + j + N * iy];
            a += xd.G[ix * N + j] * v;
            c += xd.S[ix * N + j] * v;
          }
        z0[q[k]] = a;
        z1[q[k]] = c;
      }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (own[k])
      {
        double a = 0.0, c = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j)
          {
            a += xd.S[iy * N + j] * z0[q[k] - node + ix + N * j];
            c += xd.G[iy * N + j] * z1[q[k] - node + ix + N * j];
          }
        double *e = efield + ((long long)y0 * W + q[k]) * 2;
        e[0] = a / xd.h[0];
        e[1] = c / xd.h[1];
      }
  if (sb == 0 && t == 0)
    {
      double *ds = reinterpret_cast<double *>(stats);
      const double nb = sqrt(bb) + 1e-300;
      stats[0] += it;
      stats[1] += 1;
      ds[2] = sqrt(rr) / nb;
      ds[3] = sqrt(rr_start) / nb;
      ds[4] = (guess ? sqrt(rr_warm) : sqrt(rr_start)) / nb;
      if (guess)
        {
          stats[5] += 1;
          ds[6] = alpha0;
          ds[7] = beta0;
        }
    }
}

// The work behind a marked launch: empties the inboxes and computes the
// residual image, or runs plain CG from the previous phi (a guess is left out),
// with its vectors in global memory.  One small workgroup with few registers,
// so that it is scheduled at once beside other work; slow, and only there for
// correctness.
template <int N>
__global__ __launch_bounds__(256) void marked_kernel(
  XDev xd, const double *__restrict__ tab, const double *__restrict__ rho,
  double *phi, double *__restrict__ efield, double *work,
  unsigned long long *slots, long long n_slots, int *mark, double rel_tol,
  int max_it, long long *__restrict__ stats, float *__restrict__ res_image,
  double *__restrict__ res_scale, double *__restrict__ phi_copy)
{
  constexpr int NN = N * N;
  __shared__ double red[256];
  if (*mark == 0)
    return;
  __syncthreads(); // every thread has read the mark
  for (long long i = threadIdx.x; i < n_slots; i += 256)
    slots[i] = kEmpty;
  if (threadIdx.x == 0)
    *mark = 0;
  const int n0 = xd.n[0], n1 = xd.n[1], n = (int)xd.n_cells * NN;
  double *r = work, *p = work + n, *Ap = work + 2 * n;
  auto total = [&](double v) {
    __syncthreads();
    red[threadIdx.x] = v;
    __syncthreads();
    for (int k = 128; k >= 1; k /= 2)
      {
        if ((int)threadIdx.x < k)
          red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
      }
    return red[0];
  };
  auto apply = [&](const double *in, double *out) {
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += 256)
      {
        const int c = e / NN, ix = e % N, iy = e % NN / N;
        const int cx = c % n0, cy = c / n0;
        double y = 0.0;
        for (int j = 0; j < N; ++j)
          for (int k = 0; k < 3; ++k)
            {
              const int xn = (cx + k + n0 - 1) % n0 + n0 * cy;
              const int yn = cx + n0 * ((cy + k + n1 - 1) % n1);
              for (int l = 0; l < N; ++l)
                y += tab[7 * NN + iy * N + j] * tab[k * NN + ix * N + l] *
                       in[xn * NN + l + N * j] +
                     tab[6 * NN + ix * N + j] *
                       tab[(3 + k) * NN + iy * N + l] *
                       in[yn * NN + j + N * l];
            }
        out[e] = y;
      }
    __syncthreads();
  };
  double s = 0.0;
  for (int e = threadIdx.x; e < n; e += 256)
    s += rho[e];
  const double mean_rho = total(s) / n;
  s = 0.0;
  for (int e = threadIdx.x; e < n; e += 256)
    {
      const int c = e / NN, ix = e % N, iy = e % NN / N;
      double a = 0.0;
      for (int j = 0; j < N; ++j)
        for (int l = 0; l < N; ++l)
          a += tab[7 * NN + iy * N + j] * tab[6 * NN + ix * N + l] *
               (rho[c * NN + l + N * j] - mean_rho);
      r[e] = -a;
      s -= a;
    }
  const double mean_b = total(s) / n;
  apply(phi, Ap);
  double bb = 0.0, rr = 0.0;
  for (int e = threadIdx.x; e < n; e += 256)
    {
      const double b = r[e] - mean_b;
      r[e] = p[e] = b - Ap[e];
      bb += b * b;
      rr += r[e] * r[e];
    }
  bb = total(bb);
  rr = total(rr);
  if (res_image)
    {
      s = 0.0;
      for (int e = threadIdx.x; e < n; e += 256)
        s += r[e];
      const double mean = total(s) / n;
      s = 0.0;
      for (int e = threadIdx.x; e < n; e += 256)
        s += (r[e] - mean) * (r[e] - mean);
      const double rms = sqrt(total(s) / n);
      const double inv = rms > 0.0 ? 1.0 / rms : 0.0;
      for (int e = threadIdx.x; e < n; e += 256)
        {
          const int c = e / NN, ix = e % N, iy = e % NN / N;
          res_image[(c / n0 * N + iy) * (n0 * N) + c % n0 * N + ix] =
            (float)((r[e] - mean) * inv);
          if (phi_copy)
            phi_copy[e] = phi[e];
        }
      if (threadIdx.x == 0)
        *res_scale = rms;
      return;
    }
  const double rr_start = rr;
  int it = 0;
  while (sqrt(rr) > rel_tol * sqrt(bb) && it < max_it)
    {
      apply(p, Ap);
      s = 0.0;
      for (int e = threadIdx.x; e < n; e += 256)
        s += p[e] * Ap[e];
      const double pAp = total(s);
      if (!(pAp > 0.0))
        break;
      s = 0.0;
      for (int e = threadIdx.x; e < n; e += 256)
        {
          phi[e] += rr / pAp * p[e];
          r[e] -= rr / pAp * Ap[e];
          s += r[e] * r[e];
        }
      const double rr2 = total(s);
      for (int e = threadIdx.x; e < n; e += 256)
        p[e] = r[e] + rr2 / rr * p[e];
      rr = rr2;
      ++it;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < n; e += 256)
    {
      const int c = e / NN, ix = e % N, iy = e % NN / N;
      double g0 = 0.0, g1 = 0.0;
      for (int j = 0; j < N; ++j)
        for (int l = 0; l < N; ++l)
          {
            const double v = phi[c * NN + l + N * j];
            g0 += xd.S[iy * N + j] * xd.G[ix * N + l] * v;
            g1 += xd.G[iy * N + j] * xd.S[ix * N + l] * v;
          }
      efield[(long long)e * 2] = g0 / xd.h[0];
      efield[(long long)e * 2 + 1] = g1 / xd.h[1];
    }
  if (threadIdx.x == 0)
    {
      double *ds = reinterpret_cast<double *>(stats);
      const double nb = sqrt(bb) + 1e-300;
      stats[0] += it;
      stats[1] += 1;
      ds[2] = sqrt(rr) / nb;
      ds[3] = ds[4] = sqrt(rr_start) / nb;
    }
}

int strip_rows(int n1)
{
  return (n1 + kMaxStrips - 1) / kMaxStrips;
}
int strip_count(int n1)
{
  const int rows = strip_rows(n1);
  return (n1 + rows - 1) / rows;
}
size_t row_slots(int N, const int *n)
{
  return (size_t)2 * strip_count(n[1]) * 2 * n[0] * N * N;
}
size_t sum_slots(const int *n)
{
  return (size_t)2 * strip_count(n[1]) * strip_count(n[1]) * kSums;
}
} // namespace vpcg

// Where the strips are the faster solver: one workgroup holds 512 cells at one
// per thread.  us per iteration, one workgroup and strips, k = 3: 16 x 2 cells
// 4.9 and 2.7, 32 x 32 11.0 and 3.1; two nodes per thread 64 x 2 4.9 and 4.9,
// 50 x 18 11.0 and 4.6; four 128 x 2 5.2 and 8.7, 128 x 5 9.2 and 8.9, 100 x 10
// 11.0 and 8.3, 66 x 9 9.2 and 6.7.  k = 2: 20 x 20 cells 3.0 and 3.0, 24 x 24
// 3.6 and 3.0, 32 x 32 5.0 and 3.1; two nodes per thread 60 x 9 3.6 and 4.3.
// k = 1: 32 x 32 1.9 and 2.1.
bool vp_strips_supported(int dim_x, int N, const int *n)
{
  if (dim_x != 2 || n[1] < 2)
    return false;
  const int T = vpcg::kThreads / (N * N) * (N * N);
  const long long nodes = (long long)vpcg::strip_rows(n[1]) * n[0] * N * N;
  const bool two = (long long)n[0] * n[1] > 512;
  return N == 4   ? nodes <= (two ? 4 : 2) * T
         : N == 3 ? two && nodes <= T
                  : false;
}

// 8-byte slots of the inboxes, then the mark
size_t vp_strips_bytes(int N, const int *n)
{
  return (vpcg::row_slots(N, n) + vpcg::sum_slots(n) + 1) * 8;
}

hipError_t vp_strips_reset(void *comm, int N, const int *n)
{
  const size_t slots = vpcg::row_slots(N, n) + vpcg::sum_slots(n);
  hipError_t e = hipMemset(comm, 0xff, slots * 8); // kEmpty
  if (e == hipSuccess)
    e = hipMemset(static_cast<char *>(comm) + slots * 8, 0, 8);
  // (solves may run on streams that do not wait for the null stream)
  return e == hipSuccess ? hipStreamSynchronize(nullptr) : e;
}

hipError_t vp_strips_solve(const XDev &xd, int N, const double *rho,
                           double *phi, const double *guess, double *efield,
                           double *work, void *comm, double rel_tol,
                           int max_it, long long *stats, hipStream_t stream,
                           const double *tab2d, bool guess_alone,
                           const ResidualImage *residual,
                           const GuessImage &guess_image)
{
  vpcg::Strips st{};
  st.rows = vpcg::strip_rows(xd.n[1]);
  st.count = vpcg::strip_count(xd.n[1]);
  st.row_in = static_cast<unsigned long long *>(comm);
  st.sum_in = st.row_in + vpcg::row_slots(N, xd.n);
  const size_t slots = vpcg::row_slots(N, xd.n) + vpcg::sum_slots(xd.n);
  st.mark = reinterpret_cast<int *>(st.row_in + slots);
  const int NN = N * N, T = vpcg::kThreads / NN * NN;
  const int nodes = st.rows * xd.n[0] * NN;
  const int npt = (nodes + T - 1) / T;
  // at least 100 KB: no tile of the learned start's convolutions (64 KB)
  // fits beside a strip
  const size_t lds = std::max<size_t>(100 * 1024,
    ((size_t)(st.rows + 2) * xd.n[0] * NN + 2 * (size_t)nodes +
     9 * vpcg::kSums) *
    sizeof(double));
  float *image = residual ? residual->image : nullptr;
  double *scale = residual ? residual->scale : nullptr;
  double *copy = residual ? residual->phi_copy : nullptr;
  auto go = [&](auto kernel, auto behind) {
    hipError_t e = hipFuncSetAttribute(
      reinterpret_cast<const void *>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess)
      return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)st.count),
                       dim3(vpcg::kThreads), lds, stream, xd, tab2d, rho, phi,
                       guess, efield, st, rel_tol, max_it, stats,
                       guess_alone ? 1 : 0, image, scale, copy,
                       guess_image);
    e = hipGetLastError();
    if (e != hipSuccess)
      return e;
    hipLaunchKernelGGL(behind, dim3(1), dim3(256), 0, stream, xd, tab2d, rho,
                       phi, efield, work, st.row_in, (long long)slots,
                       st.mark, rel_tol, max_it, stats, image, scale, copy);
    return hipGetLastError();
  };
#define HD_STRIP(NN_, NPT_)                                                  \
  if (N == NN_ && npt <= NPT_)                                               \
    return go(&vpcg::strip_kernel<NN_, NPT_>, &vpcg::marked_kernel<NN_>);
  HD_STRIP(3, 1) HD_STRIP(4, 1) HD_STRIP(4, 2) HD_STRIP(4, 4)
#undef HD_STRIP
  return hipErrorInvalidValue;
}
} // namespace hd
