// Standalone three-point stencils and the Jacobi anti-Laplacian sweep for
// gfx950, backing NumericalDifferentiator's public methods on any number of
// dimensions.  Semantics restate
// pararealml/operators/fdm/numerical_differentiator.py:1012-1242.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <limits>
#include <type_traits>
#include <vector>

#include "pml_common.h"

namespace pml {

static int grid_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > (1 << 20)) b = 1 << 20;
  return static_cast<int>(b < 1 ? 1 : b);
}

template <typename T>
__device__ __forceinline__ void emit(T *out, int64_t t, T r, int mode) {
  if (mode == 0) out[t] = r;
  else if (mode > 0) out[t] = out[t] + r;
  else out[t] = out[t] - r;
}

// (y[i+1] - y[i-1]) / (2 dx) at element t, index i of n along the axis with
// element stride inner, slab index `slab` in the axis' boundary arrays: zero
// halos, boundary override by lo/hi (numerical_differentiator.py:1012-1057).
template <typename T, typename I>
__device__ __forceinline__ T first_at(const T *y, I t, I i, I n, I inner, I slab, T den,
                                      const double *lo, const double *hi) {
  const T yp = i > 0 ? y[t - inner] : T(0);
  const T yn = i < n - 1 ? y[t + inner] : T(0);
  T d = (yn - yp) / den;
  if (i == 0 && lo) {
    const double g = lo[slab];
    if (g == g) d = static_cast<T>(g);
  }
  if (i == n - 1 && hi) {
    const double g = hi[slab];
    if (g == g) d = static_cast<T>(g);
  }
  return d;
}

// ((y[i+1] - 2 y[i]) + y[i-1]) / (dx dx2) with constraint ghosts
// (numerical_differentiator.py:1083-1095, 1188-1242).
template <typename T, typename I>
__device__ __forceinline__ T second_at(const T *y, I t, I i, I n, I inner, I slab, T den, T m2dx,
                                       T p2dx, const double *lo, const double *hi) {
  T yp, yn;
  if (i > 0) {
    yp = y[t - inner];
  } else {
    const double g = lo ? lo[slab] : NAN;
    yp = (g == g) ? y[t + inner] + m2dx * static_cast<T>(g) : T(0);
  }
  if (i < n - 1) {
    yn = y[t + inner];
  } else {
    const double g = hi ? hi[slab] : NAN;
    yn = (g == g) ? y[t - inner] + p2dx * static_cast<T>(g) : T(0);
  }
  return ((yn - T(2) * y[t]) + yp) / den;
}

template <typename T>
__global__ void k_first(const T *y, T *out, int64_t outer, int64_t n, int64_t inner,
                        double two_dx, const double *lo, const double *hi, int mode) {
  const int64_t total = outer * n * inner;
  const T den = static_cast<T>(two_dx);
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t o = t / (n * inner), rem = t - o * n * inner;
    const int64_t i = rem / inner, q = rem - i * inner;
    emit(out, t, first_at<T, int64_t>(y, t, i, n, inner, o * inner + q, den, lo, hi), mode);
  }
}

template <typename T>
__global__ void k_second(const T *y, T *out, int64_t outer, int64_t n, int64_t inner,
                         double dx, double den_d, const double *lo, const double *hi,
                         int mode) {
  const int64_t total = outer * n * inner;
  const T den = static_cast<T>(den_d);
  const T m2dx = static_cast<T>(-2.0 * dx), p2dx = static_cast<T>(2.0 * dx);
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t o = t / (n * inner), rem = t - o * n * inner;
    const int64_t i = rem / inner, q = rem - i * inner;
    emit(out, t,
         second_at<T, int64_t>(y, t, i, n, inner, o * inner + q, den, m2dx, p2dx, lo, hi), mode);
  }
}

// One Runge-Kutta stage of u_t = D lap(u) on a mesh whose Laplacian is a sum
// of stencils along the axes, each with an optional weight per vertex (the
// coordinate factors of polar, cylindrical and spherical meshes), fused:
// Laplacian of the stage input, the stage sum, the next stage input (or the
// step's result) and its y constraints.  The operations and their order are
// those of the separate stencil, weighted-add and set-values kernels, so the
// results are the same to the bit.
//
// Bound: the launch and one dependent pass over a grid that sits in L2
// (3 reads and 2 writes per vertex); 128 threads per block keep two
// wavefronts on every CU at the few ten thousand vertices such meshes have.
// 40 RK4 steps on 33 x 29 x 31 vertices in FP64, the whole solve: 15.8 ms by
// some 40 separate launches a step with host work between them, 0.95 ms by
// 4 a step.
struct LapTerm {
  int axis, order;
  const void *weight;  // per vertex, in the state's precision (NULL: 1)
};
struct LapGeom {
  int n[3], stride[3];
  double dx[3];
  const double *lo[3], *hi[3];
  LapTerm term[PML_LAPLACIAN_MAX_TERMS];
  int n_terms;
};
// What a stage does with k = dt D lap(s):
//   kStepEuler   out = y + k                                (the last stage
//                of forward Euler and of the midpoint method)
//   kStageHalf   out = y + k / 2                            (midpoint)
//   kRkFirst     acc = k,          out = y + k / 2
//   kRkSecond    acc = acc + 2 k,  out = y + k / 2
//   kRkThird     acc = acc + 2 k,  out = y + k
//   kRkLast      out = y + (acc + k) / 6
enum LapStage { kStepEuler, kStageHalf, kRkFirst, kRkSecond, kRkThird, kRkLast };

template <typename T, int STAGE>
__global__ void __launch_bounds__(128) k_lap_stage(LapGeom g, const T *__restrict__ s,
                                                   const T *y, T *acc, T *out, double *snap,
                                                   const double *__restrict__ ycons, T coef,
                                                   T dt, int count) {
  const int t = blockIdx.x * 128 + threadIdx.x;
  if (t >= count) return;
  int idx[3];
  idx[2] = t % g.n[2];
  const int rest = t / g.n[2];
  idx[1] = rest % g.n[1];
  idx[0] = rest / g.n[1];
  // the element's index in the boundary arrays of each axis
  const int slab[3] = {idx[1] * g.n[2] + idx[2], idx[0] * g.n[2] + idx[2],
                       idx[0] * g.n[1] + idx[1]};
  const T yv = y[t];
  const double fixed = ycons ? ycons[t] : NAN;
  T lap = T(0);
#pragma unroll
  for (int k = 0; k < PML_LAPLACIAN_MAX_TERMS; ++k) {
    if (k >= g.n_terms) break;
    const int a = g.term[k].axis;
    const int i = a == 0 ? idx[0] : (a == 1 ? idx[1] : idx[2]);
    const int q = a == 0 ? slab[0] : (a == 1 ? slab[1] : slab[2]);
    T d;
    if (g.term[k].order == 2)
      d = second_at<T, int>(s, t, i, g.n[a], g.stride[a], q, static_cast<T>(g.dx[a] * g.dx[a]),
                            static_cast<T>(-2.0 * g.dx[a]), static_cast<T>(2.0 * g.dx[a]),
                            g.lo[a], g.hi[a]);
    else
      d = first_at<T, int>(s, t, i, g.n[a], g.stride[a], q, static_cast<T>(2.0 * g.dx[a]),
                           g.lo[a], g.hi[a]);
    if (g.term[k].weight) d = static_cast<const T *>(g.term[k].weight)[t] * d;
    lap = k == 0 ? d : lap + d;
  }
  const T kk = dt * (coef * lap);
  T nv;
  if (STAGE == kStepEuler) {
    nv = yv + kk;
  } else if (STAGE == kStageHalf) {
    nv = yv + T(0.5) * kk;
  } else if (STAGE == kRkFirst) {
    acc[t] = kk;
    nv = yv + T(0.5) * kk;
  } else if (STAGE == kRkSecond) {
    acc[t] = acc[t] + T(2) * kk;
    nv = yv + T(0.5) * kk;
  } else if (STAGE == kRkThird) {
    acc[t] = acc[t] + T(2) * kk;
    nv = yv + kk;
  } else {
    nv = yv + static_cast<T>(1.0 / 6.0) * (acc[t] + kk);
  }
  if (fixed == fixed) nv = static_cast<T>(fixed);
  out[t] = nv;
  if (snap) snap[t] = static_cast<double>(nv);
}

struct JacobiGeom {
  int64_t n[3];
  int64_t stride[3];  // element strides of the three spatial axes
  double dx[3];
  double dxsq[3];
  const double *glo[3];
  const double *ghi[3];
  int active[3];
  double coef;  // sum over active axes of 2 / dx^2
  // reciprocals of dxsq and coef, rounded in the precision of the sweep, and
  // the |x| from which on div_by() gives every quotient by them
  double rdxsq[3], rcoef;
  double div_lo;
  // Curvilinear weights per vertex (NULL: Cartesian): the update is
  // (sum_a wsum[a] (prev + next) + wdiff[a] (next - prev) - lap) / wden.
  const double *wsum[3];
  const double *wdiff[3];
  const double *wden;
};

// One Jacobi update of the Cartesian anti-Laplacian
// (numerical_differentiator.py:1097-1186) followed by the y constraints
// and a sum of squared updates (872-927).
// State of a device-side Jacobi loop (pml_jacobi_solve): the sweep's
// sum of squared updates, a done flag and the number of sweeps taken.
struct JacobiState {
  double sumsq;
  double last_diff;
  long long sweeps;
  int done;
  int pad;
  double partials[PML_REDUCE_SLOTS];  // one per sweep block, summed in order
};
static_assert(sizeof(JacobiState) == PML_JACOBI_STATE_BYTES, "JacobiState layout");

// x / d with r = 1 / d rounded to nearest: the product with r, two steps of
// correction by the residual x - q d.  The first brings q within one ulp,
// after which the second rounds correctly (P. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990), so the
// result is the quotient's for |x| from div_least() on and for +0; a product
// that overflows leaves NaN.  5 operations where the compiler's division takes
// 11 and a reciprocal.
template <typename T>
__device__ __forceinline__ T div_by(T x, T d, T r) {
  T q = x * r;
  q = __builtin_elementwise_fma(__builtin_elementwise_fma(-d, q, x), r, q);
  return __builtin_elementwise_fma(__builtin_elementwise_fma(-d, q, x), r, q);
}

// The |x| from which on div_by() divides by each of the divisors as a division
// does (or gives NaN), for a type of p bits and normal numbers from 2^emin on.
// The last bit of a residual x - q d is at least 2^(e(x) - 2 p + 1), a
// multiple of the least subnormal 2^(emin - p + 1) from e(x) = emin + p on,
// and the quotient itself has to be normal.  Infinite where a divisor has no
// normal reciprocal.
template <typename T>
static double div_least(const double *divisors, int n) {
  constexpr int p = std::numeric_limits<T>::digits;
  constexpr int emin = std::numeric_limits<T>::min_exponent - 1;
  constexpr int emax = std::numeric_limits<T>::max_exponent - 1;
  int least = emin + p;
  for (int k = 0; k < n; ++k) {
    const double d = static_cast<double>(static_cast<T>(divisors[k]));
    if (!(d >= std::ldexp(1.0, emin + 2) && d <= std::ldexp(1.0, emax - 2)))
      return std::numeric_limits<double>::infinity();
    least = std::max(least, emin + 2 + std::ilogb(d));
  }
  return std::ldexp(1.0, least);
}

// The update of element t (field f of cell (idx)) from the iterate y.
template <typename T, typename I>
__device__ __forceinline__ T jacobi_update(const T *y, I t, I f, I cell, const I *idx, I nf,
                                           const JacobiGeom &g, T lap, const double *ycons) {
  // constrained vertices, most often all of an edge's, need no neighbours
  if (ycons) {
    const double c = ycons[t];
    if (c == c) return static_cast<T>(c);
  }
  T acc = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (!g.active[a]) continue;
    const I s = static_cast<I>(g.stride[a]);
    const I n = static_cast<I>(g.n[a]);
    // Slab index: the element with axis a removed.
    I slab = 0;
    for (int b = 0; b < 3; ++b) {
      if (b == a) continue;
      slab = slab * static_cast<I>(g.n[b]) + idx[b];
    }
    slab = slab * nf + f;
    T prev, next;
    if (idx[a] > 0) {
      prev = y[t - s];
    } else {
      const double gv = g.glo[a] ? g.glo[a][slab] : NAN;
      prev = (gv == gv) ? y[t + s] + static_cast<T>(-2.0 * g.dx[a]) * static_cast<T>(gv) : T(0);
    }
    if (idx[a] < n - 1) {
      next = y[t + s];
    } else {
      const double gv = g.ghi[a] ? g.ghi[a][slab] : NAN;
      next = (gv == gv) ? y[t - s] + static_cast<T>(2.0 * g.dx[a]) * static_cast<T>(gv) : T(0);
    }
    if (g.wden) {
      acc = acc + static_cast<T>(g.wsum[a][cell]) * (prev + next);
      if (g.wdiff[a]) acc = acc + static_cast<T>(g.wdiff[a][cell]) * (next - prev);
    } else {
      acc = acc + (prev + next) / static_cast<T>(g.dxsq[a]);
    }
  }
  acc = acc - lap;
  return acc / static_cast<T>(g.wden ? g.wden[cell] : g.coef);
}

// Each block writes its sum of squared updates to partials[blockIdx.x]
// (grid-stride order, then a fixed tree); k_jacobi_check adds them in block
// order, so the norm and the sweep count do not depend on scheduling.
template <typename T>
__global__ void k_jacobi(const T *y, T *yn, const T *lap, int64_t total, int nf,
                         JacobiGeom g, const double *ycons, double *partials,
                         const int *done) {
  // A loop that has converged turns its remaining sweeps into no-ops.
  if (done && *done) return;
  __shared__ double red[256];
  double acc2 = 0.0;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t f = t % nf;
    const int64_t cell = t / nf;
    int64_t idx[3];
    idx[2] = cell % g.n[2];
    idx[1] = (cell / g.n[2]) % g.n[1];
    idx[0] = cell / (g.n[2] * g.n[1]);
    const T v = jacobi_update<T, int64_t>(y, t, f, cell, idx, nf, g, lap[t], ycons);
    const double d = static_cast<double>(v) - static_cast<double>(y[t]);
    acc2 += d * d;
    yn[t] = v;
  }
  red[threadIdx.x] = acc2;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

// The whole loop in one workgroup, the iterate in LDS: a sweep is two
// barriers instead of two launches, and a caller that steps in time never
// waits for the host to see the stopping test.  y (the iterate, overwritten
// by the result) starts from `start`; the source is scale * lap.  Takes at
// most `most` sweeps; a loop that has not reached tol by then leaves
// state->done 0.  A state that holds an unfinished loop (state->pad set by an
// earlier launch of the same time loop) makes the launch a no-op.
//
// One CU works on the grid.  A sweep is bound by the instructions of its
// vertices (some 35 in 2-D, 16 wavefronts on 4 SIMDs) above 64 x 64 and by
// its reduction and two barriers (1.2 us) below 20 x 20.
// PLATE: one field on two axes, without vertex weights (grids of 3 x 3 and
// more).  Vertices inside the grid read their neighbours without a branch
// there and divide by div_by(); the general update is left to free vertices
// on an edge.  A vertex with a numerator below div_least() or a result that is
// not finite is divided as elsewhere, unless all three numerators are 0.
template <typename T, int PER, bool PLATE>
__global__ void __launch_bounds__(1024)
    k_jacobi_resident(T *y, const T *start, const T *__restrict__ lap, T scale, int total, int nf,
                      JacobiGeom g, const double *__restrict__ ycons, double tol, long long most,
                      JacobiState *state) {
  extern __shared__ unsigned char smem[];
  double *part = reinterpret_cast<double *>(smem);  // one sum per wavefront
  T *L = reinterpret_cast<T *>(smem + 16 * sizeof(double));
  if (state->pad) return;  // the same value in every thread
  const int tid = threadIdx.x, nt = blockDim.x;
  // the source and which vertices are free stay in registers: a sweep reads
  // nothing but the iterate (and boundary values where they are constrained)
  T src[PER];
  unsigned free = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int t = tid + k * nt;
    src[k] = T(0);
    if (t < total) {
      const double c = ycons ? ycons[t] : NAN;
      L[t] = c == c ? static_cast<T>(c) : start[t];
      src[k] = scale * lap[t];
      if (c != c) free |= 1u << k;
    }
  }
  __syncthreads();
  const int n2 = static_cast<int>(g.n[2]), n1 = static_cast<int>(g.n[1]);
  // Quotients by multiplication: with m = ceil(2^32 / d), t m / 2^32 exceeds
  // t / d by less than t / 2^32, which cannot reach the next integer while
  // t d < 2^32 (here both are below 2^16).
  auto inverse = [](int d) { return d == 1 ? 0u : static_cast<unsigned>(0xffffffffu / d) + 1u; };
  auto quotient = [](int t, unsigned m) {
    return m ? static_cast<int>(__umulhi(static_cast<unsigned>(t), m)) : t;
  };
  const unsigned mf = inverse(nf), m2 = inverse(n2), m1 = inverse(n1);
  const int n0 = static_cast<int>(g.n[0]);
  const T dxsq0 = static_cast<T>(g.dxsq[0]), dxsq1 = static_cast<T>(g.dxsq[1]);
  const T rdxsq0 = static_cast<T>(g.rdxsq[0]), rdxsq1 = static_cast<T>(g.rdxsq[1]);
  const T coef = static_cast<T>(g.coef), rcoef = static_cast<T>(g.rcoef);
  const T div_lo = static_cast<T>(g.div_lo);
  long long sweeps = 0;
  double norm = 0.0, sum = 0.0;
  bool done = false;
  int stuck = 0;  // consecutive norms that are not a number
  while (!done && sweeps < most && stuck < 3) {
    T nv[PER];
    double acc2 = 0.0;
    int first = tid;
    // Their indices are computed again in every sweep (kept, they are more
    // than the registers hold).
    if (PER > 2) asm volatile("" : "+v"(first));
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int t = first + k * nt;
      if (free >> k & 1u) {
        const T old = L[t];
        int idx[3] = {0, 0, 0};
        if (PLATE) {
          const T up = L[max(t - n1, 0)], down = L[min(t + n1, total - 1)];
          const T left = L[max(t - 1, 0)], right = L[min(t + 1, total - 1)];
          idx[0] = quotient(t, m1);
          idx[1] = t - idx[0] * n1;
          const T a = up + down, b = left + right;
          T acc = T(0) + div_by(a, dxsq0, rdxsq0);
          acc = acc + div_by(b, dxsq1, rdxsq1);
          const T c = acc - src[k];
          nv[k] = div_by(c, coef, rcoef);
          if (!(fmin(fmin(fabs(a), fabs(b)), fabs(c)) >= div_lo) ||
              !(fabs(nv[k]) < static_cast<T>(INFINITY))) {
            if (a != T(0) || b != T(0) || c != T(0))
              nv[k] = (((T(0) + a / dxsq0) + b / dxsq1) - src[k]) / coef;
          }
          if (idx[0] == 0 || idx[0] == n0 - 1 || idx[1] == 0 || idx[1] == n1 - 1)
            nv[k] = jacobi_update<T, int>(L, t, 0, t, idx, 1, g, src[k], nullptr);
        } else {
          const int cell = quotient(t, mf), f = t - cell * nf;
          const int row = quotient(cell, m2);
          idx[2] = cell - row * n2;
          idx[0] = quotient(row, m1);
          idx[1] = row - idx[0] * n1;
          nv[k] = jacobi_update<T, int>(L, t, f, cell, idx, nf, g, src[k], nullptr);
        }
        const double d = static_cast<double>(nv[k]) - static_cast<double>(old);
        acc2 += d * d;
      }
      if (PER > 2) __builtin_amdgcn_sched_barrier(0);
    }
    for (int s = 32; s > 0; s >>= 1) acc2 += __shfl_xor(acc2, s);
    if ((tid & 63) == 0) part[tid >> 6] = acc2;
    __syncthreads();  // every read of the iterate is done, the sums are there
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int t = tid + k * nt;
      if (free >> k & 1u) L[t] = nv[k];
    }
    sum = 0.0;
    for (int w = 0; w < nt >> 6; ++w) sum += part[w];
    norm = sqrt(sum);
    ++sweeps;
    done = norm <= tol;
    // A value that is not finite stays on its free neighbours for good (it
    // is gone after one sweep where it has none): no later sweep can stop
    // the loop, which its caller reports as not converging.
    stuck = norm != norm ? stuck + 1 : 0;
    __syncthreads();
  }
  for (int t = tid; t < total; t += nt) y[t] = L[t];
  if (tid == 0) {
    state->sumsq = sum;
    state->last_diff = norm;
    state->sweeps = sweeps;
    state->done = done ? 1 : (stuck >= 3 ? -1 : 0);
    if (!done) state->pad = 1;
  }
}

// Which grids the resident loop takes.  A sweep of two launches takes 8.0 to
// 8.5 us whatever the size (of these), and 64 are launched before the host
// looks.  Resident sweeps in FP64: plates between constrained edges 1.2 us at
// 17 x 17, 2.9 at 65 x 65, 6.1 at 100 x 100, 8.8 at 129 x 129 (7 to 9 % of it
// the test of the quotients' range); with free edges 6.8 at 65 x 65, 10.5 at
// 90 x 90; other grids 4.3 at 13^3, 7.4 at 17^3.  The lid-driven cavity on
// 65 x 65, 60 steps: 42 ms with a host round trip and 128 launches a step,
// 1.6 ms in the device loop.
constexpr int kResidentPer = 18;
// A sweep's time on two launches, and up to which the Poisson time loop stays
// in one workgroup: its steps would each pay the host's look and the launches
// beyond convergence (some 0.3 ms) outside.
constexpr double kTwoLaunchUs = 8.4, kPoissonLoopUs = 10.0;
// Sweeps of one launch at most (some 100 ms on the largest grid): the host
// looks at the loop's state in between.
constexpr int64_t kResidentSweeps = 16384;
template <typename T>
static size_t resident_lds(int64_t total) {
  return 16 * sizeof(double) + sizeof(T) * static_cast<size_t>(total);
}
static bool is_plate(const JacobiGeom &g, int nf) {
  return nf == 1 && !g.wden && g.n[0] > 1 && g.n[1] > 1 && g.n[2] == 1;
}

// A plate's resident sweep by its runs of 64 vertices, a wavefront's step
// each, of which `slow` hold a free vertex on an edge and run the general
// update as well.  Run r is on SIMD r % 4, and the fullest SIMD counts: slow
// is 4 times its share.  Measured against this, FP64 us: 129 x 129 all edges
// fixed 8.8 / 8.7, none 16.0 / 16.0; 64 x 256 one column free 20.1 / 22.4;
// 256 x 64 none fixed 22.7 / 22.4; FP32 129 x 129 6.8 / 6.7 and 12.6 / 13.1.
static double resident_us(int precision, int64_t total, int64_t slow) {
  const double runs = static_cast<double>((total + 63) / 64);
  return precision == PML_F64 ? 1.1 + 0.0292 * runs + 0.054 * slow
                              : 1.3 + 0.0208 * runs + 0.047 * slow;
}

// The slow runs of a plate with all its edges free.
static int64_t edge_runs(int n0, int n1) {
  int64_t on[4] = {0, 0, 0, 0};
  const int total = n0 * n1;
  for (int r = 0; 64 * r < total; ++r) {
    const int a = 64 * r, b = std::min(a + 63, total - 1);
    const bool inside = a / n1 == b / n1 && a >= n1 && b < total - n1 && a % n1 && (b + 1) % n1;
    if (!inside) ++on[r % 4];
  }
  return 4 * *std::max_element(on, on + 4);
}

// The same of the plate's own constraints, into st->sweeps (one block of 1024).
__global__ void __launch_bounds__(1024) k_edge_runs(const double *ycons, int n0, int n1,
                                                    JacobiState *st) {
  __shared__ int on[4];
  if (threadIdx.x < 4) on[threadIdx.x] = 0;
  __syncthreads();
  const int total = n0 * n1;
  for (int t0 = 0; t0 < total; t0 += 1024) {
    const int t = t0 + threadIdx.x;
    const int i = t / n1, j = t - i * n1;
    const bool edge = t < total && (i == 0 || i == n0 - 1 || j == 0 || j == n1 - 1);
    const bool slow = edge && ycons[t] != ycons[t];
    if (__ballot(slow) && (threadIdx.x & 63) == 0) atomicAdd(&on[(t >> 6) & 3], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) st->sweeps = 4 * max(max(on[0], on[1]), max(on[2], on[3]));
}

// Whether the resident loop takes a grid for at most `most_us` a sweep.  Where
// that depends on which edge vertices are free, they are counted (one launch
// and a look by the host, some 20 us).
static int takes_resident(int precision, int64_t total, int nf, const JacobiGeom &g,
                          const double *ycons, double most_us, JacobiState *js, hipStream_t st,
                          bool *yes) {
  *yes = false;
  if (!is_plate(g, nf)) {
    *yes = total <= 5 * 1024;
    return PML_OK;
  }
  if (total > kResidentPer * 1024 || resident_us(precision, total, 0) > most_us) return PML_OK;
  const int n0 = static_cast<int>(g.n[0]), n1 = static_cast<int>(g.n[1]);
  int64_t slow = edge_runs(n0, n1);
  if (ycons && resident_us(precision, total, slow) > most_us) {
    hipLaunchKernelGGL(k_edge_runs, dim3(1), dim3(1024), 0, st, ycons, n0, n1, js);
    PML_LAUNCH_CHECK();
    long long counted = 0;
    PML_HIP_CHECK(hipMemcpyAsync(&counted, &js->sweeps, sizeof(counted), hipMemcpyDeviceToHost,
                                 st));
    PML_HIP_CHECK(hipStreamSynchronize(st));
    slow = counted;
  }
  *yes = resident_us(precision, total, slow) <= most_us;
  return PML_OK;
}

template <typename T>
static int launch_resident(T *y, const T *start, const T *lap, T scale, int64_t total, int nf,
                           const JacobiGeom &g, const double *ycons, double tol, long long most,
                           JacobiState *state, hipStream_t st) {
  const size_t lds = resident_lds<T>(total);
  const int threads = total < 1024 ? static_cast<int>((total + 63) / 64 * 64) : 1024;
  auto launch = [&](auto kernel) -> int {
    PML_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
    hipLaunchKernelGGL(kernel, dim3(1), dim3(threads), lds, st, y, start, lap, scale,
                       static_cast<int>(total), nf, g, ycons, tol, most, state);
    PML_LAUNCH_CHECK();
    return PML_OK;
  };
  const bool plate = is_plate(g, nf);
  auto pick = [&](auto per) {
    constexpr int P = decltype(per)::value;
    return plate ? launch(&k_jacobi_resident<T, P, true>)
                 : launch(&k_jacobi_resident<T, P, false>);
  };
  if (total <= 2 * 1024) return pick(std::integral_constant<int, 2>{});
  if (total <= 5 * 1024) return pick(std::integral_constant<int, 5>{});
  return pick(std::integral_constant<int, kResidentPer>{});
}

// sum of parts[0 .. n) in a fixed order into *out (one block).
__device__ void sum_in_order(const double *parts, int n, double *out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int b = threadIdx.x; b < n; b += blockDim.x) acc += parts[b];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

__global__ void k_jacobi_sum(const double *parts, int n, double *out) {
  sum_in_order(parts, n, out);
}

__global__ void k_jacobi_init(JacobiState *st) {
  if (threadIdx.x == 0) {
    st->sumsq = 0.0;
    st->last_diff = 0.0;
    st->sweeps = 0;
    st->done = 0;
    st->pad = 0;
  }
}

// After a sweep of n_parts blocks: add its partials in order, count it,
// stop once ||y_new - y_old||_2 <= tol (the reference's loop condition).
// A loop that is already done leaves the state as it is.
__global__ void k_jacobi_check(JacobiState *st, int n_parts, double tol) {
  if (st->done) return;
  sum_in_order(st->partials, n_parts, &st->sumsq);
  __syncthreads();
  if (threadIdx.x == 0) {
    st->sweeps += 1;
    st->last_diff = sqrt(st->sumsq);
    if (st->last_diff <= tol) st->done = 1;
  }
}

// out (=, +=, -=) coef * x, element by element: the coordinate-dependent
// factors of the curvilinear operators (numerical_differentiator.py:158-173,
// 229-308, 348-400, 482-590, 636-725, 771-870) applied to stencil results
// and to field components.
template <typename T>
__global__ void k_weighted_add(const T *x, const T *coef, T *out, int64_t count, int mode) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < count;
       t += (int64_t)gridDim.x * blockDim.x)
    emit(out, t, coef[t] * x[t], mode);
}

// y[t] = v[t] where v[t] is not NaN: the static y constraints of a
// channel-last state (constraint.py:104-131 over the full grid).
template <typename T>
__global__ void k_set_values(T *y, const double *v, int64_t count) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < count;
       t += (int64_t)gridDim.x * blockDim.x) {
    const double c = v[t];
    if (c == c) y[t] = static_cast<T>(c);
  }
}

// One iteration of the element-wise secant method that
// scipy.optimize.newton runs on arrays without a derivative (the implicit
// integrators, numerical_integrator.py:135-270).  mode 0: where q1 != q0,
// p_new = p1 - q1 (p1 - p) / (q1 - q0) and fail = |dp| >= tol; where
// q1 == q0 and the element is still active, p_new = (p1 + p) / 2; elements
// with q1 == q0 become inactive.  counters[0] += elements with q1 != q0,
// counters[1] += those still failing.  mode 1: p_new = (p1 + p) / 2
// everywhere (all residual differences were zero).
template <typename T>
__global__ void k_secant(const T *p, const T *p1, const T *q0, const T *q1, T *p_new,
                         unsigned char *active, unsigned char *fail, int64_t count, double tol,
                         int mode, unsigned long long *counters) {
  unsigned long long n_nz = 0, n_fail = 0;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < count;
       t += (int64_t)gridDim.x * blockDim.x) {
    if (mode == 1) {
      p_new[t] = (p1[t] + p[t]) / T(2);
      continue;
    }
    if (mode == 2) {  // the second start point; tol carries dx
      const T dx = static_cast<T>(tol);
      p_new[t] = p[t] * (T(1) + dx) + (p[t] >= T(0) ? dx : -dx);
      continue;
    }
    if (q1[t] != q0[t]) {
      const T dp = (q1[t] * (p1[t] - p[t])) / (q1[t] - q0[t]);
      p_new[t] = p1[t] - dp;
      const bool f = fabs(static_cast<double>(dp)) >= tol;
      fail[t] = f;
      n_nz += 1;
      n_fail += f;
    } else {
      p_new[t] = active[t] ? (p1[t] + p[t]) / T(2) : p[t];
      active[t] = 0;
    }
  }
  if (mode == 0) {
    if (n_nz) atomicAdd(&counters[0], n_nz);
    if (n_fail) atomicAdd(&counters[1], n_fail);
  }
}

}  // namespace pml

using namespace pml;

extern "C" int pml_stencil_first(int precision, const void *y, void *out, int64_t outer,
                                 int64_t n, int64_t inner, double dx, const double *lo,
                                 const double *hi, int mode, void *stream) {
  if (n <= 2) return fail(PML_E_INVALID, "y must contain at least 3 points along the axis");
  if (outer <= 0 || inner <= 0 || !y || !out || !(dx > 0))
    return fail(PML_E_INVALID, "bad stencil arguments");
  hipStream_t st = as_stream(stream);
  const int nb = grid_for(outer * n * inner);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_first<double>, dim3(nb), dim3(256), 0, st, (const double *)y,
                       (double *)out, outer, n, inner, 2.0 * dx, lo, hi, mode);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_first<float>, dim3(nb), dim3(256), 0, st, (const float *)y,
                       (float *)out, outer, n, inner, 2.0 * dx, lo, hi, mode);
  else
    return fail(PML_E_INVALID, "stencils take FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_weighted_add(int precision, const void *x, const void *coef, void *out,
                                int64_t count, int mode, void *stream) {
  if (count <= 0 || !x || !coef || !out) return fail(PML_E_INVALID, "bad weighted-add arguments");
  hipStream_t st = as_stream(stream);
  const int nb = grid_for(count);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_weighted_add<double>, dim3(nb), dim3(256), 0, st, (const double *)x,
                       (const double *)coef, (double *)out, count, mode);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_weighted_add<float>, dim3(nb), dim3(256), 0, st, (const float *)x,
                       (const float *)coef, (float *)out, count, mode);
  else
    return fail(PML_E_INVALID, "weighted add takes FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_set_values(int precision, void *y, const double *values, int64_t count,
                              void *stream) {
  if (count <= 0 || !y || !values) return fail(PML_E_INVALID, "bad set-values arguments");
  hipStream_t st = as_stream(stream);
  const int nb = grid_for(count);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_set_values<double>, dim3(nb), dim3(256), 0, st, (double *)y, values,
                       count);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_set_values<float>, dim3(nb), dim3(256), 0, st, (float *)y, values,
                       count);
  else
    return fail(PML_E_INVALID, "set values takes FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_secant_step(int precision, int mode, const void *p, const void *p1,
                               const void *q0, const void *q1, void *p_new, void *active,
                               void *failing, int64_t count, double tol, void *counters,
                               void *stream) {
  if (count <= 0 || !p || !p_new || (mode != 2 && !p1) ||
      (mode == 0 && (!q0 || !q1 || !active || !failing || !counters)) || mode < 0 || mode > 2)
    return fail(PML_E_INVALID, "bad secant arguments");
  hipStream_t st = as_stream(stream);
  const int nb = grid_for(count);
  auto *act = static_cast<unsigned char *>(active);
  auto *fl = static_cast<unsigned char *>(failing);
  auto *cnt = static_cast<unsigned long long *>(counters);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_secant<double>, dim3(nb), dim3(256), 0, st, (const double *)p,
                       (const double *)p1, (const double *)q0, (const double *)q1,
                       (double *)p_new, act, fl, count, tol, mode, cnt);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_secant<float>, dim3(nb), dim3(256), 0, st, (const float *)p,
                       (const float *)p1, (const float *)q0, (const float *)q1,
                       (float *)p_new, act, fl, count, tol, mode, cnt);
  else
    return fail(PML_E_INVALID, "secant step takes FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_stencil_second(int precision, const void *y, void *out, int64_t outer,
                                  int64_t n, int64_t inner, double dx, double dx2,
                                  const double *lo, const double *hi, int mode, void *stream) {
  if (n <= 2) return fail(PML_E_INVALID, "y must contain at least 3 points along the axis");
  if (outer <= 0 || inner <= 0 || !y || !out || !(dx > 0) || !(dx2 > 0))
    return fail(PML_E_INVALID, "bad stencil arguments");
  hipStream_t st = as_stream(stream);
  const int nb = grid_for(outer * n * inner);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_second<double>, dim3(nb), dim3(256), 0, st, (const double *)y,
                       (double *)out, outer, n, inner, dx, dx * dx2, lo, hi, mode);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_second<float>, dim3(nb), dim3(256), 0, st, (const float *)y,
                       (float *)out, outer, n, inner, dx, dx * dx2, lo, hi, mode);
  else
    return fail(PML_E_INVALID, "stencils take FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

template <typename T>
static int lap_solve(const LapGeom &g, int integ, const double *ycons, double coef, double dt,
                     int64_t n_steps, T *y, T *work, double *snaps, int64_t every, int count,
                     hipStream_t st) {
  const dim3 grid((count + 127) / 128), block(128);
  const T c = static_cast<T>(coef), h = static_cast<T>(dt);
  T *cur = y, *a = work, *b = work + count, *acc = work + 2 * static_cast<size_t>(count);
  for (int64_t s = 0; s < n_steps; ++s) {
    double *snap = (s + 1) % every == 0 ? snaps + ((s + 1) / every - 1) * count : nullptr;
    double *none = nullptr;
    if (integ == PML_INT_FE) {
      T *nxt = cur == y ? a : y;
      hipLaunchKernelGGL((k_lap_stage<T, kStepEuler>), grid, block, 0, st, g, cur, cur, acc, nxt,
                         snap, ycons, c, h, count);
      cur = nxt;
    } else if (integ == PML_INT_MIDPOINT) {
      hipLaunchKernelGGL((k_lap_stage<T, kStageHalf>), grid, block, 0, st, g, y, y, acc, a, none,
                         ycons, c, h, count);
      hipLaunchKernelGGL((k_lap_stage<T, kStepEuler>), grid, block, 0, st, g, a, y, acc, y, snap,
                         ycons, c, h, count);
    } else {
      hipLaunchKernelGGL((k_lap_stage<T, kRkFirst>), grid, block, 0, st, g, y, y, acc, a, none,
                         ycons, c, h, count);
      hipLaunchKernelGGL((k_lap_stage<T, kRkSecond>), grid, block, 0, st, g, a, y, acc, b, none,
                         ycons, c, h, count);
      hipLaunchKernelGGL((k_lap_stage<T, kRkThird>), grid, block, 0, st, g, b, y, acc, a, none,
                         ycons, c, h, count);
      hipLaunchKernelGGL((k_lap_stage<T, kRkLast>), grid, block, 0, st, g, a, y, acc, y, snap,
                         ycons, c, h, count);
    }
    PML_LAUNCH_CHECK();
  }
  if (cur != y)
    PML_HIP_CHECK(hipMemcpyAsync(y, cur, sizeof(T) * count, hipMemcpyDeviceToDevice, st));
  return PML_OK;
}

extern "C" int pml_laplacian_solve(int precision, int integrator_id, const int64_t *shape,
                                   const double *dx, const double *const *ghost_lo,
                                   const double *const *ghost_hi, int n_terms,
                                   const int *term_axis, const int *term_order,
                                   const void *const *term_weight, const double *ycons,
                                   double coefficient, double dt, int64_t n_steps, void *y,
                                   void *work, double *snapshots, int64_t snapshot_every,
                                   void *stream) {
  if (!shape || !dx || !term_axis || !term_order || !y || !work || !snapshots || n_steps < 0 ||
      snapshot_every <= 0 || n_terms <= 0 || n_terms > PML_LAPLACIAN_MAX_TERMS)
    return fail(PML_E_INVALID, "bad Laplacian solve arguments");
  if (integrator_id != PML_INT_FE && integrator_id != PML_INT_MIDPOINT &&
      integrator_id != PML_INT_RK4)
    return fail(PML_E_UNSUPPORTED, "the Laplacian solve runs the explicit integrators");
  LapGeom g{};
  int64_t count = 1;
  for (int a = 0; a < 3; ++a) {
    if (shape[a] <= 0 || !(dx[a] > 0)) return fail(PML_E_INVALID, "bad Laplacian solve shape");
    if (count > (int64_t(1) << 31) / shape[a])
      return fail(PML_E_INVALID, "a grid must hold fewer than 2^31 values");
    count *= shape[a];
    g.n[a] = static_cast<int>(shape[a]);
    g.dx[a] = dx[a];
    g.lo[a] = ghost_lo ? ghost_lo[a] : nullptr;
    g.hi[a] = ghost_hi ? ghost_hi[a] : nullptr;
  }
  if (count > (int64_t(1) << 31) - 256)
    return fail(PML_E_INVALID, "a grid must hold fewer than 2^31 values");
  g.stride[2] = 1;
  g.stride[1] = g.n[2];
  g.stride[0] = g.n[1] * g.n[2];
  g.n_terms = n_terms;
  for (int k = 0; k < n_terms; ++k) {
    const int a = term_axis[k];
    if (a < 0 || a > 2 || (term_order[k] != 1 && term_order[k] != 2))
      return fail(PML_E_INVALID, "bad Laplacian term");
    if (shape[a] <= 2)
      return fail(PML_E_INVALID, "y must contain at least 3 points along the axis");
    g.term[k] = LapTerm{a, term_order[k], term_weight ? term_weight[k] : nullptr};
  }
  hipStream_t st = as_stream(stream);
  if (precision == PML_F64)
    return lap_solve<double>(g, integrator_id, ycons, coefficient, dt, n_steps,
                             static_cast<double *>(y), static_cast<double *>(work), snapshots,
                             snapshot_every, static_cast<int>(count), st);
  if (precision == PML_F32)
    return lap_solve<float>(g, integrator_id, ycons, coefficient, dt, n_steps,
                            static_cast<float *>(y), static_cast<float *>(work), snapshots,
                            snapshot_every, static_cast<int>(count), st);
  return fail(PML_E_INVALID, "the Laplacian solve takes FP32 or FP64 arrays");
}

// Geometry of a Jacobi sweep over a (shape[0], shape[1], shape[2], n_fields)
// array; returns PML_OK or the error, and the element count in *total.
static int jacobi_geom(int precision, const int64_t *shape, int n_fields, const double *dx,
                       const double *const *ghost_lo, const double *const *ghost_hi,
                       JacobiGeom *out, int64_t *total_out) {
  JacobiGeom g{};
  int64_t total = n_fields;
  g.coef = 0.0;
  for (int a = 0; a < 3; ++a) {
    g.n[a] = shape[a];
    if (shape[a] <= 0) return fail(PML_E_INVALID, "bad Jacobi shape");
    g.active[a] = shape[a] > 1;
    if (g.active[a] && shape[a] <= 2)
      return fail(PML_E_INVALID, "y must contain at least 3 points along all x axes");
    g.dx[a] = dx[a];
    g.dxsq[a] = dx[a] * dx[a];
    g.glo[a] = ghost_lo ? ghost_lo[a] : nullptr;
    g.ghi[a] = ghost_hi ? ghost_hi[a] : nullptr;
    if (g.active[a]) {
      if (!(dx[a] > 0)) return fail(PML_E_INVALID, "spacing must be positive");
      g.coef += 2.0 / g.dxsq[a];
    }
    g.rdxsq[a] = precision == PML_F32
                     ? static_cast<double>(1.0f / static_cast<float>(g.dxsq[a]))
                     : 1.0 / g.dxsq[a];
    total *= shape[a];
  }
  g.rcoef = precision == PML_F32 ? static_cast<double>(1.0f / static_cast<float>(g.coef))
                                 : 1.0 / g.coef;
  double divisors[4] = {g.coef};
  int n_div = 1;
  for (int a = 0; a < 3; ++a)
    if (g.active[a]) divisors[n_div++] = g.dxsq[a];
  g.div_lo = precision == PML_F32 ? div_least<float>(divisors, n_div)
                                  : div_least<double>(divisors, n_div);
  g.stride[2] = n_fields;
  g.stride[1] = shape[2] * n_fields;
  g.stride[0] = shape[1] * shape[2] * n_fields;
  *out = g;
  *total_out = total;
  return PML_OK;
}

extern "C" int pml_jacobi_sweep(int precision, const void *y_old, void *y_new, const void *lap,
                                const int64_t *shape, int n_fields, const double *dx,
                                const double *const *ghost_lo, const double *const *ghost_hi,
                                const double *ycons, double *sumsq_out, double *work,
                                void *stream) {
  if (!y_old || !y_new || !lap || !shape || !dx || !sumsq_out || !work || n_fields <= 0)
    return fail(PML_E_INVALID, "bad Jacobi arguments");
  JacobiGeom g{};
  int64_t total = 0;
  if (int rc = jacobi_geom(precision, shape, n_fields, dx, ghost_lo, ghost_hi, &g, &total); rc != PML_OK)
    return rc;
  hipStream_t st = as_stream(stream);
  int nb = grid_for(total);
  if (nb > PML_REDUCE_SLOTS) nb = PML_REDUCE_SLOTS;
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_jacobi<double>, dim3(nb), dim3(256), 0, st, (const double *)y_old,
                       (double *)y_new, (const double *)lap, total, n_fields, g, ycons,
                       work, nullptr);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_jacobi<float>, dim3(nb), dim3(256), 0, st, (const float *)y_old,
                       (float *)y_new, (const float *)lap, total, n_fields, g, ycons,
                       work, nullptr);
  else
    return fail(PML_E_INVALID, "Jacobi sweep takes FP32 or FP64 arrays");
  PML_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_jacobi_sum, dim3(1), dim3(256), 0, st, work, nb, sumsq_out);
  PML_LAUNCH_CHECK();
  return PML_OK;
}

static int jacobi_solve(int precision, void *y, void *work, const void *lap,
                        const int64_t *shape, int n_fields, const double *dx,
                        const double *const *ghost_lo, const double *const *ghost_hi,
                        const double *ycons, double tol, int64_t max_sweeps, int64_t batch,
                        void *state, int64_t *sweeps_out, double *diff_out,
                        const double *const *w_sum, const double *const *w_diff,
                        const double *w_den, void *stream) {
  if (!y || !work || !lap || !shape || !dx || !state || !sweeps_out || n_fields <= 0 ||
      max_sweeps <= 0 || batch <= 0 || !(tol >= 0.0))
    return fail(PML_E_INVALID, "bad Jacobi solve arguments");
  if (precision != PML_F64 && precision != PML_F32)
    return fail(PML_E_INVALID, "Jacobi solve takes FP32 or FP64 arrays");
  JacobiGeom g{};
  int64_t total = 0;
  if (int rc = jacobi_geom(precision, shape, n_fields, dx, ghost_lo, ghost_hi, &g, &total); rc != PML_OK)
    return rc;
  if (w_den) {
    if (!w_sum) return fail(PML_E_INVALID, "weighted Jacobi needs w_sum");
    for (int a = 0; a < 3; ++a) {
      if (g.active[a] && !w_sum[a])
        return fail(PML_E_INVALID, "weighted Jacobi needs w_sum for every axis");
      g.wsum[a] = w_sum[a];
      g.wdiff[a] = w_diff ? w_diff[a] : nullptr;
    }
    g.wden = w_den;
  }
  hipStream_t st = as_stream(stream);
  JacobiState *js = static_cast<JacobiState *>(state);
  int nb = grid_for(total);
  if (nb > PML_REDUCE_SLOTS) nb = PML_REDUCE_SLOTS;
  JacobiState host;
  host.done = 0;
  host.sweeps = 0;
  host.last_diff = 0.0;
  int64_t issued = 0;
  bool resident = false;
  if (int rc = takes_resident(precision, total, n_fields, g, ycons, kTwoLaunchUs, js, st,
                              &resident);
      rc != PML_OK)
    return rc;
  if (resident) {
    while (issued < max_sweeps) {
      const int64_t n = std::min<int64_t>(kResidentSweeps, max_sweeps - issued);
      hipLaunchKernelGGL(k_jacobi_init, dim3(1), dim3(64), 0, st, js);
      const int rc =
          precision == PML_F64
              ? launch_resident<double>(static_cast<double *>(y), static_cast<const double *>(y),
                                        static_cast<const double *>(lap), 1.0, total, n_fields, g,
                                        ycons, tol, n, js, st)
              : launch_resident<float>(static_cast<float *>(y), static_cast<const float *>(y),
                                       static_cast<const float *>(lap), 1.0f, total, n_fields, g,
                                       ycons, tol, n, js, st);
      if (rc) return rc;
      PML_HIP_CHECK(hipMemcpyAsync(&host, js, offsetof(JacobiState, partials),
                                   hipMemcpyDeviceToHost, st));
      PML_HIP_CHECK(hipStreamSynchronize(st));
      issued = host.done < 0 ? max_sweeps : issued + host.sweeps;
      if (host.done == 1) break;
    }
    *sweeps_out = host.done == 1 ? issued : -issued;
    if (diff_out) *diff_out = host.last_diff;
    return PML_OK;
  }
  hipLaunchKernelGGL(k_jacobi_init, dim3(1), dim3(64), 0, st, js);
  while (issued < max_sweeps) {
    const int64_t n = std::min<int64_t>(batch, max_sweeps - issued);
    for (int64_t k = 0; k < n; ++k) {
      // sweep i (0-based) reads buffer i % 2 (y, work) and writes the other
      const bool odd = ((issued + k) & 1) != 0;
      const void *src = odd ? work : y;
      void *dst = odd ? y : work;
      if (precision == PML_F64)
        hipLaunchKernelGGL(k_jacobi<double>, dim3(nb), dim3(256), 0, st,
                           static_cast<const double *>(src), static_cast<double *>(dst),
                           static_cast<const double *>(lap), total, n_fields, g, ycons,
                           js->partials, &js->done);
      else
        hipLaunchKernelGGL(k_jacobi<float>, dim3(nb), dim3(256), 0, st,
                           static_cast<const float *>(src), static_cast<float *>(dst),
                           static_cast<const float *>(lap), total, n_fields, g, ycons,
                           js->partials, &js->done);
      hipLaunchKernelGGL(k_jacobi_check, dim3(1), dim3(256), 0, st, js, nb, tol);
    }
    issued += n;
    PML_LAUNCH_CHECK();
    PML_HIP_CHECK(hipMemcpyAsync(&host, js, offsetof(JacobiState, partials),
                                 hipMemcpyDeviceToHost, st));
    PML_HIP_CHECK(hipStreamSynchronize(st));
    if (host.done) break;
  }
  // The converged iterate is the output of sweep `sweeps` (1-based): it is
  // in work when that count is odd.
  const size_t esz = precision == PML_F64 ? 8 : 4;
  if (host.done && (host.sweeps & 1))
    PML_HIP_CHECK(hipMemcpyAsync(y, work, total * esz, hipMemcpyDeviceToDevice, st));
  else if (!host.done && (issued & 1))
    PML_HIP_CHECK(hipMemcpyAsync(y, work, total * esz, hipMemcpyDeviceToDevice, st));
  *sweeps_out = host.done ? host.sweeps : -issued;
  if (diff_out) *diff_out = host.last_diff;
  return PML_OK;
}

extern "C" int pml_jacobi_solve(int precision, void *y, void *work, const void *lap,
                                const int64_t *shape, int n_fields, const double *dx,
                                const double *const *ghost_lo, const double *const *ghost_hi,
                                const double *ycons, double tol, int64_t max_sweeps,
                                int64_t batch, void *state, int64_t *sweeps_out,
                                double *diff_out, void *stream) {
  return jacobi_solve(precision, y, work, lap, shape, n_fields, dx, ghost_lo, ghost_hi, ycons,
                      tol, max_sweeps, batch, state, sweeps_out, diff_out, nullptr, nullptr,
                      nullptr, stream);
}

extern "C" int pml_jacobi_solve_weighted(int precision, void *y, void *work, const void *lap,
                                         const int64_t *shape, int n_fields, const double *dx,
                                         const double *const *ghost_lo,
                                         const double *const *ghost_hi, const double *ycons,
                                         double tol, int64_t max_sweeps, int64_t batch,
                                         void *state, int64_t *sweeps_out, double *diff_out,
                                         const double *const *w_sum,
                                         const double *const *w_diff, const double *w_den,
                                         void *stream) {
  if (!w_sum || !w_den) return fail(PML_E_INVALID, "weighted Jacobi needs w_sum and w_den");
  return jacobi_solve(precision, y, work, lap, shape, n_fields, dx, ghost_lo, ghost_hi, ycons,
                      tol, max_sweeps, batch, state, sweeps_out, diff_out, w_sum, w_diff, w_den,
                      stream);
}

extern "C" int pml_fdm_poisson_solve(int eq_id, const double *eq_params, int n_params,
                                     int integrator_id, int precision, const pml_grid *grid,
                                     const double *bc_values, void *state, void *work,
                                     int64_t total_elems, double dt, int64_t n_steps,
                                     int tile_config, int flags, int n_poisson,
                                     const int *field,
                                     const int *source, const double *scale,
                                     const double *const *ghost_lo,
                                     const double *const *ghost_hi, const double *const *ycons,
                                     double tol, double *snapshots, int64_t snapshot_every,
                                     void *jacobi_state, int64_t *sweeps_out, void *stream) {
  if (!grid || !state || !work || !field || !source || !scale || !ghost_lo || !ghost_hi ||
      !ycons || !jacobi_state || !sweeps_out || n_poisson <= 0 || n_steps < 0 || !(tol >= 0.0) ||
      (snapshots && snapshot_every <= 0))
    return fail(PML_E_INVALID, "bad Poisson time loop arguments");
  if (precision != PML_F64 && precision != PML_F32)
    return fail(PML_E_UNSUPPORTED, "LHS.Y_LAPLACIAN equations run in FP32 or FP64");
  *sweeps_out = 0;
  const int64_t plane = static_cast<int64_t>(grid->n0) * grid->n1;
  const int64_t shape[3] = {grid->n0, grid->n1, 1};
  const double dx[3] = {grid->dx0, grid->dx1, 1.0};
  if (plane <= 0 || plane > total_elems || grid->state_offset != 0)
    return fail(PML_E_INVALID, "bad grid of a Poisson time loop");
  const int64_t fields = total_elems / plane;
  std::vector<JacobiGeom> geoms(n_poisson);
  hipStream_t st = as_stream(stream);
  auto *js = static_cast<JacobiState *>(jacobi_state);
  for (int k = 0; k < n_poisson; ++k) {
    if (field[k] < 0 || field[k] >= fields || source[k] < 0 || source[k] >= fields)
      return fail(PML_E_INVALID, "bad field of a Poisson equation");
    int64_t total = 0;
    if (int rc = jacobi_geom(precision, shape, 1, dx, ghost_lo + 3 * k, ghost_hi + 3 * k, &geoms[k],
                             &total);
        rc != PML_OK)
      return rc;
    bool resident = false;
    if (int rc = takes_resident(precision, plane, 1, geoms[k], ycons[k], kPoissonLoopUs, js, st,
                                &resident);
        rc != PML_OK || !resident)
      return rc;
  }
  const size_t esz = precision == PML_F64 ? 8 : 4;
  hipLaunchKernelGGL(k_jacobi_init, dim3(1), dim3(64), 0, st, js);
  PML_LAUNCH_CHECK();
  char *cur = static_cast<char *>(state), *nxt = static_cast<char *>(work);
  for (int64_t s = 0; s < n_steps; ++s) {
    if (int rc = fdm_step(eq_id, eq_params, n_params, integrator_id, precision, 2, grid, 1,
                          bc_values, cur, nxt, total_elems, dt, tile_config,
                          flags & PML_FLAG_AUTO, stream);
        rc != PML_OK)
      return rc;
    for (int k = 0; k < n_poisson; ++k) {
      // the pre-step state's source, the iteration started from its field
      const size_t f = static_cast<size_t>(field[k]) * plane * esz;
      const size_t q = static_cast<size_t>(source[k]) * plane * esz;
      const int rc =
          precision == PML_F64
              ? launch_resident<double>(reinterpret_cast<double *>(nxt + f),
                                        reinterpret_cast<const double *>(cur + f),
                                        reinterpret_cast<const double *>(cur + q), scale[k],
                                        plane, 1, geoms[k], ycons[k], tol, kResidentSweeps, js,
                                        st)
              : launch_resident<float>(reinterpret_cast<float *>(nxt + f),
                                       reinterpret_cast<const float *>(cur + f),
                                       reinterpret_cast<const float *>(cur + q),
                                       static_cast<float>(scale[k]), plane, 1, geoms[k],
                                       ycons[k], tol, kResidentSweeps, js, st);
      if (rc) return rc;
    }
    std::swap(cur, nxt);
    if (snapshots && (s + 1) % snapshot_every == 0)
      if (int rc = pml_to_f64(precision, cur, nullptr,
                              snapshots + ((s + 1) / snapshot_every - 1) * total_elems,
                              total_elems, stream);
          rc != PML_OK)
        return rc;
  }
  if (cur != state)
    PML_HIP_CHECK(
        hipMemcpyAsync(state, cur, total_elems * esz, hipMemcpyDeviceToDevice, st));
  JacobiState host;
  PML_HIP_CHECK(hipMemcpyAsync(&host, js, offsetof(JacobiState, partials), hipMemcpyDeviceToHost,
                               st));
  PML_HIP_CHECK(hipStreamSynchronize(st));
  *sweeps_out = host.pad ? 0 : host.sweeps;
  return PML_OK;
}
