// Many steps of small grids in one launch.
//
// fdm_deep advances a region of a grid -- an output tile and a halo of one
// vertex per stage of every step, clipped to the grid -- by `steps` steps in
// one workgroup: the state in registers, the stage inputs in two LDS buffers
// that the stages alternate between, one barrier a stage.  Vertices of the
// halo are computed with neighbours missing at the region's own border, and
// are wrong by one vertex more with every stage; the output tile is beyond
// their reach.  A grid that fits the region needs no halo and takes any
// number of steps.  Snapshots are written as their steps come by.
//
// Bound: a launch per step of a small grid is bound by the launch and by the
// latency of a pass over it (5 to 12 us whatever the size), here a stage is
// an LDS round trip, the arithmetic of a few vertices per thread and a
// barrier.  The arithmetic is that of the other kernels, operation by
// operation, so results do not depend on which of them runs.
#pragma once

#include <type_traits>

#include "pml_fdm_kernels.h"

namespace pml {

constexpr int kDeepThreads = 1024;
constexpr int kDeepLds = 144 * 1024;

struct DeepArgs {
  const TileDev *tiles;
  const GridDev *grids;
  const double *bc;
  const void *in_hi;
  const void *in_lo;
  void *out_hi;
  void *out_lo;
  void *snap_hi;
  void *snap_lo;
  double dt;
  double p[6];
  int64_t total;      // elements of one snapshot
  int64_t snap_idx;   // the next snapshot's index
  int snap_every;     // steps between snapshots
  int until;          // steps to the next snapshot (never reached: no snapshots)
  int n_tiles;
  int ndim;
  int oy, ox, halo;   // output tile and halo
  int steps;
};

using DeepFn = void (*)(DeepArgs);

// The kernels of a system, for regions of up to 1024 and (NULL: none) 2048
// vertices.
struct Deep {
  DeepFn fn[2] = {nullptr, nullptr};
  int fields = 0, stages = 0, value_bytes = 0;
  int most = 0;        // the largest region's vertices
  double units = 0.0;  // arithmetic of a vertex and stage (diffusion: 1)
  // LDS of a region: two buffers of stage inputs
  size_t lds(int64_t cells) const { return 2 * static_cast<size_t>(fields) * cells * value_bytes; }
};

template <class Eq, class Integ, class P, int PER>
__global__ void __launch_bounds__(kDeepThreads) fdm_deep(DeepArgs a) {
  using C = typename P::C;
  constexpr int F = Eq::F;
  constexpr int S = Eq::kInvariant ? 1 : Integ::kStages;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  if (tile >= a.n_tiles) return;  // the whole workgroup
  const TileDev T = a.tiles[tile];
  const GridDev G = a.grids[T.g];
  const int n0 = G.n0, n1 = G.n1;
  const int64_t plane = static_cast<int64_t>(n0) * n1;
  const bool ax0 = a.ndim == 2;
  const double *bcg = a.bc + G.bc;
  using D = typename std::conditional<P::kComp || sizeof(C) == 8, double, C>::type;
  const int64_t fstride = 4 * static_cast<int64_t>(n0 + n1);
  const StencilK<C> K(G);
  C pc[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) pc[i] = static_cast<C>(a.p[i]);
  const C dt = static_cast<C>(a.dt);
  const C hdt = static_cast<C>(a.dt * 0.5);

  // the region: rows r0 .. r0 + h, columns c0 .. c0 + w
  const int r0 = max(T.i0 - a.halo, 0), c0 = max(T.j0 - a.halo, 0);
  const int h = min(T.i0 + a.oy + a.halo, n0) - r0, w = min(T.j0 + a.ox + a.halo, n1) - c0;
  const int cells = h * w;
  const int tid = threadIdx.x, nt = blockDim.x;

  C *L = reinterpret_cast<C *>(smem);

  // Per vertex: the state, the stage sums and, where the vertex lies on an
  // edge of the grid, its Dirichlet value and the Neumann values along both
  // axes (NaN: none; they do not change in a launch).
  C yh[PER][F], yl[PER][F], acc[PER][F], alg[PER][F], g0[PER][F], g1[PER][F];
  D dv[PER][F];
  int row[PER], col[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int idx = tid + k * nt;
    row[k] = r0 + idx / w;
    col[k] = c0 + idx - (idx / w) * w;
    const int i = row[k], j = col[k];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      yh[k][f] = yl[k][f] = acc[k][f] = alg[k][f] = 0;
      g0[k][f] = g1[k][f] = static_cast<C>(NAN);
      dv[k][f] = static_cast<D>(NAN);
      if (idx < cells) {
        Store<P>::load(a.in_hi, a.in_lo, G.off + f * plane + static_cast<int64_t>(i) * n1 + j,
                       yh[k][f], yl[k][f]);
        L[f * cells + idx] = yh[k][f];
        const double *fb = bcg + f * fstride, *nb = fb + 2 * (n0 + n1);
        dv[k][f] = static_cast<D>(dirichlet_at(fb, n0, n1, i, j, ax0));
        if (ax0 && (i == 0 || i == n0 - 1)) g0[k][f] = static_cast<C>(nb[i == 0 ? j : n1 + j]);
        if (j == 0 || j == n1 - 1)
          g1[k][f] = static_cast<C>(nb[2 * n1 + (j == 0 ? i : n0 + i)]);
      }
    }
  }
  __syncthreads();

  // The output tile's values of this thread, where the state has them.
  auto write = [&](void *hi, void *lo, int64_t base) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = tid + k * nt;
      const int gi = row[k], gj = col[k];
      if (idx < cells && gi >= T.i0 && gi < T.i0 + a.oy && gj >= T.j0 && gj < T.j0 + a.ox) {
#pragma unroll
        for (int f = 0; f < F; ++f)
          Store<P>::store(hi, lo, base + G.off + f * plane + static_cast<int64_t>(gi) * n1 + gj,
                          yh[k][f], yl[k][f]);
      }
    }
  };

  const C *from = L;
  C *to = L + F * cells;
  int until = a.until;
  int64_t snap = a.snap_idx;
#pragma unroll 1
  for (int step = 0; step < a.steps; ++step) {
#pragma unroll
    for (int stage = 0; stage < S; ++stage) {
      const C weight = (!Eq::kInvariant && Integ::kStages == 2 && stage == 0) ? hdt : dt;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int idx = tid + k * nt;
        if (idx < cells) {
          const int i = row[k], j = col[k];
          const bool lo1 = j == 0, hi1 = j == n1 - 1;
          const bool lo0 = ax0 && i == 0, hi0 = ax0 && i == n0 - 1;
          // neighbours beyond the region: the vertex itself (see above)
          const int west = j > c0 ? idx - 1 : idx, east = j < c0 + w - 1 ? idx + 1 : idx;
          const int north = i > r0 ? idx - w : idx, south = i < r0 + h - 1 ? idx + w : idx;
          Quant<C> q[F];
#define PML_FQD(F_)                                                                           \
  if constexpr (F_ < F) {                                                                     \
    const C *y = from + F_ * cells;                                                           \
    field_quant_sel<C, Need<Eq, F_>::kL, Need<Eq, F_>::kD>(                                   \
        q[F_], y[idx], y[west], y[east], y[north], y[south], lo1, hi1, lo0, hi0, ax0,         \
        g1[k][F_], g1[k][F_], g0[k][F_], g0[k][F_], K);                                       \
  }
          PML_FQD(0)
          PML_FQD(1)
          PML_FQD(2)
          PML_FQD(3)
#undef PML_FQD
          C rr[F], ra[F];
#pragma unroll
          for (int f = 0; f < F; ++f) rr[f] = ra[f] = 0;
          Eq::template rhs<C>(pc, q, rr);
          if (Eq::kAlg != 0u) Eq::template alg<C>(pc, q, ra);
#pragma unroll
          for (int f = 0; f < F; ++f) {
            const bool is_alg = (Eq::kAlg >> f) & 1u;
            if (is_alg && stage == 0) alg[k][f] = ra[f];
            C nv = stage_update<Eq, Integ, P>(f, stage, weight * rr[f], alg[k][f], yh[k][f],
                                              yl[k][f], acc[k][f]);
            const bool fixed = dv[k][f] == dv[k][f];
            if (stage == S - 1 || is_alg) {
              C sh, sl;
              state_set<P>(sh, sl, static_cast<double>(dv[k][f]));
              yh[k][f] = fixed ? sh : yh[k][f];
              yl[k][f] = fixed ? sl : yl[k][f];
              nv = yh[k][f];
            } else {
              nv = fixed ? static_cast<C>(dv[k][f]) : nv;
            }
            to[f * cells + idx] = nv;
          }
        }
      }
      __syncthreads();
      C *t = const_cast<C *>(from);
      from = to;
      to = t;
    }
    if (--until == 0 && a.snap_hi) {
      write(a.snap_hi, a.snap_lo, snap * a.total);
      ++snap;
      until = a.snap_every;
    }
  }
  write(a.out_hi, a.out_lo, 0);
}

template <class EQ, class IN, class PR>
Deep deep_for() {
  Deep d;
  // two vertices a thread where they fit its 128 registers
  constexpr bool two =
      EQ::F == 1 || (EQ::F == 2 && (EQ::kD == 0u || sizeof(typename PR::C) == 4));
  d.fn[0] = &fdm_deep<EQ, IN, PR, 1>;
  if constexpr (two) d.fn[1] = &fdm_deep<EQ, IN, PR, 2>;
  d.fields = EQ::F;
  d.stages = EQ::kInvariant ? 1 : IN::kStages;
  d.value_bytes = sizeof(typename PR::C);
  d.most = (two ? 2 : 1) * kDeepThreads;
  d.units = __builtin_popcount(EQ::kLap) + 1.5 * __builtin_popcount(EQ::kD);
  return d;
}

template <class EQ, class PR>
Deep deep_by_int(int integ) {
  switch (integ) {
    case PML_INT_FE: return deep_for<EQ, IntFE, PR>();
    case PML_INT_MIDPOINT: return deep_for<EQ, IntMidpoint, PR>();
    case PML_INT_RK4: return deep_for<EQ, IntRK4, PR>();
    default: return Deep{};
  }
}

template <class PR>
Deep deep_table(int eq, int integ, int ndim) {
  switch (eq) {
    case PML_EQ_DIFFUSION: return deep_by_int<EqDiffusion, PR>(integ);
    case PML_EQ_CONVECTION_DIFFUSION: return deep_by_int<EqConvectionDiffusion, PR>(integ);
    case PML_EQ_WAVE: return deep_by_int<EqWave, PR>(integ);
    case PML_EQ_CAHN_HILLIARD: return deep_by_int<EqCahnHilliard, PR>(integ);
    case PML_EQ_BURGERS:
      return ndim == 1 ? deep_by_int<EqBurgers1, PR>(integ) : deep_by_int<EqBurgers2, PR>(integ);
    case PML_EQ_SHALLOW_WATER: return deep_by_int<EqShallowWater, PR>(integ);
    case PML_EQ_NAVIER_STOKES: return deep_by_int<EqNavierStokes, PR>(integ);
    default: return Deep{};
  }
}

// One per precision (pml_fdm_deep_<prec>.hip).
Deep fdm_deep_f32(int eq, int integ, int ndim);
Deep fdm_deep_f64(int eq, int integ, int ndim);
Deep fdm_deep_f32c(int eq, int integ, int ndim);

}  // namespace pml
