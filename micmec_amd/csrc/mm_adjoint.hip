// Differentiation form: energy, node gradient, virial, domain-vector gradient and the gradient
// with respect to every cell-type parameter, optionally in dual numbers.
//
// Energy model: micmec/pes/nanocell.py:40-132 (eight corner matrices) and
// nanocell_original.py:46-132 (averaged matrix), combined over metastable states by the
// free-energy log-sum-exp of micmec/pes/mmff.py:380-398. The reference differentiates only with
// respect to positions (mmff.py:384-398; mmff_jax.py:249-250 also with respect to a deformation);
// the parameter derivatives have no counterpart there.
//
// In double precision the kernel returns first derivatives of the energy. With dual numbers
// (value, tangent) and a tangent direction (dpos, drvecs) the same pass also returns the
// directional derivative of each first derivative: the tangent of gpos is a Hessian-vector
// product and the tangent of dE/dtheta is (d^2E / dtheta dr) . dr, the quantity the parameter
// gradient of a loss on forces and stresses needs (forward-over-reverse).
//
// Parameter entries per (table row, state), kNps = 32 of them:
//   [0..20]  dE/dCv, Cv the 6x6 Voigt matrix in u = e.Cv.e / 2: 1/2 sum e_I e_J for I <= J
//            (upper triangle, row by row); the full 6x6 gradient is that entry at (I,J) and (J,I)
//   [21..29] dE/dP, P = h0^-1 (row-major)
//   [30]     dE/dw, w = det(h0)/8 (eight-corner model) or det(h0) (averaged model)
//   [31]     dE/d(free energy) = p_s, the state's Boltzmann weight
// followed by one entry per row, dE/d(kT). The caller maps (Cv, P, w, kT) to (Cv, h0, T_eff).
// They are bilinear in the corners' strains, so the kernel works in the metric of the edges as
// the force kernels do (mm_device.h): with x the six Gram entries of a corner less the state's
// rest metric and p_s the state's weight it sums p_s x_I x_J (21), p_s x_I (6) and p_s, and
// metric_entries_kernel turns the sums of a (row, state) into its 32 entries.
//
// Lanes: one per cell, one wave per block. Blocks lie inside one 256-slot segment of the work
// order, so the type row and the system are uniform per block.
//
// HBM layout of the outputs:
//   part   [2 * kSysQ][W / 64]     per block: energy, virial (9), domain-vector gradient (9);
//                                  rows kSysQ.. hold the tangents
//   ppart  [2 * npar][W / 64]      per block: row 2i value, 2i + 1 tangent of metric sum i of a
//                                  state's 32 (0..20 x x, 21..26 x, 27 p), or of dE/d(kT)
//   gcell, gcell2 [4][3][S]        vertex gradients and their tangents, as the cell pass's
//                                  face-class records (mm_force.hip), gathered into gpos
// All sums run in a fixed order; there are no floating-point atomics.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "../../include/micmec_amd.h"
#include "mm_cell.h"
#include "mm_device.h"
#include "mm_internal.h"
#include "mm_kernels.h"

namespace mm {

struct Dual {
  double v, d;
};

__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ Dual operator-(Dual a) { return {-a.v, -a.d}; }
__device__ __forceinline__ Dual operator*(Dual a, Dual b) {
  return {a.v * b.v, a.v * b.d + a.d * b.v};
}
__device__ __forceinline__ Dual operator*(double a, Dual b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ Dual operator-(Dual a, double b) { return {a.v - b, a.d}; }
__device__ __forceinline__ Dual operator-(double a, Dual b) { return {a - b.v, -b.d}; }
__device__ __forceinline__ Dual operator+(Dual a, double b) { return {a.v + b, a.d}; }
__device__ __forceinline__ Dual operator/(Dual a, double b) { return {a.v / b, a.d / b}; }
__device__ __forceinline__ Dual operator/(Dual a, Dual b) {
  const double q = a.v / b.v;
  return {q, (a.d - q * b.d) / b.v};
}
__device__ __forceinline__ Dual dexp(Dual a) {
  const double e = exp(a.v);
  return {e, e * a.d};
}
__device__ __forceinline__ Dual dlog(Dual a) { return {log(a.v), a.d / a.v}; }
__device__ __forceinline__ double dexp(double a) { return exp(a); }
__device__ __forceinline__ double dlog(double a) { return log(a); }
__device__ __forceinline__ double val(double a) { return a; }
__device__ __forceinline__ double val(Dual a) { return a.v; }
__device__ __forceinline__ double tan_(double) { return 0.0; }
__device__ __forceinline__ double tan_(Dual a) { return a.d; }
template <typename T> __device__ __forceinline__ T make(double v, double d);
template <> __device__ __forceinline__ double make<double>(double v, double) { return v; }
template <> __device__ __forceinline__ Dual make<Dual>(double v, double d) { return {v, d}; }
template <typename T> struct IsDual { static constexpr bool value = false; };
template <> struct IsDual<Dual> { static constexpr bool value = true; };

// a b + c, fused in every component.
__device__ __forceinline__ double mad(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__device__ __forceinline__ Dual mad(Dual a, Dual b, Dual c) {
  return {__builtin_fma(a.v, b.v, c.v), __builtin_fma(a.v, b.d, __builtin_fma(a.d, b.v, c.d))};
}
__device__ __forceinline__ Dual mad(double a, Dual b, Dual c) {
  return {__builtin_fma(a, b.v, c.v), __builtin_fma(a, b.d, c.d)};
}
// Keeps the work on either side of it apart.
__device__ __forceinline__ void fence(double& a) { asm("" : "+v"(a)); }
__device__ __forceinline__ void fence(Dual& a) { asm("" : "+v"(a.v), "+v"(a.d)); }

// Upper triangle of the 6x6 Voigt matrix, row by row: entry q is (kUpperI[q], kUpperJ[q]).
__device__ constexpr int kUpperI[21] = {0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 3, 4, 4, 5};
__device__ constexpr int kUpperJ[21] = {0, 1, 2, 3, 4, 5, 1, 2, 3, 4, 5, 2, 3, 4, 5, 3, 4, 5, 4, 5, 5};

constexpr int kAdjCells = 64;  // cells per block
constexpr int kAdjPerSeg = kCellBlock / kAdjCells;  // adjoint blocks per cell-pass block
static_assert(kCellBlock % kAdjCells == 0, "cell-pass blocks hold whole adjoint blocks");
constexpr int kNps = 32;       // parameter entries per (row, state)
constexpr int kSysQ = 19;      // energy, virial (9), domain-vector gradient (9)

// Sums over the wave of NQ quantities q(0), q(1), ... (dual numbers: values and tangents) by the
// reduce-scatter butterfly; put(i, half, sum) is called on one lane per quantity and half.
// Without dual numbers the tangents are zero.
template <int NQ, typename T, typename Quantity, typename Put>
__device__ __forceinline__ void wave_sums(Quantity q, Put put) {
  const int lane = threadIdx.x & 63, at = scatter_index(lane);
  constexpr int n0 = NQ < 16 ? NQ : 16, n1 = NQ - n0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    auto part = [&](int i) { return h == 0 ? val(q(i)) : tan_(q(i)); };
    double t = 0.0, u = 0.0;
    if (h == 0 || IsDual<T>::value) {
      double c[n0];
#pragma unroll
      for (int i = 0; i < n0; ++i) c[i] = part(i);
      t = wave_reduce_scatter<n0>(c, lane);
      if constexpr (n1 > 0) {
        double d[n1];
#pragma unroll
        for (int i = 0; i < n1; ++i) d[i] = part(16 + i);
        u = wave_reduce_scatter<n1>(d, lane);
      }
    }
    if ((lane & 3) == 0) {
      if (at < n0) put(at, h, t);
      if (n1 > 0 && at < n1) put(16 + at, h, u);
    }
  }
}

// Strain x of the i-th corner in the metric of the edges (Gram entries less the rest metric,
// halved on the diagonal) from the edges E and their strains q against that of the type's first
// state, its stress K x: the diagonal entries added to their edges' D, the others
// in O; returns x . K x.
template <typename T, int kModel>
__device__ __forceinline__ T adjoint_corner(const const_f64 ts, int i,
                                            const T (&E)[Frame<kModel>::NE][3],
                                            const T (&q)[Frame<kModel>::NE], T (&x)[6],
                                            T (&D)[Frame<kModel>::NE], T (&O)[3]) {
  using F = Frame<kModel>;
  const const_f64 K = ts + kMetricOffset, R = ts + kRestOffset;
  const int a = F::corner(i);
#pragma unroll
  for (int d = 0; d < 3; ++d) x[d] = q[F::edge(a, d)] + ts[kShiftOffset + d];
#pragma unroll
  for (int o = 0; o < 3; ++o) {
    const T(&A)[3] = E[F::edge(a, F::axis0(o))];
    const T(&B)[3] = E[F::edge(a, F::axis1(o))];
    x[3 + o] = mad(A[2], B[2], mad(A[1], B[1], mad(A[0], B[0], make<T>(-R[3 + o], 0.0)))) -
               ts[kRestLowOffset + 3 + o];
  }
  T u = make<T>(0.0, 0.0);
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    T t = K[6 * I] * x[0];
#pragma unroll
    for (int J = 1; J < 6; ++J) t = mad(K[6 * I + J], x[J], t);
    u = mad(x[I], t, u);
    if (I < 3) {
      const int e = F::edge(a, I);
      D[e] = F::first(e) < i ? D[e] + t : t;
    } else {
      O[I < 3 ? 0 : I - 3] = t;
    }
  }
  return u;
}

// Column q of a lane's LDS (64 lanes side by side; a dual number takes two).
template <typename T>
__device__ __forceinline__ T get_column(const double* col, int q) {
  return IsDual<T>::value ? make<T>(col[128 * q], col[128 * q + 64]) : make<T>(col[64 * q], 0.0);
}
template <typename T>
__device__ __forceinline__ void put_column(double* col, int q, T v) {
  col[(IsDual<T>::value ? 128 : 64) * q] = val(v);
  if (IsDual<T>::value) col[128 * q + 64] = tan_(v);
}

// Energy of a cell, dE/dkT, the stresses weighted by the states' p_s in the lane's columns (edge
// e's diagonal in e, the others of the i-th corner behind them, then the states' energies), and
// the metric sums of every state over the wave (put_sum(state, quantity, half, sum)).
template <typename T, int kModel, bool kMulti, typename PutSum>
__device__ __forceinline__ void adjoint_states(const const_f64 tab, int ns, double kt,
                                               const T (&E)[Frame<kModel>::NE][3],
                                               const T (&sq)[Frame<kModel>::NE], bool valid,
                                               double* col, T& ecell, T& dkt, PutSum put_sum) {
  using F = Frame<kModel>;
  constexpr int NE = F::NE, NC = F::NC, NS = NE + 3 * NC;
  T zsum = make<T>(1.0, 0.0);
  double emin = 0.0;
  if (kMulti) {
    // pass 1: E_s = sum_a w u_a + f_s (mmff.py:380-384) and Z = sum_s exp(-(E_s - E_min)/kT), which
    // the weights of pass 2 need first; E = E_min - kT ln Z (mmff.py:386-395)
    for (int s = 0; s < ns; ++s) {
      const const_f64 ts = tab + s * kTabStride;
      T D[NE], u = make<T>(0.0, 0.0);
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        T x[6], O[3];
        u = u + adjoint_corner<T, kModel>(ts, i, E, sq, x, D, O);
        fence(u);
      }
      const T es = 0.5 * u + ts[10];
      put_column(col, NS + s, es);
      emin = (s == 0 || val(es) < emin) ? val(es) : emin;
    }
    zsum = make<T>(0.0, 0.0);
    for (int s = 0; s < ns; ++s) zsum = zsum + dexp(-(get_column<T>(col, NS + s) - emin) / kt);
    const T lnz = dlog(zsum);
    ecell = emin - kt * lnz;
    // dE/dkT = -ln Z - sum_s p_s (E_s - E_min) / kT
    dkt = -lnz;
  }
  if (kMulti) {
#pragma unroll
    for (int q = 0; q < NS; ++q) put_column(col, q, make<T>(0.0, 0.0));
  }
  // pass 2: stresses weighted by p_s (mmff.py:396-398) and the metric sums
  for (int s = 0; s < ns; ++s) {
    const const_f64 ts = tab + s * kTabStride;
    T D[NE], u = make<T>(0.0, 0.0), ps = make<T>(1.0, 0.0);
    if (kMulti) {
      const T d = get_column<T>(col, NS + s) - emin;
      ps = dexp(-d / kt) / zsum;
      dkt = dkt - (ps * d) / kt;
    }
    auto add = [&](int q, T v) {
      if (kMulti) v = mad(ps, v, get_column<T>(col, q));
      put_column(col, q, v);
    };
    T X2[21], X1[6];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      T x[6], O[3];
      u = u + adjoint_corner<T, kModel>(ts, i, E, sq, x, D, O);
#pragma unroll
      for (int q = 0; q < 21; ++q)
        X2[q] = i == 0 ? x[kUpperI[q]] * x[kUpperJ[q]] : mad(x[kUpperI[q]], x[kUpperJ[q]], X2[q]);
#pragma unroll
      for (int I = 0; I < 6; ++I) X1[I] = i == 0 ? x[I] : X1[I] + x[I];
#pragma unroll
      for (int o = 0; o < 3; ++o) add(NE + 3 * i + o, O[o]);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int e = F::edge(F::corner(i), d);
        if (F::last(e) == i) add(e, D[e]);
      }
      fence(u);
#pragma unroll
      for (int q = 0; q < 21; ++q) fence(X2[q]);
    }
    if (!kMulti) ecell = 0.5 * u + ts[10];
    if (kMulti) {
#pragma unroll
      for (int q = 0; q < 21; ++q) X2[q] = ps * X2[q];
#pragma unroll
      for (int I = 0; I < 6; ++I) X1[I] = ps * X1[I];
    }
    wave_sums<28, T>(
        [&](int q) -> T {
          const T v = q < 21 ? X2[q] : q < 27 ? X1[q - 21] : ps;
          return valid ? v : make<T>(0.0, 0.0);
        },
        [&](int q, int half, double t) { put_sum(s, q, half, t); });
  }
}

// One lane a cell, one wave a block: the eight corners of a cell follow each other on the lane, so
// that its sums over the corners need no exchange between lanes and an edge's square and gradient
// are formed once; the 56 sums of a state over the wave are one butterfly for 64 cells. The edges
// (36 dual numbers) stay in registers, in part in accumulation registers, one wave a SIMD; the
// stresses, weighted over the states, go through LDS (36 KB a wave, four waves a CU). The waves' own
// instructions bound it (5000 for one state, 9500 for two, six in ten of them FP64): 64
// configurations of 16^3 cells, eight-corner model with tangents, 206 us with one lane a corner and
// products with P per corner, 154 us with one lane a corner in the metric of the edges, 103 us so
// (94 us where positions need no gradient and no records are stored);
// 5 of 7^3 cells with the averaged model 18.7, 13.1 and 15.5 us. A field of a few waves takes one
// wave's time, which the cells' lanes make longer: eight-corner model, 2 of 5^3 cells 14.9 us with
// one lane a corner, 24.6 us so, 8 of 12^3 19.9 and 26.7 us (a product of either, DiffField.vjp, 43.5
// and 46 us, the launches being fewer).
template <typename T, int kModel>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1)))
adjoint_kernel(const double* __restrict__ pos, const double* __restrict__ dpos,
               const double* __restrict__ rvecs, const double* __restrict__ drvecs,
               const int32_t* __restrict__ blk_sys, const int32_t* __restrict__ cnode,
               const int32_t* __restrict__ cwrap, const int32_t* __restrict__ blk_row,
               const double* __restrict__ tab_g, const double* __restrict__ kt_g,
               const int32_t* __restrict__ nstates_g, int32_t max_states, int64_t W,
               const int32_t* __restrict__ cbase, int64_t S, double* __restrict__ gcell,
               double* __restrict__ gcell2, double* __restrict__ part,
               double* __restrict__ ppart) {
  using F = Frame<kModel>;
  constexpr int NE = F::NE, NC = F::NC;
  extern __shared__ double st_sh[];  // columns: the stresses, then the states' energies
  const int64_t nblk = gridDim.x;
  const int seg = blockIdx.x / kAdjPerSeg;
  const int trow = blk_row[seg];
  const int sys = blk_sys[seg];
  const int ns = nstates_g[trow];
  const double kt = kt_g[trow];
  const const_f64 tab = (const_f64)tab_g + (int64_t)trow * max_states * kTabStride;
  const int lane = threadIdx.x;
  const int64_t w = (int64_t)blockIdx.x * kAdjCells + lane;
  int n[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) n[k] = cnode[w * 8 + k];
  const bool valid = n[0] >= 0;
  const int wrap = valid ? cwrap[w] : 0;
  auto stress = [&](int q) -> T { return get_column<T>(st_sh + lane, q); };

  // edges (mmff.py:347-371): differences of the corners' positions plus the domain vector of the
  // edge's axis when the cell wraps along it (a factor 0 or 1; a padding slot reads node 0)
  T E[NE][3], sq[NE];
  {
    T p[8][3], t[12][3];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t i = 3 * (int64_t)(valid ? n[k] : 0);
#pragma unroll
      for (int j = 0; j < 3; ++j) p[k][j] = make<T>(pos[i + j], dpos ? dpos[i + j] : 0.0);
    }
#pragma unroll
    for (int e = 0; e < 12; ++e) {
      const int d = e / 4;
      const double f = (double)((wrap >> d) & 1);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int q = 9 * sys + 3 * d + j;
        t[e][j] = mad(f, make<T>(rvecs[q], drvecs ? drvecs[q] : 0.0),
                      p[kEdgeHi[e]][j] - p[kEdgeLo[e]][j]);
      }
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        E[e][j] = kModel == 0 ? t[e][j]
                              : 0.25 * ((t[4 * e % 12][j] + t[(4 * e + 1) % 12][j]) +
                                        (t[(4 * e + 2) % 12][j] + t[(4 * e + 3) % 12][j]));
      // the strain (E.E)/2 - R, the sum begun as in edge_strain
      const int d = F::along(e), b = d == 0 ? 1 : 0, c = d == 2 ? 1 : 2;
      const T r = make<T>(-tab[kRestOffset + d], 0.0);
      sq[e] = mad(0.5, mad(E[e][c], E[e][c], mad(E[e][b], E[e][b], mad(E[e][d], E[e][d], r))),
                  make<T>(-tab[kRestLowOffset + d], 0.0));
    }
  }

  T ecell = make<T>(0.0, 0.0), dkt = make<T>(0.0, 0.0);
  auto put_sum = [&](int s, int q, int half, double t) {
    ppart[((int64_t)2 * (s * kNps + q) + half) * nblk + blockIdx.x] = t;
  };
  if (ns > 1)
    adjoint_states<T, kModel, true>(tab, ns, kt, E, sq, valid, st_sh + lane, ecell, dkt, put_sum);
  else
    adjoint_states<T, kModel, false>(tab, 1, kt, E, sq, valid, st_sh + lane, ecell, dkt, put_sum);

  // dE/d(edge) = D_e E_e + the rows of S M off the diagonal (edge_gradient): an edge closes at its
  // second corner and pulls at its upper vertex, pushes at its lower one (averaged model: a
  // quarter of the mean edge's at every vertex), adds gE (x) E to the virial and, when the cell
  // wraps along its axis, gE to that domain vector's gradient
  T gE[NE][3], g[8][3], vir[6], gdom[3][3];
#pragma unroll
  for (int v = 0; v < 8; ++v)
#pragma unroll
    for (int j = 0; j < 3; ++j) g[v][j] = make<T>(-0.0, -0.0);
#pragma unroll
  for (int v = 0; v < 6; ++v) vir[v] = make<T>(0.0, 0.0);
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int j = 0; j < 3; ++j) gdom[d][j] = make<T>(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int a = F::corner(i);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::first(e) == i) {
        const T De = stress(e);
#pragma unroll
        for (int j = 0; j < 3; ++j) gE[e][j] = De * E[e][j];
      }
    }
#pragma unroll
    for (int o = 0; o < 3; ++o) {
      const int e0 = F::edge(a, F::axis0(o)), e1 = F::edge(a, F::axis1(o));
      const T Oo = stress(NE + 3 * i + o);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        gE[e0][j] = mad(Oo, E[e1][j], gE[e0][j]);
        gE[e1][j] = mad(Oo, E[e0][j], gE[e1][j]);
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::last(e) != i) continue;
      constexpr int kK[6] = {0, 1, 2, 1, 0, 0}, kL[6] = {0, 1, 2, 2, 2, 1};
#pragma unroll
      for (int v = 0; v < 6; ++v) vir[v] = mad(gE[e][kK[v]], E[e][kL[v]], vir[v]);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        gdom[d][j] = gdom[d][j] + gE[e][j];
        if (kModel == 0) {
          g[kEdgeHi[e]][j] = g[kEdgeHi[e]][j] + gE[e][j];
          g[kEdgeLo[e]][j] = g[kEdgeLo[e]][j] - gE[e][j];
        } else {
          const T t = 0.25 * gE[e][j];
#pragma unroll
          for (int v = 0; v < 8; ++v) g[v][j] = kOff[v][d] ? g[v][j] + t : g[v][j] - t;
        }
      }
    }
  }
  wave_sums<17, T>(
      [&](int q) -> T {
        T t = q == 0 ? ecell : q < 7 ? vir[(q - 1) % 6] : q < 16 ? gdom[(q - 7) / 3 % 3][(q - 7) % 3] : dkt;
        if (q >= 7 && q < 16) t = (double)((wrap >> ((q - 7) / 3)) & 1) * t;
        return valid ? t : make<T>(0.0, 0.0);
      },
      [&](int q, int half, double t) {
        if (q == 16) {
          ppart[((int64_t)2 * max_states * kNps + half) * nblk + blockIdx.x] = t;
          return;
        }
        // rows of the energy, of the full 3x3 virial (both copies of an off-diagonal entry) and of
        // the domain-vector gradient, as nibbles
        const int row = q < 7 ? (int)(0x2369510ull >> (4 * q)) & 0xf : q + 3;
        double* out = part + (int64_t)(half * kSysQ) * nblk + blockIdx.x;
        out[(int64_t)row * nblk] = t;
        if (q >= 4 && q < 7) out[(int64_t)((int)(0x478ull >> (4 * (q - 4))) & 0xf) * nblk] = t;
      });
  if (!gcell) return;  // no position gradient wanted
  double gv[8][3];
#pragma unroll
  for (int v = 0; v < 8; ++v)
#pragma unroll
    for (int j = 0; j < 3; ++j) gv[v][j] = valid ? val(g[v][j]) : -0.0;
  store_cell(w, wrap, valid, cbase, W, S, gcell, gv);
  if (IsDual<T>::value) {
#pragma unroll
    for (int v = 0; v < 8; ++v)
#pragma unroll
      for (int j = 0; j < 3; ++j) gv[v][j] = valid ? tan_(g[v][j]) : -0.0;
    store_cell(w, wrap, valid, cbase, W, S, gcell2, gv);
  }
}

// Where the gradients of the parameter tensors go (mm_adjoint_param_grads; cv null: not wanted).
struct GradOut {
  const double* h0;
  int corner8;
  double boltzmann;
  double *cv, *h, *free, *teff;
};

// Gradients of (Cv, h0, free energy) of (row, state) t from its 32 entries ent (LDS), by one wave:
// the 21 upper-triangle entries give the symmetric Voigt gradient, P^T = cof / det with the rows
// r1 x r2, r2 x r0, r0 x r1 of cof, dE/dh0 = -P^T (dE/dP) P^T + (dE/dw) w P^T with w = det / 8
// (corner8) or det, an entry a lane; zeros for a state that the row does not have (!on).
__device__ __forceinline__ void state_gradients(const double* ent, bool on, int64_t t,
                                                const GradOut& o) {
  const int lane = threadIdx.x;
  if (lane < 36) {
    const int I = lane / 6, J = lane % 6, a = I < J ? I : J, b = I < J ? J : I;
    o.cv[t * 36 + lane] = on ? ent[6 * a - a * (a - 1) / 2 + b - a] : 0.0;
  }
  if (lane < 9) {
    const double* h = o.h0 + t * 9;
    const int i = lane / 3, j = lane % 3;
    double pt[9], m1[3];
    for (int a = 0; a < 3; ++a) {
      const double* u = h + 3 * ((a + 1) % 3);
      const double* v = h + 3 * ((a + 2) % 3);
      pt[3 * a + 0] = u[1] * v[2] - u[2] * v[1];
      pt[3 * a + 1] = u[2] * v[0] - u[0] * v[2];
      pt[3 * a + 2] = u[0] * v[1] - u[1] * v[0];
    }
    const double det = (h[0] * pt[0] + h[1] * pt[1]) + h[2] * pt[2];
    for (int k = 0; k < 9; ++k) pt[k] = pt[k] / det;
    const double p0 = pt[3 * i], p1 = pt[3 * i + 1], p2 = pt[3 * i + 2];
    for (int k = 0; k < 3; ++k) m1[k] = (p0 * ent[21 + k] + p1 * ent[24 + k]) + p2 * ent[27 + k];
    const double m2 = (m1[0] * pt[j] + m1[1] * pt[3 + j]) + m1[2] * pt[6 + j];
    const double w = o.corner8 ? det / 8.0 : det;
    o.h[t * 9 + lane] = on ? -m2 + ent[30] * w * pt[3 * i + j] : 0.0;
  }
  if (lane == 0) o.free[t] = on ? ent[31] : 0.0;
}

// The 32 parameter entries of every (row, state) from its metric sums, in place in params
// [nrows][npar][2]: with T the map of x to the engineering strain e = T x (metric_entry),
// X2 = sum p x x^T and X1 = sum p x, S = Cv T x the stress and G = 2 x + R the Gram matrix,
//   dE/dCv = w T X2 T^T / 2,  dE/dP_ik = w sum_mn P_mn (sum p S_im G_nk),
//   dE/dw = tr(Cv^T T X2 T^T) / 2,
// all linear in the sums, so values and tangents alike; zeros for a state that the row does not
// have. One wave per (row, state); lane 32 h + i works on half h. With grads.cv the gradients of the
// parameter tensors, from values plus tangents, are formed too.
__global__ void __launch_bounds__(64)
metric_entries_kernel(const double* __restrict__ tab, const int32_t* __restrict__ nstates,
                      int max_states, int64_t npar, double* __restrict__ params, GradOut grads) {
  const int row = blockIdx.x / max_states, s = blockIdx.x % max_states;
  __shared__ double ent[32];
  if (grads.cv && s == 0 && threadIdx.x == 0) {
    const double* e = params + 2 * (row * npar + (int64_t)max_states * kNps);
    grads.teff[row] = (e[0] + e[1]) * grads.boltzmann;
  }
  double* out = params + 2 * (row * npar + (int64_t)s * kNps);
  if (s >= nstates[row]) {
    // the sums of a state that the row no longer has are those of an earlier evaluation
    out[threadIdx.x] = 0.0;
    if (grads.cv) state_gradients(ent, false, blockIdx.x, grads);
    return;
  }
  const double* ts = tab + (int64_t)blockIdx.x * kTabStride;
  const double* C = ts + kCvOffset;
  const double* R = ts + kRestOffset;
  const double w = ts[9];
  __shared__ double T[36], P[9], X2[2][36], X1[2][6], A[2][36], E[2][36], Q[2][36], B[2][6], p[2];
  const int h = threadIdx.x >> 5, i = threadIdx.x & 31;
  if (threadIdx.x < 9) P[threadIdx.x] = ts[threadIdx.x];
  if (i < 28) {
    const double v = out[2 * i + h];
    if (i < 21)
      X2[h][6 * kUpperI[i] + kUpperJ[i]] = X2[h][6 * kUpperJ[i] + kUpperI[i]] = v;
    else if (i < 27)
      X1[h][i - 21] = v;
    else
      p[h] = v;
  }
  __syncthreads();
  if (threadIdx.x < 36) T[threadIdx.x] = strain_map(P, threadIdx.x / 6, threadIdx.x % 6);
  __syncthreads();
  for (int q = i; q < 36; q += 32) {
    double t = 0.0;
    for (int k = 0; k < 6; ++k) t += T[6 * (q / 6) + k] * X2[h][6 * k + q % 6];
    A[h][q] = t;
  }
  __syncthreads();
  for (int q = i; q < 36; q += 32) {
    double t = 0.0, c = 0.0;
    for (int k = 0; k < 6; ++k) {
      t += A[h][6 * (q / 6) + k] * T[6 * (q % 6) + k];
      c += C[6 * (q / 6) + k] * A[h][6 * k + q % 6];
    }
    E[h][q] = t;
    Q[h][q] = c;
  }
  if (i < 6) {
    double t = 0.0;
    for (int k = 0; k < 6; ++k)
      for (int l = 0; l < 6; ++l) t += (C[6 * i + k] * T[6 * k + l]) * X1[h][l];
    B[h][i] = t;
  }
  __syncthreads();
  double v = 0.0;
  if (i < 21) {
    v = 0.5 * (w * E[h][6 * kUpperI[i] + kUpperJ[i]]);
  } else if (i < 30) {
    constexpr int kVoigt[9] = {0, 5, 4, 5, 1, 3, 4, 3, 2};
    const int a = (i - 21) / 3, k = (i - 21) % 3;
    for (int m = 0; m < 3; ++m)
      for (int n = 0; n < 3; ++n) {
        const int sm = kVoigt[3 * a + m], gn = kVoigt[3 * n + k];
        const double q = Q[h][6 * sm + gn];
        v += P[3 * m + n] * (B[h][sm] * R[gn] + (n == k ? 2.0 * q : q));
      }
    v *= w;
  } else if (i == 30) {
    for (int q = 0; q < 36; ++q) v += C[q] * E[h][q];
    v *= 0.5;
  } else {
    v = p[h];
  }
  out[2 * i + h] = v;
  if (!grads.cv) return;
  const double d = __shfl_down(v, 32, 64);
  if (h == 0) ent[i] = v + d;
  __syncthreads();
  state_gradients(ent, true, blockIdx.x, grads);
}

// Row sums of per-block partials over lists of segments (kAdjPerSeg blocks each). Rows q with
// q % weight_every == 0 are scaled per segment by weight[system of the segment] when weight is given.
struct SegmentSums {
  const double* part;
  int lists, nrows_part;  // outputs [list][row of part]
  const int32_t *list_ptr, *list_idx;
  const double* weight;
  int weight_every;
  double* out;
};

// One block per (list, row): first those of x, then those of y.
__global__ void __launch_bounds__(256)
segment_sum_kernel(SegmentSums x, SegmentSums y, int64_t nblk, const int32_t* __restrict__ blk_sys) {
  __shared__ double red[4];
  const int nx = x.lists * x.nrows_part;
  const bool first = (int)blockIdx.x < nx;
  const SegmentSums a = first ? x : y;
  const int at = first ? blockIdx.x : blockIdx.x - nx;
  const int li = at / a.nrows_part;
  const int q = at % a.nrows_part;
  const bool weighted = a.weight != nullptr && (q % a.weight_every) == 0;
  const int i0 = a.list_ptr[li], i1 = a.list_ptr[li + 1];
  double acc = 0.0;
  for (int i = i0 + threadIdx.x; i < i1; i += 256) {
    const int seg = a.list_idx[i];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kAdjPerSeg; ++k)
      s += a.part[(int64_t)q * nblk + (int64_t)seg * kAdjPerSeg + k];
    acc += weighted ? a.weight[blk_sys[seg]] * s : s;
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) a.out[at] = ((red[0] + red[1]) + red[2]) + red[3];
}

// A force-and-stress loss (mm_fit_loss) whose cotangents are formed where they are used:
//   gG = gl 2 (g - gt) / (3 N f_scale),  gV = gl 2 (v inv - vt) inv / (9 nsys s_scale).
struct FitTerms {
  const double *g, *gt, *v, *vt, *inv;  // [N][3], [N][3], [nsys][9], [nsys][9], [nsys]
  const double* gl;                     // the loss' own cotangent
  double cf, cs;                        // 2 / (3 N f_scale), 2 / (9 nsys s_scale)
  double* gV;                           // [nsys][9], for the kernels after the direction
  __device__ double stress(int64_t sy, int q) const {
    return *gl * cs * (v[9 * sy + q] * inv[sy] - vt[9 * sy + q]) * inv[sy];
  }
};

// Tangent direction of a vector-Jacobian product from the cotangents (gE, gG, gV) of
// (E, gpos, vtens): dpos_n = gG_n + pos_n gV_s^T (s = node_sys[n]), and for the threads past the
// nodes drvecs_s = rvecs_s gV_s^T. gG or gV may be null (zero); kFit: those of the loss.
template <bool kFit>
__global__ void __launch_bounds__(256)
vjp_direction_kernel(const double* __restrict__ pos, const double* __restrict__ rvecs,
                     const int32_t* __restrict__ node_sys, const double* __restrict__ gG,
                     const double* __restrict__ gV, FitTerms fit, int64_t N, int nsys,
                     double* __restrict__ dpos, double* __restrict__ drv) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  auto stress = [&](int64_t sy, int q) { return kFit ? fit.stress(sy, q) : gV[9 * sy + q]; };
  if (t < N) {
    const bool on = kFit || gV;
    const int64_t sy = on ? node_sys[t] : 0;
    const double cf = kFit ? *fit.gl * fit.cf : 0.0;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      double d = kFit ? cf * (fit.g[3 * t + l] - fit.gt[3 * t + l]) : gG ? gG[3 * t + l] : 0.0;
      if (on)
        d += (pos[3 * t] * stress(sy, 3 * l) + pos[3 * t + 1] * stress(sy, 3 * l + 1)) +
             pos[3 * t + 2] * stress(sy, 3 * l + 2);
      dpos[3 * t + l] = d;
    }
  } else if (t < N + 9 * (int64_t)nsys) {
    const int64_t q = t - N;
    const int64_t sy = q / 9;
    const int dd = (int)(q % 9) / 3, l = (int)(q % 3);
    const double* R = rvecs + 9 * sy;
    double d = 0.0;
    if (kFit || gV)
      d = (R[3 * dd] * stress(sy, 3 * l) + R[3 * dd + 1] * stress(sy, 3 * l + 1)) +
          R[3 * dd + 2] * stress(sy, 3 * l + 2);
    drv[q] = d;
    if (kFit) fit.gV[q] = stress(sy, (int)(q % 9));
  }
}

// The product's position cotangent, g_n = gE_s gpos_n + dgpos_n + gpos_n gV_s, from the vertex
// gradients' and their tangents' records (nb blocks, none when g_pos is null), and beyond them the
// domain vectors' (g_rv, null: none), dL/drvecs = gE dE/drvecs + d(dE/drvecs) + (dE/drvecs) gV,
// from sys_out. gV may be null: zero. One pass in place of two gathers and a pass over their
// results.
template <bool kAllLoads>
__global__ void __launch_bounds__(256)
vjp_output_kernel(const int32_t* __restrict__ ncell, const double* __restrict__ gcell,
                  const double* __restrict__ gcell2, int64_t N, int64_t RS,
                  const int32_t* __restrict__ node_sys, const double* __restrict__ gE,
                  const double* __restrict__ gV, const double* __restrict__ sys_out, int nsys,
                  int nb, double* __restrict__ g_pos, double* __restrict__ g_rv,
                  int* __restrict__ nanflag) {
  if ((int)blockIdx.x >= nb) {
    const int q = ((int)blockIdx.x - nb) * 256 + threadIdx.x;
    if (q >= 9 * nsys) return;
    const int sy = q / 9, i = q % 9;
    const double* r = sys_out + (int64_t)sy * 2 * kSysQ + 10;
    double v = gE[sy] * r[i] + r[kSysQ + i];
    if (gV) {
      const double *a = r + 3 * (i / 3), *V = gV + 9 * (int64_t)sy + i % 3;
      v += (a[0] * V[0] + a[1] * V[3]) + a[2] * V[6];
    }
    g_rv[q] = v;
    return;
  }
  const int64_t n = (int64_t)xcd_block((int)blockIdx.x, nb) * 256 + threadIdx.x;
  if (n >= N) return;
  double g[3], d[3];
  sum_node_records<kAllLoads>(ncell, gcell, N, RS, n, g);
  sum_node_records<kAllLoads>(ncell, gcell2, N, RS, n, d);
  bool bad = false;
#pragma unroll
  for (int l = 0; l < 3; ++l) bad |= g[l] != g[l] || d[l] != d[l];
  if (bad) atomicOr(nanflag, 2);
  const int sy = node_sys[n];
  const double e = gE[sy];
  const double* V = gV ? gV + 9 * (int64_t)sy : nullptr;
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    double v = e * g[l] + d[l];
    if (V) v += (g[0] * V[l] + g[1] * V[3 + l]) + g[2] * V[6 + l];
    g_pos[3 * n + l] = v;
  }
}

// Sums of squares for the force-and-stress loss. Per block of the node terms (g - gt)^2:
constexpr int kLossBlocks = 1024;
__global__ void __launch_bounds__(256)
fit_loss_partial_kernel(const double* __restrict__ g, const double* __restrict__ gt, int64_t n,
                        double* __restrict__ part) {
  __shared__ double red[4];
  double acc[1] = {0.0};
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double d = g[i] - gt[i];
    acc[0] += d * d;
  }
  wave_reduce<1>(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc[0];
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// loss = mean (g - gt)^2 / f_scale + mean (v inv - vt)^2 / s_scale over n and m values; one block.
__global__ void __launch_bounds__(256)
fit_loss_kernel(const double* __restrict__ part, int nb, int64_t n, const double* __restrict__ v,
                const double* __restrict__ vt, const double* __restrict__ inv, int m,
                double f_scale, double s_scale, double* __restrict__ loss) {
  __shared__ double red[8];
  double acc[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < nb; i += 256) acc[0] += part[i];
  for (int i = threadIdx.x; i < m; i += 256) {
    const double d = v[i] * inv[i / 9] - vt[i];
    acc[1] += d * d;
  }
  wave_reduce<2>(acc);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = acc[0];
    red[4 + (threadIdx.x >> 6)] = acc[1];
  }
  __syncthreads();
  if (threadIdx.x == 0)
    *loss = (((red[0] + red[1]) + red[2]) + red[3]) / (double)n / f_scale +
            (((red[4] + red[5]) + red[6]) + red[7]) / (double)m / s_scale;
}

}  // namespace mm

using namespace mm;

// Gradients of (Cv, h0, free energy, T_eff) from parameter entries, one wave per (row, state).
__global__ void __launch_bounds__(64)
param_grads_kernel(const double* __restrict__ entries, int64_t stride, int add_next, int64_t npar,
                   int max_states, const int32_t* __restrict__ nstates, GradOut grads) {
  const int row = blockIdx.x / max_states, s = blockIdx.x % max_states;
  const double* er = entries + (int64_t)row * npar * stride;
  auto get = [&](int64_t q) {
    return add_next ? er[q * stride] + er[q * stride + 1] : er[q * stride];
  };
  __shared__ double ent[32];
  if (threadIdx.x < 32) ent[threadIdx.x] = get((int64_t)s * kNps + threadIdx.x);
  if (s == 0 && threadIdx.x == 0)
    grads.teff[row] = get((int64_t)max_states * kNps) * grads.boltzmann;
  __syncthreads();
  state_gradients(ent, s < nstates[row], blockIdx.x, grads);
}

struct mm_adjoint {
  mm_field* field = nullptr;
  int64_t npar = 0;            // parameter entries per row: max_states * 32 + 1
  int64_t nblk = 0;            // W / 64
  double* part = nullptr;      // [2 kSysQ][nblk]
  double* ppart = nullptr;     // [2 npar][nblk]
  double* gcell2 = nullptr;    // [4][3][S]
  int32_t* row_ptr = nullptr;  // [nrows + 1] CSR of the segments of every table row
  int32_t* row_idx = nullptr;  // [W / kCellBlock]
  // of the products: direction [N][3] and [nsys][9], sys_out [nsys][2 kSysQ], params
  // [nrows][npar][2], stress cotangents [nsys][9], loss partials [kLossBlocks]
  double *vjp = nullptr, *drv = nullptr, *sys_out = nullptr, *params = nullptr, *gV = nullptr,
         *lpart = nullptr;
};

extern "C" {

int mm_adjoint_create(mm_adjoint** out, mm_field* field, int64_t* npar) {
  if (!out || !field) return set_error(MM_ERR_ARG, "missing argument");
  *out = nullptr;
  const int64_t nseg = field->W / kCellBlock;
  std::vector<int32_t> blk_row(nseg > 0 ? nseg : 1, 0);
  int cur = 0;
  (void)hipGetDevice(&cur);
  (void)hipSetDevice(field->device);
  hipError_t e = hipSuccess;
  if (nseg > 0)
    e = hipMemcpy(blk_row.data(), field->blk_row, sizeof(int32_t) * nseg, hipMemcpyDeviceToHost);
  if (e != hipSuccess) {
    (void)hipSetDevice(cur);
    return hip_error(e, "mm_adjoint_create");
  }
  std::vector<int32_t> row_ptr(field->nrows + 1, 0), row_idx;
  for (int t = 0; t < field->nrows; ++t) {
    for (int64_t s = 0; s < nseg; ++s)
      if (blk_row[s] == t) row_idx.push_back((int32_t)s);
    row_ptr[t + 1] = (int32_t)row_idx.size();
  }
  mm_adjoint* a = new mm_adjoint();
  a->field = field;
  a->npar = (int64_t)field->max_states * kNps + 1;
  a->nblk = field->W / kAdjCells;
  const size_t nb = (size_t)(a->nblk > 0 ? a->nblk : 1);
  e = hipMalloc((void**)&a->part, sizeof(double) * 2 * kSysQ * nb);
  if (e == hipSuccess) e = hipMalloc((void**)&a->ppart, sizeof(double) * 2 * a->npar * nb);
  if (e == hipSuccess)
    e = hipMalloc((void**)&a->gcell2, sizeof(double) * 12 * (field->S > 0 ? field->S : 1));
  if (e == hipSuccess)
    e = hipMalloc((void**)&a->vjp,
                  sizeof(double) * (3 * (size_t)field->N + (18 + 2 * kSysQ) * (size_t)field->nsys +
                                    2 * (size_t)a->npar * field->nrows + kLossBlocks));
  if (e == hipSuccess) {
    a->drv = a->vjp + 3 * field->N;
    a->sys_out = a->drv + 9 * (int64_t)field->nsys;
    a->gV = a->sys_out + 2 * kSysQ * (int64_t)field->nsys;
    a->params = a->gV + 9 * (int64_t)field->nsys;
    a->lpart = a->params + 2 * a->npar * field->nrows;
  }
  if (e == hipSuccess) e = hipMalloc((void**)&a->row_ptr, sizeof(int32_t) * row_ptr.size());
  if (e == hipSuccess)
    e = hipMalloc((void**)&a->row_idx, sizeof(int32_t) * (row_idx.empty() ? 1 : row_idx.size()));
  if (e == hipSuccess)
    e = hipMemcpy(a->row_ptr, row_ptr.data(), sizeof(int32_t) * row_ptr.size(),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess && !row_idx.empty())
    e = hipMemcpy(a->row_idx, row_idx.data(), sizeof(int32_t) * row_idx.size(),
                  hipMemcpyHostToDevice);
  // rows of states that a type does not have are summed too (metric_entries_kernel drops the sums)
  if (e == hipSuccess) e = hipMemset(a->ppart, 0, sizeof(double) * 2 * a->npar * nb);
  (void)hipSetDevice(cur);
  if (e != hipSuccess) {
    mm_adjoint_destroy(a);
    return hip_error(e, "mm_adjoint_create");
  }
  if (npar) *npar = a->npar;
  *out = a;
  return MM_OK;
}

}  // extern "C"

namespace {

// The adjoint kernel and its sums on the current device: sys_out, params (and grads from them),
// and with records the vertex gradients' and tangents' records.
hipError_t adjoint_passes(mm_adjoint* a, const double* pos, const double* dpos,
                          const double* rvecs, const double* drvecs, const double* energy_weight,
                          double* sys_out, double* params, bool records, const GradOut& grads,
                          hipStream_t s) {
  mm_field* f = a->field;
  const bool dual = dpos != nullptr;
  const int64_t nblk = a->nblk;
  if (nblk == 0) {
    hipError_t e = hipMemsetAsync(sys_out, 0, sizeof(double) * 2 * kSysQ * f->nsys, s);
    if (e == hipSuccess)
      e = hipMemsetAsync(params, 0, sizeof(double) * 2 * a->npar * f->nrows, s);
    return e;
  }
  const size_t lds = sizeof(double) * 64 * (dual ? 2 : 1) *
                     ((f->model == 0 ? 36 : 6) + (f->max_states > 1 ? f->max_states : 0));
#define MM_ADJ(T, MODEL)                                                                        \
  hipLaunchKernelGGL((adjoint_kernel<T, MODEL>), dim3((unsigned)nblk), dim3(64), lds, s, pos,   \
                     dpos, rvecs, drvecs, f->blk_sys, f->cnode, f->cwrap, f->blk_row, f->tab,  \
                     f->kt, f->nstates, f->max_states, f->W, f->cbase, f->S,                   \
                     records ? f->gcell : nullptr, a->gcell2, a->part, a->ppart)
  if (dual) {
    if (f->model == 0) MM_ADJ(Dual, 0); else MM_ADJ(Dual, 1);
  } else {
    if (f->model == 0) MM_ADJ(double, 0); else MM_ADJ(double, 1);
  }
#undef MM_ADJ
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // per system: energy, virial, domain-vector gradient (value rows, then tangent rows); per
  // table row: parameter entries (value rows scaled by the system's energy weight)
  const SegmentSums x{a->part, f->nsys, 2 * kSysQ, f->sys_cblk_ptr, f->sys_cblk_idx, nullptr, 1,
                      sys_out};
  const SegmentSums y{a->ppart, f->nrows, (int)(2 * a->npar), a->row_ptr, a->row_idx,
                      energy_weight, 2, params};
  hipLaunchKernelGGL(segment_sum_kernel,
                     dim3((unsigned)(x.lists * x.nrows_part + y.lists * y.nrows_part)), dim3(256),
                     0, s, x, y, nblk, f->blk_sys);
  e = hipGetLastError();
  if (e != hipSuccess || f->nrows == 0) return e;
  hipLaunchKernelGGL(metric_entries_kernel, dim3((unsigned)(f->nrows * f->max_states)), dim3(64),
                     0, s, f->tab, f->nstates, f->max_states, a->npar, params, grads);
  return hipGetLastError();
}

hipError_t launch_param_grads(mm_adjoint* a, const double* entries, int64_t stride, int add_next,
                              const GradOut& grads, hipStream_t s) {
  const mm_field* f = a->field;
  const int n = f->nrows * f->max_states;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(param_grads_kernel, dim3((unsigned)n), dim3(64), 0, s, entries, stride,
                     add_next, a->npar, f->max_states, f->nstates, grads);
  return hipGetLastError();
}

// A vector-Jacobian product on the current device (fit: of the loss; then gG and gV are not read).
// g_pos, g_rv and grads.cv may be null. Five launches: direction, adjoint kernel, sums, entries with
// the parameter gradients, outputs. The host's work per launch and tensor bounds both uses: nine
// launches and some fifteen torch kernels for loss, cotangents and domain gradients took 500 us a
// fit step (64 configurations of 16^3 cells; its parameters alone need a gradient, so no records
// are stored nor gathered) and 430 us for all gradients of 5 of 7^3 cells, now 349 and 351 us.
hipError_t vjp_passes(mm_adjoint* a, const double* pos, const double* rvecs,
                      const int32_t* node_sys, const double* gE, const double* gG,
                      const double* gV, const FitTerms* fit, double* sys_out, double* params,
                      double* g_pos, double* g_rv, const GradOut& grads, hipStream_t s) {
  mm_field* f = a->field;
  const int64_t nt = f->N + 9 * (int64_t)f->nsys;
  const dim3 grid((unsigned)((nt + 255) / 256));
  if (fit) {
    hipLaunchKernelGGL(vjp_direction_kernel<true>, grid, dim3(256), 0, s, pos, rvecs, node_sys, gG,
                       gV, *fit, f->N, f->nsys, a->vjp, a->drv);
    gV = a->gV;
  } else {
    hipLaunchKernelGGL(vjp_direction_kernel<false>, grid, dim3(256), 0, s, pos, rvecs, node_sys,
                       gG, gV, FitTerms{}, f->N, f->nsys, a->vjp, a->drv);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = adjoint_passes(a, pos, a->vjp, rvecs, a->drv, gE, sys_out, params, g_pos != nullptr,
                       grads, s);
  if (e == hipSuccess && a->nblk == 0 && grads.cv)
    e = launch_param_grads(a, params, 2, 1, grads, s);
  if (e != hipSuccess) return e;
  const int nb = g_pos ? (int)((f->N + 255) / 256) : 0;
  const int nr = g_rv ? (9 * f->nsys + 255) / 256 : 0;
  if (nb + nr == 0) return hipSuccess;
#define MM_OUT(A)                                                                               \
  hipLaunchKernelGGL(vjp_output_kernel<A>, dim3(nb + nr), dim3(256), 0, s, f->nrec, f->gcell,     \
                     a->gcell2, f->N, f->S, node_sys, gE, gV, sys_out, f->nsys, nb, g_pos, g_rv, \
                     f->nanflag)
  if (nb <= kGatherAllLoadsMaxBlocks) MM_OUT(true); else MM_OUT(false);
#undef MM_OUT
  return hipGetLastError();
}

struct CurrentDevice {
  int cur = 0;
  explicit CurrentDevice(int device) {
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(device);
  }
  ~CurrentDevice() { (void)hipSetDevice(cur); }
};

int grad_out(const mm_adjoint* a, const double* h0, double boltzmann, double* g_cv, double* g_h0,
             double* g_free, double* g_teff, GradOut& out) {
  if ((g_cv || g_h0 || g_free || g_teff) && !(h0 && g_cv && g_h0 && g_free && g_teff))
    return set_error(MM_ERR_ARG, "h0, g_cv, g_h0, g_free and g_teff go together");
  out = GradOut{h0, a->field->model == MM_MODEL_CORNER8 ? 1 : 0, boltzmann, g_cv, g_h0, g_free,
                g_teff};
  return MM_OK;
}

}  // namespace

extern "C" {

int mm_adjoint_compute(mm_adjoint* a, const double* pos, const double* dpos, const double* rvecs,
                       const double* drvecs, const double* energy_weight, double* sys_out,
                       double* gpos, double* dgpos, double* params, void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  mm_field* f = a->field;
  if ((f->N > 0 && !pos) || !rvecs || !sys_out || !params)
    return set_error(MM_ERR_ARG, "missing argument");
  if ((dpos == nullptr) != (drvecs == nullptr))
    return set_error(MM_ERR_ARG, "dpos and drvecs go together");
  if (dgpos && !dpos) return set_error(MM_ERR_ARG, "dgpos needs a tangent direction");
  const CurrentDevice device(f->device);
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = adjoint_passes(a, pos, dpos, rvecs, drvecs, energy_weight, sys_out, params,
                                gpos != nullptr, GradOut{}, s);
  if (e == hipSuccess && a->nblk > 0 && f->N > 0 && gpos) {
    ForceArgs g{};
    g.ncell = f->nrec;
    g.gcell = f->gcell;
    g.rstride = f->S;
    g.N = f->N;
    g.W = f->W;
    g.gpos = gpos;
    g.accumulate = 0;
    g.nanflag = f->nanflag;
    e = launch_gather(g, ReduceList{}, s);
    if (e == hipSuccess && dgpos) {
      g.gcell = a->gcell2;
      g.gpos = dgpos;
      e = launch_gather(g, ReduceList{}, s);
    }
  }
  if (e != hipSuccess) return hip_error(e, "adjoint kernels");
  return MM_OK;
}

int mm_adjoint_vjp(mm_adjoint* a, const double* pos, const double* rvecs,
                   const int32_t* node_sys, const double* gE, const double* gG, const double* gV,
                   double* sys_out, double* g_pos, double* params, void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  mm_field* f = a->field;
  if ((f->N > 0 && (!pos || !node_sys || !g_pos)) || !rvecs || !gE || !sys_out || !params)
    return set_error(MM_ERR_ARG, "missing argument (gE is required: zeros for none)");
  const CurrentDevice device(f->device);
  const hipError_t e = vjp_passes(a, pos, rvecs, node_sys, gE, gG, gV, nullptr, sys_out, params,
                                  g_pos, nullptr, GradOut{}, (hipStream_t)stream);
  if (e != hipSuccess) return hip_error(e, "vector-Jacobian product kernels");
  return MM_OK;
}

int mm_adjoint_backward(mm_adjoint* a, const double* pos, const double* rvecs,
                        const int32_t* node_sys, const double* gE, const double* gG,
                        const double* gV, const double* h0, double boltzmann, double* g_pos,
                        double* g_rv, double* g_cv, double* g_h0, double* g_free, double* g_teff,
                        void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  mm_field* f = a->field;
  if ((f->N > 0 && (!pos || !node_sys)) || !rvecs || !gE)
    return set_error(MM_ERR_ARG, "missing argument (gE is required: zeros for none)");
  GradOut grads;
  const int rc = grad_out(a, h0, boltzmann, g_cv, g_h0, g_free, g_teff, grads);
  if (rc != MM_OK) return rc;
  const CurrentDevice device(f->device);
  const hipError_t e = vjp_passes(a, pos, rvecs, node_sys, gE, gG, gV, nullptr, a->sys_out,
                                  a->params, g_pos, g_rv, grads, (hipStream_t)stream);
  if (e != hipSuccess) return hip_error(e, "backward kernels");
  return MM_OK;
}

int mm_fit_loss(mm_adjoint* a, const double* g, const double* g_target, const double* v,
                const double* v_target, const double* inv_volume, double f_scale, double s_scale,
                double* loss, void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  mm_field* f = a->field;
  if ((f->N > 0 && (!g || !g_target)) || !v || !v_target || !inv_volume || !loss)
    return set_error(MM_ERR_ARG, "missing argument");
  const CurrentDevice device(f->device);
  const hipStream_t s = (hipStream_t)stream;
  const int64_t n = 3 * f->N;
  const int nb = (int)std::min<int64_t>((n + 1023) / 1024, kLossBlocks);
  if (nb > 0)
    hipLaunchKernelGGL(fit_loss_partial_kernel, dim3(nb), dim3(256), 0, s, g, g_target, n,
                       a->lpart);
  hipLaunchKernelGGL(fit_loss_kernel, dim3(1), dim3(256), 0, s, a->lpart, nb, n, v, v_target,
                     inv_volume, 9 * f->nsys, f_scale, s_scale, loss);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_error(e, "loss kernels");
  return MM_OK;
}

int mm_fit_backward(mm_adjoint* a, const double* pos, const double* rvecs,
                    const int32_t* node_sys, const double* gE, const double* g,
                    const double* g_target, const double* v, const double* v_target,
                    const double* inv_volume, double f_scale, double s_scale, const double* gl,
                    const double* h0, double boltzmann, double* g_pos, double* g_rv, double* g_cv,
                    double* g_h0, double* g_free, double* g_teff, void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  mm_field* f = a->field;
  if ((f->N > 0 && (!pos || !node_sys || !g || !g_target)) || !rvecs || !gE || !v || !v_target ||
      !inv_volume || !gl)
    return set_error(MM_ERR_ARG, "missing argument (gE is required: zeros)");
  GradOut grads;
  const int rc = grad_out(a, h0, boltzmann, g_cv, g_h0, g_free, g_teff, grads);
  if (rc != MM_OK) return rc;
  const CurrentDevice device(f->device);
  const FitTerms fit{g, g_target, v, v_target, inv_volume, gl,
                     2.0 / (3.0 * (double)f->N * f_scale), 2.0 / (9.0 * f->nsys * s_scale),
                     a->gV};
  const hipError_t e = vjp_passes(a, pos, rvecs, node_sys, gE, nullptr, nullptr, &fit, a->sys_out,
                                  a->params, g_pos, g_rv, grads, (hipStream_t)stream);
  if (e != hipSuccess) return hip_error(e, "backward kernels of the loss");
  return MM_OK;
}

int mm_adjoint_param_grads(mm_adjoint* a, const double* entries, int64_t stride, int add_next,
                           const double* h0, double boltzmann, double* g_cv, double* g_h0,
                           double* g_free, double* g_teff, void* stream) {
  if (!a) return set_error(MM_ERR_ARG, "adjoint is NULL");
  if (!entries || !h0 || !g_cv || !g_h0 || !g_free || !g_teff)
    return set_error(MM_ERR_ARG, "missing argument");
  if (stride < 1 || (add_next && stride < 2))
    return set_error(MM_ERR_ARG, "stride %lld with add_next %d", (long long)stride, add_next);
  GradOut grads;
  const int rc = grad_out(a, h0, boltzmann, g_cv, g_h0, g_free, g_teff, grads);
  if (rc != MM_OK) return rc;
  const CurrentDevice device(a->field->device);
  const hipError_t e = launch_param_grads(a, entries, stride, add_next, grads,
                                          (hipStream_t)stream);
  if (e != hipSuccess) return hip_error(e, "parameter gradient kernel");
  return MM_OK;
}

void mm_adjoint_destroy(mm_adjoint* a) {
  if (!a) return;
  if (a->part) (void)hipFree(a->part);
  if (a->ppart) (void)hipFree(a->ppart);
  if (a->gcell2) (void)hipFree(a->gcell2);
  if (a->row_ptr) (void)hipFree(a->row_ptr);
  if (a->row_idx) (void)hipFree(a->row_idx);
  if (a->vjp) (void)hipFree(a->vjp);
  delete a;
}

}  // extern "C"
