// Device-side building blocks of the nanocell force field (CDNA4 / gfx950, FP64).
//
// Geometry conventions follow micmec/pes/nanocell.py:40-132 and micmec/utils.py:43-52:
//   corner k of a cell sits at lattice offset OFF[k] = (000,100,010,001,110,101,011,111);
//   the corner matrix M_a has as rows the three edges through corner a, each oriented along
//   +x, +y, +z (micmec/pes/nanocell_utils.py:32-75);
//   B_a = h0^-1 M_a, eps_a = (B_a B_a^T - I)/2 (Green-Lagrange), u_a = eps_a : C0 : eps_a / 2.
// The gradient is the adjoint of that chain: dE/dB = S B with S the symmetric stress built from
// the Voigt vector C e, and dE/dM = h0^-T dE/dB; it equals the derivative-table route of
// nanocell.py:98-132. The force kernels evaluate both in the metric of the edges (state_stress).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mm {

// Doubles per (type, state) entry of the parameter table.
//   [0..8]   P = h0^-1 (row-major)
//   [9]      w  = det(h0) / 8 (corner8) or det(h0) (original)
//   [10]     free energy of the state
//   [11]     unused
//   [12..47] Voigt matrix Cv[6][6] (row-major), averaged over index orderings
//   [48..83] K = T^T (w Cv) T, the weighted matrix of the force kernels (metric_entry)
//   [84..89] rest metric R (rest_entry): R00, R11, R22, R12, R02, R01
//   [90..95] what they lack: half of it for R00, R11, R22, all of it for the others
//   [96..98] the diagonal of R/2 of the type's first state less this state's
//   [99..103] unused (entries begin at cache lines)
constexpr int kTabStride = 104;
constexpr int kCvOffset = 12;
constexpr int kMetricOffset = 48;
constexpr int kRestOffset = 84;
constexpr int kRestLowOffset = 90;
constexpr int kShiftOffset = 96;

// Tables that no kernel of a launch writes: read with scalar loads wherever the index is uniform,
// also where other memory changes during the launch.
typedef const __attribute__((address_space(4))) double* const_f64;
typedef const __attribute__((address_space(4))) int32_t* const_i32;

// 3x3 inverse (row-major) by cofactors; returns the determinant. Shared by the host and the
// device table builders, without contraction, so both round the same way.
__host__ __device__ inline double inverse3_cof(const double* h, double* inv) {
#pragma clang fp contract(off)
  const double a = h[0], b = h[1], c = h[2], d = h[3], e = h[4], f = h[5], g = h[6], k = h[7],
               l = h[8];
  const double c00 = e * l - f * k, c01 = f * g - d * l, c02 = d * k - e * g;
  const double det = a * c00 + b * c01 + c * c02;
  inv[0] = c00 / det;
  inv[1] = (c * k - b * l) / det;
  inv[2] = (b * f - c * e) / det;
  inv[3] = c01 / det;
  inv[4] = (a * l - c * g) / det;
  inv[5] = (c * d - a * f) / det;
  inv[6] = c02 / det;
  inv[7] = (b * g - a * k) / det;
  inv[8] = (a * e - b * d) / det;
  return det;
}

// Entry IJ of the map T of the Gram entries e6 to the engineering strain: eps_ij = sum_ab P_ia P_jb
// e_ab, i.e. with (i,j) and (a,b) the pairs of rows I and columns J, T_IJ = P_ia P_ja (a = b) or
// (P_ia P_jb + P_ib P_ja) / 2 (a != b, where e6 holds 2 e_ab), doubled for the shear rows I >= 3.
__host__ __device__ inline double strain_map(const double* P, int I, int J) {
#pragma clang fp contract(off)
  const int pi[6] = {0, 1, 2, 1, 0, 0}, pj[6] = {0, 1, 2, 2, 2, 1};
  const double* a = P + 3 * pi[I];
  const double* b = P + 3 * pj[I];
  const double cross = a[pi[J]] * b[pj[J]] + a[pj[J]] * b[pi[J]];
  return (I < 3) == (J < 3) ? (I < 3 ? a[pi[J]] * b[pi[J]] : cross)
                            : (I < 3 ? 0.5 * cross : cross);
}

// Entries IJ of CT = (w Cv) T and of K = T^T CT.
__host__ __device__ inline double stiffness_half(double w, const double* Cv, const double* T, int I,
                                                 int J) {
#pragma clang fp contract(off)
  double t = 0.0;
  for (int L = 0; L < 6; ++L) t += (w * Cv[6 * I + L]) * T[6 * L + J];
  return t;
}
__host__ __device__ inline double stiffness_entry(const double* T, const double* CT, int I, int J) {
#pragma clang fp contract(off)
  double t = 0.0;
  for (int L = 0; L < 6; ++L) t += T[6 * L + I] * CT[6 * L + J];
  return t;
}
// start + sum_k a[k sa] b[k sb] as the sum of the result and lo, from exact products and sums.
__host__ __device__ inline double dot3_exact(const double* a, int sa, const double* b, int sb,
                                             double start, double& lo) {
#pragma clang fp contract(off)
  double s = start, c = 0.0;
  for (int k = 0; k < 3; ++k) {
    const double p = a[k * sa] * b[k * sb], e = __builtin_fma(a[k * sa], b[k * sb], -p);
    const double t = s + p, z = t - s;
    c += ((s - (t - z)) + (p - z)) + e;
    s = t;
  }
  lo = c;
  return s;
}
// R is the metric that P, rounded as it is, takes to the identity, R = P^-1 P^-T: with the rounding
// of h0 h0^T in its place every cell would carry the same strain of 1e-17, which a virial of
// small strains of either sign does not average out. P h0 = I + E, so to first order in E (1e-16)
// R = h0 h0^T - h0 (E + E^T) h0^T. Returns the entry rounded, the rest (half of it on the diagonal,
// as the strains take it) in lo.
__host__ __device__ inline double inverse_residual(const double* P, const double* h0, int q) {
#pragma clang fp contract(off)
  double lo;  // entry q of E
  const double hi = dot3_exact(P + 3 * (q / 3), 1, h0 + q % 3, 3, q % 4 == 0 ? -1.0 : 0.0, lo);
  return hi + lo;
}
__host__ __device__ inline double rest_entry(const double* h0, const double* E, int I, double& lo) {
#pragma clang fp contract(off)
  const int pi[6] = {0, 1, 2, 1, 0, 0}, pj[6] = {0, 1, 2, 2, 2, 1};
  const double* a = h0 + 3 * pi[I];
  const double* b = h0 + 3 * pj[I];
  double c = 0.0, l;
  for (int m = 0; m < 3; ++m)
    for (int n = 0; n < 3; ++n) c += a[m] * (E[3 * m + n] + E[3 * n + m]) * b[n];
  const double r = dot3_exact(a, 1, b, 1, 0.0, l);
  l -= c;
  const double hi = r + l;
  lo = (r - hi) + l;
  if (I < 3) lo *= 0.5;
  return hi;
}
// Half of the first state's diagonal entry r0, l0 less this one's r1, l1.
__host__ __device__ inline double rest_shift(double r0, double l0, double r1, double l1) {
#pragma clang fp contract(off)
  return 0.5 * (r0 - r1) + (l0 - l1);
}

// K (36) and the rest entries (15, from kRestOffset) of a table entry from h0, P = h0^-1, w and Cv, and
// those of the type's first state. Shared by the host and the device table builders, without
// contraction, so both round the same way.
inline void metric_entry(const double* h0, const double* P, double w, const double* Cv,
                         const double* h00, const double* P00, double* K, double* R) {
  double T[36], CT[36];
  for (int q = 0; q < 36; ++q) T[q] = strain_map(P, q / 6, q % 6);
  for (int q = 0; q < 36; ++q) CT[q] = stiffness_half(w, Cv, T, q / 6, q % 6);
  for (int q = 0; q < 36; ++q) K[q] = stiffness_entry(T, CT, q / 6, q % 6);
  double E[9], E0[9], lo, lo0;
  for (int q = 0; q < 9; ++q) {
    E[q] = inverse_residual(P, h0, q);
    E0[q] = inverse_residual(P00, h00, q);
  }
  for (int I = 0; I < 6; ++I) {
    R[I] = rest_entry(h0, E, I, lo);
    R[kRestLowOffset - kRestOffset + I] = lo;
    if (I >= 3) continue;
    const double r0 = rest_entry(h00, E0, I, lo0);
    R[kShiftOffset - kRestOffset + I] = rest_shift(r0, lo0, R[I], lo);
  }
}

// Edge endpoints: corner a, axis d -> lower / upper corner of the edge along d through a.
__device__ constexpr int kLo[8][3] = {
    {0, 0, 0}, {0, 1, 1}, {2, 0, 2}, {3, 3, 0}, {2, 1, 4}, {3, 5, 1}, {6, 3, 2}, {6, 5, 4}};
__device__ constexpr int kHi[8][3] = {
    {1, 2, 3}, {1, 4, 5}, {4, 2, 6}, {5, 6, 3}, {4, 4, 7}, {5, 7, 5}, {7, 6, 6}, {7, 7, 7}};
// Corner offsets along x, y, z.
__device__ constexpr int kOff[8][3] = {
    {0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {1, 1, 0}, {1, 0, 1}, {0, 1, 1}, {1, 1, 1}};
// The twelve edges: four along x, y and z each; edge kEdge[a][d] is the edge along d through
// corner a, from corner kEdgeLo to corner kEdgeHi (so kEdgeLo/Hi[kEdge[a][d]] = kLo/kHi[a][d]).
__device__ constexpr int kEdgeLo[12] = {0, 2, 3, 6, 0, 1, 3, 5, 0, 1, 2, 4};
__device__ constexpr int kEdgeHi[12] = {1, 4, 5, 7, 2, 4, 6, 7, 3, 5, 6, 7};
__device__ constexpr int kEdge[8][3] = {{0, 4, 8},  {0, 5, 9},  {1, 4, 10}, {2, 6, 8},
                                        {1, 5, 11}, {2, 7, 9},  {3, 6, 10}, {3, 7, 11}};

// A cell's energy in the metric of its edges. With M_a the corner matrix (rows = edges) and
// G = M M^T its Gram matrix, the Green-Lagrange strain of the corner is
//   eps = (P M M^T P^T - I)/2 = P e P^T,  e = (G - h0 h0^T)/2,
// linear in G, so the energy w u = e6 . K e6 / 2 and the stress S6 = K e6 need only the Gram
// entries e6 = (e00, e11, e22, 2 e12, 2 e02, 2 e01) and one matrix K = T^T (w Cv) T per (type,
// state), T the map of e6 to the engineering strain (metric_entry); and dU/dM = S M with S the
// symmetric matrix of S6. No B = P M and no products with P remain per corner, an edge's
// length is shared by its two corners, and several states share the whole geometry: about 830
// FP64 instructions a cell instead of 1500 for one state.
//
// kModel 0 (corner8, nanocell.py) has 8 corners and 12 edges, kModel 1 (original,
// nanocell_original.py) one averaged corner with 3 edges H_d (the mean of the four edges along d).
template <int kModel>
struct Frame {
  static constexpr int NC = kModel == 0 ? 8 : 1;
  static constexpr int NE = kModel == 0 ? 12 : 3;
  // the i-th corner: neighbours on the cube follow each other, so that an edge's two corners
  // come close together and few edges are open at a time
  __device__ static constexpr int corner(int i) {
    constexpr int kOrder[8] = {0, 1, 4, 2, 3, 5, 7, 6};
    return kModel == 0 ? kOrder[i] : 0;
  }
  __device__ static constexpr int rank(int a) {
    constexpr int kRank[8] = {0, 1, 3, 4, 2, 5, 7, 6};
    return kRank[a];
  }
  __device__ static constexpr int edge(int a, int d) { return kModel == 0 ? kEdge[a][d] : d; }
  // the two axes of off-diagonal entry q: 12, 02, 01
  __device__ static constexpr int axis0(int q) { return q == 0 ? 1 : 0; }
  __device__ static constexpr int axis1(int q) { return q == 2 ? 1 : 2; }
  // axis along which edge e runs, and the ranks of its first and last corner
  __device__ static constexpr int along(int e) { return kModel == 0 ? e / 4 : e; }
  __device__ static constexpr int first(int e) {
    return kModel != 0 ? 0 : rank(kEdgeLo[e]) < rank(kEdgeHi[e]) ? rank(kEdgeLo[e]) : rank(kEdgeHi[e]);
  }
  __device__ static constexpr int last(int e) {
    return kModel != 0 ? 0 : rank(kEdgeLo[e]) > rank(kEdgeHi[e]) ? rank(kEdgeLo[e]) : rank(kEdgeHi[e]);
  }
};

// Stress of the i-th corner from its strain x: the diagonal entries are added to their edges' D,
// the off-diagonal ones go to O, and their energy terms to u.
template <int kModel>
__device__ __forceinline__ void corner_stress(const_f64 K, int i,
                                              const double (&x)[6],
                                              double (&D)[Frame<kModel>::NE], double (&O)[3],
                                              double& u) {
#pragma clang fp contract(off)
  using F = Frame<kModel>;
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    const int e = I < 3 ? F::edge(F::corner(i), I) : 0;
    double t = I < 3 && F::first(e) < i ? __builtin_fma(K[6 * I], x[0], D[e]) : K[6 * I] * x[0];
#pragma unroll
    for (int J = 1; J < 6; ++J) t = __builtin_fma(K[6 * I + J], x[J], t);
    if (I < 3) D[e] = t;
    else O[I < 3 ? 0 : I - 3] = t;
  }
#pragma unroll
  for (int o = 0; o < 3; ++o) u = __builtin_fma(x[3 + o], O[o], u);
}

// Off-diagonal strain of a corner's edges A and B: their dot product less the rest metric's g0 + lo.
__device__ __forceinline__ double edge_dot(const double (&A)[3], const double (&B)[3], double g0,
                                           double lo) {
#pragma clang fp contract(off)
  return __builtin_fma(A[2], B[2], __builtin_fma(A[1], B[1], __builtin_fma(A[0], B[0], -g0))) - lo;
}
// Diagonal strain of an edge along d against its rest metric g0 + 2 lo: (A.A - g0)/2 - lo, the sum
// begun with the component along d less g0. That product is exact inside the fused multiply-add,
// so where the rest cell is near the axes the error is relative to the strain, not to the edge.
__device__ __forceinline__ double edge_strain(const double (&A)[3], int d, double g0, double lo) {
#pragma clang fp contract(off)
  const int b = d == 0 ? 1 : 0, c = d == 2 ? 1 : 2;
  const double t = __builtin_fma(A[c], A[c],
                                 __builtin_fma(A[b], A[b], __builtin_fma(A[d], A[d], -g0)));
  return __builtin_fma(0.5, t, -lo);
}

// Energy (weighted, without the free-energy offset) and stress of one (type, state) at all
// corners, from the edges E and their strains q against the rest metric of the type's first
// state: D[e] = the diagonal stress along edge e summed over its corners, O[a][q] the
// off-diagonal stresses of corner a. The sums are fused
// multiply-adds in a fixed order, so every kernel that evaluates a state gets the same bits.
template <int kModel>
__device__ __forceinline__ double state_stress(const_f64 tab,
                                               const double (&E)[Frame<kModel>::NE][3],
                                               const double (&q)[Frame<kModel>::NE],
                                               double (&D)[Frame<kModel>::NE],
                                               double (&O)[Frame<kModel>::NC][3]) {
#pragma clang fp contract(off)
  using F = Frame<kModel>;
  const const_f64 g0 = tab + kRestOffset;
  double u = 0.0;
#pragma unroll
  for (int i = 0; i < F::NC; ++i) {
    const int a = F::corner(i);
    double x[6];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = q[F::edge(a, d)] + tab[kShiftOffset + d];
#pragma unroll
    for (int o = 0; o < 3; ++o)
      x[3 + o] = edge_dot(E[F::edge(a, F::axis0(o))], E[F::edge(a, F::axis1(o))], g0[3 + o],
                          tab[kRestLowOffset + 3 + o]);
    corner_stress<kModel>(tab + kMetricOffset, i, x, D, O[a], u);
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (F::last(F::edge(a, d)) == i) u = __builtin_fma(x[d], D[F::edge(a, d)], u);
    asm("" : "+v"(u));
  }
  return 0.5 * u;
}

// The virial sum_e gE_e (x) E_e (= sum_a M^T S M, symmetric) as (00, 11, 22, 12, 02, 01).
__device__ __forceinline__ void edge_virial(const double (&gE)[3], const double (&E)[3],
                                            double (&vir)[6]) {
#pragma clang fp contract(off)
  constexpr int kK[6] = {0, 1, 2, 1, 0, 0}, kL[6] = {0, 1, 2, 2, 2, 1};
#pragma unroll
  for (int v = 0; v < 6; ++v) vir[v] = __builtin_fma(gE[kK[v]], E[kL[v]], vir[v]);
}

// An edge pulls at its upper corner and pushes at its lower one (averaged model: a quarter of
// H_d's derivative at every corner). g starts at -0.0, the identity of addition.
template <int kModel>
__device__ __forceinline__ void edge_to_vertices(int e, const double (&gE)[3],
                                                 double (&g)[8][3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (kModel == 0) {
      g[kEdgeHi[e]][j] += gE[j];
      g[kEdgeLo[e]][j] -= gE[j];
    } else {
      const double t = 0.25 * gE[j];
#pragma unroll
      for (int v = 0; v < 8; ++v) g[v][j] += kOff[v][e] ? t : -t;
    }
  }
}

// dU/d(edge) of every edge from the stresses, gE_e = D_e E_e + the rows of S M off the diagonal,
// its share of the virial, and with kGrad of the vertex gradient g.
template <int kModel, bool kGrad>
__device__ __forceinline__ void edge_gradient(const double (&E)[Frame<kModel>::NE][3],
                                              const double (&D)[Frame<kModel>::NE],
                                              const double (&O)[Frame<kModel>::NC][3],
                                              double (&vir)[6], double (&g)[8][3]) {
#pragma clang fp contract(off)
  using F = Frame<kModel>;
  double gE[F::NE][3];
#pragma unroll
  for (int i = 0; i < F::NC; ++i) {
    const int a = F::corner(i);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::first(e) == i) {
#pragma unroll
        for (int j = 0; j < 3; ++j) gE[e][j] = D[e] * E[e][j];
      }
    }
#pragma unroll
    for (int o = 0; o < 3; ++o) {
      const int e0 = F::edge(a, F::axis0(o)), e1 = F::edge(a, F::axis1(o));
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        gE[e0][j] = __builtin_fma(O[a][o], E[e1][j], gE[e0][j]);
        gE[e1][j] = __builtin_fma(O[a][o], E[e0][j], gE[e1][j]);
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::last(e) == i) {
        edge_virial(gE[e], E[e], vir);
        if (kGrad) edge_to_vertices<kModel>(e, gE[e], g);
      }
    }
  }
}

// Edge e of a cell: the difference of its corners' positions plus f * rv, the domain vector of
// its axis when the cell wraps along it (f = 0 or 1).
__device__ __forceinline__ void form_edge(const double (&p)[8][3], int e, double f,
                                          const double* rv, double (&E)[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < 3; ++j)
    E[j] = __builtin_fma(f, rv[j], p[kEdgeHi[e]][j] - p[kEdgeLo[e]][j]);
}

// One state of an eight-corner cell in one sweep over its corners: an edge is formed at its
// first corner and gives its energy, virial and vertex terms at its second, so that at most five
// of the twelve edges are held at a time (kOut as the cell pass's: 0 energy, 1 and virial, 2 and
// vertex gradient). f, rv: wrap factors and domain vectors.
template <int kOut>
__device__ __forceinline__ double sweep_cell(const_f64 tab,
                                             const double (&p)[8][3], const double (&f)[3],
                                             const double (&rv)[9], double (&vir)[6],
                                             double (&g)[8][3]) {
#pragma clang fp contract(off)
  using F = Frame<0>;
  const const_f64 g0 = tab + kRestOffset;
  double E[12][3], q[12], D[12], gE[12][3];
  double u = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int a = F::corner(i);
    double x[6], O[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::first(e) == i) {
        form_edge(p, e, f[d], &rv[3 * d], E[e]);
        q[e] = edge_strain(E[e], d, g0[d], tab[kRestLowOffset + d]);
      }
      x[d] = q[e];
    }
#pragma unroll
    for (int o = 0; o < 3; ++o)
      x[3 + o] = edge_dot(E[F::edge(a, F::axis0(o))], E[F::edge(a, F::axis1(o))], g0[3 + o],
                          tab[kRestLowOffset + 3 + o]);
    corner_stress<0>(tab + kMetricOffset, i, x, D, O, u);
    if (kOut != 0) {
      bool open[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) open[d] = F::first(F::edge(a, d)) < i;
#pragma unroll
      for (int o = 0; o < 3; ++o) {
        const int d0 = F::axis0(o), d1 = F::axis1(o);
        const int e0 = F::edge(a, d0), e1 = F::edge(a, d1);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          gE[e0][j] = open[d0] ? __builtin_fma(O[o], E[e1][j], gE[e0][j]) : O[o] * E[e1][j];
          gE[e1][j] = open[d1] ? __builtin_fma(O[o], E[e0][j], gE[e1][j]) : O[o] * E[e0][j];
        }
        open[d0] = open[d1] = true;
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int e = F::edge(a, d);
      if (F::last(e) == i) {
        u = __builtin_fma(q[e], D[e], u);
        if (kOut != 0) {
#pragma unroll
          for (int j = 0; j < 3; ++j) gE[e][j] = __builtin_fma(D[e], E[e][j], gE[e][j]);
          edge_virial(gE[e], E[e], vir);
          if (kOut == 2) edge_to_vertices<0>(e, gE[e], g);
        }
      }
    }
    // keeps the corners apart: moved into each other they would need 200 registers
    asm("" : "+v"(u));
  }
  return 0.5 * u;
}

template <int NV>
__device__ __forceinline__ void wave_reduce(double (&v)[NV]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] += __shfl_down(v[q], off, 64);
  }
}

// Row vector times 3x3 matrix, without contractions: the position and velocity transforms of
// the barostat (npt.py:700-702, 725-726) give the same bits in every kernel that applies them.
__device__ __forceinline__ void vecmat(const double v[3], const double* M, double out[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < 3; ++j) out[j] = (v[0] * M[j] + v[1] * M[3 + j]) + v[2] * M[6 + j];
}

// g = the sum of node n's records in k order (mmff.py:303-318): record e = ncell[k * N + n]
// (none when e < 0) holds the three components gcell[(3 * (e & 3) + j) * RS + (e >> 2)];
// g starts at +0.0 and takes the records present in k order.
// kAllLoads: the eight indices are loaded first and then all 24 components, a none reading those
// of record 0 (always allocated) and left out of the sum, so that every load of the lane is in
// flight at once (two memory round trips instead of up to sixteen), at the cost of about 50
// more VGPRs; the same bits as skipping the nones. Without it each record is loaded behind
// the test of its index, which keeps the registers few: the form for passes with enough
// waves to hide the latency. (Two or four records at a time there, nones read too, whole evaluation:
// 72x80x96 cells 76.6 -> 74.1 us, but 80^3 66.4 -> 69.7, 96^3 99.8 -> 102, 128^3 202 -> 211 and 160^3
// 401 -> 431 us.)
// The loads carry the non-temporal hint.
template <bool kAllLoads>
__device__ __forceinline__ void sum_node_records(const int32_t* __restrict__ ncell,
                                                 const double* gcell, int64_t N, int64_t RS,
                                                 int64_t n, double g[3]) {
  auto load = [](const auto* p) { return __builtin_nontemporal_load(p); };
#pragma unroll
  for (int j = 0; j < 3; ++j) g[j] = 0.0;
  if (!kAllLoads) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int32_t e = load(&ncell[k * N + n]);
      if (e >= 0) {
        const int64_t w = e >> 2;
        const int p = e & 3;
#pragma unroll
        for (int j = 0; j < 3; ++j)
          g[j] += load(&gcell[(int64_t)(3 * p + j) * RS + w]);
      }
    }
    return;
  }
  int32_t e[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) e[k] = load(&ncell[k * N + n]);
  double r[8][3];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int32_t c = e[k] >= 0 ? e[k] : 0;
    const int64_t w = c >> 2;
    const int p = c & 3;
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r[k][j] = load(&gcell[(int64_t)(3 * p + j) * RS + w]);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int j = 0; j < 3; ++j) g[j] = e[k] >= 0 ? g[j] + r[k][j] : g[j];
}

// Workgroups are dealt to the 8 XCDs of the device in turn (block b runs on XCD b mod 8), and
// every XCD has its own L2. Neighbouring blocks share cache lines (the cell segments share
// nodes, the node blocks' record gathers share the lines at their ends), so each XCD is given
// one contiguous range of the n blocks: block b -> (b mod 8) * (n / 8) + min(b mod 8, n mod 8)
// + b / 8. The map is a bijection of [0, n) for any n.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int n) {
  const int q = n / kXcds, r = n % kXcds, x = b % kXcds, i = b / kXcds;
  return x * q + (x < r ? x : r) + i;
}

// 64-bit DPP move (two 32-bit moves): the lanes that kBanks enables take v from the lane kCtrl
// names (row_shl:N reads lane + N, row_shr:N lane - N, quad_perm within four lanes), the others
// keep old. A register-to-register exchange, no LDS round trip.
template <int kCtrl, int kBanks>
__device__ __forceinline__ double dpp_f64(double old, double v) {
  const long long o = __double_as_longlong(old), x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, kCtrl, 0xF, kBanks, false);
  const int hi =
      __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), kCtrl, 0xF, kBanks, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                          (unsigned long long)(unsigned)lo));
}

// Row swap of two registers (v_permlane32_swap / v_permlane16_swap): with kDist 32 lanes 32-63
// of x trade places with lanes 0-31 of y, with kDist 16 the odd 16-lane rows of x with the even
// rows of y. Afterwards a lane whose bit kDist is clear holds its own x in x and its partner's
// (lane ^ kDist) x in y; a lane whose bit is set holds its own y in y and its partner's y in x.
template <int kDist>
__device__ __forceinline__ void row_swap(double& x, double& y) {
  static_assert(kDist == 16 || kDist == 32, "row swaps across 16 or 32 lanes");
  const unsigned long long xb = (unsigned long long)__double_as_longlong(x);
  const unsigned long long yb = (unsigned long long)__double_as_longlong(y);
  const unsigned xl = (unsigned)xb, xh = (unsigned)(xb >> 32);
  const unsigned yl = (unsigned)yb, yh = (unsigned)(yb >> 32);
  unsigned xl2, xh2, yl2, yh2;
  if (kDist == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap(xl, yl, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(xh, yh, false, false);
    xl2 = lo[0], yl2 = lo[1], xh2 = hi[0], yh2 = hi[1];
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap(xl, yl, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(xh, yh, false, false);
    xl2 = lo[0], yl2 = lo[1], xh2 = hi[0], yh2 = hi[1];
  }
  x = __longlong_as_double((long long)(((unsigned long long)xh2 << 32) | xl2));
  y = __longlong_as_double((long long)(((unsigned long long)yh2 << 32) | yl2));
}

// Wave sums of up to 16 values by a reduce-scatter butterfly: returns in lane l the wave total
// of value q(l) = 8 b5 + 4 b4 + 2 b3 + b2 (bk = bit k of l); values q >= NV are zero. At each
// level a lane keeps the upper half of its values when its bit is set, the lower half
// otherwise, and adds its partner's copy of them: across 32 and 16 lanes by row swaps, across
// 8 and 4 lanes by two bank-masked DPP row shifts, the last two levels (a plain butterfly on
// one value) by quad permutations. Every exchange stays in registers; the pairs and the order
// of every addition are fixed, so the sums are deterministic.
template <int NV>
__device__ __forceinline__ double wave_reduce_scatter(const double (&v)[NV], int lane) {
  static_assert(NV >= 1 && NV <= 16, "1 to 16 values");
  constexpr int L1 = NV < 8 ? NV : 8, L2 = L1 < 4 ? L1 : 4, L3 = L2 < 2 ? L2 : 2;
  double a[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) a[q] = q < NV ? v[q] : 0.0;
  // lane ^ 32, pairs (i, 8 + i); a pair of zeros stays zero
#pragma unroll
  for (int i = 0; i < L1; ++i) {
    double x = a[i], y = a[8 + i];
    row_swap<32>(x, y);
    a[i] = x + y;
  }
  // lane ^ 16, pairs (i, 4 + i)
#pragma unroll
  for (int i = 0; i < L2; ++i) {
    double x = a[i], y = a[4 + i];
    row_swap<16>(x, y);
    a[i] = x + y;
  }
  // lane ^ 8, pairs (i, 2 + i): lanes 0-7 of a row read lane + 8's a[i], lanes 8-15 lane - 8's
  // a[2 + i]
  const bool up8 = (lane & 8) != 0;
#pragma unroll
  for (int i = 0; i < L3; ++i) {
    const double t = dpp_f64<0x118, 0xC>(dpp_f64<0x108, 0x3>(0.0, a[i]), a[2 + i]);
    a[i] = (up8 ? a[2 + i] : a[i]) + t;
  }
  // lane ^ 4, the pair (0, 1): banks 0 and 2 read lane + 4, banks 1 and 3 lane - 4
  const bool up4 = (lane & 4) != 0;
  const double t = dpp_f64<0x114, 0xA>(dpp_f64<0x104, 0x5>(0.0, a[0]), a[1]);
  double s = (up4 ? a[1] : a[0]) + t;
  s += dpp_f64<0x4E, 0xF>(s, s);  // lane ^ 2
  s += dpp_f64<0xB1, 0xF>(s, s);  // lane ^ 1
  return s;
}

__device__ __forceinline__ int scatter_index(int lane) {
  return ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 2) & 1);
}

}  // namespace mm
