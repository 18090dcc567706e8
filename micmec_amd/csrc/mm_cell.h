// The work of one cell of the force field on one lane: energy, virial and vertex gradient, and the
// storing of the gradient's face-class records. Shared by the cell pass (mm_force.hip) and the
// one-launch MD loop (mm_md.hip), which thereby give the same bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mm_device.h"
#include "mm_kernels.h"

namespace mm {

// What a cell pass forms: the energy, the virial too, the vertex gradient (and records) too.
constexpr int kOutEnergy = 0, kOutVirial = 1, kOutGradient = 2;

// The node positions of a cell's eight corners. All 24 loads are issued before any arithmetic.
// With on every position is taken through the pending transforms: xm2 (with on2), then xm (vecmat,
// the products the scaling pass stores, in its order).
__device__ __forceinline__ void load_corners(const double* pos, const int n[8],
                                             double (&p)[8][3], bool on, const double* xm,
                                             bool on2, const double* xm2) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    // 3 n < 2^32 (n < 2^30): a 32-bit product
    const double* t = pos + (uint64_t)(3u * (uint32_t)n[k]);
#pragma unroll
    for (int j = 0; j < 3; ++j) p[k][j] = t[j];
  }
  if (on2) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      double t[3];
      vecmat(p[k], xm2, t);
#pragma unroll
      for (int j = 0; j < 3; ++j) p[k][j] = t[j];
    }
  }
  if (on) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      double t[3];
      vecmat(p[k], xm, t);
#pragma unroll
      for (int j = 0; j < 3; ++j) p[k][j] = t[j];
    }
  }
}

// The edges of a cell (or the averaged matrix): pos[n_hi] - pos[n_lo] of the edge's corners, plus
// rvecs[d] for the edges along d when the cell is in the last layer along the periodic axis d
// (mmff.py:347-371 with get_mic 258-286). The reference forms vertices relative to corner 0
// and then edge differences; taking the differences of the positions directly avoids the
// vertices' rounding. The shifts use factors f of 0 or 1 (exact products) rather than
// data-dependent selects.
template <int kModel>
__device__ __forceinline__ void form_edges(const double (&p)[8][3], const double (&f)[3],
                                           const double (&rv)[9],
                                           double (&E)[Frame<kModel>::NE][3]) {
#pragma clang fp contract(off)
  double t[12][3];
#pragma unroll
  for (int e = 0; e < 12; ++e) form_edge(p, e, f[e / 4], &rv[3 * (e / 4)], t[e]);
#pragma unroll
  for (int e = 0; e < Frame<kModel>::NE; ++e)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      E[e][j] = kModel == 0 ? t[e][j]
                            : 0.25 * ((t[4 * e % 12][j] + t[(4 * e + 1) % 12][j]) +
                                      (t[(4 * e + 2) % 12][j] + t[(4 * e + 3) % 12][j]));
}

// Corners of the lower (z = 0) and upper (z = 1) face of a cell, in face-class order: upper
// corner kUpperCorner[q] of a cell is lower corner kLowerCorner[q] of its +z neighbour.
__device__ constexpr int kLowerCorner[4] = {0, 1, 2, 4};
__device__ constexpr int kUpperCorner[4] = {3, 5, 6, 7};

// Entry i of a gradient plane (S < 2^29, so that the byte offset fits 32 bits beside the plane's
// uniform base), with the non-temporal hint.
__device__ __forceinline__ void store_record(double* plane, uint32_t i, double v) {
  double* t = reinterpret_cast<double*>(reinterpret_cast<char*>(plane) + (size_t)(i * 8u));
  __builtin_nontemporal_store(v, t);
}

// Energies of all states of a cell, combined by the log-sum-exp of mmff.py:386-398, with virial
// (00, 11, 22, 12, 02, 01) and vertex gradient as kOut asks. tab: the table entries of the cell's
// type, ns its states; valid: false for a padding slot, which gives zeros; corners(p) puts the node
// positions of the cell's corners into p; acc: the lane's column of an LDS array
// [NE + 3 NC][kStride] (kMulti with a virial only).
template <int kModel, int kOut, bool kMulti, int kStride, typename Corners>
__device__ __forceinline__ void cell_eval(const_f64 tab, int ns, double kt, bool valid,
                                          Corners corners, int wrap, const double (&rv)[9],
                                          double* acc, double& ecell, double (&vir)[6],
                                          double (&gacc)[8][3]) {
#pragma clang fp contract(off)
  using F = Frame<kModel>;
  constexpr bool kGrad = kOut == kOutGradient, kVir = kOut != kOutEnergy;
  ecell = 0.0;
#pragma unroll
  for (int q = 0; q < 6; ++q) vir[q] = 0.0;
#pragma unroll
  for (int v = 0; v < 8; ++v)
#pragma unroll
    for (int j = 0; j < 3; ++j) gacc[v][j] = -0.0;
  if (valid) {
    double p[8][3], f[3];
    corners(p);
#pragma unroll
    for (int d = 0; d < 3; ++d) f[d] = (double)((wrap >> d) & 1);
    if constexpr (kModel == 0 && !kMulti) {
      ecell = tab[10] + sweep_cell<kOut>(tab, p, f, rv, vir, gacc);
    } else {
      double E[F::NE][3], q[F::NE], D[F::NE], O[F::NC][3];
      form_edges<kModel>(p, f, rv, E);
#pragma unroll
      for (int e = 0; e < F::NE; ++e)
        q[e] = edge_strain(E[e], F::along(e), tab[kRestOffset + F::along(e)],
                           tab[kRestLowOffset + F::along(e)]);
      if (!kMulti) {
        ecell = tab[10] + state_stress<kModel>(tab, E, q, D, O);
      } else {
        // one pass over the states (mmff.py:386-398): E = E_min - kT ln Z with Z = sum_s c_s,
        // c_s = exp(-(E_s - E_min)/kT), and the stresses sum_s c_s S_s accumulated in LDS, both
        // relative to the lowest energy so far and rescaled when it moves
        double emin = 0.0, zsum = 0.0;
        for (int s = 0; s < ns; ++s) {
          const const_f64 ts = tab + s * kTabStride;
          const double es = ts[10] + state_stress<kModel>(ts, E, q, D, O);
          double keep = 0.0, c = 1.0;  // factors of the sums so far and of this state
          if (s == 0) {
            emin = es;
            zsum = 1.0;
          } else if (es < emin) {
            keep = exp(-(emin - es) / kt);
            zsum = zsum * keep + 1.0;
            emin = es;
          } else {
            keep = 1.0;
            c = exp(-(es - emin) / kt);
            zsum += c;
          }
          if (kVir) {
            if (s == 0) {
#pragma unroll
              for (int e = 0; e < F::NE; ++e) acc[e * kStride] = D[e];
#pragma unroll
              for (int q = 0; q < 3 * F::NC; ++q) acc[(F::NE + q) * kStride] = O[q / 3][q % 3];
            } else {
#pragma unroll
              for (int e = 0; e < F::NE; ++e) {
                if (e % 6 == 0) __builtin_amdgcn_sched_barrier(0);
                acc[e * kStride] = __builtin_fma(c, D[e], keep * acc[e * kStride]);
              }
#pragma unroll
              for (int q = 0; q < 3 * F::NC; ++q) {
                // six columns in flight at a time: all of them would not fit the registers
                if (q % 6 == 0) __builtin_amdgcn_sched_barrier(0);
                double* t = acc + (F::NE + q) * kStride;
                *t = __builtin_fma(c, O[q / 3][q % 3], keep * *t);
              }
            }
          }
        }
        ecell = emin - kt * log(zsum);
        if (kVir) {
          const double inv = 1.0 / zsum;
#pragma unroll
          for (int e = 0; e < F::NE; ++e) D[e] = acc[e * kStride] * inv;
#pragma unroll
          for (int q = 0; q < 3 * F::NC; ++q) O[q / 3][q % 3] = acc[(F::NE + q) * kStride] * inv;
        }
      }
      if (kVir) edge_gradient<kModel, kGrad>(E, D, O, vir, gacc);
    }
  }
}

// The upper face (corners 3, 5, 6, 7) of the slot below is added to this slot's lower face (corners
// 0, 1, 2, 4) when that slot holds the -z neighbour (wrap bit 3). The move from lane - 1 is a DPP
// wave shift (lane 0, which never folds, keeps its own value). Every lane of the wave calls this.
__device__ __forceinline__ void fold_cell(int wrap, double (&gacc)[8][3]) {
#pragma clang fp contract(off)
  const bool fold = (wrap & 8) != 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double up = gacc[kUpperCorner[q]][j];
      const double t = dpp_f64<0x138, 0xF>(up, up);  // wave_shr:1
      const double lo = gacc[kLowerCorner[q]][j];
      gacc[kLowerCorner[q]][j] = fold ? lo + t : lo;
    }
  }
}

// The vertex gradient of the cell in slot w as records (every lane of the wave calls this).
__device__ __forceinline__ void store_cell(int64_t w, int wrap, bool valid,
                                           const int32_t* __restrict__ cbase, int64_t W,
                                           int64_t S, double* gcell, double (&gacc)[8][3]) {
  // the lower faces go to their class planes, the upper faces that were not folded (wrap bit 4
  // clear) to the wave's compact slots, in lane order
  fold_cell(wrap, gacc);
  if (valid) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        store_record(gcell + (int64_t)(3 * q + j) * S, (uint32_t)w, gacc[kLowerCorner[q]][j]);
  }
  const bool open_top = valid && !(wrap & 16);
  const uint64_t tops = __ballot(open_top);
  if (open_top) {
    const int lane = threadIdx.x & 63;
    const uint32_t ci =
        (uint32_t)W + (uint32_t)cbase[w >> 6] + __popcll(tops & ((1ull << lane) - 1ull));
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        store_record(gcell + (int64_t)(3 * q + j) * S, ci, gacc[kUpperCorner[q]][j]);
  }
}

// Wave totals of the energy and the six virial entries (the reduce-scatter butterfly) into red[7].
__device__ __forceinline__ void cell_wave_totals(double ecell, const double (&vir)[6],
                                                 double* red) {
  const double v[7] = {ecell, vir[0], vir[1], vir[2], vir[3], vir[4], vir[5]};
  const int lane = threadIdx.x & 63;
  const double t = wave_reduce_scatter<7>(v, lane);
  const int q = scatter_index(lane);
  if ((lane & 3) == 0 && q < 7) red[q] = t;
}

// Where a wave's totals (cell_wave_totals) hold entry q < 10 of the energy and the full 3x3 virial:
// {0, 1, 6, 5, 6, 2, 4, 5, 4, 3}, as nibbles (a table would be a load from memory).
__device__ __forceinline__ int total_entry(int q) {
  return (int)(0x3454265610ull >> (4 * q)) & 0xf;
}

// Entry q < 10 of a block's totals from its waves' red[4][7], in wave order.
__device__ __forceinline__ double cell_block_total(const double* red, int q) {
  const int e = total_entry(q);
  double s = red[e];
#pragma unroll
  for (int w = 1; w < kCellBlock / 64; ++w) s += red[w * 7 + e];
  return s;
}

}  // namespace mm
