// Device MD engine: velocity Verlet with Nose-Hoover chain or Langevin thermostat and MTK or
// Langevin barostat (FP64).
//
// Reference sequence (one step, micmec/sampling/verlet.py:140-166):
//   pre hooks  -> v += a dt/2 -> x += v dt -> force -> v += a dt/2 -> ekin -> post hooks
// With a thermostat and a barostat the hooks run as TBCombination (micmec/sampling/npt.py:99-148):
//   pre  = MTK.baro (npt.py:653-736) then NHC chain (nvt.py:410-451);
//   post = NHC chain then MTK.baro. Each MTK.baro call evaluates the force once more.
// Node-wise work runs in wide kernels; every scalar update (chain, barostat velocity, 3x3
// symmetric exponentials, energies, conserved-quantity tracking) runs in a small kernel on the
// scalar block S between the node kernels (its blocks reduce the partial sums, the last one
// runs the phase), so a whole step can be captured in a HIP graph. Velocity/position
// transforms produced by a scalar phase (thermostat factors, barostat matrices) are stored in
// S and applied by the next pass that reads the array; kinetic sums after a pending barostat
// matrix follow from the sums before it. The Langevin thermostat's noise is drawn inside the
// node passes that already touch the velocities (pre: the kick-drift pass, with a barostat
// the gather that is the kick-drift; post: the gather-kick pass), from a counter-based
// generator keyed by node and hook call, so it costs no extra pass over the nodes.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/micmec_amd.h"
#include "mm_cell.h"
#include "mm_device.h"
#include "mm_internal.h"
#include "mm_kernels.h"
#include "mm_rng.h"

namespace mm {

constexpr int kNodeBlock = 256;   // nodes per block (system boundaries are block aligned)
// What a node gather does with the face-class records (gather_kick_kernel).
constexpr int kGatherNone = 0, kGatherKeep = 1, kGatherStore = 2;
constexpr int kNodeThreads = 64;  // one wave per block, kNodeBlock / kNodeThreads nodes a lane
// node sums: [0] ekin [1..9] sum m v(x)v [10] sum g^2 [11] sum d^2 [12] nan
// [13] ekin before the Langevin post update [14] ekin after the Langevin pre update
constexpr int kNodePartial = 16;
constexpr int kNodeSums = 16;
constexpr int kScalarThreads = 256;
constexpr int kScalarSlices = 32;  // most blocks a scalar phase spreads its reduction over
// Systems of at most this many cell and node blocks run the phases of a row of steps inside the
// kernels after them (and sum a phase's partials in one block otherwise).
constexpr int kMergeMaxBlocks = 512;
constexpr int kSliceQ = 10 + kNodeSums;  // force and node sums per slice

enum NodeMode {
  kScalePos = 1,
  kVV = 3,
  kApplyV = 4,
  kRmsd = 5,
};

enum Phase {
  kPhInitForce = 0,      // epot (+ vtens) after an initial force evaluation
  kPhInitProps = 1,      // node sums -> ekin, svv; properties without advancing time
  kPhNveEnd = 2,         // force + node sums after the second kick; properties
  kPhNvtPre = 3,         // NHC pre
  kPhNvtEnd = 4,         // force + node sums; NHC post; properties
  kPhBaroPre = 5,        // TBC pre, barostat: v_g update, position/domain and velocity transforms
  kPhBaroEndPre = 7,     // force; kinetic sums after the pending velocity matrix; v_g; NHC pre
  kPhMainEndNpt = 8,     // force + node sums; NHC post; barostat transforms of the post call
  kPhBaroEndPost = 9,    // force (+ gather NaN flag); kinetic sums after the matrix; v_g; econs
  kPhRmsd = 10,          // rmsd_gpos / rmsd_delta
  kPhApplied = 11,       // pending transforms were applied
  kPhBaroEndPostPre = 12,  // kPhBaroEndPost, then the next step's kPhBaroPre (steps in a row)
  kPhNvtEndPre = 13,       // kPhNvtEnd, then the next step's kPhNvtPre (steps in a row)
  // kPhNvtEnd of a Langevin step in a row of steps: the thermostat's pre update is accounted for in
  // the phase of the step whose gather made it (nd[14]), the first step's (nd[15]) in its own
  kPhLtFirst = 14,
  kPhLtNext = 15,
  kPhLtLast = 16,
};

// ----------------------------------------------------------------------------- node kernels

// Block totals of a node pass (one wave per block), written SoA: out[q * gridDim.x + blockIdx.x].
template <int NV>
__device__ __forceinline__ void block_sum_store(double (&v)[NV], double* part) {
  const int lane = threadIdx.x & 63;
  const double t = wave_reduce_scatter<NV>(v, lane);
  const int q = scatter_index(lane);
  if ((lane & 3) == 0 && q < NV) part[(int64_t)q * gridDim.x + blockIdx.x] = t;
}

// The same for blocks of kNodeBlock threads (waves summed in order through LDS), into the
// partial slot of logical block blk.
template <int NV>
__device__ __forceinline__ void block_sum_store_wide(double (&v)[NV], double* part, int blk) {
  __shared__ double red[NV * (kNodeBlock / 64)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  {
    const double t = wave_reduce_scatter<NV>(v, lane);
    const int q = scatter_index(lane);
    if ((lane & 3) == 0 && q < NV) red[wave * NV + q] = t;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double s = red[threadIdx.x];
    for (int w = 1; w < kNodeBlock / 64; ++w) s += red[w * NV + threadIdx.x];
    part[(int64_t)threadIdx.x * gridDim.x + blk] = s;
  }
}

// Kinetic-energy and m v (x) v sums of one node, in the reference's operation order:
// 0.5 * (v**2 * m) (verlet.py:169) and (v.T * m) . v (verlet.py:187-188, npt.py:661-663).
template <int NA>
__device__ __forceinline__ void node_vv(const double v[3], double m, double (&acc)[NA]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < 3; ++j) acc[0] += 0.5 * ((v[j] * v[j]) * m);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[1 + 3 * i + j] += (v[i] * m) * v[j];
}

// LangevinThermostat.thermo (nvt.py:211-218): v = c1 v + sqrt((1 - c1^2) T k_B / m) xi with
// xi the standard normals of node n at hook call 2 counter + call (0: pre, 1: post, 2: the next
// step's pre, before the counter moves).
__device__ __forceinline__ void langevin_thermo(const double* S, int64_t n, int call, double m,
                                                double v[3]) {
#pragma clang fp contract(off)
  const uint64_t ctr[4] = {(uint64_t)n, 2ull * (uint64_t)S[MM_S_COUNTER] + (uint64_t)call, 0ull,
                           0ull};
  double z[4];
  normals4(ctr, seed_from(S + MM_S_LT_SEED), kStreamThermostat, z);
  const double c1 = S[MM_S_LT_C1];
  const double c2 = sqrt(S[MM_S_LT_A] / m);
#pragma unroll
  for (int j = 0; j < 3; ++j) v[j] = c1 * v[j] + c2 * z[j];
}

__device__ __forceinline__ double node_ekin(const double v[3], double m) {
#pragma clang fp contract(off)
  double e = 0.0;
#pragma unroll
  for (int j = 0; j < 3; ++j) e += 0.5 * ((v[j] * v[j]) * m);
  return e;
}

// Pending velocity transforms, applied in the order the reference performs them:
// factor A (thermostat post of the previous half), matrix M (barostat), matrix M2 (the next
// barostat call, when M still waits), factor B (thermostat pre). A null pointer is a transform
// that is off.
__device__ __forceinline__ void apply_vtransform(const double* fa, const double* M,
                                                 const double* M2, const double* fb,
                                                 double v[3]) {
#pragma clang fp contract(off)
  if (fa) {
    const double f = *fa;
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = v[j] * f;
  }
  if (M) {
    double t[3];
    vecmat(v, M, t);
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = t[j];
  }
  if (M2) {
    double t[3];
    vecmat(v, M2, t);
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = t[j];
  }
  if (fb) {
    const double f = *fb;
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = v[j] * f;
  }
}

// The transforms as the scalar block holds them, read where they are applied.
__device__ __forceinline__ void apply_vtransform(const double* __restrict__ S, double v[3]) {
  apply_vtransform(S[MM_S_VSCALE_A_ON] != 0.0 ? S + MM_S_VSCALE_A : nullptr,
                   S[MM_S_VMAT_ON] != 0.0 ? S + MM_S_VMAT : nullptr,
                   S[MM_S_VMAT2_ON] != 0.0 ? S + MM_S_VMAT2 : nullptr,
                   S[MM_S_VSCALE_B_ON] != 0.0 ? S + MM_S_VSCALE_B : nullptr, v);
}

// What a step does to one node, on values that the caller has loaded; S is the system's scalar
// block (in HBM or LDS).

// First half kick and drift (verlet.py:141-146): with kLT the Langevin thermostat's pre update (its
// kinetic energy after it added to lt), then v += a dt / 2 and x += dt v.
template <bool kLT>
__device__ __forceinline__ void half_step_node(const double* S, int64_t n, int call, double mass,
                                               const double g[3], double v[3], double x[3],
                                               double& lt) {
#pragma clang fp contract(off)
  const double dt = S[MM_S_TIMESTEP];
  if (kLT) {
    langevin_thermo(S, n, call, mass, v);
    lt += node_ekin(v, mass);
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double a = -g[j] / mass;
    v[j] = v[j] + (0.5 * a) * dt;
    x[j] = x[j] + dt * v[j];
  }
}

// The same after the pending velocity transforms.
template <bool kLT>
__device__ __forceinline__ void kick_drift_node(const double* S, int64_t n, double mass,
                                                const double g[3], double v[3], double x[3],
                                                double& lt) {
  apply_vtransform(S, v);
  half_step_node<kLT>(S, n, 0, mass, g, v, x, lt);
}

// The pending position transforms: an earlier call's when it still waits (the previous post
// call's, of steps in a row), then the last one's.
__device__ __forceinline__ void scale_position(const double* S, double x[3]) {
  double t[3];
  if (S[MM_S_XMAT2_ON] != 0.0) {
    vecmat(x, S + MM_S_XMAT2, t);
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] = t[j];
  }
  vecmat(x, S + MM_S_XMAT, t);
#pragma unroll
  for (int j = 0; j < 3; ++j) x[j] = t[j];
}

// Second half kick (verlet.py:152-153) and the node sums acc[0..9] of the new velocities; with
// kLT the Langevin thermostat's post update in between (the kinetic energy before it in lt).
template <bool kLT, int NA>
__device__ __forceinline__ void kick_node(const double* S, int64_t n, double mass,
                                          const double g[3], double v[3], double (&acc)[NA],
                                          double& lt) {
#pragma clang fp contract(off)
  const double dt = S[MM_S_TIMESTEP];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double a = -g[j] / mass;
    v[j] = v[j] + (0.5 * a) * dt;
  }
  if (kLT) {
    lt += node_ekin(v, mass);
    langevin_thermo(S, n, 1, mass, v);
  }
  node_vv(v, mass, acc);
}

template <int kMode>
__global__ void __launch_bounds__(kNodeThreads)
node_kernel(double* __restrict__ x, double* __restrict__ v, const double* __restrict__ g,
            const double* __restrict__ m, const double* __restrict__ xold,
            const double* __restrict__ S0, const int32_t* __restrict__ blk_sys, int64_t N,
            double* __restrict__ partials) {
#pragma clang fp contract(off)
  const double* S = S0 + (blk_sys ? (int64_t)blk_sys[blockIdx.x] * MM_S_COUNT : 0);
  double acc[13];
#pragma unroll
  for (int q = 0; q < 13; ++q) acc[q] = 0.0;
  constexpr int kIt = kNodeBlock / kNodeThreads;
  const int64_t n0 = (int64_t)blockIdx.x * kNodeBlock + threadIdx.x;
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int64_t n = n0 + it * kNodeThreads;
    if (n >= N) break;
    if (kMode == kScalePos) {
      double p[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) p[j] = x[3 * n + j];
      scale_position(S, p);
#pragma unroll
      for (int j = 0; j < 3; ++j) x[3 * n + j] = p[j];
    } else if (kMode == kVV || kMode == kApplyV) {
      double vv[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) vv[j] = v[3 * n + j];
      if (kMode != kVV) {
        apply_vtransform(S, vv);
#pragma unroll
        for (int j = 0; j < 3; ++j) v[3 * n + j] = vv[j];
      }
      if (kMode != kApplyV) node_vv(vv, m[n], acc);
    } else if (kMode == kRmsd) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const double gj = g[3 * n + j];
        const double d = x[3 * n + j] - xold[3 * n + j];
        acc[10] += gj * gj;
        acc[11] += d * d;
      }
    }
  }
  if (kMode == kVV || kMode == kRmsd) {
    block_sum_store<13>(acc, partials);
  }
}

// ----------------------------------------------------------------------------- scalar math
//
// The scalar phases are one long dependence chain on a few dozen numbers, and every kernel of the
// step waits for them. They run on the 64 lanes of one wave: what is one number is computed by
// all lanes alike, the nine entries of a 3x3 matrix by nine lanes at once (entry_of), the beads of
// a chain by a lane each, the two exponentials of a barostat call by the two halves of the wave,
// and the divisions of the properties together, so that the chain holds few divisions and few
// waits for LDS; the scalar block is in LDS, where a wave's accesses keep their order. A wave
// alone on its SIMD issues an instruction every four to eight cycles, so the length of this code is
// its time: all phases of a step took 5.4 us (NVT-NHC) and 23 us (NPT) on one lane, now 3.4 and
// 10.7 us; 32^3 NVT step 37.7 -> 34.8 us, 24x19x27 NPT 82 -> 72 us, 128^3 NPT 579 -> 572 us.

// The scalar block of a phase, in LDS; six more doubles behind it are scratch.
typedef __attribute__((address_space(3))) double lds_f64;
constexpr int kScratch = MM_S_COUNT;

// Lane l's copy of v.
__device__ __forceinline__ double lane_value(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The matrix entry of a lane: lanes 0..8 own one each, the others repeat the last.
__device__ __forceinline__ int entry_of(int lane) { return lane < 9 ? lane : 8; }
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// exp(x): for |x| <= 1/16, where the chains' and barostats' arguments lie, the Taylor polynomial of
// degree 11 (first omitted term below 2e-22) as 1 + (x + x^2 q), a dozen instructions in six
// dependent steps; the general function otherwise.
__device__ __attribute__((noinline)) double exp_far(double x) { return exp(x); }
__device__ __forceinline__ double exp_near0(double x) {
  if (__any(!(fabs(x) <= 0.0625))) return exp_far(x);
  const double x2 = x * x, x4 = x2 * x2;
  const double a0 = __builtin_fma(x, 1.0 / 6, 1.0 / 2), a1 = __builtin_fma(x, 1.0 / 120, 1.0 / 24),
               a2 = __builtin_fma(x, 1.0 / 5040, 1.0 / 720),
               a3 = __builtin_fma(x, 1.0 / 362880, 1.0 / 40320),
               a4 = __builtin_fma(x, 1.0 / 39916800, 1.0 / 3628800);
  const double b0 = __builtin_fma(x2, a1, a0), b1 = __builtin_fma(x2, a3, a2);
  const double q = __builtin_fma(x4, __builtin_fma(x4, a4, b1), b0);
  return 1.0 + __builtin_fma(x2, q, x);
}

// D = C + A B (D may be C).
__device__ __forceinline__ void fma_matmul(const double (&A)[9], const double (&B)[9],
                                           const double (&C)[9], double (&D)[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      D[3 * i + j] = __builtin_fma(
          A[3 * i + 2], B[6 + j],
          __builtin_fma(A[3 * i + 1], B[3 + j],
                        __builtin_fma(A[3 * i + 0], B[0 + j], C[3 * i + j])));
}

// R = exp(sign * A * dt / 2) for symmetric A: the matrix the reference forms from
// eigh(A) = (w, Q) as Q diag(exp(sign w dt / 2)) Q^T (npt.py:686-690, 709-726), here by scaling
// and squaring, one matrix a lane. X = sign * A * dt / 2 is halved s times until
// r = ||X||_inf <= 1/2, exp(X) is the Taylor polynomial of degree 6 where r <= 1/80 on every lane
// (its first omitted term r^7 / 7! is then below 1e-17; a barostat velocity times dt / 2 is of
// order 1e-5 to 1e-3), as I + X + X^2 / 2 + X^3 (I / 6 + X / 24 + X^2 / 120 + X^3 / 720), and of
// degree 14 otherwise (the remainder is at most e^r times the first omitted term against
// ||exp(X)|| >= e^-r: below 7e-17 relative at r = 1/2); the result is squared s times.
__device__ __forceinline__ void expm_sym_half(const double (&A)[9], double sign, double dt,
                                              double (&P)[9]) {
#pragma clang fp contract(off)
  const double h = (sign * dt) / 2.0;
  double X[9];
  double nrm = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double r = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      X[3 * i + j] = h * A[3 * i + j];
      r += fabs(X[3 * i + j]);
    }
    nrm = fmax(nrm, r);
  }
  if (__all(nrm <= 0.0125)) {
    double X2[9], X3[9], B[9];
    const double zero[9] = {};
    fma_matmul(X, X, zero, X2);
    fma_matmul(X2, X, zero, X3);
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      const double one = (q % 4 == 0) ? 1.0 : 0.0;
      P[q] = __builtin_fma(X2[q], 0.5, one + X[q]);
      B[q] = __builtin_fma(X3[q], 1.0 / 720,
                           __builtin_fma(X2[q], 1.0 / 120,
                                         __builtin_fma(X[q], 1.0 / 24, one * (1.0 / 6))));
    }
    fma_matmul(X3, B, P, P);
    return;
  }
  int s = 0;
  double scale = 1.0;
  while (nrm * scale > 0.5 && s < 64) {
    scale *= 0.5;
    ++s;
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) X[q] *= scale;
#pragma unroll
  for (int q = 0; q < 9; ++q) P[q] = (q % 4 == 0) ? 1.0 : 0.0;
#pragma unroll 1
  for (int k = 14; k >= 1; --k) {
    // P <- I + X P / k
    double T[9];
    const double zero[9] = {};
    fma_matmul(X, P, zero, T);
#pragma unroll
    for (int q = 0; q < 9; ++q) P[q] = __builtin_fma(T[q], 1.0 / k, (q % 4 == 0) ? 1.0 : 0.0);
  }
  for (int t = 0; t < s; ++t) {
    double T[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        T[3 * i + j] =
            (P[3 * i + 0] * P[0 + j] + P[3 * i + 1] * P[3 + j]) + P[3 * i + 2] * P[6 + j];
#pragma unroll
    for (int q = 0; q < 9; ++q) P[q] = T[q];
  }
}

// |det| of the domain vectors, as micmec/pes/domain.c:42-48.
__device__ double volume3(const lds_f64* r) {
#pragma clang fp contract(off)
  return fabs(r[0] * (r[4] * r[8] - r[5] * r[7]) + r[1] * (r[5] * r[6] - r[3] * r[8]) +
              r[2] * (r[3] * r[7] - r[4] * r[6]));
}

// Where a Nose-Hoover chain keeps its state in the scalar block: the particle thermostat's
// chain, or the MTK barostat's own chain (baro_thermo), which acts on the barostat alone.
struct ChainSlots {
  int len, temp, ndof, mass, pos, vel;
};
constexpr ChainSlots kThermoChain{MM_S_CHAIN_LEN, MM_S_THERMO_TEMP, MM_S_CHAIN_NDOF,
                                  MM_S_CHAIN_MASS, MM_S_CHAIN_POS, MM_S_CHAIN_VEL};
constexpr ChainSlots kBaroChain{MM_S_BCHAIN_LEN, MM_S_BCHAIN_TEMP, MM_S_BCHAIN_NDOF,
                                MM_S_BCHAIN_MASS, MM_S_BCHAIN_POS, MM_S_BCHAIN_VEL};

// The value of the next / previous lane (a DPP wave shift; the end lane keeps its own).
__device__ __forceinline__ double next_lane(double v) { return dpp_f64<0x130, 0xF>(v, v); }
__device__ __forceinline__ double previous_lane(double v) { return dpp_f64<0x138, 0xF>(v, v); }

// NHChain.__call__ (nvt.py:410-451): the velocity factor and the new kinetic energy. Lane k holds
// bead k. The sweep from the last bead to the first takes each bead's force from the old velocity
// of the bead before it, so all forces are formed at once and only the factors (from the new
// velocity of the bead behind) follow each other; the sweep back the other way round. The forces
// are divided by the masses through their reciprocals with one correction step, which rounds
// as the division does; (g dt) / 4 and (v dt) / 8 round as g (dt / 4) and v (dt / 8).
struct ChainStep {
  double factor, ekin;
};
__device__ __forceinline__ ChainStep nhc_chain(lds_f64* S, double ekin, bool has_g1, double g1,
                                               const ChainSlots& c) {
#pragma clang fp contract(off)
  const int lane = lane_id(), own = lane & 7;
  const int L = __builtin_amdgcn_readfirstlane((int)S[c.len]);
  const double dt = S[MM_S_TIMESTEP], dt4 = dt / 4.0, dt8 = dt / 8.0;
  const double kt = S[c.temp] * S[MM_S_BOLTZMANN];
  const double nkt = (S[c.ndof] * S[c.temp]) * S[MM_S_BOLTZMANN];
  const double mass = S[c.mass + own];
  double vel = S[c.vel + own];
  const double pos = S[c.pos + own];
  const double inv = 1.0 / mass, mass_before = previous_lane(mass);
  auto kick = [&](double v_before, double ek) {
    double first = 2.0 * ek - nkt;
    if (has_g1) first += g1;
    const double g = lane == 0 ? first : mass_before * (v_before * v_before) - kt;
    const double q = g * inv;
    return __builtin_fma(__builtin_fma(-q, mass, g), inv, q) * dt4;
  };
  auto damping = [&](double v) {
    const double e = exp_near0((-next_lane(v)) * dt8);
    return lane == L - 1 ? 1.0 : e;
  };
  const double down = kick(previous_lane(vel), ekin);
#pragma unroll 1
  for (int k = L - 1; k >= 0; --k) {
    const double e = damping(vel);
    const double v = (vel * e + down) * e;
    vel = lane == k ? v : vel;
  }
  if (lane < L) S[c.pos + own] = pos + (vel * dt) / 2.0;
  const double factor = exp_near0(((-lane_value(vel, 0)) * dt) / 2.0);
  ekin *= factor * factor;
  const double e = damping(vel);
#pragma unroll 1
  for (int k = 0; k < L; ++k) {
    const double v = (vel * e + kick(previous_lane(vel), ekin)) * e;
    vel = lane == k ? v : vel;
  }
  if (lane < L) S[c.vel + own] = vel;
  return {factor, ekin};
}

// NHChain.get_econs_correction (nvt.py:453-458)
__device__ __forceinline__ double nhc_econs(const lds_f64* S, const ChainSlots& c = kThermoChain) {
#pragma clang fp contract(off)
  const int L = __builtin_amdgcn_readfirstlane((int)S[c.len]);
  const int own = lane_id() & 7;
  const double kt = S[MM_S_BOLTZMANN] * S[c.temp];
  const double vel = S[c.vel + own], pos = S[c.pos + own];
  const double twice = (vel * vel) * S[c.mass + own];
  double kin = 0.0, rest = 0.0;
#pragma unroll 1
  for (int k = 0; k < L; ++k) {
    kin += lane_value(twice, k);
    if (k > 0) rest += lane_value(pos, k);
  }
  return 0.5 * kin + kt * (S[c.ndof] * lane_value(pos, 0) + rest);
}

__device__ __forceinline__ bool baro_chain_on(const lds_f64* S) {
  return S[MM_S_BCHAIN_ON] != 0.0;
}

// MTKBarostat._compute_ekin_baro (npt.py:748-757): W tr(v_g^T v_g) / 2, or W v_g^2 / 2 in the
// isotropic form.
__device__ __forceinline__ double baro_ekin(const lds_f64* S) {
#pragma clang fp contract(off)
  if (S[MM_S_BARO_ANISO] == 0.0)
    return (0.5 * S[MM_S_MASS_PRESS]) * (S[MM_S_VEL_PRESS] * S[MM_S_VEL_PRESS]);
  double v[9], tr = 0.0;
#pragma unroll
  for (int i = 0; i < 9; ++i) v[i] = S[MM_S_VEL_PRESS + i];
#pragma unroll
  for (int i = 0; i < 9; ++i) tr += v[i] * v[i];
  return (0.5 * S[MM_S_MASS_PRESS]) * tr;
}

// MTKBarostat.add_press_cont (npt.py:738-746); with its own chain the barostat is decoupled
// from the particle thermostat and contributes 0.
__device__ double add_press_cont(const lds_f64* S) {
#pragma clang fp contract(off)
  if (baro_chain_on(S)) return 0.0;
  return 2.0 * baro_ekin(S) - S[MM_S_BARO_NDOF] * (S[MM_S_BARO_TEMP] * S[MM_S_BOLTZMANN]);
}

// The barostat chain's half step on the barostat kinetic energy (npt.py:625-629, 634-638): the
// chain advances, the velocity factor it returns is discarded (v_g is damped inside
// update_baro_vel through chainvel0).
__device__ void baro_chain_step(lds_f64* S) {
  (void)nhc_chain(S, baro_ekin(S), true, 0.0, kBaroChain);
}

__device__ __forceinline__ bool baro_langevin(const lds_f64* S) {
  return S[MM_S_BARO] == (double)MM_BARO_LANGEVIN;
}
__device__ __forceinline__ bool baro_aniso(const lds_f64* S) {
  return S[MM_S_BARO_ANISO] != 0.0;
}
__device__ __forceinline__ bool thermo_nhc(const lds_f64* S) {
  return S[MM_S_THERMO] == (double)MM_THERMO_NHC;
}

// LangevinBarostat.getR (npt.py:489-505): a symmetric matrix whose lower triangle is a draw of
// N(0, 1) x RSCALE, here the normals of system sys at hook call 2 counter + post, update sub:
// the triangle row by row (00, 10, 11, 20, 21, 22).
__device__ __attribute__((noinline)) void langevin_random_force(const lds_f64* S, int sys,
                                                                 int post, int sub,
                                                                 lds_f64* R) {
#pragma clang fp contract(off)
  const uint64_t call = 2ull * (uint64_t)S[MM_S_COUNTER] + (uint64_t)post;
  const double seed[2] = {S[MM_S_LB_SEED], S[MM_S_LB_SEED + 1]};
  const uint64_t key = seed_from(seed);
  double z[8];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const uint64_t ctr[4] = {(uint64_t)sys, call, (uint64_t)sub, (uint64_t)b};
    normals4(ctr, key, kStreamBarostat, z + 4 * b);
  }
  const double sc = S[MM_S_LB_RSCALE];
#pragma unroll
  for (int k = 0; k < 6; ++k) R[k] = z[k] * sc;
}

// update_baro_vel of MTKBarostat.baro (npt.py:654-681) and of LangevinBarostat.baro
// (npt.py:394-432: friction exp(-dt / 8 tau) on both sides, random force R, optional volume
// constraint and isotropic form). sub is 0 for the first and 1 for the second update of a call.
// One entry of v_g a lane (the isotropic form has one for all).
__device__ __forceinline__ void update_baro_vel(lds_f64* S, int sys, int post, int sub) {
#pragma clang fp contract(off)
  const int q = entry_of(lane_id()), i = q / 3, j = q - 3 * i, qt = 3 * j + i;
  const double dt = S[MM_S_TIMESTEP], W = S[MM_S_MASS_PRESS];
  const bool lb = baro_langevin(S), aniso = baro_aniso(S), volcon = S[MM_S_BARO_VOLCON] != 0.0;
  const bool has = S[MM_S_HAS_CHAINVEL0] != 0.0;
  const double fric = lb ? exp_near0((-dt) / (8.0 * S[MM_S_LB_TIMECON])) : 1.0;
  // the chain's damping factor, applied before and after the force term
  const double fchain = has ? exp_near0(((-dt) * S[MM_S_CHAINVEL0]) / 8.0) : 1.0;
  lds_f64* slot = S + MM_S_VEL_PRESS + (aniso ? q : 0);
  double vp = *slot;
  if (lb) vp *= fric;
  if (has) vp *= fchain;
  const double diag = (2.0 * S[MM_S_EKIN]) / S[MM_S_NDOF] - S[MM_S_BARO_PRESS] * S[MM_S_VOLUME];
  const double Pq = S[MM_S_SVV + q] - S[MM_S_VTENS + q];
  const double Pt = S[MM_S_SVV + qt] - S[MM_S_VTENS + qt];
  double p = 0.5 * (Pt + Pq);
  if (i == j) p = p + diag;
  double G = p / W;
  const double trace = (lane_value(G, 0) + lane_value(G, 4)) + lane_value(G, 8);
  if (!lb) {
    // MTK (npt.py:671-676): the isotropic form takes the trace, the volume constraint removes
    // it (the two together are refused at construction, utils.py:498-500)
    if (!aniso) {
      G = trace;
    } else if (volcon) {
      const double tg = trace / S[MM_S_NVEC];
      if (i == j) G -= tg;
    }
    vp += (G * dt) / 4.0;
  } else {
    lds_f64* R = S + kScratch;
    langevin_random_force(S, sys, post, sub, R);
    double r = R[i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i];
    double r00 = R[0];
    if (volcon) {
      const double dim = S[MM_S_NVEC];
      const double tg = trace / dim, tr = ((R[0] + R[2]) + R[5]) / dim;
      if (i == j) {
        G -= tg;
        r -= tr;
      }
      r00 -= tr;
    }
    if (aniso) {
      vp += ((G - r / W) * dt) / 4.0;
    } else {
      const double g = (lane_value(G, 0) + lane_value(G, 4)) + lane_value(G, 8);
      vp += ((g - r00 / W) * dt) / 4.0;
    }
    vp *= fric;
  }
  if (has) vp *= fchain;
  *slot = vp;
}

// First half of a barostat call: v_g update, then its two transforms. The positions and the domain
// are scaled by exp(v_g dt / 2) (npt.py:683-702, 434-452); the position transform is left in XMAT.
// The velocities are taken through exp(-(v_g + tr(v_g)/ndof) dt / 2) (npt.py:709-726; without
// the trace term under a volume constraint, and exp(-(1 + 3/ndof) v_g dt / 2) in the isotropic
// form, npt.py:466-484), which does not depend on the call's force: it stays pending after any
// pending velocity factor and matrix (in the second matrix slot when the previous call's matrix
// still waits). The lower half of the wave forms the first transform, the upper half the second.
__device__ __forceinline__ void baro_transforms(lds_f64* S, int sys, int post) {
#pragma clang fp contract(off)
  update_baro_vel(S, sys, post, 0);
  const bool upper = lane_id() >= 32;
  const double dt = S[MM_S_TIMESTEP];
  const bool second = S[MM_S_VMAT_ON] != 0.0;
  lds_f64* out = S + (upper ? (second ? MM_S_VMAT2 : MM_S_VMAT) : MM_S_XMAT);
  double R[9];
  if (baro_aniso(S)) {
    double A[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) A[k] = S[MM_S_VEL_PRESS + k];
    if (S[MM_S_BARO_VOLCON] == 0.0) {
      const double sh = ((A[0] + A[4]) + A[8]) / S[MM_S_NDOF];
      if (upper) {
        A[0] += sh;
        A[4] += sh;
        A[8] += sh;
      }
    }
    expm_sym_half(A, upper ? -1.0 : 1.0, dt, R);
  } else {
    const double v0 = S[MM_S_VEL_PRESS];
    const double x = upper ? -((1.0 + 3.0 / S[MM_S_NDOF]) * v0) : v0;
    const double c = exp_near0((x * dt) / 2.0);
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = (k % 4 == 0) ? c : 0.0;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) out[k] = R[k];
  S[second ? MM_S_VMAT2_ON : MM_S_VMAT_ON] = 1.0;
  const int q = entry_of(lane_id()), i = q / 3, j = q - 3 * i;
  const lds_f64* rv = S + MM_S_RVECS;
  const lds_f64* X = S + MM_S_XMAT;
  const double r =
      (rv[3 * i + 0] * X[0 + j] + rv[3 * i + 1] * X[3 + j]) + rv[3 * i + 2] * X[6 + j];
  S[MM_S_RVECS + q] = r;
  S[MM_S_VOLUME] = volume3(S + MM_S_RVECS);
}

// LangevinBarostat.pre/post bookkeeping (npt.py:374-392): energies at the start of the call.
__device__ void baro_call_begin(lds_f64* S) {
  if (baro_langevin(S)) {
    S[MM_S_BARO_EPOT0] = S[MM_S_EPOT];
    S[MM_S_BARO_EKIN0] = S[MM_S_EKIN];
  }
}

// ... and the econs correction at its end: += epot0 - epot1 + ekin0 - ekin1.
__device__ void baro_call_end(lds_f64* S) {
#pragma clang fp contract(off)
  if (baro_langevin(S))
    S[MM_S_ECONS_BARO] += ((S[MM_S_BARO_EPOT0] - S[MM_S_EPOT]) + S[MM_S_BARO_EKIN0]) - S[MM_S_EKIN];
}

// LangevinThermostat.pre/post bookkeeping (nvt.py:197-209) for the two updates of a step made
// in the node passes: econs += ekin0 - ekin1 for each.
__device__ void langevin_thermo_econs(lds_f64* S, double ekin_before_pre, const lds_f64* nd) {
#pragma clang fp contract(off)
  S[MM_S_ECONS_THERMO] += ekin_before_pre - nd[15];
  S[MM_S_ECONS_THERMO] += nd[13] - S[MM_S_EKIN];
}

__device__ void clear_vtransforms(lds_f64* S) {
  S[MM_S_VSCALE_A_ON] = 0.0;
  S[MM_S_VMAT_ON] = 0.0;
  S[MM_S_VSCALE_B_ON] = 0.0;
  // the second matrix slot is used only by steps in a row; clearing its entries as well keeps
  // the scalar block the same as after steps taken one per call
  S[MM_S_VMAT2_ON] = 0.0;
  S[MM_S_VMAT2 + entry_of(lane_id())] = 0.0;
}

__device__ void set_vscale(lds_f64* S, int slot, double f) {
  S[slot] = f;
  S[slot + 1] = 1.0;
}

// Hook econs corrections as summed by compute_properties (verlet.py:176-181, npt.py:135-148).
__device__ double econs_correction(const lds_f64* S) {
#pragma clang fp contract(off)
  const bool th = S[MM_S_THERMO] != 0.0, ba = S[MM_S_BARO] != 0.0;
  if (th && ba) {
    const double corr = S[MM_S_ECONS_THERMO] + S[MM_S_ECONS_BARO];
    if (!thermo_nhc(S) || baro_chain_on(S)) return corr;
    // particle NHC thermostat also thermostats the barostat (npt.py:139-148)
    const double kt = S[MM_S_BOLTZMANN] * S[MM_S_THERMO_TEMP];
    return corr + S[MM_S_BARO_NDOF] * kt * S[MM_S_CHAIN_POS];
  }
  if (th) return S[MM_S_ECONS_THERMO];
  if (ba) return S[MM_S_ECONS_BARO];
  return 0.0;
}

// VerletIntegrator.compute_properties (verlet.py:171-190) minus the rmsd terms. The divisions are
// made together: lanes 0..8 the pressure tensor's, lanes 9..12 those of the temperature and of
// the running means, then two lanes the pressure's and the error ratio's.
__device__ __forceinline__ void properties(lds_f64* S, bool advance) {
#pragma clang fp contract(off)
  if (advance) {
    S[MM_S_TIME] += S[MM_S_TIMESTEP];
    S[MM_S_COUNTER] += 1.0;
  }
  const int lane = lane_id(), e = entry_of(lane);
  const double ekin = S[MM_S_EKIN];
  const double etot = ekin + S[MM_S_EPOT];
  const double corr = econs_correction(S);
  const double econs = etot + corr;
  lds_f64* ce = S + MM_S_CE;  // ConsErrTracker (verlet.py:275-307)
  const double count = ce[0];
  double ekin_m = ce[1], ekin_s = ce[2], econs_m = ce[3], econs_s = ce[4];
  const double t1 = ekin - ekin_m, t2 = econs - econs_m;
  double num = S[MM_S_SVV + e] - S[MM_S_VTENS + e], den = S[MM_S_VOLUME];
  if (lane == 9) num = ekin, den = S[MM_S_NDOF];
  if (lane == 10) num = 2.0, den = S[MM_S_BOLTZMANN];
  if (lane == 11) num = t1, den = count + 1.0;
  if (lane == 12) num = t2, den = count + 1.0;
  const double r = num / den;
  if (count == 0.0) {
    ekin_m = ekin;
    econs_m = econs;
  } else {
    ekin_m += lane_value(r, 11);
    ekin_s += t1 * (ekin - ekin_m);
    econs_m += lane_value(r, 12);
    econs_s += t2 * (econs - econs_m);
  }
  const double trace = (lane_value(r, 0) + lane_value(r, 4)) + lane_value(r, 8);
  const double r2 = lane == 0 ? trace / 3.0 : econs_s / ekin_s;
  S[MM_S_TEMP] = lane_value(r, 9) * lane_value(r, 10);
  S[MM_S_ETOT] = etot;
  S[MM_S_ECONS_CORR] = corr;
  S[MM_S_ECONS] = econs;
  ce[0] = count + 1.0;
  ce[1] = ekin_m;
  ce[2] = ekin_s;
  ce[3] = econs_m;
  ce[4] = econs_s;
  S[MM_S_CONS_ERR] = count + 1.0 > 1.0 ? sqrt(lane_value(r2, 1)) : 0.0;
  if (S[MM_S_NVEC] > 0.0) {
    if (lane < 9) S[MM_S_PTENS + lane] = r;
    S[MM_S_PRESS] = lane_value(r2, 0);
  }
}

// Energy and virial from the force sums f (in LDS), plus the external-pressure part (P V, P V I).
__device__ __forceinline__ void take_force(lds_f64* S, const lds_f64* f, bool with_vtens) {
#pragma clang fp contract(off)
  const int q = entry_of(lane_id());
  const double e = f[0];
  S[MM_S_EPOT_MECH] = e;
  const double P = S[MM_S_EXT_PRESS];
  const double pv = P * S[MM_S_VOLUME];
  S[MM_S_EPOT] = P != 0.0 ? e + S[MM_S_VOLUME] * P : e;
  bool bad = e != e;
  if (with_vtens) {
    double v = f[1 + q];
    bad = bad || v != v;
    if (P != 0.0 && q % 4 == 0) v += pv;
    S[MM_S_VTENS + q] = v;
  }
  if (__any(bad)) S[MM_S_NAN] = 1.0;
}

__device__ __forceinline__ void take_nodes(lds_f64* S, const lds_f64* nd) {
  const int q = entry_of(lane_id());
  S[MM_S_EKIN] = nd[0];
  S[MM_S_SVV + q] = nd[1 + q];
  if (nd[12] != 0.0) S[MM_S_NAN] = 1.0;
}

// The node sums after the last pending barostat matrix M, from those before it: the barostat
// call changes every velocity to v M (row vectors, npt.py:709-726), so sum m (v M) (x) (v M) =
// M^T (sum m v (x) v) M and the kinetic energy is half its trace. Only the NaN flag comes from
// the node pass (the gather of the same force), when there is one.
__device__ __forceinline__ void take_nodes_after_vmat(lds_f64* S, const lds_f64* nd) {
#pragma clang fp contract(off)
  const bool second = S[MM_S_VMAT2_ON] != 0.0;
  if (second || S[MM_S_VMAT_ON] != 0.0) {
    const int q = entry_of(lane_id()), i = q / 3, j = q - 3 * i;
    const lds_f64* M = S + (second ? MM_S_VMAT2 : MM_S_VMAT);
    const lds_f64* V = S + MM_S_SVV;
    double T[3];  // column j of V M
#pragma unroll
    for (int k = 0; k < 3; ++k)
      T[k] = (V[3 * k + 0] * M[0 + j] + V[3 * k + 1] * M[3 + j]) + V[3 * k + 2] * M[6 + j];
    const double r = (M[0 + i] * T[0] + M[3 + i] * T[1]) + M[6 + i] * T[2];
    S[MM_S_SVV + q] = r;
    S[MM_S_EKIN] = 0.5 * ((lane_value(r, 0) + lane_value(r, 4)) + lane_value(r, 8));
  }
  if (nd[12] != 0.0) S[MM_S_NAN] = 1.0;
}

// This thread's share of a phase's sums, of at least kScalarThreads threads (the first of them sum):
// the force partials fpart[q * nbf + b] over the blocks b = fidx[ff + i] (or ff + i), i < fc, and
// the node partials npart[q * nbn + nf + i], i < nc, each in index order.
__device__ __forceinline__ void load_partials(const double* fpart, int nbf,
                                              const int32_t* __restrict__ fidx, int ff, int fc,
                                              const double* npart, int nbn, int nf, int nc,
                                              double (&acc)[kSliceQ]) {
#pragma unroll
  for (int q = 0; q < kSliceQ; ++q) acc[q] = 0.0;
  const bool on = threadIdx.x < kScalarThreads;
  for (int i = threadIdx.x; on && i < fc; i += kScalarThreads) {
    const int b = fidx ? fidx[ff + i] : ff + i;
#pragma unroll
    for (int q = 0; q < 10; ++q) acc[q] += fpart[(int64_t)q * nbf + b];
  }
  for (int i = threadIdx.x; on && i < nc; i += kScalarThreads) {
#pragma unroll
    for (int q = 0; q < kNodeSums; ++q) acc[10 + q] += npart[(int64_t)q * nbn + nf + i];
  }
}

// The shares summed in a fixed order (the wave by the reduce-scatter butterfly, then the waves in
// order) into tot[kSliceQ] in LDS; red: kSliceQ * kScalarThreads / 64 doubles of LDS. kNodes: with
// the node sums (zero otherwise).
template <bool kNodes>
__device__ __forceinline__ void sum_partials(const double (&acc)[kSliceQ], double* red,
                                             double* tot) {
  constexpr int kWaves = kScalarThreads / 64;
  constexpr int NV = kSliceQ, NL = kNodes ? 16 : 10;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool on = threadIdx.x < kScalarThreads;
  const int q = scatter_index(lane);
  {
    double lo[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) lo[k] = acc[k];
    const double t = wave_reduce_scatter<NL>(lo, lane);
    if (on && (lane & 3) == 0 && q < NL) red[wave * NV + q] = t;
  }
  if (kNodes) {
    double hi[NV - 16];
#pragma unroll
    for (int k = 16; k < NV; ++k) hi[k - 16] = acc[k];
    const double t = wave_reduce_scatter<NV - 16>(hi, lane);
    if (on && (lane & 3) == 0 && q < NV - 16) red[wave * NV + 16 + q] = t;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double t = 0.0;
    if (kNodes || threadIdx.x < 10) {
      t = red[threadIdx.x];
      for (int w = 1; w < kWaves; ++w) t += red[w * NV + threadIdx.x];
    }
    tot[threadIdx.x] = t;
  }
  __syncthreads();
}

__device__ __forceinline__ constexpr bool phase_uses_force(int phase) {
  return phase == kPhInitForce || phase == kPhNveEnd || phase == kPhNvtEnd ||
         phase == kPhBaroEndPre || phase == kPhMainEndNpt || phase == kPhBaroEndPost ||
         phase == kPhBaroEndPostPre || phase >= kPhNvtEndPre;
}
__device__ __forceinline__ constexpr bool phase_uses_nodes(int phase) {
  return phase == kPhInitProps || phase == kPhNveEnd || phase == kPhNvtEnd ||
         phase == kPhMainEndNpt || phase == kPhBaroEndPost || phase >= kPhNvtEndPre ||
         phase == kPhRmsd;
}

// The scalar update of one phase on the scalar block S of system sys. chained: the phase closes
// a step that another step of the same call follows (kPhBaroEndPost: its velocity transforms
// stay pending for the next kick-drift pass).
__device__ void run_phase(int phase, lds_f64* S, const lds_f64* f,
                          const lds_f64* nd, int with_vtens, int sys,
                          bool chained = false) {
  const bool nhc = thermo_nhc(S);
  const bool lt = S[MM_S_THERMO] == (double)MM_THERMO_LANGEVIN;
  // the barostat's pressure contribution enters the chain only for MTK (npt.py:109-113)
  const bool g1_on = S[MM_S_BARO] == (double)MM_BARO_MTK;
  switch (phase) {
    case kPhInitForce:
      take_force(S, f, with_vtens != 0);
      break;
    case kPhInitProps:
      take_nodes(S, nd);
      properties(S, false);
      break;
    case kPhNveEnd:
      clear_vtransforms(S);
      take_force(S, f, true);
      take_nodes(S, nd);
      properties(S, true);
      break;
    case kPhNvtPre: {
      const ChainStep step = nhc_chain(S, S[MM_S_EKIN], false, 0.0, kThermoChain);
      const double fac = step.factor;
      S[MM_S_EKIN] = step.ekin;
      set_vscale(S, MM_S_VSCALE_B, fac);
      break;
    }
    case kPhNvtEnd: {
      clear_vtransforms(S);
      take_force(S, f, true);
      if (lt) {
        const double ekin0 = S[MM_S_EKIN];
        take_nodes(S, nd);
        langevin_thermo_econs(S, ekin0, nd);
        properties(S, true);
        break;
      }
      take_nodes(S, nd);
      const ChainStep step = nhc_chain(S, S[MM_S_EKIN], false, 0.0, kThermoChain);
      const double fac = step.factor;
      set_vscale(S, MM_S_VSCALE_A, fac);
      S[MM_S_SVV + entry_of(lane_id())] *= fac * fac;
      S[MM_S_EKIN] = step.ekin;
      S[MM_S_ECONS_THERMO] = nhc_econs(S);
      properties(S, true);
      break;
    }
    case kPhLtFirst:
    case kPhLtNext:
    case kPhLtLast: {
      clear_vtransforms(S);
      take_force(S, f, true);
      const double ekin0 = S[MM_S_EKIN];
      take_nodes(S, nd);
      if (phase == kPhLtFirst) S[MM_S_ECONS_THERMO] += ekin0 - nd[15];
      S[MM_S_ECONS_THERMO] += nd[13] - S[MM_S_EKIN];
      properties(S, true);
      if (phase != kPhLtLast) S[MM_S_ECONS_THERMO] += S[MM_S_EKIN] - nd[14];
      break;
    }
    case kPhBaroPre:
      // TBC.pre: chainvel0 = chain.vel[0] before the barostat (npt.py:101-107); the
      // barostat's own chain overrules it (npt.py:616-619)
      S[MM_S_HAS_CHAINVEL0] = nhc ? 1.0 : 0.0;
      S[MM_S_CHAINVEL0] = nhc ? S[MM_S_CHAIN_VEL] : 0.0;
      if (baro_chain_on(S)) {
        S[MM_S_HAS_CHAINVEL0] = 1.0;
        S[MM_S_CHAINVEL0] = S[MM_S_BCHAIN_VEL];
      }
      // (a pending thermostat factor is already in m v (x) v: the phases that set one scale
      // the sums by its square)
      baro_call_begin(S);
      // the velocity transform stays pending for the kick-drift pass, which applies it before
      // the chain's factor
      baro_transforms(S, sys, 0);
      break;
    case kPhBaroEndPre: {
      // the barostat's velocity transform is still pending (see kPhBaroPre): the node sums
      // after it follow from those before it. The gather of this force comes after the phase
      // (it is the kick-drift pass), so a NaN gradient shows here through the virial.
      take_force(S, f, true);
      take_nodes_after_vmat(S, nd);
      update_baro_vel(S, sys, 0, 1);
      baro_call_end(S);
      if (baro_chain_on(S)) baro_chain_step(S);
      // a Langevin thermostat's pre update follows in the kick-drift pass
      if (nhc) {
        const double g1 = g1_on ? add_press_cont(S) : 0.0;
        const ChainStep step = nhc_chain(S, S[MM_S_EKIN], g1_on, g1, kThermoChain);
        const double fac = step.factor;
        S[MM_S_EKIN] = step.ekin;
        set_vscale(S, MM_S_VSCALE_B, fac);
      }
      break;
    }
    case kPhMainEndNpt: {
      // gather_drift has stored the positions through a pending earlier position transform; its
      // slot is cleared, entries included, as after steps taken one per call
      S[MM_S_XMAT2_ON] = 0.0;
      S[MM_S_XMAT2 + entry_of(lane_id())] = 0.0;
      clear_vtransforms(S);
      take_force(S, f, true);
      const double ekin0 = S[MM_S_EKIN];
      take_nodes(S, nd);
      if (nhc) {
        const double g1 = g1_on ? add_press_cont(S) : 0.0;
        const ChainStep step = nhc_chain(S, S[MM_S_EKIN], g1_on, g1, kThermoChain);
        const double fac = step.factor;
        S[MM_S_EKIN] = step.ekin;
        set_vscale(S, MM_S_VSCALE_A, fac);
        S[MM_S_SVV + entry_of(lane_id())] *= fac * fac;
        S[MM_S_ECONS_THERMO] = nhc_econs(S);
      } else if (lt) {
        langevin_thermo_econs(S, ekin0, nd);
      }
      // TBC.post: chainvel0 after the thermostat (npt.py:128-133); the barostat's own chain
      // steps first and overrules it (npt.py:631-639)
      S[MM_S_HAS_CHAINVEL0] = nhc ? 1.0 : 0.0;
      S[MM_S_CHAINVEL0] = nhc ? S[MM_S_CHAIN_VEL] : 0.0;
      if (baro_chain_on(S)) {
        baro_chain_step(S);
        S[MM_S_HAS_CHAINVEL0] = 1.0;
        S[MM_S_CHAINVEL0] = S[MM_S_BCHAIN_VEL];
      }
      baro_call_begin(S);
      baro_transforms(S, sys, 1);
      break;
    }
    case kPhBaroEndPost:
      // the node sums after the call's velocity transform follow from those before it (as in
      // kPhBaroEndPre), whether the gather applied it (a call's last step) or it stays
      // pending (chained)
      take_force(S, f, true);
      take_nodes_after_vmat(S, nd);
      if (!chained) clear_vtransforms(S);
      // chained, the positions still wait for this call's transform (its force evaluation
      // applied it on the fly): it moves to the earlier slot, before the next call's
      if (chained) {
        const int q = entry_of(lane_id());
        S[MM_S_XMAT2 + q] = S[MM_S_XMAT + q];
        S[MM_S_XMAT2_ON] = 1.0;
      }
      update_baro_vel(S, sys, 1, 1);
      if (baro_langevin(S)) {
        baro_call_end(S);
      } else {
        // MTKBarostat.post (npt.py:640-651)
        double e = baro_ekin(S);
        if (S[MM_S_BARO_VOLCON] == 0.0) e += S[MM_S_BARO_PRESS] * S[MM_S_VOLUME];
        if (baro_chain_on(S)) e += nhc_econs(S, kBaroChain);
        S[MM_S_ECONS_BARO] = e;
      }
      properties(S, true);
      break;
    case kPhRmsd: {
      const double denom = 3.0 * S[MM_S_NNODES];
      S[MM_S_RMSD_GPOS] = sqrt(nd[10] / denom);
      S[MM_S_RMSD_DELTA] = sqrt(nd[11] / denom);
      break;
    }
    case kPhApplied:
      clear_vtransforms(S);
      break;
  }
}

// One phase, or the end of one step and the start of the next on the same copy of the block; tot
// holds the force and node sums.
__device__ __forceinline__ void run_phases(int phase, lds_f64* S, const lds_f64* tot,
                                           int with_vtens, int sys) {
  const lds_f64 *f = tot, *nd = tot + 10;
  const bool chained = phase == kPhBaroEndPostPre;
  const int next = chained ? kPhBaroPre : phase == kPhNvtEndPre ? kPhNvtPre : -1;
  int now = chained ? kPhBaroEndPost : phase == kPhNvtEndPre ? kPhNvtEnd : phase;
  for (;;) {
    run_phase(now, S, f, nd, with_vtens, sys, chained);
    if (now == next || next < 0) break;
    now = next;
  }
}

// Grid (slices, systems). Block (g, sys) reduces slice g of that system's force and node
// partials; the last block of the system to finish (counted with an atomic counter, which it
// resets) sums the slices in slice order and runs the phase on a copy of the system's scalar
// block in LDS, written back at the end.
__global__ void __launch_bounds__(kScalarThreads)
scalar_kernel(int phase, double* __restrict__ S0, const double* __restrict__ fpart, int nbf,
              const int32_t* __restrict__ fsys_ptr, const int32_t* __restrict__ fsys_idx,
              const double* __restrict__ npart, int nbn, const int32_t* __restrict__ nsys_ptr,
              int with_vtens, double* __restrict__ slices, unsigned int* __restrict__ counters) {
  static_assert(MM_S_COUNT <= kScalarThreads, "one scalar-block entry per thread");
  __shared__ double Sl[MM_S_COUNT + 6];
  __shared__ double tot[kSliceQ];
  __shared__ int is_last;
  const int sys = blockIdx.y;
  const int G = gridDim.x, gi = blockIdx.x;
  double* Sg = S0 + (int64_t)sys * MM_S_COUNT;
  // the scalar block is loaded up front, so that its latency hides behind the reduction
  const double s_own = threadIdx.x < MM_S_COUNT ? Sg[threadIdx.x] : 0.0;
  {
    int ff = 0, fc = 0, nf = 0, nc = 0;
    if (phase_uses_force(phase)) {
      const int b0 = fsys_ptr[sys], cnt = fsys_ptr[sys + 1] - b0;
      ff = b0 + (int)((int64_t)cnt * gi / G);
      fc = b0 + (int)((int64_t)cnt * (gi + 1) / G) - ff;
    }
    if (phase_uses_nodes(phase)) {
      const int b0 = nsys_ptr[sys], cnt = nsys_ptr[sys + 1] - b0;
      nf = b0 + (int)((int64_t)cnt * gi / G);
      nc = b0 + (int)((int64_t)cnt * (gi + 1) / G) - nf;
    }
    __shared__ double red[kSliceQ * (kScalarThreads / 64)];
    double acc[kSliceQ];
    load_partials(fpart, nbf, fsys_idx, ff, fc, npart, nbn, nf, nc, acc);
    sum_partials<true>(acc, red, tot);
  }
  if (G > 1) {
    if (threadIdx.x == 0) {
      double* sl = slices + ((int64_t)sys * G + gi) * kSliceQ;
      for (int q = 0; q < kSliceQ; ++q) sl[q] = tot[q];
      __threadfence();
      const unsigned int prev = atomicAdd(&counters[sys], 1u);
      is_last = prev == (unsigned int)(G - 1);
    }
    __syncthreads();
    if (!is_last) return;
    __threadfence();
    // all slices into LDS in one parallel pass, then each total summed in slice order
    __shared__ double sl_sh[kScalarSlices * kSliceQ];
    const double* sl = slices + (int64_t)sys * G * kSliceQ;
    for (int i = threadIdx.x; i < G * kSliceQ; i += kScalarThreads) sl_sh[i] = sl[i];
    __syncthreads();
    if (threadIdx.x < kSliceQ) {
      double t = 0.0;
      for (int k = 0; k < G; ++k) t += sl_sh[k * kSliceQ + threadIdx.x];
      tot[threadIdx.x] = t;
    }
    if (threadIdx.x == 0) counters[sys] = 0u;
  }
  if (threadIdx.x < MM_S_COUNT) Sl[threadIdx.x] = s_own;
  __syncthreads();
  if (threadIdx.x < 64) {
    run_phases(phase, (lds_f64*)Sl, (const lds_f64*)tot, with_vtens, sys);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < MM_S_COUNT; q += kScalarThreads) Sg[q] = Sl[q];
}

// ----------------------------------------------------------------------------- merged phases
//
// On a mid-sized system a step of three to eight kernels is bound by their number: each waits for
// the one before it to drain, starts (2.3 us from kernel to kernel) and then for its first loads.
// In a row of steps the scalar phases are therefore no kernels of their own. The kernel after a
// phase begins with it: every block sums the partials and runs the phase on a copy of the scalar
// block in LDS, all alike, so that nothing has to be handed from block to block, and block 0
// stores the result to the other of two copies in memory (the rest of the grid still reads the
// first); the block's own loads are under way meanwhile. Where a phase gates nothing (NVE, the
// Langevin thermostat) one extra block of the next cell pass runs it beside the others. A cell
// pass that reads the sums of the pass before stores its own to a second buffer; a gather copies
// back what the next kernels expect in the first (Carry). The arithmetic and the order of all sums
// are those of the separate kernels: the same bits. Kernels of a step: NVE and Langevin 3 -> 2,
// NVT 4 -> 3, NPT 8 -> 5. Step at 10^3 / 32^3 / 48^3 cells: NVE 23.6 / 25.8 / 36.0 -> 19.0 / 21.0 /
// 28.1 us, Langevin 27.5 / 29.6 / 41.7 -> 22.6 / 24.6 / 33.7, NVT 31.2 / 33.6 / 45.4 -> 25.9 / 29.0
// / 42.3, NPT 64.1 / 68.5 / 90.4 -> 54.8 / 59.1 / 79.5. (A cell pass that moved the nodes as it
// read them, for an NVT step of two kernels, took three loads a corner value instead of one: 26.6 /
// 31.9 / 50.6 us.) With more than kMergeMaxBlocks blocks the cells run as two launches side by
// side and a block's share of the repeated sums grows with the system; there a phase is a kernel.

// What a gather copies for the kernels after it: the scalar block and the cell passes' sums.
struct Carry {
  double* s = nullptr;  // destination of the scalar block (null: stays)
  const double* f_src = nullptr;
  double* f_dst = nullptr;
  int f_count = 0;
};
__device__ __forceinline__ void carry(const Carry& c, const double* S, int blk, int blocks) {
  if (c.s && blk == 0 && threadIdx.x < MM_S_COUNT) c.s[threadIdx.x] = S[threadIdx.x];
  for (int i = blk * kNodeBlock + threadIdx.x; i < c.f_count; i += blocks * kNodeBlock)
    c.f_dst[i] = c.f_src[i];
}

// The partials and the copies of the scalar block of a merged phase.
struct PhaseArgs {
  const double* s_in = nullptr;
  double* s_out = nullptr;
  const double* fpart = nullptr;
  const double* npart = nullptr;
  int nbf = 0, nbn = 0;
};

// Phase kPhase on Sl (LDS, MM_S_COUNT + 6 doubles; s_own is the thread's entry of the block as it
// came from memory), from the threads' shares acc of the partials. Every thread calls this.
template <int kPhase>
__device__ __forceinline__ void merged_phase(double s_own, const double (&acc)[kSliceQ],
                                             double* Sl) {
  __shared__ double red[kSliceQ * (kScalarThreads / 64)];
  __shared__ double tot[kSliceQ];
  if (threadIdx.x < MM_S_COUNT) Sl[threadIdx.x] = s_own;
  sum_partials<phase_uses_nodes(kPhase)>(acc, red, tot);
  if (threadIdx.x < 64) run_phases(kPhase, (lds_f64*)Sl, (const lds_f64*)tot, 1, 0);
  __syncthreads();
}
template <int kPhase>
__device__ __forceinline__ void load_merged(const PhaseArgs& a, double (&acc)[kSliceQ]) {
  load_partials(a.fpart, a.nbf, nullptr, 0, phase_uses_force(kPhase) ? a.nbf : 0, a.npart, a.nbn, 0,
                phase_uses_nodes(kPhase) ? a.nbn : 0, acc);
}

// Half kick and drift from a stored gradient, one node a thread: latency bounds it on a small
// system, above all with the Langevin noise (some 300 dependent instructions a node), so the
// nodes are spread over as many waves as there are. 40x36x47 Langevin step 52 -> 46 us against
// four nodes a lane; without noise and on large systems the two are equal (128^3 and the batch of
// 192 replicas within 0.5%).
// kPhase >= 0: the kernel begins with that scalar phase (merged_phase), on the loads' time.
template <bool kLT, int kPhase = -1>
__global__ void __launch_bounds__(kNodeBlock, kPhase >= 0 ? 2 : 1)
kick_drift_kernel(double* __restrict__ x, double* __restrict__ v, const double* __restrict__ g,
                  const double* __restrict__ m, const double* __restrict__ S0,
                  const int32_t* __restrict__ blk_sys, int64_t N, double* __restrict__ partials,
                  PhaseArgs ph) {
  __shared__ double Sl[kPhase >= 0 ? MM_S_COUNT + 6 : 1];
  const double* S =
      kPhase >= 0 ? Sl : S0 + (blk_sys ? (int64_t)blk_sys[blockIdx.x] * MM_S_COUNT : 0);
  double s_own = 0.0, share[kSliceQ];
  if constexpr (kPhase >= 0) {
    if (threadIdx.x < MM_S_COUNT) s_own = ph.s_in[threadIdx.x];
    load_merged<kPhase>(ph, share);
  }
  const int64_t n = (int64_t)blockIdx.x * kNodeBlock + threadIdx.x;
  double lt[1] = {0.0};
  double mass = 1.0, vv[3], gg[3], xx[3];
  if (n < N) {
    mass = m[n];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      vv[j] = v[3 * n + j];
      gg[j] = g[3 * n + j];
      xx[j] = x[3 * n + j];
    }
  }
  if constexpr (kPhase >= 0) {
    merged_phase<kPhase>(s_own, share, Sl);
    if (blockIdx.x == 0 && threadIdx.x < MM_S_COUNT) ph.s_out[threadIdx.x] = Sl[threadIdx.x];
  }
  if (n < N) {
    kick_drift_node<kLT>(S, n, mass, gg, vv, xx, lt[0]);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      v[3 * n + j] = vv[j];
      x[3 * n + j] = xx[j];
    }
  }
  if (kLT) block_sum_store_wide<1>(lt, partials + (int64_t)15 * gridDim.x, blockIdx.x);
}

// gpos[n] = sum of the node's face-class records (mmff.py:303-318; the cell pass has already
// added the faces shared along z), fused with the second half kick
// v += a dt / 2 (verlet.py:152-153) and the node sums of the new velocities; with kLT also
// the Langevin thermostat's post update (the node sums then hold the ekin before it in [13]).
// With kScaleV instead (a barostat call, npt.py:704-735), the pending velocity transforms are
// applied (the barostat's exp(-(v_g + tr(v_g)/ndof) dt / 2), known before its force) in the
// same pass; the phase after it takes the kinetic sums from those before the matrix, so this
// pass leaves only the NaN flag of the gradient.
// gmode: kGatherStore sums the records and stores gpos; kGatherKeep sums them for the kick only
// (the step overwrites gpos before anything reads it); kGatherNone (kScaleV only) reads no
// records: the force evaluation fed only the energy and the virial.
// With kDrift instead, the first half kick and the drift of the step (verlet.py:141-146) with
// the barostat's pre-call gradient, which nothing else reads: the pending velocity transforms
// (and the Langevin thermostat's pre update, its ekin after the update in partial row 15),
// then v += a dt / 2 and x += dt v, as kick_drift_kernel does from a stored gpos, with
// x first taken through the barostat call's pending position scaling (the previous post
// call's when it still waits, then the pre call's), which its cell pass applied on the fly.
// With kKick and kDrift, the second half kick of a step and the first half kick and drift of the next
// (with kLT the thermostat's pre update too, its ekin in partial row 14), for a step in a row of
// steps whose scalar phase moves neither: the node sums are those in between. The kick-drift pass
// with its launch and its trip to memory for x, v and g falls away: NVE / Langevin step 28.5 / 30.8
// -> 23.5 / 27.5 us at 10^3 cells, 42.8 / 48.3 -> 35.8 / 41.2 us at 48^3, 274 / 306 -> 237 / 289 us
// at 128^3.
// One node per thread (the gathers need every wave in flight that they can get); the node
// blocks are dealt to the XCDs in contiguous ranges (xcd_block), and the partial sums are
// stored per logical block.
// kPhase >= 0: the kernel begins with that scalar phase (merged_phase), after the loads that do not
// depend on it.
template <bool kKick, bool kLT, bool kScaleV, bool kDrift, bool kAllLoads, int kPhase = -1>
__global__ void __launch_bounds__(kNodeBlock, kPhase >= 0 ? 2 : 1)
gather_kick_kernel(const int32_t* __restrict__ ncell, const double* __restrict__ gcell,
                   int64_t N, int64_t RS, double* __restrict__ gpos, double* __restrict__ v,
                   const double* __restrict__ m, const double* __restrict__ S0,
                   const int32_t* __restrict__ blk_sys, double* __restrict__ partials,
                   int gmode, double* __restrict__ x, Carry c, PhaseArgs ph) {
  const int blk = xcd_block((int)blockIdx.x, (int)gridDim.x);
  __shared__ double Sl[kPhase >= 0 ? MM_S_COUNT + 6 : 1];
  const double* S = kPhase >= 0 ? Sl : S0 + (blk_sys ? (int64_t)blk_sys[blk] * MM_S_COUNT : 0);
  double s_own = 0.0, share[kSliceQ];
  if constexpr (kPhase >= 0) {
    if (threadIdx.x < MM_S_COUNT) s_own = ph.s_in[threadIdx.x];
    load_merged<kPhase>(ph, share);
  } else {
    carry(c, S, blk, (int)gridDim.x);
  }
  constexpr int NA = kLT ? (kKick && kDrift ? 15 : 14) : 13;
  double acc[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) acc[q] = 0.0;
  const int64_t n = (int64_t)blk * kNodeBlock + threadIdx.x;
  const bool own = n < N;
  // the node's own values: with kAllLoads loaded before the records, so that they arrive with them
  double mass = 1.0, v0[3] = {0.0, 0.0, 0.0}, x0[3] = {0.0, 0.0, 0.0}, g[3] = {0.0, 0.0, 0.0};
  auto load_node = [&]() {
    if (kKick || kDrift) mass = m[n];
    if (kKick || kDrift || kScaleV) {
#pragma unroll
      for (int j = 0; j < 3; ++j) v0[j] = v[3 * n + j];
    }
    if (kDrift) {
#pragma unroll
      for (int j = 0; j < 3; ++j) x0[j] = x[3 * n + j];
    }
  };
  if (own) {
    if (kAllLoads) load_node();
    if (gmode != kGatherNone) {
      sum_node_records<kAllLoads>(ncell, gcell, N, RS, n, g);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if (gmode == kGatherStore) gpos[3 * n + j] = g[j];
        if (g[j] != g[j]) acc[12] = 1.0;
      }
    }
    if (!kAllLoads) load_node();
  }
  if constexpr (kPhase >= 0) {
    merged_phase<kPhase>(s_own, share, Sl);
    if (blk == 0 && threadIdx.x < MM_S_COUNT) ph.s_out[threadIdx.x] = Sl[threadIdx.x];
  }
  if (own) {
    if (kKick) {
      double lt = 0.0;
      kick_node<kLT>(S, n, mass, g, v0, acc, lt);
      if (kLT) acc[13] += lt;
      if (kDrift) {
        lt = 0.0;
        half_step_node<kLT>(S, n, 2, mass, g, v0, x0, lt);
        if (kLT) acc[NA - 1] += lt;
#pragma unroll
        for (int j = 0; j < 3; ++j) x[3 * n + j] = x0[j];
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) v[3 * n + j] = v0[j];
    }
    if (kScaleV) {
      apply_vtransform(S, v0);
#pragma unroll
      for (int j = 0; j < 3; ++j) v[3 * n + j] = v0[j];
    }
    if (kDrift && !kKick) {
      // the positions as the cell pass read them: the pending scaling(s) of the barostat call
      scale_position(S, x0);
      kick_drift_node<kLT>(S, n, mass, g, v0, x0, acc[0]);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        v[3 * n + j] = v0[j];
        x[3 * n + j] = x0[j];
      }
    }
  }
  if (kDrift && !kKick) {
    if (kLT) {
      double lt[1] = {acc[0]};
      block_sum_store_wide<1>(lt, partials + (int64_t)15 * gridDim.x, blk);
    }
  } else if (kKick) {
    block_sum_store_wide<NA>(acc, partials, blk);
  } else {
    // only the NaN flag: any lane's flag, per block
    const unsigned long long bad = __ballot(acc[12] != 0.0);
    __shared__ int any_bad;
    if (threadIdx.x == 0) any_bad = 0;
    __syncthreads();
    if ((threadIdx.x & 63) == 0 && bad) any_bad = 1;
    __syncthreads();
    if (threadIdx.x < 13)
      partials[(int64_t)threadIdx.x * gridDim.x + blk] =
          (threadIdx.x == 12 && any_bad) ? 1.0 : 0.0;
  }
}

// The cells of one system as the step's own cell passes read them.
struct CellPass {
  const int32_t *cnode, *cwrap, *blk_row, *nstates, *cbase;
  const double *tab, *kt;
  int32_t max_states;
  int64_t W, S;
  double* gcell;
};

// The cell pass of a row of steps, both kinds of block in one launch (as cell_kernel_both), with
// the scalar phase before it. kPhBaroEndPostPre and kPhMainEndNpt gate the pass and open every
// block; the positions are then taken through the pending transforms. The other phases run in
// block 0,
// beside the cells of the blocks behind it, and store all of the scalar block but the domain
// vectors, which they leave alone and the others read.
constexpr bool phase_gates(int phase) {
  return phase == kPhBaroEndPostPre || phase == kPhMainEndNpt;
}
template <int kModel, int kOut, int kPhase>
__global__ void __launch_bounds__(kCellBlock, 2)
md_cells_kernel(CellPass c, const double* __restrict__ x, PhaseArgs ph,
                double* __restrict__ partials) {
  using F = Frame<kModel>;
  constexpr int NS = F::NE + 3 * F::NC;
  constexpr bool kGates = phase_gates(kPhase), kPost = kPhase == kPhBaroEndPostPre;
  __shared__ double st_sh[NS * kCellBlock];
  __shared__ double cred[7 * (kCellBlock / 64)];
  __shared__ double Sl[MM_S_COUNT + 6];
  const int t = threadIdx.x;
  double s_own = 0.0, share[kSliceQ];
  if (kGates || blockIdx.x == 0) {
    if (t < MM_S_COUNT) s_own = ph.s_in[t];
    load_merged<kPhase>(ph, share);
  }
  if (!kGates && blockIdx.x == 0) {
    merged_phase<kPhase>(s_own, share, Sl);
    if (t < MM_S_COUNT && (t < MM_S_RVECS || t >= MM_S_RVECS + 9)) ph.s_out[t] = Sl[t];
    return;
  }
  const int extra = kGates ? 0 : 1, nblocks = (int)gridDim.x - extra;
  const int bid = xcd_block((int)blockIdx.x - extra, nblocks);
  const int64_t w = (int64_t)bid * kCellBlock + t;
  int n[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) n[k] = c.cnode[w * 8 + k];
  const bool valid = n[0] >= 0;
  const int wrap = valid ? c.cwrap[w] : 0;
  if constexpr (kGates) {
    // one word of every corner's position: the lines are in the cache by the time they are needed
    uint32_t word[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      word[k] = reinterpret_cast<const uint32_t*>(x + 3 * (int64_t)(valid ? n[k] : 0))[0];
    merged_phase<kPhase>(s_own, share, Sl);
    if (bid == 0 && t < MM_S_COUNT) ph.s_out[t] = Sl[t];
#pragma unroll
    for (int k = 0; k < 8; ++k) asm volatile("" ::"v"(word[k]));
  }
  const int trow = ((const_i32)c.blk_row)[bid];
  const int ns = ((const_i32)c.nstates)[trow];
  const double kt = ((const_f64)c.kt)[trow];
  const const_f64 tab = (const_f64)c.tab + (int64_t)trow * c.max_states * kTabStride;
  double rv[9];
#pragma unroll
  for (int q = 0; q < 9; ++q)
    rv[q] = kGates ? lane_value(Sl[MM_S_RVECS + q], 0) : ((const_f64)ph.s_in)[MM_S_RVECS + q];
  auto corners = [&](double (&p)[8][3]) {
    load_corners(x, n, p, kGates, Sl + MM_S_XMAT, kPost && Sl[MM_S_XMAT2_ON] != 0.0,
                 Sl + MM_S_XMAT2);
  };
  double ecell, vir[6], gacc[8][3];
  if (ns > 1)
    cell_eval<kModel, kOut, true, kCellBlock>(tab, ns, kt, valid, corners, wrap, rv, st_sh + t,
                                              ecell, vir, gacc);
  else
    cell_eval<kModel, kOut, false, kCellBlock>(tab, ns, kt, valid, corners, wrap, rv, st_sh + t,
                                               ecell, vir, gacc);
  if (kOut == kOutGradient) store_cell(w, wrap, valid, c.cbase, c.W, c.S, c.gcell, gacc);
  cell_wave_totals(ecell, vir, cred + 7 * (t >> 6));
  __syncthreads();
  if (t < 10) partials[(int64_t)t * nblocks + bid] = cell_block_total(cred, t);
}

// ----------------------------------------------------------------------------- small systems

// The steps of a call in one launch by one workgroup, for a system of at most kSmall work slots
// and nodes. Such a system leaves the chip idle whatever the launches are: its step is bound by
// the four to eight launches, the gaps between them (2.3 us each) and the trips to memory that
// hand over the results. Thread t owns cell slot t and node t: the node's velocity, gradient and
// mass stay in its registers, positions, vertex-gradient records, wave sums and the scalar block
// in LDS (a slot's column holds its multistate sums, then its records: lower faces in rows 0..11,
// upper in 12..23). Arithmetic, blocks and the order of all sums are those of the step's kernels:
// the same bits. What is left is one wave's instruction stream a SIMD: cells 15k cycles (corner8
// with a two-state type) or 7k (original), node passes 4k to 6k, scalar phases 2k (NVE) to 22k
// (NPT). Per step, launches -> this kernel, corner8 / original model: 3^3 NVE 24.4 -> 10.0 /
// 23.1 -> 5.8 us, 3^3 NVT 27.2 -> 12.0 / 23.6 -> 8.2 us, 3^3 NPT 54.6 -> 34.8 / 48.8 -> 23.6 us;
// 7^3 (two types, at the limit) NVE 27.2 -> 10.6 / 24.7 -> 6.9 us, NPT 62.3 -> 35.7 / 53.2 -> 24.9
// us. The limit is what LDS holds: 36 columns of 512 sums are 144 of its 160 KB.
constexpr int kSmall = 512;

struct SmallArgs {
  const int32_t *cnode, *cwrap, *blk_row, *nstates, *nrec, *cbase;
  const double *tab, *kt;
  int32_t max_states;
  int W, N;
  double *pos, *vel, *gpos;
  const double* masses;
  double* S;
  int thermo, baro, nsteps;
};

enum SmallGather { kSmallNone = 0, kSmallKick, kSmallDrift, kSmallScale };

template <int kModel, bool kLT>
__global__ void __launch_bounds__(kSmall, 2) small_kernel(SmallArgs a) {
  using F = Frame<kModel>;
  constexpr int NS = F::NE + 3 * F::NC;
  constexpr int NR = NS > 24 ? NS : 24;
  constexpr int NA = kLT ? 14 : 13;
  constexpr int kWaves = kSmall / 64;
  __shared__ double col[NR * kSmall];
  __shared__ double xs[3 * kSmall];
  __shared__ double Sl[MM_S_COUNT + 6];
  // sums of every wave, zero where nothing writes: energy and virial, node sums, thermostat ekin
  __shared__ double red[24 * kWaves];
  __shared__ double tot[kSliceQ];
  double *cred = red, *nred = red + 7 * kWaves, *lred = red + 23 * kWaves;
  unsigned short* top_slot = reinterpret_cast<unsigned short*>(col);  // before the first step only
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  if (t < MM_S_COUNT) Sl[t] = a.S[t];
  if (t < 24 * kWaves) red[t] = 0.0;
  // the slot
  const bool has_slot = 64 * wave < a.W;  // W is a multiple of the block size
  uint32_t nodes[4];  // its nodes, two to a word
  const bool valid = has_slot && a.cnode[8 * t] >= 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    nodes[k] = valid ? (uint32_t)a.cnode[8 * t + 2 * k] | (uint32_t)a.cnode[8 * t + 2 * k + 1] << 16
                     : 0u;
  const int wrap = valid ? a.cwrap[t] : 0;
  const int trow = has_slot ? ((const_i32)a.blk_row)[wave >> 2] : 0;
  const int ns = ((const_i32)a.nstates)[trow];
  const double kt = ((const_f64)a.kt)[trow];
  const_f64 tab = (const_f64)a.tab + (int64_t)trow * a.max_states * kTabStride;
  {
    const bool open_top = valid && !(wrap & 16);
    const uint64_t tops = __ballot(open_top);
    if (open_top)
      top_slot[((const_i32)a.cbase)[wave] + __popcll(tops & ((1ull << lane) - 1ull))] = t;
  }
  __syncthreads();
  // the node: its records as places in col, two to a word, 0xffff for none
  const bool own = t < a.N;
  uint32_t places[4] = {};
  double mass = 1.0, v[3] = {0.0, 0.0, 0.0}, g[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int e = own ? a.nrec[k * a.N + t] : -1;
    const int slot = e >> 2, row = 3 * (e & 3);
    const int place = e < 0 ? 0xffff
                      : slot < a.W ? row * kSmall + slot
                                   : (12 + row) * kSmall + top_slot[slot - a.W];
    places[k / 2] |= (uint32_t)place << (16 * (k & 1));
  }
  if (own) {
    mass = a.masses[t];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      v[j] = a.vel[3 * t + j];
      g[j] = a.gpos[3 * t + j];
      xs[3 * t + j] = a.pos[3 * t + j];
    }
  }
  __syncthreads();

  const bool opens = a.baro != 0 || a.thermo == MM_THERMO_NHC;
  int step = 0, seg = opens ? -1 : 0;
  while (step < a.nsteps) {
    const bool last = step + 1 == a.nsteps;
    // the parts of this segment, in order: a node pass (half kick and drift, or the position
    // scaling), a cell pass, a scalar phase, a gather, a scalar phase
    bool cells = true, records = true, drift0 = false, scale0 = false, on = false, on2 = false;
    int gather = kSmallKick, phase0 = -1, phase1 = -1;
    if (seg < 0) {
      cells = false;
      gather = kSmallNone;
      phase0 = a.baro ? kPhBaroPre : kPhNvtPre;
    } else if (!a.baro) {
      drift0 = true;
      phase1 = a.thermo == MM_THERMO_NONE ? kPhNveEnd
               : a.thermo == MM_THERMO_NHC && !last ? kPhNvtEndPre : kPhNvtEnd;
    } else if (seg == 0) {
      on = true;
      on2 = Sl[MM_S_XMAT2_ON] != 0.0;
      phase0 = kPhBaroEndPre;
      gather = kSmallDrift;
    } else if (seg == 1) {
      phase1 = kPhMainEndNpt;
    } else if (!last) {
      on = true;
      records = false;
      gather = kSmallNone;
      phase0 = kPhBaroEndPostPre;
    } else {
      scale0 = true;
      gather = kSmallScale;
      phase1 = kPhBaroEndPost;
    }

    if (drift0 || scale0) {
      double lt[1] = {0.0};
      if (own) {
        double x[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) x[j] = xs[3 * t + j];
        if (drift0)
          kick_drift_node<kLT>(Sl, t, mass, g, v, x, lt[0]);
        else
          scale_position(Sl, x);
#pragma unroll
        for (int j = 0; j < 3; ++j) xs[3 * t + j] = x[j];
      }
      if (kLT && drift0) {
        const double s = wave_reduce_scatter<1>(lt, lane);
        if (lane == 0) lred[wave] = s;
      }
      __syncthreads();
    }

    if (cells) {
      if (has_slot) {
        double rv[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) rv[q] = lane_value(Sl[MM_S_RVECS + q], 0);
        // the table and the packed words are taken anew in every step: hoisted out of the loop
        // they would not fit the registers
        asm volatile("" : "+s"(tab));
        int n[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          asm volatile("" : "+v"(nodes[k]));
          n[2 * k] = valid ? (int)(nodes[k] & 0xffffu) : -1;
          n[2 * k + 1] = (int)(nodes[k] >> 16);
        }
        double* acc = col + t;
        double ecell, vir[6], gacc[8][3];
        auto corners = [&](double (&p)[8][3]) {
          load_corners(xs, n, p, on, Sl + MM_S_XMAT, on2, Sl + MM_S_XMAT2);
        };
        if (ns > 1)
          cell_eval<kModel, kOutGradient, true, kSmall>(tab, ns, kt, valid, corners, wrap, rv, acc,
                                                        ecell, vir, gacc);
        else
          cell_eval<kModel, kOutGradient, false, kSmall>(tab, ns, kt, valid, corners, wrap, rv,
                                                         acc, ecell, vir, gacc);
        if (records) {
          fold_cell(wrap, gacc);
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              acc[(3 * q + j) * kSmall] = gacc[kLowerCorner[q]][j];
              acc[(12 + 3 * q + j) * kSmall] = gacc[kUpperCorner[q]][j];
            }
        }
        cell_wave_totals(ecell, vir, cred + 7 * wave);
      }
      __syncthreads();
    }

    for (int part = 0; part < 2; ++part) {
      if (part == 1) {
        if (gather == kSmallNone) break;
        double acc[NA];
#pragma unroll
        for (int q = 0; q < NA; ++q) acc[q] = 0.0;
        double lt = 0.0;
        if (own) {
#pragma unroll
          for (int j = 0; j < 3; ++j) g[j] = 0.0;
#pragma unroll
          for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(places[k]));
          double r[8][3];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const int place = places[k / 2] >> (16 * (k & 1)) & 0xffffu;
#pragma unroll
            for (int j = 0; j < 3; ++j) r[k][j] = col[(place == 0xffff ? 0 : place) + j * kSmall];
          }
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const bool none = (places[k / 2] >> (16 * (k & 1)) & 0xffffu) == 0xffffu;
#pragma unroll
            for (int j = 0; j < 3; ++j) g[j] = none ? g[j] : g[j] + r[k][j];
          }
#pragma unroll
          for (int j = 0; j < 3; ++j)
            if (g[j] != g[j]) acc[12] = 1.0;
          if (gather == kSmallKick) {
            kick_node<kLT>(Sl, t, mass, g, v, acc, lt);
            if (kLT) acc[NA - 1] = lt;
          } else if (gather == kSmallDrift) {
            double x[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) x[j] = xs[3 * t + j];
            scale_position(Sl, x);
            kick_drift_node<kLT>(Sl, t, mass, g, v, x, lt);
#pragma unroll
            for (int j = 0; j < 3; ++j) xs[3 * t + j] = x[j];
          } else {
            apply_vtransform(Sl, v);
          }
        }
        if (gather == kSmallDrift) {
          if (kLT) {
            const double one[1] = {lt};
            const double s = wave_reduce_scatter<1>(one, lane);
            if (lane == 0) lred[wave] = s;
          }
        } else {
          const double s = wave_reduce_scatter<NA>(acc, lane);
          const int q = scatter_index(lane);
          if ((lane & 3) == 0 && q < NA)
            nred[16 * wave + q] = gather == kSmallKick ? s : q == 12 && s != 0.0 ? 1.0 : 0.0;
        }
        __syncthreads();
      }
      const int ph = part ? phase1 : phase0;
      if (ph < 0) continue;
      if (wave == 0) {
        // the blocks' sums (their waves in order), the two blocks in order
        static_assert(kWaves == 8 && kCellBlock == 256 && kNodeBlock == 256, "two blocks of sums");
        const bool force = lane < 10, ltq = lane == 25;
        const int each = force ? 7 : ltq ? 1 : 16;
        const double* w = force ? cred + total_entry(lane)
                          : ltq ? lred : nred + (lane < 26 ? lane - 10 : 0);
        double p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = w[k * each];
        double s = 0.0 + (((p[0] + p[1]) + p[2]) + p[3]);
        s += ((p[4] + p[5]) + p[6]) + p[7];
        if (!(force ? phase_uses_force(ph) : phase_uses_nodes(ph))) s = 0.0;
        if (lane < kSliceQ) tot[lane] = s;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        run_phases(ph, (lds_f64*)Sl, (const lds_f64*)tot, 1, 0);
      }
      __syncthreads();
    }
    if (seg >= 0 && (!a.baro || seg == 2)) {
      ++step;
      seg = 0;
    } else {
      ++seg;
    }
  }
  if (own) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      a.pos[3 * t + j] = xs[3 * t + j];
      a.vel[3 * t + j] = v[j];
      a.gpos[3 * t + j] = g[j];
    }
  }
  if (t < MM_S_COUNT) a.S[t] = Sl[t];
}

}  // namespace mm

using namespace mm;

struct mm_md {
  mm_field* field = nullptr;
  double* pos = nullptr;
  double* vel = nullptr;
  double* gpos = nullptr;
  const double* masses = nullptr;
  double* posold = nullptr;
  double* S = nullptr;
  double* npart = nullptr;
  int thermo = 0, baro = 0;
  int64_t N = 0;
  int nbn = 0;
  int32_t nsys = 1;
  int32_t* node_blk_sys = nullptr;   // [nbn] system of every node block
  int32_t* sys_nblk = nullptr;       // [nsys + 1] node-block range of every system
  int slices = 1;                    // blocks per system of a reducing scalar phase
  double* slice_buf = nullptr;       // [nsys][slices][kSliceQ]
  unsigned int* counters = nullptr;  // [nsys] last-block counters (kept at zero between calls)
  bool merge = false;                // phases of a row of steps merged into the kernels after them
  double* S2 = nullptr;              // [MM_S_COUNT] the scalar block's other copy (merge)
  double* fpart2 = nullptr;          // the second cell pass's sums (merge)
  hipStream_t stream = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  // One step alone; a call of several replays the lean step without its opening part (the scalar
  // phase or the kick-drift pass that the step before has done) and ends with a full step
  // without it.
  hipGraph_t graph = nullptr, graph_lean = nullptr, graph_last = nullptr;
  hipGraphExec_t exec = nullptr, exec_lean = nullptr, exec_last = nullptr;
  int graph_split = 0;                // the field's block split the graphs were captured with
};

namespace {

struct Dev {
  int prev = -1;
  explicit Dev(int d) {
    (void)hipGetDevice(&prev);
    if (prev != d) (void)hipSetDevice(d);
  }
  ~Dev() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

ForceArgs force_args(mm_md* md) {
  mm_field* f = md->field;
  ForceArgs a;
  a.pos = md->pos;
  a.rvecs = md->S + MM_S_RVECS;
  a.rvecs_stride = MM_S_COUNT;
  a.blk_sys = f->blk_sys;
  a.cnode = f->cnode;
  a.cwrap = f->cwrap;
  a.blk_row = f->blk_row;
  a.tab = f->tab;
  a.kt = f->kt;
  a.nstates = f->nstates;
  a.max_states = f->max_states;
  a.W = f->W;
  a.N = f->N;
  a.ncell = f->nrec;
  a.gcell = f->gcell;
  a.rstride = f->S;
  a.cbase = f->cbase;
  a.partials = f->partials;
  a.energy = nullptr;
  a.gpos = nullptr;
  a.vtens = nullptr;
  a.accumulate = 0;
  a.model = f->model;
  a.nanflag = f->nanflag;
  a.force_grad = 1;
  schedule_args(f, a);
  return a;
}

hipError_t node(mm_md* md, int mode, hipStream_t s) {
  const dim3 grid(md->nbn), block(kNodeThreads);
#define MM_NODE(M)                                                                          \
  hipLaunchKernelGGL((node_kernel<M>), grid, block, 0, s, md->pos, md->vel, md->gpos,        \
                     md->masses, md->posold, md->S, md->node_blk_sys, md->N, md->npart)
  switch (mode) {
    case kScalePos: MM_NODE(kScalePos); break;
    case kVV: MM_NODE(kVV); break;
    case kApplyV: MM_NODE(kApplyV); break;
    case kRmsd: MM_NODE(kRmsd); break;
  }
#undef MM_NODE
  return hipGetLastError();
}

hipError_t kick_drift(mm_md* md, bool lt, hipStream_t s) {
#define MM_KD(T, P, A)                                                                      \
  hipLaunchKernelGGL((kick_drift_kernel<T, P>), dim3(md->nbn), dim3(kNodeBlock), 0, s, md->pos, \
                     md->vel, md->gpos, md->masses, md->S, md->node_blk_sys, md->N, md->npart, A)
  if (lt)
    MM_KD(true, -1, PhaseArgs{});
  else
    MM_KD(false, -1, PhaseArgs{});
  return hipGetLastError();
}

// The same, begun with the phase kPhNvtEndPre on the sums of the step before.
hipError_t kick_drift_merged(mm_md* md, hipStream_t s) {
  const mm_field* f = md->field;
  const PhaseArgs ph{md->S, md->S2, f->partials, md->npart, (int)(f->W / kCellBlock), md->nbn};
  MM_KD(false, kPhNvtEndPre, ph);
#undef MM_KD
  return hipGetLastError();
}

bool reduces(int phase) {
  return phase == kPhInitForce || phase == kPhNveEnd || phase == kPhNvtEnd ||
         phase == kPhMainEndNpt || phase == kPhInitProps || phase == kPhBaroEndPre ||
         phase == kPhBaroEndPost || phase == kPhBaroEndPostPre || phase >= kPhNvtEndPre ||
         phase == kPhRmsd;
}

hipError_t scalar(mm_md* md, int phase, int with_vtens, hipStream_t s) {
  const int nbf = (int)(md->field->W / kCellBlock);
  const int G = reduces(phase) ? md->slices : 1;
  // one system owns every cell block, in order: its block list is the identity
  const int32_t* cidx = md->nsys == 1 ? nullptr : md->field->sys_cblk_idx;
  hipLaunchKernelGGL(scalar_kernel, dim3(G, md->nsys), dim3(kScalarThreads), 0, s, phase, md->S,
                     md->field->partials, nbf, md->field->sys_cblk_ptr, cidx, md->npart, md->nbn,
                     md->sys_nblk, with_vtens, md->slice_buf, md->counters);
  return hipGetLastError();
}

// force evaluation: cells, then gather (+ second half kick when kick, + the Langevin
// thermostat's post update when lt; with next also the next step's kick and drift; + the pending
// velocity transforms when scale_v). gmode
// (gather_kick_kernel): kGatherNone leaves out the records altogether, so the cell pass skips
// them too, and without scale_v there is then no node pass at all (energy and virial only).
hipError_t gather_kick(mm_md* md, bool kick, bool lt, hipStream_t s, bool scale_v, int gmode,
                       bool next, const double* S, const Carry& c) {
  const mm_field* f = md->field;
  const bool all = md->nbn <= kGatherAllLoadsMaxBlocks;
#define MM_GATHER1(K, T, V, D, A)                                                            \
  hipLaunchKernelGGL((gather_kick_kernel<K, T, V, D, A>), dim3(md->nbn), dim3(kNodeBlock), 0, s, \
                     f->nrec, f->gcell, md->N, f->S, md->gpos, md->vel, md->masses, S,        \
                     md->node_blk_sys, md->npart, gmode, md->pos, c, PhaseArgs{})
#define MM_GATHER(K, T, V, D)          \
  do {                                 \
    if (all)                           \
      MM_GATHER1(K, T, V, D, true);    \
    else                               \
      MM_GATHER1(K, T, V, D, false);   \
  } while (0)
  if (kick && next && lt)
    MM_GATHER(true, true, false, true);
  else if (kick && next)
    MM_GATHER(true, false, false, true);
  else if (kick && lt)
    MM_GATHER(true, true, false, false);
  else if (kick)
    MM_GATHER(true, false, false, false);
  else if (scale_v)
    MM_GATHER(false, false, true, false);
  else
    MM_GATHER(false, false, false, false);
#undef MM_GATHER
#undef MM_GATHER1
  return hipGetLastError();
}

hipError_t force(mm_md* md, bool kick, bool lt, hipStream_t s, bool scale_v = false,
                 int gmode = kGatherStore, const double* xmat = nullptr, bool next = false) {
  ForceArgs a = force_args(md);
  a.xmat = xmat;
  if (gmode == kGatherNone) {
    if (kick) return hipErrorInvalidValue;
    a.store_records = 0;
  }
  hipError_t e = launch_cells(a, s);
  if (e != hipSuccess) return e;
  // with no records, no transform to apply and no kick, the evaluation has no node pass
  if (md->N > 0 && !(gmode == kGatherNone && !scale_v && !kick))
    e = gather_kick(md, kick, lt, s, scale_v, gmode, next, md->S, Carry{});
  return e;
}

#define MM_TRY(x)                         \
  do {                                    \
    hipError_t _e = (x);                  \
    if (_e != hipSuccess) return _e;      \
  } while (0)

// The first half kick and the drift from the records of the last cell pass (the barostat's
// pre call, whose gradient nothing else reads), after that call's scalar phase has set the
// pending velocity transforms; with lt also the Langevin thermostat's pre update.
hipError_t gather_drift(mm_md* md, bool lt, hipStream_t s) {
  if (md->N == 0) return hipSuccess;
  mm_field* f = md->field;
  const bool all = md->nbn <= kGatherAllLoadsMaxBlocks;
#define MM_DRIFT(T, A, P, C)                                                                 \
  hipLaunchKernelGGL((gather_kick_kernel<false, T, false, true, A, P>), dim3(md->nbn),       \
                     dim3(kNodeBlock), 0, s, f->nrec, f->gcell, md->N, f->S, md->gpos,       \
                     md->vel, md->masses, md->S, md->node_blk_sys, md->npart, kGatherKeep,   \
                     md->pos, Carry{}, C)
  if (lt && all)
    MM_DRIFT(true, true, -1, PhaseArgs{});
  else if (lt)
    MM_DRIFT(true, false, -1, PhaseArgs{});
  else if (all)
    MM_DRIFT(false, true, -1, PhaseArgs{});
  else
    MM_DRIFT(false, false, -1, PhaseArgs{});
  return hipGetLastError();
}

// The same, begun with the phase kPhBaroEndPre on the sums of the last cell pass.
hipError_t gather_drift_merged(mm_md* md, bool lt, hipStream_t s) {
  mm_field* f = md->field;
  const PhaseArgs ph{md->S, md->S2, f->partials, md->npart, (int)(f->W / kCellBlock), md->nbn};
  if (lt)
    MM_DRIFT(true, true, kPhBaroEndPre, ph);
  else
    MM_DRIFT(false, true, kPhBaroEndPre, ph);
#undef MM_DRIFT
  return hipGetLastError();
}

// The barostat call MTKBarostat.baro after its first scalar phase: positions scaled, force,
// then the second barostat-velocity update. The pre call (pre_call) scales no positions in a
// pass of its own: its cell pass reads them through the pending transforms, and it leaves its
// records for gather_drift, which stores the scaled positions and applies the velocity
// transform with the kick. The post call's velocity transform is applied by its gather
// (scale_v) or stays pending; with defer_x (a post call without records) its position scaling
// also waits (the cell pass applies it on the fly, the next gather_drift stores it).
hipError_t baro_call(mm_md* md, int end_phase, hipStream_t s, bool scale_v,
                     int gmode = kGatherStore, bool pre_call = false,
                     bool defer_x = false) {
  if (!defer_x && !pre_call) MM_TRY(node(md, kScalePos, s));
  if (pre_call) {
    // the pre call's scaling (after a pending post-call one) is applied by its cell pass as it
    // reads the positions and stored by gather_drift
    ForceArgs a = force_args(md);
    a.xmat = md->S + MM_S_XMAT;
    a.xmat2 = md->S + MM_S_XMAT2;
    a.xmat2_on = md->S + MM_S_XMAT2_ON;
    MM_TRY(launch_cells(a, s));
  } else {
    MM_TRY(force(md, false, false, s, scale_v, gmode, defer_x ? md->S + MM_S_XMAT : nullptr));
  }
  MM_TRY(scalar(md, end_phase, 1, s));
  return hipSuccess;
}

// One step. lean: a step that another step of the same call follows, so that nothing reads
// the node gradients or the scalar block in between. With a barostat, the gradient of its main
// force evaluation is then used only by the kick in the gather, and that of the barostat's post
// call by nothing (the next step's pre call evaluates the force again before its kick,
// verlet.py:141-143 with npt.py:616-620), so those evaluations keep their gradients out of
// HBM; and a lean step ends with the next step's opening phase (kPhBaroEndPostPre,
// kPhNvtEndPre) or, where no phase opens a step, with its kick and drift, so that step is enqueued
// with pre = false. Positions, velocities, energies,
// virials and every scalar are those of full steps, bit for bit.
hipError_t enqueue_step(mm_md* md, hipStream_t s, bool lean = false, bool pre = true) {
  const bool lt = md->thermo == MM_THERMO_LANGEVIN;
  if (md->baro) {
    if (pre) MM_TRY(scalar(md, kPhBaroPre, 1, s));
    // the pre call's gradient drives only the first half kick: its gather is the kick-drift
    MM_TRY(baro_call(md, kPhBaroEndPre, s, false, kGatherKeep, true));
    MM_TRY(gather_drift(md, lt, s));
    MM_TRY(force(md, true, lt, s, false, lean ? kGatherKeep : kGatherStore));
    MM_TRY(scalar(md, kPhMainEndNpt, 1, s));
    // the post call's velocity transform stays pending in a lean step (its node sums follow
    // from the ones before it), and so does its position scaling (the cell pass applies it
    // as it reads the positions, the next step's scaling pass stores it), so its force
    // evaluation has no node pass at all and forms no vertex gradient (the virial comes from
    // the edges, the same bits either way)
    MM_TRY(baro_call(md, lean ? kPhBaroEndPostPre : kPhBaroEndPost, s, !lean,
                     lean ? kGatherNone : kGatherStore, false, lean));
  } else if (md->thermo == MM_THERMO_NHC) {
    if (pre) MM_TRY(scalar(md, kPhNvtPre, 1, s));
    MM_TRY(kick_drift(md, false, s));
    MM_TRY(force(md, true, false, s));
    MM_TRY(scalar(md, lean ? kPhNvtEndPre : kPhNvtEnd, 1, s));
  } else {
    // no scalar phase stands between the second kick of a step and the first of the next: the
    // gather of a lean step does both, and the drift
    if (pre) MM_TRY(kick_drift(md, lt, s));
    MM_TRY(force(md, true, lt, s, false, lean ? kGatherKeep : kGatherStore, nullptr, lean));
    const int end = !lt ? kPhNveEnd
                    : pre ? (lean ? kPhLtFirst : kPhNvtEnd) : (lean ? kPhLtNext : kPhLtLast);
    MM_TRY(scalar(md, end, 1, s));
  }
  return hipSuccess;
}

// A merged cell pass: phase on the sums fin (and the node sums) from s_in to s_out, its own to fout.
hipError_t md_cells(mm_md* md, int phase, const double* s_in, double* s_out, const double* fin,
                    double* fout, hipStream_t s) {
  const mm_field* f = md->field;
  const CellPass c{f->cnode, f->cwrap, f->blk_row, f->nstates, f->cbase, f->tab, f->kt,
                   f->max_states, f->W, f->S, f->gcell};
  const int nb = (int)(f->W / kCellBlock);
  const PhaseArgs ph{s_in, s_out, fin, md->npart, nb, md->nbn};
  const dim3 grid(nb + (phase_gates(phase) ? 0 : 1)), block(kCellBlock);
#define MM_CELLS(M, O, P)                                                                     \
  hipLaunchKernelGGL((md_cells_kernel<M, O, P>), grid, block, 0, s, c, md->pos, ph, fout)
#define MM_CELLS_PHASE(M)                                                   \
  switch (phase) {                                                          \
    case kPhNveEnd: MM_CELLS(M, kOutGradient, kPhNveEnd); break;            \
    case kPhLtFirst: MM_CELLS(M, kOutGradient, kPhLtFirst); break;          \
    case kPhLtNext: MM_CELLS(M, kOutGradient, kPhLtNext); break;            \
    case kPhBaroEndPostPre: MM_CELLS(M, kOutGradient, kPhBaroEndPostPre); break; \
    case kPhMainEndNpt: MM_CELLS(M, kOutVirial, kPhMainEndNpt); break;      \
    default: return hipErrorInvalidValue;                                   \
  }
  if (f->model == 0) {
    MM_CELLS_PHASE(0)
  } else {
    MM_CELLS_PHASE(1)
  }
#undef MM_CELLS_PHASE
#undef MM_CELLS
  return hipGetLastError();
}

// The barostat's main force evaluation and the cell pass of its post call, from the positions
// and velocities of gather_drift_merged on: the scalar block is in S2.
hipError_t row_main(mm_md* md, bool last, hipStream_t s) {
  const bool lt = md->thermo == MM_THERMO_LANGEVIN;
  ForceArgs a = force_args(md);
  a.rvecs = md->S2 + MM_S_RVECS;
  MM_TRY(launch_cells(a, s));
  MM_TRY(gather_kick(md, true, lt, s, false, last ? kGatherStore : kGatherKeep, false, md->S2,
                     Carry{md->S}));
  if (last) return hipSuccess;
  return md_cells(md, kPhMainEndNpt, md->S, md->S2, md->field->partials, md->fpart2, s);
}

// The first step of a row of merged steps, without its closing phase.
hipError_t row_open(mm_md* md, hipStream_t s) {
  const bool lt = md->thermo == MM_THERMO_LANGEVIN;
  if (md->baro) {
    MM_TRY(scalar(md, kPhBaroPre, 1, s));
    ForceArgs a = force_args(md);
    a.xmat = md->S + MM_S_XMAT;
    a.xmat2 = md->S + MM_S_XMAT2;
    a.xmat2_on = md->S + MM_S_XMAT2_ON;
    MM_TRY(launch_cells(a, s));
    MM_TRY(gather_drift_merged(md, lt, s));
    return row_main(md, false, s);
  }
  if (md->thermo == MM_THERMO_NHC) {
    MM_TRY(scalar(md, kPhNvtPre, 1, s));
    MM_TRY(kick_drift(md, false, s));
    return force(md, true, false, s);
  }
  MM_TRY(kick_drift(md, lt, s));
  return force(md, true, lt, s, false, kGatherKeep, nullptr, true);
}

// A further step, from the closing phase of the one before it on; first: that one opened the row;
// last: this one ends it (with its closing phase).
hipError_t row_next(mm_md* md, bool first, bool last, hipStream_t s) {
  const bool lt = md->thermo == MM_THERMO_LANGEVIN;
  double* f0 = md->field->partials;
  const int nf = 10 * (int)(md->field->W / kCellBlock);
  if (md->baro) {
    MM_TRY(md_cells(md, kPhBaroEndPostPre, md->S2, md->S, md->fpart2, f0, s));
    MM_TRY(gather_drift_merged(md, lt, s));
    MM_TRY(row_main(md, last, s));
    if (!last) return hipSuccess;
    MM_TRY(scalar(md, kPhMainEndNpt, 1, s));
    return baro_call(md, kPhBaroEndPost, s, true);
  }
  if (md->thermo == MM_THERMO_NHC) {
    MM_TRY(kick_drift_merged(md, s));
    MM_TRY(launch_cells(force_args(md), s));
    MM_TRY(gather_kick(md, true, false, s, false, kGatherStore, false, md->S2, Carry{md->S}));
    return last ? scalar(md, kPhNvtEnd, 1, s) : hipSuccess;
  }
  MM_TRY(md_cells(md, !lt ? kPhNveEnd : first ? kPhLtFirst : kPhLtNext, md->S, md->S, f0,
                  md->fpart2, s));
  MM_TRY(gather_kick(md, true, lt, s, false, last ? kGatherStore : kGatherKeep, !last, md->S,
                     Carry{nullptr, md->fpart2, f0, nf}));
  return last ? scalar(md, lt ? kPhLtLast : kPhNveEnd, 1, s) : hipSuccess;
}

// Whether the one-workgroup kernel steps this system.
bool small_system(const mm_md* md) {
  return md->nsys == 1 && md->N > 0 && md->N <= kSmall && md->field->W > 0 &&
         md->field->W <= kSmall;
}

// nsteps steps (the last one full), at most kSmallSteps in a launch (some 20 to 80 ms: a call can be
// any number of steps, a kernel should end within a reasonable time).
constexpr int kSmallSteps = 2048;
hipError_t run_small(mm_md* md, int nsteps, hipStream_t s) {
  for (; nsteps > kSmallSteps; nsteps -= kSmallSteps) MM_TRY(run_small(md, kSmallSteps, s));
  const mm_field* f = md->field;
  const SmallArgs a{f->cnode, f->cwrap, f->blk_row, f->nstates, f->nrec, f->cbase, f->tab, f->kt,
                    f->max_states, (int)f->W, (int)md->N, md->pos, md->vel, md->gpos,
                    md->masses, md->S, md->thermo, md->baro, nsteps};
  const dim3 block(std::max(f->W, md->N) > kSmall / 2 ? kSmall : kSmall / 2);
  const bool lt = md->thermo == MM_THERMO_LANGEVIN;
#define MM_SMALL(M, T) hipLaunchKernelGGL((small_kernel<M, T>), dim3(1), block, 0, s, a)
  if (f->model == 0) {
    if (lt) MM_SMALL(0, true); else MM_SMALL(0, false);
  } else {
    if (lt) MM_SMALL(1, true); else MM_SMALL(1, false);
  }
#undef MM_SMALL
  return hipGetLastError();
}

int begin(mm_md* md, void* stream) {
  hipError_t e = hipEventRecord(md->ev_in, (hipStream_t)stream);
  if (e == hipSuccess) e = hipStreamWaitEvent(md->stream, md->ev_in, 0);
  return e == hipSuccess ? MM_OK : hip_error(e, "stream ordering");
}

int end(mm_md* md, void* stream) {
  hipError_t e = hipEventRecord(md->ev_out, md->stream);
  if (e == hipSuccess) e = hipStreamWaitEvent((hipStream_t)stream, md->ev_out, 0);
  return e == hipSuccess ? MM_OK : hip_error(e, "stream ordering");
}

}  // namespace

namespace {

// Capture what enqueue puts on the engine's stream into an executable graph.
template <typename Enqueue>
hipError_t capture(mm_md* md, hipGraph_t* graph, hipGraphExec_t* exec, Enqueue enqueue) {
  hipError_t e = hipStreamBeginCapture(md->stream, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return e;
  const hipError_t e2 = enqueue();
  e = hipStreamEndCapture(md->stream, graph);
  if (e2 != hipSuccess) e = e2;
  if (e == hipSuccess) e = hipGraphInstantiate(exec, *graph, nullptr, nullptr, 0);
  return e;
}

void drop_graph(mm_md* md) {
  if (md->exec) (void)hipGraphExecDestroy(md->exec);
  if (md->graph) (void)hipGraphDestroy(md->graph);
  if (md->exec_lean) (void)hipGraphExecDestroy(md->exec_lean);
  if (md->graph_lean) (void)hipGraphDestroy(md->graph_lean);
  if (md->exec_last) (void)hipGraphExecDestroy(md->exec_last);
  if (md->graph_last) (void)hipGraphDestroy(md->graph_last);
  md->exec = md->exec_lean = md->exec_last = nullptr;
  md->graph = md->graph_lean = md->graph_last = nullptr;
}

}  // namespace

extern "C" {

int mm_md_create_batch(mm_md** out, mm_field* field, int32_t nsys, const int64_t* sys_node_start,
                       double* pos, double* vel, double* gpos, const double* masses,
                       double* posold, double* scalars, int thermo, int baro) {
  if (!out || !field || !scalars || !sys_node_start) return set_error(MM_ERR_ARG, "missing argument");
  if (nsys != field->nsys)
    return set_error(MM_ERR_ARG, "field holds %d systems, not %d", field->nsys, nsys);
  if (field->N > 0 && (!pos || !vel || !gpos || !masses || !posold))
    return set_error(MM_ERR_ARG, "missing node buffer");
  if (thermo != MM_THERMO_NONE && thermo != MM_THERMO_NHC && thermo != MM_THERMO_LANGEVIN)
    return set_error(MM_ERR_ARG, "unknown thermostat %d", thermo);
  if (baro != MM_BARO_NONE && baro != MM_BARO_MTK && baro != MM_BARO_LANGEVIN)
    return set_error(MM_ERR_ARG, "unknown barostat %d", baro);
  if (sys_node_start[0] != 0 || sys_node_start[nsys] != field->N)
    return set_error(MM_ERR_ARG, "node ranges must cover [0, %lld)", (long long)field->N);
  const int nbn_total = (int)((field->N + kNodeBlock - 1) / kNodeBlock);
  std::vector<int32_t> node_blk_sys(nbn_total > 0 ? nbn_total : 1, 0), sys_nblk(nsys + 1, 0);
  for (int s = 0; s < nsys; ++s) {
    const int64_t a = sys_node_start[s], b = sys_node_start[s + 1];
    if (b < a || (nsys > 1 && a % kNodeBlock != 0))
      return set_error(MM_ERR_ARG, "system %d: node range [%lld, %lld) invalid", s,
                       (long long)a, (long long)b);
    const int blo = (int)(a / kNodeBlock), bhi = (int)((b + kNodeBlock - 1) / kNodeBlock);
    sys_nblk[s] = blo;
    sys_nblk[s + 1] = bhi;
    for (int k = blo; k < bhi; ++k) node_blk_sys[k] = s;
  }
  Dev dev(field->device);
  mm_md* md = new mm_md();
  md->field = field;
  md->pos = pos;
  md->vel = vel;
  md->gpos = gpos;
  md->masses = masses;
  md->posold = posold;
  md->S = scalars;
  md->thermo = thermo;
  md->baro = baro;
  md->N = field->N;
  md->nbn = nbn_total > 0 ? nbn_total : 1;
  md->nsys = nsys;
  // slices of a reducing scalar phase: about 256 partial blocks each, at most kScalarSlices
  std::vector<int32_t> cptr(nsys + 1, 0);
  hipError_t e = hipMemcpy(cptr.data(), field->sys_cblk_ptr, sizeof(int32_t) * (nsys + 1),
                           hipMemcpyDeviceToHost);
  int most = 0;
  for (int s = 0; s < nsys; ++s) {
    most = std::max(most, cptr[s + 1] - cptr[s]);
    most = std::max(most, sys_nblk[s + 1] - sys_nblk[s]);
  }
  md->slices = most <= kMergeMaxBlocks ? 1 : std::min(kScalarSlices, (most + 255) / 256);
  md->merge = nsys == 1 && md->slices == 1 && field->W > 0 && field->N > 0 && !small_system(md);
  if (e == hipSuccess && md->merge)
    e = hipMalloc((void**)&md->S2, sizeof(double) * MM_S_COUNT);
  if (e == hipSuccess && md->merge)
    e = hipMalloc((void**)&md->fpart2, sizeof(double) * 10 * (field->W / kCellBlock));
  if (e == hipSuccess) e = hipMalloc((void**)&md->npart, sizeof(double) * kNodePartial * md->nbn);
  if (e == hipSuccess) e = hipMemset(md->npart, 0, sizeof(double) * kNodePartial * md->nbn);
  if (e == hipSuccess)
    e = hipMalloc((void**)&md->slice_buf, sizeof(double) * kSliceQ * md->slices * nsys);
  if (e == hipSuccess) e = hipMalloc((void**)&md->counters, sizeof(unsigned int) * nsys);
  if (e == hipSuccess) e = hipMemset(md->counters, 0, sizeof(unsigned int) * nsys);
  if (e == hipSuccess) e = hipMalloc((void**)&md->node_blk_sys, sizeof(int32_t) * md->nbn);
  if (e == hipSuccess) e = hipMalloc((void**)&md->sys_nblk, sizeof(int32_t) * (nsys + 1));
  if (e == hipSuccess)
    e = hipMemcpy(md->node_blk_sys, node_blk_sys.data(), sizeof(int32_t) * md->nbn,
                  hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(md->sys_nblk, sys_nblk.data(), sizeof(int32_t) * (nsys + 1),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&md->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&md->ev_in, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&md->ev_out, hipEventDisableTiming);
  if (e != hipSuccess) {
    mm_md_destroy(md);
    return hip_error(e, "mm_md_create");
  }
  *out = md;
  return MM_OK;
}

int mm_md_create(mm_md** out, mm_field* field, double* pos, double* vel, double* gpos,
                 const double* masses, double* posold, double* scalars, int thermo, int baro) {
  if (!field) return set_error(MM_ERR_ARG, "missing argument");
  if (field->nsys != 1) return set_error(MM_ERR_ARG, "batched field: use mm_md_create_batch");
  const int64_t range[2] = {0, field->N};
  return mm_md_create_batch(out, field, 1, range, pos, vel, gpos, masses, posold, scalars,
                            thermo, baro);
}

int mm_md_init_force(mm_md* md, int with_vtens, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = force(md, false, false, md->stream);
  if (e == hipSuccess) e = scalar(md, kPhInitForce, with_vtens, md->stream);
  if (e != hipSuccess) return hip_error(e, "mm_md_init_force");
  return end(md, stream);
}

int mm_md_init_properties(mm_md* md, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = node(md, kVV, md->stream);
  if (e == hipSuccess) e = scalar(md, kPhInitProps, 1, md->stream);
  if (e != hipSuccess) return hip_error(e, "mm_md_init_properties");
  return end(md, stream);
}

int mm_md_step(mm_md* md, int32_t nsteps, int use_graph, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  if (nsteps < 0) return set_error(MM_ERR_ARG, "negative step count");
  if (nsteps == 0) return MM_OK;
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = hipSuccess;
  if (use_graph && small_system(md)) {
    e = run_small(md, nsteps, md->stream);
  } else if (use_graph) {
    // the launch ranges of the cell pass follow the field's block split: a new split (new
    // state counts through mm_field_set_params) needs a new graph
    if (md->graph_split != md->field->split) drop_graph(md);
    md->graph_split = md->field->split;
    // every step but the last is followed by another before the call returns
    hipStream_t q = md->stream;
    const bool row = nsteps > 1;
    if (!row && !md->exec)
      e = capture(md, &md->graph, &md->exec, [&] { return enqueue_step(md, q); });
    if (row && !md->exec_lean)
      e = capture(md, &md->graph_lean, &md->exec_lean, [&] {
        return md->merge ? row_next(md, false, false, q) : enqueue_step(md, q, true, false);
      });
    if (row && e == hipSuccess && !md->exec_last)
      e = capture(md, &md->graph_last, &md->exec_last, [&] {
        return md->merge ? row_next(md, false, true, q) : enqueue_step(md, q, false, false);
      });
    if (e != hipSuccess) return hip_error(e, "capturing the MD step");
    if (row) {
      // the first step, or its opening phase, is like no other, and with the Langevin thermostat
      // the second merged one
      int i = 0;
      const bool lt = md->thermo == MM_THERMO_LANGEVIN && !md->baro;
      if (md->merge) {
        e = row_open(md, q);
        i = 1;
        if (e == hipSuccess && lt) {
          e = row_next(md, true, nsteps == 2, q);
          i = 2;
        }
      } else if (md->baro || md->thermo == MM_THERMO_NHC) {
        e = scalar(md, md->baro ? kPhBaroPre : kPhNvtPre, 1, q);
      } else {
        e = enqueue_step(md, q, true, true);
        i = 1;
      }
      for (; i + 1 < nsteps && e == hipSuccess; ++i) e = hipGraphLaunch(md->exec_lean, q);
      if (i < nsteps && e == hipSuccess) e = hipGraphLaunch(md->exec_last, q);
    } else {
      e = hipGraphLaunch(md->exec, q);
    }
  } else {
    const bool lean = nsteps > 1;
    for (int i = 0; i < nsteps && e == hipSuccess; ++i)
      e = enqueue_step(md, md->stream, lean && i + 1 < nsteps, !lean || i == 0);
  }
  if (e != hipSuccess) return hip_error(e, "mm_md_step");
  return end(md, stream);
}

int mm_md_sync(mm_md* md, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = node(md, kApplyV, md->stream);
  if (e == hipSuccess) e = scalar(md, kPhApplied, 0, md->stream);
  if (e != hipSuccess) return hip_error(e, "mm_md_sync");
  return end(md, stream);
}

int mm_md_snapshot(mm_md* md, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = hipMemcpyAsync(md->posold, md->pos, sizeof(double) * 3 * md->N,
                                hipMemcpyDeviceToDevice, md->stream);
  if (e != hipSuccess) return hip_error(e, "mm_md_snapshot");
  return end(md, stream);
}

int mm_md_rmsd(mm_md* md, void* stream) {
  if (!md) return set_error(MM_ERR_ARG, "md is NULL");
  Dev dev(md->field->device);
  int rc = begin(md, stream);
  if (rc) return rc;
  hipError_t e = node(md, kRmsd, md->stream);
  if (e == hipSuccess) e = scalar(md, kPhRmsd, 0, md->stream);
  if (e != hipSuccess) return hip_error(e, "mm_md_rmsd");
  return end(md, stream);
}

void mm_md_destroy(mm_md* md) {
  if (!md) return;
  drop_graph(md);
  if (md->stream) {
    (void)hipStreamSynchronize(md->stream);
    (void)hipStreamDestroy(md->stream);
  }
  if (md->ev_in) (void)hipEventDestroy(md->ev_in);
  if (md->ev_out) (void)hipEventDestroy(md->ev_out);
  if (md->npart) (void)hipFree(md->npart);
  if (md->slice_buf) (void)hipFree(md->slice_buf);
  if (md->counters) (void)hipFree(md->counters);
  if (md->S2) (void)hipFree(md->S2);
  if (md->fpart2) (void)hipFree(md->fpart2);
  if (md->node_blk_sys) (void)hipFree(md->node_blk_sys);
  if (md->sys_nblk) (void)hipFree(md->sys_nblk);
  delete md;
}

}  // extern "C"
