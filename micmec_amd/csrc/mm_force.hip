// Force-field kernels: per-cell energies and vertex gradients, node gather, reductions.
//
// Reference path: ForcePartMechanical._internal_compute (micmec/pes/mmff.py:288-323) and
// deformation (mmff.py:326-403). Layout in HBM (all FP64 unless noted):
//   pos      [N][3]              node positions (caller's buffer)
//   rvecs    [3][3]              domain vectors, rows (device copy)
//   cnode    [W][8] int32        node at corner k of work slot w (-1 = padding slot)
//   cwrap    [W]    int32        wrap bits of the cell in slot w
//   blk_row  [W/256] int32       parameter-table row shared by all cells of a block
//   ncell    [8][N] int32        node n -> record (slot << 2 | face class) of its corner k, -1
//                                none or folded into the +z neighbour's record
//   gcell    [4][3][S]           vertex gradients by face class: the lower face (corners 0, 1,
//                                2, 4) of slot w at w, with the upper face of the -z neighbour
//                                in slot w - 1 added when the two share a wave; the other upper
//                                faces (corners 3, 5, 6, 7) at compact slots W + i (S = W + their
//                                number)
//   cbase    [W/64] int32        first compact slot of every wave
//   partials [16][W/256]         per-block energy (0) and virial (1..9), SoA
//   cgpart   [8][(N+255)/256]    per-workgroup sums of the line-search kernels (cg_*)
// Cells are grouped by type into 256-slot segments, so the type, its number of states and its
// parameter row are uniform per block and the parameters are read with scalar loads.
//
// One lane per cell: the lane gathers the cell's eight nodes, evaluates strains and stresses of
// every corner in the metric of the edges (mm_device.h) and forms the eight vertex gradients in
// registers (for multistate cells the stresses' weighted sum over the states is kept in LDS).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mm_cell.h"
#include "mm_device.h"
#include "mm_kernels.h"

namespace mm {

// One lane per cell. Energies of all states of the block's cell type, combined by the
// log-sum-exp of mmff.py:386-398; the vertex gradient of the combined energy goes to gcell and
// the cell's energy and virial (symmetric, from the edges) enter the block partials. A block holds
// one cell type; single-state and multistate blocks run in separate instances (kMulti), each
// launched over its own range of blocks (blk0 + blockIdx.x) when the work order allows, so that
// the single-state instance does not carry the registers of the state combination.
// kOut: kOutEnergy, kOutVirial (energy and virial, no vertex gradient) or kOutGradient (the vertex
// gradient too); the energies and virials of all three are the same bits. The latter two take the
// node positions through the pending transforms xmat (and xmat2 first, when its flag is set) when
// they are given: a barostat call whose position scaling is stored by a later node pass.
// The single-state instance sweeps the corners (sweep_cell) in 163 VGPRs, three waves a SIMD (168
// without the gradient); the multistate one keeps the stresses of all corners for the state sum
// (223 VGPRs and 72 KB of LDS a block, two waves). The compiler's default scheduler is the one that
// keeps both free of vector spills. HBM bounds the gradient pass: 469 MB at 128^3 (20% two-state,
// 5% empty) in 100 to 115 us, with 1185 / 1910 VALU instructions a wave (67 us of issue); the form
// with B = P M per corner took 1735 / 4000 and 150 us, and 120 us for the pass without
// gradient that now takes 83 us.
#define MM_CELL_PARAMS                                                                        \
  const double *__restrict__ pos, const double *__restrict__ rvecs, int64_t rvecs_stride,     \
      const int32_t *__restrict__ blk_sys, const int32_t *__restrict__ cnode,                 \
      const int32_t *__restrict__ cwrap, const int32_t *__restrict__ blk_row,                 \
      const double *__restrict__ tab_g, const double *__restrict__ kt_g,                      \
      const int32_t *__restrict__ nstates_g, int32_t max_states, int64_t W,                   \
      const int32_t *__restrict__ cbase, int64_t S, double *__restrict__ gcell,               \
      double *__restrict__ partials, int blk0, int nblocks, const double *__restrict__ xmat,  \
      const double *__restrict__ xmat2, const double *__restrict__ xmat2_on
#define MM_CELL_ARGS                                                                          \
  pos, rvecs, rvecs_stride, blk_sys, cnode, cwrap, blk_row, tab_g, kt_g, nstates_g,            \
      max_states, W, cbase, S, gcell, partials, blk0, nblocks, xmat, xmat2, xmat2_on

// The work of cell block bid (see cell_kernel).
template <int kModel, int kOut, bool kMulti>
__device__ __forceinline__ void cell_body(int bid, MM_CELL_PARAMS) {
  using F = Frame<kModel>;
  constexpr bool kVir = kOut != kOutEnergy;
  constexpr int NS = F::NE + 3 * F::NC;  // stresses of a cell
  __shared__ double red[7 * (kCellBlock / 64)];
  // running weighted sum of the states' stresses, one column a lane: [NS][kCellBlock]
  __shared__ double st_sh[(kMulti && kVir) ? NS * kCellBlock : 1];
  const int trow = blk_row[bid];
  // a block of the other kind (full-range launches only) leaves its partials to the other
  // instance
  if (kMulti != (nstates_g[trow] > 1)) return;
  const int ns = nstates_g[trow];
  const double kt = kt_g[trow];
  const const_f64 tab = (const_f64)tab_g + (int64_t)trow * max_states * kTabStride;
  const int64_t soff = blk_sys ? (int64_t)blk_sys[bid] * rvecs_stride : 0;
  const double* rvb = rvecs + soff;
  double rv[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) rv[q] = rvb[q];
  const bool on = kVir && xmat, on2 = on && xmat2 && xmat2_on[soff] != 0.0;

  const int64_t w = (int64_t)bid * kCellBlock + threadIdx.x;
  int n[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) n[k] = cnode[w * 8 + k];
  const bool valid = n[0] >= 0;
  const int wrap = valid ? cwrap[w] : 0;
  double ecell, vir[6], gacc[8][3];
  cell_eval<kModel, kOut, kMulti, kCellBlock>(
      tab, ns, kt, valid,
      [&](double (&p)[8][3]) { load_corners(pos, n, p, on, xmat + soff, on2, xmat2 + soff); },
      wrap, rv, st_sh + threadIdx.x, ecell, vir, gacc);
  if (kOut == kOutGradient) store_cell(w, wrap, valid, cbase, W, S, gcell, gacc);
  cell_wave_totals(ecell, vir, red + 7 * (threadIdx.x >> 6));
  __syncthreads();
  if (threadIdx.x < 10)
    partials[(int64_t)threadIdx.x * nblocks + bid] = cell_block_total(red, threadIdx.x);
}

template <int kModel, int kOut, bool kMulti>
__global__ void __launch_bounds__(kCellBlock, kMulti ? 2 : 3) cell_kernel(MM_CELL_PARAMS) {
  cell_body<kModel, kOut, kMulti>(blk0 + xcd_block((int)blockIdx.x, (int)gridDim.x),
                                  MM_CELL_ARGS);
}

// Both kinds of block in one launch, each block running the body of its own kind: for a pass
// that the device holds at once, where the two instances would otherwise run one after the
// other, each taking about one block's time.
template <int kModel, int kOut>
__global__ void __launch_bounds__(kCellBlock, 2) cell_kernel_both(MM_CELL_PARAMS) {
  const int bid = blk0 + xcd_block((int)blockIdx.x, (int)gridDim.x);
  if (nstates_g[blk_row[bid]] > 1)
    cell_body<kModel, kOut, true>(bid, MM_CELL_ARGS);
  else
    cell_body<kModel, kOut, false>(bid, MM_CELL_ARGS);
}
#undef MM_CELL_ARGS
#undef MM_CELL_PARAMS

// NaN-propagating maximum (the result is NaN when either operand is).
__device__ __forceinline__ double nan_max(double a, double b) {
  return (a > b || a != a) ? a : b;
}

// Block reduction of NS sums (fixed order) followed by NM NaN-propagating maxima; thread q
// writes total q to part[q * stride] (256-thread blocks).
template <int NS, int NM>
__device__ __forceinline__ void block_sum_max_store(double (&v)[NS + NM], double* part,
                                                    int64_t stride) {
  constexpr int NV = NS + NM;
  __shared__ double red[4 * NV];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const double o = __shfl_down(v[q], off, 64);
      v[q] = q < NS ? v[q] + o : nan_max(v[q], o);
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) red[wave * NV + q] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    const int q = threadIdx.x;
    double t = red[q];
    for (int w = 1; w < 4; ++w) t = q < NS ? t + red[w * NV + q] : nan_max(t, red[w * NV + q]);
    part[q * stride] = t;
  }
}

// One block of 256 threads reduces an item's src[0..n) (sum in a fixed order, or a NaN-propagating
// maximum) into dst[0] (added to it when acc). A NaN total sets the item's bit in nanflag.
__device__ __forceinline__ void reduce_item(const ReduceItem it, int* __restrict__ nanflag) {
  constexpr int kUnroll = 8;
  __shared__ double red[4];
  const bool is_max = it.op == kReduceMax;
  const double zero = is_max ? -HUGE_VAL : 0.0;
  double acc = zero;
  for (int64_t base = threadIdx.x; base < it.n; base += 256 * kUnroll) {
    double v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t i = base + (int64_t)u * 256;
      v[u] = i < it.n ? it.src[i] : zero;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) acc = is_max ? nan_max(acc, v[u]) : acc + v[u];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_down(acc, off, 64);
    acc = is_max ? nan_max(acc, o) : acc + o;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = red[0];
    for (int w = 1; w < 4; ++w) t = is_max ? nan_max(t, red[w]) : t + red[w];
    if (it.acc) t += it.dst[0];
    it.dst[0] = t;
    if (it.host) *it.host = t;
    if (t != t && it.nanbit) atomicOr(nanflag, it.nanbit);
  }
}

// One block per item.
__global__ void __launch_bounds__(256)
reduce_items_kernel(ReduceList list, int* __restrict__ nanflag) {
  reduce_item(list.item[blockIdx.x], nanflag);
}

// Per-system totals of a batch: one block per system sums its own cell blocks in list order.
__device__ __forceinline__ void batch_totals(const BatchTotals& a, int s,
                                             int* __restrict__ nanflag) {
  __shared__ double red[10 * 4];
  const double* partials = a.partials;
  const int32_t *sys_ptr = a.sys_ptr, *sys_idx = a.sys_idx;
  double *energies = a.energies, *vtens = a.vtens;
  const int nb = a.nb;
  const int b0 = sys_ptr[s], b1 = sys_ptr[s + 1];
  double acc[10];
#pragma unroll
  for (int q = 0; q < 10; ++q) acc[q] = 0.0;
  for (int i = b0 + threadIdx.x; i < b1; i += 256) {
    const int b = sys_idx[i];
#pragma unroll
    for (int q = 0; q < 10; ++q) acc[q] += partials[(int64_t)q * nb + b];
  }
  wave_reduce<10>(acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 10; ++q) red[wave * 10 + q] = acc[q];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int bad = 0;
    for (int q = 0; q < 10; ++q) {
      const double t = ((red[q] + red[10 + q]) + red[20 + q]) + red[30 + q];
      if (t != t) bad |= q == 0 ? 1 : 4;
      if (q == 0 && energies) energies[s] = t;
      if (q > 0 && vtens) vtens[9 * (int64_t)s + q - 1] = t;
    }
    if (bad) atomicOr(nanflag, bad);
  }
}

__global__ void __launch_bounds__(256)
batch_totals_kernel(BatchTotals a, int* __restrict__ nanflag) {
  batch_totals(a, blockIdx.x, nanflag);
}

// gpos[n] (+)= sum_{k=0..7} gcell[k][:][w(n,k)] in fixed k order (mmff.py:303-318). A workgroup
// owns 256 consecutive nodes; their 768 gpos values (and, with DOT, dir and gold values) move
// between HBM and LDS in contiguous runs, and each thread takes its node's three from LDS. With
// DOT (a line-search trial), also the workgroup partials of sum_n gpos_n . dir_n,
// sum_n |gpos_n|^2, sum_n gpos_n . gold_n and max_n |gpos_n|^2 into dpart rows 0-3 (row stride =
// workgroups). The launch's blocks from gb on reduce an item of the cell pass's partials each
// (energy and virial), beside the gather: a launch less than a reduction behind it (72x80x96
// 79.3 -> 75.0 us).
template <bool DOT, bool kAllLoads>
__global__ void __launch_bounds__(256)
gather_kernel(const int32_t* __restrict__ ncell, const double* __restrict__ gcell, int64_t N,
              int64_t RS, double* __restrict__ gpos, int accumulate, int* __restrict__ nanflag,
              const double* __restrict__ dir, const double* __restrict__ gold,
              double* __restrict__ dpart, int gb, ReduceList list, BatchTotals batch) {
  if (!DOT && (int)blockIdx.x >= gb) {
    const int i = (int)blockIdx.x - gb;
    if (i < list.count)
      reduce_item(list.item[i], nanflag);
    else
      batch_totals(batch, i - list.count, nanflag);
    return;
  }
  __shared__ double sg[768];
  __shared__ double sd[DOT ? 768 : 1], so[DOT ? 768 : 1];
  const int t = threadIdx.x;
  // node blocks dealt to the XCDs in contiguous ranges: neighbouring blocks share record lines
  const int blk = xcd_block((int)blockIdx.x, gb);
  const int64_t n0 = (int64_t)blk * 256, n = n0 + t;
  const int64_t e0 = 3 * n0;
  const int64_t ne = 3 * (N < n0 + 256 ? N - n0 : (int64_t)256);  // values of this workgroup
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int li = r * 256 + t;
    if (li < ne) {
      if (accumulate) sg[li] = gpos[e0 + li];
      if (DOT) {
        sd[li] = dir[e0 + li];
        so[li] = gold[e0 + li];
      }
    }
  }
  double g[3] = {0.0, 0.0, 0.0};
  if (n < N) sum_node_records<kAllLoads>(ncell, gcell, N, RS, n, g);
  __syncthreads();
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (n < N) {
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      bad |= (g[j] != g[j]);
      const double v = accumulate ? sg[3 * t + j] + g[j] : g[j];
      sg[3 * t + j] = v;
      if (DOT) {
        acc[0] += v * sd[3 * t + j];
        acc[1] += v * v;
        acc[2] += v * so[3 * t + j];
      }
    }
    acc[3] = acc[1];
    if (bad) atomicOr(nanflag, 2);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int li = r * 256 + t;
    if (li < ne) gpos[e0 + li] = sg[li];
  }
  if (DOT) block_sum_max_store<3, 1>(acc, dpart + blk, gb);
}

hipError_t launch_cells(const ForceArgs& a, hipStream_t stream) {
  const int nb = (int)(a.W / kCellBlock);
  const int out = (a.gpos != nullptr || a.force_grad) && a.store_records ? kOutGradient
                  : a.vtens != nullptr || a.force_grad                     ? kOutVirial
                                                                           : kOutEnergy;
  if (nb == 0) return hipSuccess;
  // Multistate blocks [0, split), single-state blocks [split, nb) when the work order is so
  // partitioned (split >= 0); otherwise both instances cover every block.
  const bool part = a.split >= 0;
  const int m0 = 0, mn = part ? a.split : nb;
  const int s0 = part ? a.split : 0, sn = part ? nb - a.split : nb;
  // The second instance runs on the side stream, concurrently with the first, when the pass
  // has more cell blocks than the device holds at once (256 CUs x 2 blocks of 256 lanes at two
  // waves a SIMD). A smaller pass takes the time of one block per instance, less than the fork
  // and join cost: it runs both kinds of block in one launch (cell_kernel_both). NVT-NHC step, NPT
  // step and evaluation, one launch / fork, a fifth of the cells two-state: 32^3 (122 blocks) 34 / 43,
  // 67 / 79 and 16 / 45 us, 48^3 (410) 48 / 53, 92 / 100 and 21 / 46 us; above the line 56^3 (652)
  // 64 / 64, 130 / 140 and 29 / 46 us, 64^3 (974) 73 / 74, 155 / 162 and 38 / 48 us, 72^3 (1385)
  // 88 / 83, 188 / 187 and 52 / 57 us, 80^3 (1900) 104 / 98, 219 / 206 and 65 / 67 us, 96^3 154 / 140,
  // 330 / 293 and 104 / 101 us, 128^3 310 / 279, 675 / 564 and 224 / 202 us: between 512 and some
  // 1000 blocks one launch would still be the faster in NPT and single evaluations.
  // The averaged model's kernels are short in either kind and the
  // device holds twice as many, so that the fork pays later: one launch against two, a fifth of
  // the cells two-state, whole evaluation of 61x64x67 (1022 blocks) 27 / 50 us, 96^3 88 / 94,
  // 104^3 108 / 115, 112^3 136 / 136, 128^3 197 / 197, 160^3 419 / 396 (with seven of ten cells
  // two-state 85 / 98, 101 / 112, 130 / 139, 188 / 199, 416 / 412); NVT-NHC step, where a graph's
  // fork costs less, 64^3 64 / 68, 96^3 137 / 132, 104^3 168 / 164, 112^3 199 / 188, 128^3 285 / 277;
  // NPT 123 / 147, 265 / 263, 328 / 320, 385 / 365, 549 / 522. The results are the same bits in
  // every form.
  const int one = a.model == 0 ? kForkMinBlocks : kForkMinBlocksAveraged;
  const bool fork = a.side != nullptr && a.ev_fork != nullptr && a.ev_join != nullptr &&
                    mn > 0 && sn > 0 && nb > one;
  hipStream_t ms = fork ? a.side : stream;
  hipError_t e = hipSuccess;
  if (fork) {
    e = hipEventRecord(a.ev_fork, stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(a.side, a.ev_fork, 0);
    if (e != hipSuccess) return e;
  }
#define MM_LAUNCH_CELL(MODEL, OUT, MULTI, S, B0, NBL)                                        \
  hipLaunchKernelGGL((cell_kernel<MODEL, OUT, MULTI>), dim3(NBL), dim3(kCellBlock), 0, S,       \
                     a.pos, a.rvecs, a.rvecs_stride, a.blk_sys, a.cnode, a.cwrap, a.blk_row, \
                     a.tab, a.kt, a.nstates, a.max_states, a.W, a.cbase, a.rstride, a.gcell,  \
                     a.partials, B0, nb, a.xmat, a.xmat2, a.xmat2_on)
  // pending position transforms: xmat with every use, xmat2 with its flag, and not for the
  // energy alone
  if ((a.xmat2 != nullptr) != (a.xmat2_on != nullptr)) return hipErrorInvalidValue;
  if (a.xmat2 != nullptr && a.xmat == nullptr) return hipErrorInvalidValue;
  if (a.xmat != nullptr && out == kOutEnergy) return hipErrorInvalidValue;
  // The multistate instance is launched first, on the caller's stream: its blocks hold twice the
  // time and 74 KB of LDS each, and started behind the single-state instance they find their
  // place only as that drains (npt 128^3 step 0.580 -> 0.576 ms; equal at 72x80x96 with seven
  // of ten cells two-state). Passes of few blocks of both kinds: one launch.
  const bool both = mn > 0 && sn > 0 && nb <= one;
#define MM_LAUNCH_BOTH(MODEL, OUT)                                                           \
  hipLaunchKernelGGL((cell_kernel_both<MODEL, OUT>), dim3(nb), dim3(kCellBlock), 0, stream,     \
                     a.pos, a.rvecs, a.rvecs_stride, a.blk_sys, a.cnode, a.cwrap,              \
                     a.blk_row, a.tab, a.kt, a.nstates, a.max_states, a.W, a.cbase, a.rstride, \
                     a.gcell, a.partials, 0, nb, a.xmat, a.xmat2, a.xmat2_on)
#define MM_LAUNCH_PAIR(MODEL, OUT)                                                           \
  do {                                                                                       \
    if (both) {                                                                              \
      MM_LAUNCH_BOTH(MODEL, OUT);                                                            \
    } else {                                                                                 \
      if (mn > 0) MM_LAUNCH_CELL(MODEL, OUT, true, stream, m0, mn);                         \
      if (sn > 0) MM_LAUNCH_CELL(MODEL, OUT, false, ms, s0, sn);                            \
    }                                                                                        \
  } while (0)
#define MM_LAUNCH_MODEL(MODEL)                                                                \
  do {                                                                                        \
    if (out == kOutGradient) MM_LAUNCH_PAIR(MODEL, kOutGradient);                            \
    else if (out == kOutVirial) MM_LAUNCH_PAIR(MODEL, kOutVirial);                           \
    else MM_LAUNCH_PAIR(MODEL, kOutEnergy);                                                  \
  } while (0)
  if (a.model == 0) MM_LAUNCH_MODEL(0); else MM_LAUNCH_MODEL(1);
#undef MM_LAUNCH_MODEL
#undef MM_LAUNCH_PAIR
#undef MM_LAUNCH_BOTH
#undef MM_LAUNCH_CELL
  e = hipGetLastError();
  if (e == hipSuccess && fork) {
    e = hipEventRecord(a.ev_join, a.side);
    if (e == hipSuccess) e = hipStreamWaitEvent(stream, a.ev_join, 0);
  }
  return e;
}

template <bool DOT>
static hipError_t gather(const ForceArgs& a, const double* dir, const double* gold, double* dpart,
                         const ReduceList& list, const BatchTotals& batch, hipStream_t stream) {
  const int gb = (int)((a.N + 255) / 256);
  const dim3 grid(gb + list.count + batch.nsys);
  if (gb <= kGatherAllLoadsMaxBlocks)
    hipLaunchKernelGGL((gather_kernel<DOT, true>), grid, dim3(256), 0, stream, a.ncell, a.gcell,
                       a.N, a.rstride, a.gpos, a.accumulate, a.nanflag, dir, gold, dpart, gb, list,
                       batch);
  else
    hipLaunchKernelGGL((gather_kernel<DOT, false>), grid, dim3(256), 0, stream, a.ncell, a.gcell,
                       a.N, a.rstride, a.gpos, a.accumulate, a.nanflag, dir, gold, dpart, gb, list,
                       batch);
  return hipGetLastError();
}

static bool no_gather(const ForceArgs& a) { return a.gpos == nullptr || a.N <= 0 || a.W <= 0; }

hipError_t launch_gather(const ForceArgs& a, const ReduceList& list, hipStream_t stream) {
  if (no_gather(a)) return launch_reduce(list, a.nanflag, stream);
  return gather<false>(a, nullptr, nullptr, nullptr, list, BatchTotals{}, stream);
}

hipError_t launch_gather_batch(const ForceArgs& a, const BatchTotals& batch, hipStream_t stream) {
  if (!no_gather(a))
    return gather<false>(a, nullptr, nullptr, nullptr, ReduceList{}, batch, stream);
  if (batch.nsys <= 0) return hipSuccess;
  hipLaunchKernelGGL(batch_totals_kernel, dim3(batch.nsys), dim3(256), 0, stream, batch,
                     a.nanflag);
  return hipGetLastError();
}

hipError_t launch_gather_dot(const ForceArgs& a, const double* dir, const double* gold,
                             double* dpart, hipStream_t stream) {
  if (no_gather(a)) return hipSuccess;
  return gather<true>(a, dir, gold, dpart, ReduceList{}, BatchTotals{}, stream);
}

hipError_t launch_reduce(const ReduceList& list, int* nanflag, hipStream_t stream) {
  if (list.count <= 0) return hipSuccess;
  hipLaunchKernelGGL(reduce_items_kernel, dim3(list.count), dim3(256), 0, stream, list, nanflag);
  return hipGetLastError();
}

void add_force_totals(ReduceList& list, const ForceArgs& a, int nb) {
  if (a.energy) list.add(a.partials, nb, kReduceSum, a.energy, a.accumulate, 1);
  if (a.vtens)
    for (int q = 0; q < 9; ++q)
      list.add(a.partials + (int64_t)(1 + q) * nb, nb, kReduceSum, a.vtens + q, a.accumulate, 4);
}

// One force evaluation in one launch by one workgroup, for a field of at most kSmallForce work
// slots and nodes: three launches (cells, gather, totals) and the trips to memory between them take
// longer than its arithmetic. Thread t owns slot t and node t; positions, stresses or vertex
// records and the wave sums stay in LDS (a slot's column holds its multistate sums, then its
// records: lower faces in rows 0..11, upper in 12..23). pos, rvecs and the outputs may be host
// memory that the device maps: every word of it is read and written once, side by side. Same
// arithmetic and order of sums as the separate kernels, so the same bits. The limit is what LDS
// holds: 36 columns of 512 sums are 144 of its 160 KB. 5^3 cells from host arrays, whole plugin
// call: 111 us with three launches and five waiting copies, 44 us so (some 20 us of it Python).
struct ForceSmallArgs {
  const double *pos, *rvecs;
  const int32_t *cnode, *cwrap, *blk_row, *nstates, *nrec, *cbase;
  const double *tab, *kt;
  int32_t max_states;
  int W, N;
  double *energy, *gpos, *vtens;
  int accumulate;
  int* nanflag;
};

template <int kModel, int kOut>
__global__ void __launch_bounds__(kSmallForce, 2) force_small_kernel(ForceSmallArgs a) {
  using F = Frame<kModel>;
  constexpr int NS = F::NE + 3 * F::NC;
  constexpr int NR = NS > 24 ? NS : 24;
  constexpr int kWaves = kSmallForce / 64;
  __shared__ double col[NR * kSmallForce];
  __shared__ double xs[3 * kSmallForce];
  __shared__ double rvs[9];
  __shared__ double red[7 * kWaves];  // zero where no wave writes
  unsigned short* top_slot = reinterpret_cast<unsigned short*>(col);  // before the cells only
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  for (int i = t; i < 3 * a.N; i += blockDim.x) xs[i] = a.pos[i];
  if (t < 9) rvs[t] = a.rvecs[t];
  if (t < 7 * kWaves) red[t] = 0.0;
  const bool has_slot = 64 * wave < a.W;  // W is a multiple of the block size
  int n[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) n[k] = has_slot ? a.cnode[8 * t + k] : -1;
  const bool valid = n[0] >= 0;
  const int wrap = valid ? a.cwrap[t] : 0;
  const int trow = has_slot ? ((const_i32)a.blk_row)[wave >> 2] : 0;
  const int ns = ((const_i32)a.nstates)[trow];
  const double kt = ((const_f64)a.kt)[trow];
  const const_f64 tab = (const_f64)a.tab + (int64_t)trow * a.max_states * kTabStride;
  {
    const bool open_top = valid && !(wrap & 16);
    const uint64_t tops = __ballot(open_top);
    if (open_top) top_slot[((const_i32)a.cbase)[wave] + __popcll(tops & ((1ull << lane) - 1ull))] = t;
  }
  __syncthreads();
  // the node's records as places in col, -1 for none
  const bool own = kOut == kOutGradient && t < a.N;
  int place[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int e = own ? a.nrec[k * a.N + t] : -1;
    const int slot = e >> 2, row = 3 * (e & 3);
    place[k] = e < 0 ? -1
                     : slot < a.W ? row * kSmallForce + slot
                                  : (12 + row) * kSmallForce + top_slot[slot - a.W];
  }
  __syncthreads();
  if (has_slot) {
    double rv[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) rv[q] = rvs[q];
    double ecell, vir[6], gacc[8][3];
    auto corners = [&](double (&p)[8][3]) {
      load_corners(xs, n, p, false, nullptr, false, nullptr);
    };
    if (ns > 1)
      cell_eval<kModel, kOut, true, kSmallForce>(tab, ns, kt, valid, corners, wrap, rv, col + t,
                                                 ecell, vir, gacc);
    else
      cell_eval<kModel, kOut, false, kSmallForce>(tab, ns, kt, valid, corners, wrap, rv, col + t,
                                                  ecell, vir, gacc);
    if (kOut == kOutGradient) {
      fold_cell(wrap, gacc);
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          col[(3 * q + j) * kSmallForce + t] = gacc[kLowerCorner[q]][j];
          col[(12 + 3 * q + j) * kSmallForce + t] = gacc[kUpperCorner[q]][j];
        }
    }
    cell_wave_totals(ecell, vir, red + 7 * wave);
  }
  __syncthreads();
  if (t < 10) {
    // the totals of the slots' blocks, in block order
    double s = cell_block_total(red, t);
    for (int b = 1; b < a.W / kCellBlock; ++b)
      s += cell_block_total(red + 7 * b * (kCellBlock / 64), t);
    double* dst = t == 0 ? a.energy : a.vtens ? a.vtens + (t - 1) : nullptr;
    if (dst) {
      if (a.accumulate) s += *dst;
      *dst = s;
      if (s != s) atomicOr(a.nanflag, t == 0 ? 1 : 4);
    }
  }
  if (own) {
    double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (place[k] >= 0) g[j] += col[place[k] + j * kSmallForce];
    if (g[0] != g[0] || g[1] != g[1] || g[2] != g[2]) atomicOr(a.nanflag, 2);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double* dst = a.gpos + 3 * t + j;
      *dst = a.accumulate ? *dst + g[j] : g[j];
    }
  }
}

static hipError_t launch_force_small(const ForceArgs& a, hipStream_t stream) {
  const ForceSmallArgs s{a.pos, a.rvecs, a.cnode, a.cwrap, a.blk_row, a.nstates, a.ncell,
                         a.cbase, a.tab, a.kt, a.max_states, (int)a.W, (int)a.N, a.energy,
                         a.gpos, a.vtens, a.accumulate, a.nanflag};
  const dim3 block(a.W > kSmallForce / 2 || a.N > kSmallForce / 2 ? kSmallForce : kSmallForce / 2);
#define MM_SMALL(M, O) hipLaunchKernelGGL((force_small_kernel<M, O>), dim3(1), block, 0, stream, s)
  if (a.model == 0) {
    if (a.gpos) MM_SMALL(0, kOutGradient); else MM_SMALL(0, kOutVirial);
  } else {
    if (a.gpos) MM_SMALL(1, kOutGradient); else MM_SMALL(1, kOutVirial);
  }
#undef MM_SMALL
  return hipGetLastError();
}

hipError_t launch_force(const ForceArgs& a, hipStream_t stream) {
  if (a.energy && a.N > 0 && a.N <= kSmallForce && a.W > 0 && a.W <= kSmallForce)
    return launch_force_small(a, stream);
  hipError_t err = launch_cells(a, stream);
  if (err != hipSuccess) return err;
  ReduceList list;
  add_force_totals(list, a, (int)(a.W / kCellBlock));
  return launch_gather(a, list, stream);
}

// Inputs of a host call from mapped host memory into device buffers.
__global__ void __launch_bounds__(256)
stage_kernel(const double* __restrict__ src, double* __restrict__ dst, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

hipError_t launch_stage(const double* src, double* dst, int64_t n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(stage_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, src,
                     dst, n);
  return hipGetLastError();
}

// Trial point of a line search over 256 nodes a workgroup: optionally d <- beta d - g first,
// then xa <- x + alpha d, in contiguous runs of the workgroup's 768 values; the squared
// displacements go through LDS to the node threads for the workgroup partials of
// sum_n |xa_n - x_n|^2 and max_n |xa_n - x_n|^2 (part rows 0-1, row stride = workgroups).
__global__ void __launch_bounds__(256)
cg_trial_kernel(const double* __restrict__ x, const double* __restrict__ g,
                double* __restrict__ d, double beta, int set_dir, double alpha,
                double* __restrict__ xa, int64_t N, double* __restrict__ part) {
  __shared__ double dx2[768];
  const int t = threadIdx.x;
  const int64_t n0 = (int64_t)blockIdx.x * 256;
  const int64_t e0 = 3 * n0;
  const int64_t ne = 3 * (N < n0 + 256 ? N - n0 : (int64_t)256);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int li = r * 256 + t;
    double v = 0.0;
    if (li < ne) {
      const int64_t i = e0 + li;
      double di;
      if (set_dir) {
        di = beta != 0.0 ? beta * d[i] - g[i] : -g[i];  // beta = 0: d is not read
        d[i] = di;
      } else {
        di = d[i];
      }
      const double xi = x[i];
      const double xn = xi + alpha * di;
      xa[i] = xn;
      const double dx = xn - xi;
      v = dx * dx;
    }
    dx2[li] = v;
  }
  __syncthreads();
  double acc[2];
  acc[0] = (dx2[3 * t] + dx2[3 * t + 1]) + dx2[3 * t + 2];
  acc[1] = acc[0];
  block_sum_max_store<1, 1>(acc, part + blockIdx.x, gridDim.x);
}

hipError_t launch_cg_trial(const double* x, const double* g, double* d, double beta, int set_dir,
                           double alpha, double* xa, int64_t N, double* part,
                           hipStream_t stream) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(cg_trial_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream,
                     x, g, d, beta, set_dir, alpha, xa, N, part);
  return hipGetLastError();
}

// Per-block partials over the nodes n of |g_n|^2, g_n . go_n, |x_n - xo_n|^2 (sums, rows 0-2)
// and of |g_n|^2, |x_n - xo_n|^2 (maxima, rows 3-4); part is [5][nb].
__global__ void __launch_bounds__(256)
cg_stats_kernel(const double* __restrict__ x, const double* __restrict__ xo,
                const double* __restrict__ g, const double* __restrict__ go, int64_t N,
                double* __restrict__ part) {
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (n < N) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double gj = g[3 * n + j], dj = x[3 * n + j] - xo[3 * n + j];
      v[0] += gj * gj;
      v[1] += gj * go[3 * n + j];
      v[2] += dj * dj;
    }
    v[3] = v[0];
    v[4] = v[2];
  }
  block_sum_max_store<3, 2>(v, part + blockIdx.x, gridDim.x);
}

hipError_t launch_cg_stats(const double* x, const double* xo, const double* g, const double* go,
                           int64_t N, double* part, double* out, double* host, int* nanflag,
                           hipStream_t stream) {
  if (N <= 0) return hipSuccess;
  const int nb = (int)((N + 255) / 256);
  hipLaunchKernelGGL(cg_stats_kernel, dim3(nb), dim3(256), 0, stream, x, xo, g, go, N, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ReduceList list;
  for (int q = 0; q < 5; ++q)
    list.add(part + (int64_t)q * nb, nb, q < 3 ? kReduceSum : kReduceMax, out + q, 0, 0,
             host ? host + q : nullptr);
  return launch_reduce(list, nanflag, stream);
}

// Parameter table entries (row t, state s) from device arrays, one wave per entry and one lane per
// matrix element, with the arithmetic of the host builder (Voigt input, metric_entry), so both give
// the same bits; entries of states beyond nstates[t] are zero. kt[t] = boltzmann * temp_eff[t]. A
// serial chain bounds it, the inverse and its residual above all: 5.9 to 6.7 us; one thread per entry,
// without the residual, took 6.5 us.
__global__ void __launch_bounds__(64)
build_table_kernel(int corner8, int max_states, const int32_t* __restrict__ nstates,
                   const double* __restrict__ h0, const double* __restrict__ cv,
                   const double* __restrict__ free_energy, const double* __restrict__ temp_eff,
                   double boltzmann, double* __restrict__ tab, double* __restrict__ kt) {
#pragma clang fp contract(off)
  // of this state and of the type's first one: rest cell, inverse, its residual, rest metric
  __shared__ double H[2][9], P[2][9], E[2][9], R[2][6], low[2][6];
  __shared__ double T[36], CT[36], C[36], W;
  const int ts = blockIdx.x, q = threadIdx.x;
  const int t = ts / max_states, s = ts % max_states;
  double* e = tab + (int64_t)ts * kTabStride;
  if (s == 0 && q == 0) kt[t] = boltzmann * temp_eff[t];
  if (s >= nstates[t]) {
    for (int i = q; i < kTabStride; i += 64) e[i] = 0.0;
    return;
  }
  if (q < 36) C[q] = cv[(int64_t)ts * 36 + q];
  if (q < 18) H[q / 9][q % 9] = h0[(int64_t)(q < 9 ? ts : t * max_states) * 9 + q % 9];
  __syncthreads();
  if (q < 2) {
    double inv[9];
    const double det = inverse3_cof(H[q], inv);
    if (q == 0) W = corner8 ? 0.125 * det : det;
    for (int i = 0; i < 9; ++i) P[q][i] = inv[i];
  }
  __syncthreads();
  if (q < 36) {
    T[q] = strain_map(P[0], q / 6, q % 6);
    e[kCvOffset + q] = C[q];
  }
  if (q < 18) E[q / 9][q % 9] = inverse_residual(P[q / 9], H[q / 9], q % 9);
  if (q < 9) e[q] = P[0][q];
  if (q == 9) e[9] = W;
  if (q == 10) e[10] = free_energy[ts];
  if (q == 11) e[11] = 0.0;
  __syncthreads();
  if (q < 12) R[q / 6][q % 6] = rest_entry(H[q / 6], E[q / 6], q % 6, low[q / 6][q % 6]);
  __syncthreads();
  if (q < 6) {
    e[kRestOffset + q] = R[0][q];
    e[kRestLowOffset + q] = low[0][q];
  }
  if (q < 8)
    e[kShiftOffset + q] = q < 3 ? rest_shift(R[1][q], low[1][q], R[0][q], low[0][q]) : 0.0;
  __syncthreads();
  if (q < 36) CT[q] = stiffness_half(W, C, T, q / 6, q % 6);
  __syncthreads();
  if (q < 36) e[kMetricOffset + q] = stiffness_entry(T, CT, q / 6, q % 6);
}

hipError_t launch_build_table(int corner8, int nrows, int max_states, const int32_t* nstates,
                              const double* h0, const double* cv, const double* free_energy,
                              const double* temp_eff, double boltzmann, double* tab, double* kt,
                              hipStream_t stream) {
  const int n = nrows * max_states;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(build_table_kernel, dim3(n), dim3(64), 0, stream, corner8, max_states,
                     nstates, h0, cv, free_energy, temp_eff, boltzmann, tab, kt);
  return hipGetLastError();
}

}  // namespace mm
