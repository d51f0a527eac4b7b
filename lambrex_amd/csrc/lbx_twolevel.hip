// lbx_twolevel.hip -- device kernels of the two-level Rohde cycle
// (src/AmrSim.cpp:430-631) on gfx950, FP64 or FP32-shifted storage.
//
// Storage.  The coarse level is a periodic level array (lbx_lattice.hip).
// Each fine box is a patch of its own, grown by 2 ghost layers like the
// reference's FABs (population-major, x fastest, per-patch population
// stride).  The fine ghosts must be separate per box because the reference
// lets them go stale between the two fine substeps (they are filled once per
// coarse step and never collided), so a cell seen as a ghost by one box and
// as valid by its neighbour evolves differently in the two places.
//
// One coarse step at refinement ratio 2, in the reference's order of effects:
//   k_fine_step           both fine substeps (FillPatchTwoLevels, collide,
//                         Stream(1), collide, Stream(1),
//                         ZeroInvalidComponents) in one pass from the current
//                         state to the next, with the 1/8 weighted sum of
//                         every 2x2x2 block of the result
//   k_coarse_push         CoarseCollide(0) (masked cells -> 0) + Stream(0) in
//                         push form; pulls across a box face read the
//                         pre-collision ghost copies, as the reference's
//                         RohdeCycle does (no FillBoundary between collide and
//                         stream)
//   k_sum_apply           SumFromFine(0): ADD those block averages (fine valid
//                         + ghosts) into coarse next, contributions to one
//                         coarse cell in a fixed order
// Only valid cells are stored, packed (PatchDesc): the ghosts live in the pass.
//
// Deeper hierarchies (RohdeCycle's recursion, src/AmrSim.cpp:453-455) run the
// same kernel on patched "middle" levels, which have both a parent and a
// child: one step of them, with the cells under the child's mask zeroed
// (MASK) and the child's block averages added into the valid cells (SUM).
//
// At ratios above 2 (r substeps, no fine ghosts in the average-down) a level's
// patches are stored grown and a step is one pass per substep:
// k_fine_fill_collide, k_fine_stream_collide, then k_fine_stream_valid and
// k_fine_avg_valid on the finest level, k_fine_stream_zero on a middle one.
//
// Storage type S is double (FP64, bit-exact with the oracle) or float (the
// shifted deviation d = f - w rho0 of the FP32 path).  Either way the block
// sums and the coarse additions of SumFromFine are done in FP64 on
// reconstructed f, and a population set to zero means f = 0 (d = -w rho0).
#include <hip/hip_runtime.h>

#include "d3q15.h"
#include "lbx_internal.h"

#pragma clang fp contract(off)

namespace lbx {
namespace {

// f of a stored value, and the stored value of f, for population q.
template <typename S>
__device__ __forceinline__ double to_f64(S v, int q, double rho0) {
  if constexpr (sizeof(S) == 8)
    return v;
  else
    return kT.W[q] * rho0 + double(v);
}

template <typename S>
__device__ __forceinline__ S from_f64(double f, int q, double rho0) {
  if constexpr (sizeof(S) == 8)
    return f;
  else
    return float(f - kT.W[q] * rho0);
}

// The stored value of f_q = 0.
template <typename S>
__device__ __forceinline__ S zero_pop(int q, double rho0) {
  return from_f64<S>(0.0, q, rho0);
}

template <typename S>
__device__ __forceinline__ void collide_s(S* f, const Relax& r) {
  if constexpr (sizeof(S) == 8)
    collide_f64(f, r.omega_s, r.omega_b);
  else
    collide_f32_shifted(f, float(r.rho0), float(r.omega_s), float(r.omega_b));
}

// n / d for 0 <= n < 2^22 and d >= 1: the float estimate from the hardware
// reciprocal (relative error below 2^-22 with the product's rounding) is
// off by less than one, and one correction makes it exact.
__device__ __forceinline__ int div_small(int n, int d) {
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)d));
  const int r = n - q * d;
  q += (r >= d) - (r < 0);
  return q;
}

// Chunk of its patch handled by this workgroup.  Workgroups go to the 8
// XCDs round-robin by linear id; with gridDim.x a multiple of 8, XCD k takes
// chunks [k G/8, (k+1) G/8) of every patch (G = gridDim.x): a contiguous
// slab, so neighbouring chunks, and the same rows of neighbouring patches,
// share that XCD's L2.  The identity for any other grid.
__device__ __forceinline__ int xcd_chunk() {
  const int G = gridDim.x, c = blockIdx.x;
  return (G & 7) ? c : (c & 7) * (G >> 3) + (c >> 3);
}

// (x, y, z) of index i < n of a box with rows of n0 and planes of n1 rows;
// n is uniform over the workgroup, so the branch is too.
__device__ __forceinline__ void split3(int i, int n, int n0, int n1, int& x, int& y, int& z) {
  if (n <= (1 << 22)) {
    const int t = div_small(i, n0);
    x = i - t * n0;
    z = div_small(t, n1);
    y = t - z * n1;
  } else {
    x = i % n0;
    const int t = i / n0;
    y = t % n1;
    z = t / n1;
  }
}

__device__ __forceinline__ void patch_coords(const PatchDesc& P, int i, int& gx, int& gy, int& gz) {
  split3(i, P.cells, P.g[0], P.g[1], gx, gy, gz);
}

__device__ __forceinline__ bool patch_valid(const PatchDesc& P, int gx, int gy, int gz) {
  return gx >= 2 && gx < P.g[0] - 2 && gy >= 2 && gy < P.g[1] - 2 && gz >= 2 && gz < P.g[2] - 2;
}

__device__ __forceinline__ bool patch_outer(const PatchDesc& P, int gx, int gy, int gz) {
  return gx == 0 || gy == 0 || gz == 0 || gx == P.g[0] - 1 || gy == P.g[1] - 1 || gz == P.g[2] - 1;
}

// Collide of a level at a ratio above 2.  Every lane first picks where its 15 populations come from (its own valid
// cell, the fine valid cell holding its periodic image, or the coarse
// parent) so the loads of valid and ghost lanes issue together; valid cells
// are then collided.  Coarse sources are -1 - (element of population 0) in
// a level array, or with PC -1 - ((coarse patch << 32) | grown index).  With
// MASK, a valid cell whose mask byte is set is zeroed instead of collided
// (CoarseCollide on a level that has a finer one, src/AmrSim.cpp:499-500).
// The patch is own[first + blockIdx.y] (`own` lists the level's patches in
// launch order); `patches` is the level's table by box index, which the
// fill sources refer to.
template <typename S, bool PC, bool MASK>
__global__ __launch_bounds__(256) void k_fine_fill_collide(
    const S* __restrict__ fnow, S* __restrict__ fnext, const S* __restrict__ cnow, Lattice clat,
    const PatchDesc* __restrict__ cpatches, const PatchDesc* __restrict__ patches,
    const PatchDesc* __restrict__ own, int first, const long long* __restrict__ fill,
    const unsigned char* __restrict__ mask, Relax r) {
  // P is read in place: with a by-value copy the PC variants merged the
  // loads of base / qs from P, patches[s] and cpatches[] into one load through
  // a selected pointer, which kept the copy in 80 B of scratch per lane.
  const PatchDesc& P = own[first + blockIdx.y];
  const int i = xcd_chunk() * 256 + threadIdx.x;
  if (i >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  const bool valid = patch_valid(P, gx, gy, gz);
  const S* src;
  long long stride;
  if (valid) {
    src = fnow + P.base + i;
    stride = P.qs;
  } else {
    const long long d = fill[P.fill_base + i];
    if (d >= 0) {
      const int s = int(d >> 32);
      src = fnow + patches[s].base + (d & 0xffffffffll);
      stride = patches[s].qs;
    } else if constexpr (PC) {
      const long long e = -1 - d;
      const PatchDesc& CP = cpatches[e >> 32];
      src = cnow + CP.base + (e & 0xffffffffll);
      stride = CP.qs;
    } else {
      src = cnow + (-1 - d);  // coarse element of population 0
      stride = clat.ps;
    }
  }
  S f[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) f[q] = src[q * stride];
  if (valid) {
    if (MASK && mask[P.fill_base + i]) {
#pragma unroll
      for (int q = 0; q < NV; ++q) f[q] = zero_pop<S>(q, r.rho0);
    } else {
      collide_s(f, r);
    }
  } else if (patch_outer(P, gx, gy, gz)) {
    f[0] = zero_pop<S>(0, r.rho0);
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) fnext[P.base + q * P.qs + i] = f[q];
}

// Pull of grown cell i over valid + 1 ghost layer, from the patch stored at
// element `base` of `in`; the outer ghost layer of the fresh array is
// defined as zero.  Returns whether i is a valid cell.
template <typename S>
__device__ __forceinline__ bool fine_pull(const PatchDesc& P, const S* __restrict__ in, long long base, int i,
                                          int gx, int gy, int gz, double rho0, S* f) {
  if (patch_outer(P, gx, gy, gz)) {
#pragma unroll
    for (int q = 0; q < NV; ++q) f[q] = zero_pop<S>(q, rho0);
    return false;
  }
  const int sx = 1, sy = P.g[0], sz = P.g[0] * P.g[1];
#pragma unroll
  for (int q = 0; q < NV; ++q) f[q] = in[base + q * P.qs + i - kC[q][0] * sx - kC[q][1] * sy - kC[q][2] * sz];
  return patch_valid(P, gx, gy, gz);
}

// fine_pull for an input whose outer ghost layer is not stored (the first
// substep's output, k_fine_stream_collide): a population whose upstream cell
// lies on the outer layer takes that layer's defined value, zero, without
// reading that layer.
template <typename S>
__device__ __forceinline__ bool fine_pull_inner(const PatchDesc& P, const S* __restrict__ in, long long base,
                                                int i, int gx, int gy, int gz, double rho0, S* f) {
  if (patch_outer(P, gx, gy, gz)) {
#pragma unroll
    for (int q = 0; q < NV; ++q) f[q] = zero_pop<S>(q, rho0);
    return false;
  }
  const int sx = 1, sy = P.g[0], sz = P.g[0] * P.g[1];
  // One load per population for every lane (a wave holds valid and ghost
  // cells alike): a lane whose upstream cell is on the outer layer (never
  // the case for a valid cell) loads its own cell instead and keeps zero.
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const bool outer = patch_outer(P, gx - kC[q][0], gy - kC[q][1], gz - kC[q][2]);
    const int off = outer ? 0 : kC[q][0] * sx + kC[q][1] * sy + kC[q][2] * sz;
    const S v = in[base + q * P.qs + i - off];
    f[q] = outer ? zero_pop<S>(q, rho0) : v;
  }
  return patch_valid(P, gx, gy, gz);
}

// A fine substep's stream + the next one's collision (refinement ratios above
// 2): pull, then collide valid cells.  The outer ghost layer of the result is
// zero by definition (Stream's fresh array) and is not stored: the next pass
// reads it as zero.  With INNER the input is itself such a result (a later
// substep), whose outer layer is read as zero.
template <typename S, bool INNER = false>
__global__ __launch_bounds__(256) void k_fine_stream_collide(const S* __restrict__ in, S* __restrict__ out,
                                                             const PatchDesc* __restrict__ patches, int first,
                                                             Relax r) {
  const PatchDesc P = patches[first + blockIdx.y];
  const int i = xcd_chunk() * 256 + threadIdx.x;
  if (i >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  if (patch_outer(P, gx, gy, gz)) return;
  S f[NV];
  const bool valid = INNER ? fine_pull_inner(P, in, P.base, i, gx, gy, gz, r.rho0, f)
                           : fine_pull(P, in, P.base, i, gx, gy, gz, r.rho0, f);
  if (valid) collide_s(f, r);
#pragma unroll
  for (int q = 0; q < NV; ++q) out[P.base + q * P.qs + i] = f[q];
}

// SumFromFine's addition into one valid cell of a patched level: `span` names
// its contributions (the first in the high 32 bits, their number in the low
// ones), the block averages avg[q * avg_stride + contrib[j]], added in FP64
// in that order to the cell's streamed value.
template <typename S>
__device__ __forceinline__ void add_block_sums(S* f, long long span, const double* __restrict__ avg,
                                               long long avg_stride, const int* __restrict__ contrib, double rho0) {
  double acc[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) acc[q] = to_f64(f[q], q, rho0);
  const int first = int(span >> 32), n = int(span & 0xffffffffll);
  for (int j = first; j < first + n; ++j) {
    const long long a = contrib[j];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] += avg[q * avg_stride + a];
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) f[q] = from_f64<S>(acc[q], q, rho0);
}

// A middle level's Stream + ZeroInvalidComponents (src/AmrSim.cpp:459-463)
// in a step whose result needs no block averages: the pull of the valid
// cells.  The ghost shell the reference computes (populations that came
// from valid cells) is not formed: nothing reads a patched level's ghost
// cells from its state (its next fill rewrites them, a finer level's fill
// and every read-back take valid cells only).  Fused with the second half
// of SumFromFine into this level (src/AmrSim.cpp:464-466, 592-602): a valid
// cell with a span (per grown cell, -1 if none) adds the child's block
// averages it names to its streamed value in FP64, in the same order as
// k_sum_apply.
template <typename S>
__global__ __launch_bounds__(256) void k_fine_stream_zero(const S* __restrict__ in, S* __restrict__ out,
                                                          const PatchDesc* __restrict__ patches, int first,
                                                          double rho0, const long long* __restrict__ spans,
                                                          const double* __restrict__ avg, long long avg_stride,
                                                          const int* __restrict__ contrib) {
  const PatchDesc P = patches[first + blockIdx.y];
  const int i = xcd_chunk() * 256 + threadIdx.x;
  if (i >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  if (!patch_valid(P, gx, gy, gz)) return;
  S f[NV];
  fine_pull(P, in, P.base, i, gx, gy, gz, rho0, f);
  const long long span = spans[P.fill_base + i];
  if (span >= 0) add_block_sums(f, span, avg, avg_stride, contrib, rho0);
#pragma unroll
  for (int q = 0; q < NV; ++q) out[P.base + q * P.qs + i] = f[q];
}

// One whole step of a patched level at ratio 2, from its parent's and its own
// current states: with FINEST the finest level's two substeps of a step of
// its parent, else one step of a level between level 0 and the finest.  In
// the reference's terms, per grown cell:
//   A  FillPatchTwoLevels, comp 0 zeroed on the outer ghost layer, collide of
//      the valid cells (a cell under the child's mask is zeroed: MASK)
//   B  (FINEST) Stream(1) over valid + 1 ghost layer of a fresh array, whose
//      outer layer is zero, and the second substep's collide
//   C  Stream(1); with SUM the child's block averages added into the valid
//      cells (SumFromFine), ZeroInvalidComponents, the valid cells stored,
//      and with AVG the 1/8-weighted sum of each 2x2x2 block of the grown
//      patch for the parent (children in (k, j, i) order in FP64)
// A patch's ghosts are filled once, so no patch's A, B or C depends on
// another's, and nothing but the valid cells of C and the block averages has
// to reach memory.  A workgroup takes a tile (FineTile: a range of grown
// cells in x, y and z, even on both ends) and walks z: it forms plane k of A
// over the tile and 2 cells around it, plane k - 1 of B over the tile and 1
// cell around it, and plane k - 2 of C, each handed to the next through one
// LDS plane; of the three planes a pull reads, the upper one is in LDS and
// the populations with c_z = 0 and +1 of the other two are carried in
// registers.  A wave holds whole 2x2 columns, so the 4 children of a block in
// a plane meet in the wave's own part of the A plane, which is free by then,
// without a barrier; its two halves hold a row each, so that its loads and
// stores run along x (with the 4 children in neighbouring lanes a load took
// 110 cycles to issue).  A
// population that does not move (q = 0) stays in its lane.
//
// Bound: per plane two collisions of each cell (and the ring's) against one
// read of the grown patch and one write of its valid cells.  The passes this
// replaces (fill + collide, stream + collide, stream + average; each reading
// and writing every patch, in groups kept in the MALL) moved 7.7 valid-cell
// transfers per pair of substeps and ran at the fabric's rate.  128 patches of
// 36^3 grown cells (64x256x256 in boxes of 32^3), two substeps: FP64 750 us
// before, 437 us so, of which a plane's two collisions and pulls are about 60 %; one
// workgroup a CU (114 KB of LDS, 2 waves a SIMD at 256 registers).  Slower: 12
// waves on tiles of 36 x 20 cells at 168 registers (484 us), the loads of a
// plane in one piece or after the first barrier (503 to 627 us).

// Orders a wave's LDS accesses among its own lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// to_f64 for a population known at run time only.
template <typename S>
__device__ __forceinline__ double to_f64_any(S v, int q, double rho0) {
  if constexpr (sizeof(S) == 8)
    return v;
  else
    return (q == 0 ? kT.W[0] : q <= 6 ? kT.W[1] : kT.W[7]) * rho0 + double(v);
}

// Number of a population's (c_x, c_y).
__device__ constexpr int lateral(int q) { return (kC[q][1] + 1) * 3 + kC[q][0] + 1; }

// First of the populations that share (c_x, c_y): 1 to 4, then 5, 7, 9, 11, 13.
__device__ constexpr int pull_first(int c) { return c < 4 ? c + 1 : 2 * c - 3; }

template <typename S, bool FINEST, bool MASK, bool SUM, bool AVG, int CELLS>
__global__ __launch_bounds__(CELLS) void k_fine_step(
    const S* __restrict__ fnow, S* __restrict__ fnext, const S* __restrict__ cnow,
    const PatchDesc* __restrict__ own, const FineTile* __restrict__ tiles, int ntiles,
    const unsigned long long* __restrict__ fill, const unsigned* __restrict__ strides, long long parent_stride,
    const unsigned char* __restrict__ mask, Relax r, double* __restrict__ avg,
    long long avg_stride, const long long* __restrict__ spans, const double* __restrict__ cavg, long long cavg_stride,
    const int* __restrict__ contrib) {
  // plane A of population q, then plane B of it
  constexpr int kSets = FINEST ? 2 : 1;
  constexpr int kFineCells = CELLS;
  __shared__ S planes[NV - 1][kSets][kFineCells];
  constexpr int kB = kSets - 1;
  constexpr int kCut1 = 5, kCut2 = 10;
  const int w = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // an XCD takes neighbouring tiles
  if (w >= ntiles) return;
  const FineTile T = tiles[w];
  const PatchDesc& P = own[T.patch];
  const int gx = P.g[0], gy = P.g[1], gz = P.g[2];
  // A region in x and y, and this thread's cell of it
  const int ax = max(T.lo[0] - 2, 0), ay = max(T.lo[1] - 2, 0);
  const int wb = (min(T.hi[0] + 2, gx) - ax) >> 1, hb = (min(T.hi[1] + 2, gy) - ay) >> 1;  // 2x2 columns
  // A wave holds 16 consecutive 2x2 columns: its lower half their lower rows,
  // its upper half the upper rows, each 32 cells along x.
  const int t = threadIdx.x, col = (t >> 6) * 16 + ((t & 31) >> 1);
  const bool on = col < wb * hb;
  const int x = ax + 2 * (col % wb) + (t & 1), y = ay + 2 * (col / wb) + ((t >> 5) & 1);
  const bool outer_xy = x == 0 || y == 0 || x == gx - 1 || y == gy - 1;
  const bool valid_xy = on && x >= 2 && x < gx - 2 && y >= 2 && y < gy - 2;
  const bool in_c = on && x >= T.lo[0] && x < T.hi[0] && y >= T.lo[1] && y < T.hi[1];
  const bool in_b = on && x >= T.lo[0] - 1 && x <= T.hi[0] && y >= T.lo[1] - 1 && y <= T.hi[1];
  // Where this lane pulls from: the cell at x - c_x, y - c_y of the same
  // plane.  Every lane pulls, so that the carried populations see no branch;
  // one whose neighbours lie outside the tile reads itself and is not used.
  // One address serves the populations that differ in c_z only (5 and 6, 7
  // and 8, ...) in both planes; kept opaque, or the compiler holds a sum per
  // population in registers it does not have.
  const bool inside = in_b && !outer_xy;
  int from[9];
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    const int q = pull_first(c);
    const int nx = x - ax - kC[q][0], ny = y - ay - kC[q][1];
    const int ncol = (ny >> 1) * wb + (nx >> 1);
    const int at = inside ? (ncol >> 4) * 64 + (ny & 1) * 32 + (ncol & 15) * 2 + (nx & 1) : t;
    from[c] = ((q - 1) * kSets * kFineCells + at) * (int)sizeof(S);
    asm volatile("" : "+v"(from[c]));
  }
  auto pulled = [&](int set, int q) {
    const int c = q <= 4 ? q - 1 : 4 + (q - 5) / 2;
    const int more = ((q - pull_first(c)) * kSets + set) * kFineCells * (int)sizeof(S);
    return *(const S*)((const char*)&planes[0][0][0] + from[c] + more);
  };
  const int sz = gx * gy;
  const unsigned stored = y * P.row + x;
  const unsigned ixy = y * gx + x;  // 8 * ixy < 2^32: a patch has fewer than 2^31 cells and at least 6 planes
  const int a0 = max(T.lo[2] - (FINEST ? 2 : 1), 0), a1 = min(T.hi[2] + (FINEST ? 2 : 1), gz);

  // Ghost cells take their source from the fill table; the entry of a plane
  // is loaded a plane ahead, so that its latency is not added to the data's.
  auto load_fill = [&](int z) -> unsigned long long {
    if (!on || z >= a1 || (valid_xy && z >= 2 && z < gz - 2)) return 0;
    return *(const unsigned long long*)((const char*)(fill + (P.fill_base + (long long)z * sz)) + ixy * 8u);
  };
  auto source = [&](int z, unsigned long long d, const S*& src, long long& stride) {
    src = (const S*)((const char*)(fnow + (P.origin + (long long)z * P.plane)) + stored * (unsigned)sizeof(S));
    stride = P.qs;
    if (!(valid_xy && z >= 2 && z < gz - 2)) {
      src = ((long long)d < 0 ? cnow : fnow) + (d & kFillElement);
      stride = strides ? strides[(d & ~kFillParent) >> kFillStrideShift]
                       : ((long long)d < 0 ? parent_stride : P.qs);
    }
  };
  // Populations [q0, q1) from src on, which moves on to q1.
  auto load_some = [&](int q0, int q1, const S*& src, long long stride, S* f) {
#pragma unroll
    for (int q = 0; q < NV; ++q)
      if (q >= q0 && q < q1) {
        f[q] = *src;
        src += stride;
      }
  };

  // carried for B (FINEST) and for C: next plane's c_z = 0 and +1
  // populations, and the c_z = +1 ones of the plane after it
  S b1[NV], b2[NV], c1[NV], c2[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) b1[q] = b2[q] = c1[q] = c2[q] = S(0);
  // pulls from the plane in LDS: f = the populations of the plane below it;
  // `rest` is this lane's own q = 0 there
  auto advance = [&](int set, S rest, S* p1, S* p2, S* f) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const S v = q == 0 ? rest : pulled(set, q);
      if (kC[q][2] < 0) {
        f[q] = v;
      } else {
        f[q] = p1[q];
        p1[q] = kC[q][2] == 0 ? v : p2[q];
        if (kC[q][2] > 0) p2[q] = v;
      }
    }
  };

  // bit lateral(q): the cell - 2 c_q is valid in x and y
  int keep_xy = 0;
  if constexpr (AVG) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const int xq = x - 2 * kC[q][0], yq = y - 2 * kC[q][1];
      if (xq >= 2 && xq < gx - 2 && yq >= 2 && yq < gy - 2) keep_xy |= 1 << lateral(q);
    }
  }
  // this lane's column of the block sums
  const int tc = (t >> 6) * 16 + (t & 15);
  const int tx = ax + 2 * (tc % wb), ty = ay + 2 * (tc / wb);
  const bool task = tc < wb * hb && tx >= T.lo[0] && tx < T.hi[0] && ty >= T.lo[1] && ty < T.hi[1];
  const int task_block = (ty >> 1) * (gx >> 1) + (tx >> 1);

  S next[NV];  // A's next plane, loading
  double sum[4] = {0.0, 0.0, 0.0, 0.0};  // this lane's block sums, between a block's two planes
  const S* src = fnow;
  long long stride = 0;
  if (on) {
    source(a0, load_fill(a0), src, stride);
    load_some(0, NV, src, stride, next);
  }
  unsigned long long fill_next = load_fill(a0 + 1);
  // MASK: this cell's byte; SUM: its span in C's plane; both a plane ahead
  auto load_mask = [&](int z) -> int {
    return MASK && valid_xy && z >= 2 && z < gz - 2 ? mask[P.fill_base + (long long)z * sz + ixy] : 0;
  };
  auto load_span = [&](int z) -> long long {
    return SUM && in_c && valid_xy && z >= max(T.lo[2], 2) && z < min(T.hi[2], gz - 2)
               ? spans[P.fill_base + (long long)z * sz + ixy]
               : -1;
  };
  int mask_next = load_mask(a0);
  long long span_next = load_span(a0 - 1);
  if (FINEST && on) {  // B is zero on the outer layer, first and last planes included
#pragma unroll
    for (int q = 1; q < NV; ++q) planes[q - 1][kB][t] = zero_pop<S>(q, r.rho0);
  }
  // A plane's loads are waited for before its predecessor's stores are issued:
  // a wait after them would be for the stores as well.
  auto arrived = [&] {
#pragma unroll
    for (int q = 0; q < NV; ++q) asm volatile("" : "+v"(next[q]));
    asm volatile("" : "+v"(fill_next));
    if constexpr (MASK) asm volatile("" : "+v"(mask_next));
    if constexpr (SUM) asm volatile("" : "+v"(span_next));
  };
  arrived();
  const int steps_behind = FINEST ? 2 : 1;
  for (int k = a0; k < T.hi[2] + steps_behind; ++k) {
    const bool more = k + 1 < a1;
    // A: plane k.  Valid and ghost lanes hand their values over separately:
    // joining them first costs a copy of every population.
    S f[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) f[q] = next[q];
    // A's next plane is loaded in three parts, before each stage: a wave that
    // issues all of it at once waits ~50 cycles per load for the ones before.
    const bool load = on && more;
    if (load) {
      source(k + 1, fill_next, src, stride);
      load_some(0, kCut1, src, stride, next);
    }
    fill_next = load_fill(k + 2);
    const bool masked = mask_next;
    long long span = span_next;
    int block = 0;  // the span's first contribution
    if constexpr (MASK) mask_next = load_mask(k + 1);
    if constexpr (SUM) {
      if (span >= 0) block = contrib[span >> 32];
      span_next = load_span(k);
    }
    S rest = zero_pop<S>(0, r.rho0);
    auto hand_over = [&](int set) {
#pragma unroll
      for (int q = 1; q < NV; ++q) planes[q - 1][set][t] = f[q];
      rest = f[0];
    };
    if (on && k < a1) {
      if (valid_xy && k >= 2 && k < gz - 2) {
        if (MASK && masked) {
#pragma unroll
          for (int q = 0; q < NV; ++q) f[q] = zero_pop<S>(q, r.rho0);
        } else {
          collide_s(f, r);
        }
        hand_over(0);
      } else {
        if (outer_xy || k == 0 || k == gz - 1) f[0] = zero_pop<S>(0, r.rho0);
        hand_over(0);
      }
    }
    if (load) load_some(kCut1, kCut2, src, stride, next);
    // SUM: the span's first block (most cells have no other), loading
    double added[NV];
    if constexpr (SUM) {
      if (span >= 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) added[q] = cavg[q * cavg_stride + block];
      }
    }
    __syncthreads();
    const int zc = k - steps_behind;
    if constexpr (FINEST) {
      // B: plane k - 1
      const int zb = k - 1;
      advance(0, rest, b1, b2, f);
      rest = zero_pop<S>(0, r.rho0);
      if (inside) {
        if (zb < 1 || zb >= gz - 1) {  // an outer layer
          if (zb == gz - 1) {
#pragma unroll
            for (int q = 1; q < NV; ++q) planes[q - 1][kB][t] = zero_pop<S>(q, r.rho0);
          }
        } else if (valid_xy && zb >= 2 && zb < gz - 2) {
          collide_s(f, r);
          hand_over(kB);
        } else {
          hand_over(kB);
        }
      }
      __syncthreads();
    }
    if (load) load_some(kCut2, NV, src, stride, next);
    // C: plane zc
    S g[NV];
    advance(kB, rest, c1, c2, g);
    if constexpr (!FINEST) __syncthreads();  // C has read the A plane
    const bool valid_c = valid_xy & (zc >= 2) & (zc < gz - 2);
    if constexpr (SUM) {
      if (span >= 0) {
        double acc[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) acc[q] = to_f64(g[q], q, r.rho0) + added[q];
        const int first = int(span >> 32), n = int(span & 0xffffffffll);
        for (int j = first + 1; j < first + n; ++j) {
          const long long c = contrib[j];
#pragma unroll
          for (int q = 0; q < NV; ++q) acc[q] += cavg[q * cavg_stride + c];
        }
#pragma unroll
        for (int q = 0; q < NV; ++q) g[q] = from_f64<S>(acc[q], q, r.rho0);
      }
    }
    if constexpr (AVG) {
      // The wave's 16 columns x 15 populations are 240 tasks: in round j lane
      // l sums population 1 + 4 j + l / 16 of the wave's column l % 16 (0 for
      // 15, which passes through the first plane once its population is done).
      // The outer layer is zero; ZeroInvalidComponents: population q of
      // another ghost cell survives only if the cell - 2 c_q is valid.
      if (zc >= T.lo[2]) {
        const bool outer = outer_xy | (zc <= 0) | (zc >= gz - 1);
        auto meet = [&](int q, int at) {
          const int zq = zc - 2 * kC[q][2];
          const bool keep = valid_c | (!outer & ((keep_xy & 1 << lateral(q)) != 0) & (zq >= 2) & (zq < gz - 2));
          if (in_c) {
            planes[at][0][t] = g[q];
            if (!keep) planes[at][0][t] = zero_pop<S>(q, r.rho0);
          }
        };
        int lane = t;
        asm volatile("" : "+v"(lane));  // no address per round held in registers
        const int task_cell = (lane & ~63) + 2 * (lane & 15);
#pragma unroll
        for (int q = 1; q < NV; ++q) meet(q, q - 1);
        wave_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j == 3) {
            wave_sync();
            meet(0, 0);
            wave_sync();
          }
          const int q = 1 + 4 * j + (lane >> 4 & 3), qq = q < NV ? q : 0;
          if (task && q <= NV) {
            double s = (zc & 1) ? sum[j] : 0.0;
#pragma unroll
            for (int c = 0; c < 4; ++c)
              s += to_f64_any(planes[q < NV ? q - 1 : 0][0][task_cell + (c & 1) + 32 * (c >> 1)], qq, r.rho0);
            sum[j] = s;
          }
        }
      }
    }
    arrived();
    if constexpr (AVG) {
      if (task & (zc >= T.lo[2]) & (zc & 1)) {
        double* here = avg + P.avg_base + (long long)(zc >> 1) * ((gx >> 1) * (gy >> 1)) + task_block;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int q = 1 + 4 * j + (t >> 4 & 3);
          if (q <= NV) here[(q < NV ? q : 0) * avg_stride] = sum[j] * 0.125;
        }
      }
    }
    if (in_c & valid_c & (zc >= T.lo[2])) {
      S* out = fnext + (P.origin + (long long)zc * P.plane);
#pragma unroll
      for (int q = 0; q < NV; ++q) *(S*)((char*)(out + q * P.qs) + stored * (unsigned)sizeof(S)) = g[q];
    }
  }
}

// Coarse cell flags: bit 0/1 = the cell is on its box's high/low x face
// (x+1 / x-1 leaves the box), bits 2/3 the same in y, 4/5 in z; bit 7 = the
// cell lies under the fine mask.
constexpr unsigned kMasked = 0x80u;

__device__ constexpr unsigned leave_bits(int q) {
  return (kC[q][0] > 0 ? 1u : 0u) | (kC[q][0] < 0 ? 2u : 0u) | (kC[q][1] > 0 ? 4u : 0u) |
         (kC[q][1] < 0 ? 8u : 0u) | (kC[q][2] > 0 ? 16u : 0u) | (kC[q][2] < 0 ? 32u : 0u);
}

// Over the whole coarse level array, shaped like the stream-collide launch.
template <typename S>
__global__ __launch_bounds__(512) void k_coarse_push(const S* __restrict__ cnow, S* __restrict__ cnext,
                                                     Lattice L, const unsigned char* __restrict__ flags,
                                                     Relax r) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= L.nx || y >= L.ny) return;
  const long long self = L.at(0, y * L.nx + x, z);
  const unsigned fl = flags[((long long)z * L.ny + y) * L.nx + x];
  S pre[NV], post[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) pre[q] = post[q] = __builtin_nontemporal_load(cnow + self + q * L.ps);
  if (fl & kMasked) {
#pragma unroll
    for (int q = 0; q < NV; ++q) post[q] = zero_pop<S>(q, r.rho0);
  } else {
    collide_s(post, r);
  }
  const int xs[3] = {(x == 0) ? L.nx - 1 : x - 1, x, (x == L.nx - 1) ? 0 : x + 1};
  const int ys[3] = {((y == 0) ? L.ny - 1 : y - 1) * L.nx, y * L.nx, ((y == L.ny - 1) ? 0 : y + 1) * L.nx};
  const int zs[3] = {(z == 0) ? L.nz - 1 : z - 1, z, (z == L.nz - 1) ? 0 : z + 1};
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const long long dest = L.at(q, ys[1 + kC[q][1]] + xs[1 + kC[q][0]], zs[1 + kC[q][2]]);
    __builtin_nontemporal_store((fl & leave_bits(q)) ? pre[q] : post[q], cnext + dest);
  }
}

// Second half of SumFromFine: thread per touched coarse cell; its
// contributions [start[u], start[u+1]) (indices into avg, in the order the
// reference's loops add them) are added in FP64 to the streamed coarse value.
// A coarse cell is the element of population 0 in the level array.
template <typename S>
__global__ __launch_bounds__(256) void k_sum_apply(const double* __restrict__ avg, long long avg_stride,
                                                   S* __restrict__ cnext, Lattice L,
                                                   const long long* __restrict__ cell,
                                                   const int* __restrict__ start,
                                                   const int* __restrict__ contrib, int ncell, double rho0) {
  const int u = xcd_chunk() * 256 + threadIdx.x;
  if (u >= ncell) return;
  const long long c = cell[u], stride = L.ps;
  double acc[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) acc[q] = to_f64(cnext[c + q * stride], q, rho0);
  for (int j = start[u]; j < start[u + 1]; ++j) {
    const long long a = contrib[j];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] += avg[q * avg_stride + a];
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) cnext[c + q * stride] = from_f64<S>(acc[q], q, rho0);
}

// The finest level's last substep at a refinement ratio r above 2: the
// stream of its valid cells (the input's outer layer read as zero) into
// `out`.  Its ghost cells need no ZeroInvalidComponents: at such a ratio the
// average-down reads valid cells only (nGrow = 2 / r = 0) and the next
// fill-collide rewrites the ghosts.
template <typename S>
__global__ __launch_bounds__(256) void k_fine_stream_valid(const S* __restrict__ in, S* __restrict__ out,
                                                           const PatchDesc* __restrict__ patches, int first,
                                                           double rho0) {
  const PatchDesc& P = patches[first + blockIdx.y];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  if (!patch_valid(P, gx, gy, gz)) return;
  S f[NV];
  fine_pull_inner(P, in, P.base, i, gx, gy, gz, rho0, f);
#pragma unroll
  for (int q = 0; q < NV; ++q) out[P.base + q * P.qs + i] = f[q];
}

// The first half of SumFromFine at a refinement ratio r above 2
// (amrex_avgdown over the valid box only, nGrow = 2 / r = 0): per r x r x r
// block of valid cells, the FP64 sum of its children in (k, j, i) order
// times 1/r^3, to avg[q * avg_stride + P.avg_base + block] (blocks x
// fastest over the coarsened valid box).
// A lane takes one block of one population (blockIdx.z), all children in
// flight at once: bound by the patches' one read, strided over the lanes by r
// elements.  A group of 18 patches of 24^3 at ratio 3, FP64: 103 us with a lane for all
// populations of a block, one child after the other, and 8.9 us so.
template <typename S, int R>
__global__ __launch_bounds__(256) void k_fine_avg_valid(const S* __restrict__ f, double* __restrict__ avg,
                                                        long long avg_stride, const PatchDesc* __restrict__ patches,
                                                        int first, double rho0) {
  const PatchDesc& P = patches[first + blockIdx.y];
  const int c0 = (P.hi[0] - P.lo[0] + 1) / R, c1 = (P.hi[1] - P.lo[1] + 1) / R, c2 = (P.hi[2] - P.lo[2] + 1) / R;
  const int u = blockIdx.x * 256 + threadIdx.x, q = blockIdx.z;
  const int nblk = c0 * c1 * c2;
  if (u >= nblk) return;
  int cx, cy, cz;
  split3(u, nblk, c0, c1, cx, cy, cz);
  const int sy = P.g[0], sz = P.g[0] * P.g[1];
  const S* from = f + P.base + q * P.qs + (long long)(2 + R * cz) * sz + (long long)(2 + R * cy) * sy + (2 + R * cx);
  S child[R * R * R];
#pragma unroll
  for (int c = 0; c < R * R * R; ++c) child[c] = from[(long long)(c / (R * R)) * sz + (c / R % R) * sy + c % R];
  double sum = 0.0;
#pragma unroll
  for (int c = 0; c < R * R * R; ++c) sum += to_f64_any(child[c], q, rho0);
  avg[q * avg_stride + P.avg_base + u] = sum * (1.0 / (double)(R * R * R));
}

// DistFnFillFromCoarse (src/AmrSim.cpp:393-411): valid fine cells take the
// coarse value of their parent (ghosts are filled before they are read).
template <typename S>
__global__ __launch_bounds__(256) void k_fine_from_coarse(S* __restrict__ fnow, const S* __restrict__ cnow,
                                                          Lattice clat, const PatchDesc* __restrict__ patches,
                                                          int ratio) {
  const PatchDesc P = patches[blockIdx.y];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  if (patch_valid(P, gx, gy, gz)) {
    const int x = (P.lo[0] - 2 + gx) / ratio, y = (P.lo[1] - 2 + gy) / ratio, z = (P.lo[2] - 2 + gz) / ratio;
    const long long c = clat.at(0, y * clat.nx + x, z), to = P.at(gx, gy, gz);
#pragma unroll
    for (int q = 0; q < NV; ++q) fnow[to + q * P.qs] = cnow[c + q * clat.ps];
  }
}

// The patches of boxes [0, n) that meet the box [lo, hi], listed by the
// workgroup in `list`, which has room for kNear; their number, or -1 if it has
// not.  A barrier at either end.
constexpr int kNear = 512;
__device__ __forceinline__ int near_boxes(const PatchDesc* __restrict__ boxes, int n, const int* lo, const int* hi,
                                          int* list, int* count) {
  __syncthreads();
  if (threadIdx.x == 0) *count = 0;
  __syncthreads();
  for (int b = threadIdx.x; b < n; b += 256) {
    const PatchDesc& B = boxes[b];
    bool meets = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) meets &= B.lo[d] <= hi[d] && B.hi[d] >= lo[d];
    if (meets) {
      const int k = atomicAdd(count, 1);
      if (k < kNear) list[k] = b;
    }
  }
  __syncthreads();
  return *count <= kNear ? *count : -1;
}

// RemakeLevel's fill (src/AmrSim.cpp:715-744 via DistFnFillPatch) and, with no
// old patches, DistFnFillFromCoarse (src/AmrSim.cpp:393-411) from a patched
// parent: each valid cell of the new patches takes the value of the old patch
// that holds it, else of its parent.  A workgroup first lists the old and the
// parent's patches that meet its own, of which every lane then looks for the
// one that holds its cell (boxes of a level are disjoint).  A table of the
// sources, made cell by cell on the host, took 14 ms for the 2 M cells of
// 32x256x256; this takes 0.1.
template <typename S, bool PC>
__global__ __launch_bounds__(256) void k_fine_remake(S* __restrict__ fnew, const S* __restrict__ fold,
                                                     const S* __restrict__ cnow, Lattice clat,
                                                     const PatchDesc* __restrict__ cpatches, int ncoarse,
                                                     const PatchDesc* __restrict__ patches,
                                                     const PatchDesc* __restrict__ old_patches, int nold, int ratio) {
  __shared__ int list[kNear], count;
  const PatchDesc& P = patches[blockIdx.y];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if ((int)blockIdx.x * 256 >= P.cells) return;
  int gx, gy, gz;
  patch_coords(P, i, gx, gy, gz);
  const bool valid = i < P.cells && patch_valid(P, gx, gy, gz);
  const S* from = nullptr;
  long long stride = 0;
  auto look = [&](const PatchDesc* boxes, int n, const S* state, int r) {
    const int lo[3] = {P.lo[0] / r, P.lo[1] / r, P.lo[2] / r}, hi[3] = {P.hi[0] / r, P.hi[1] / r, P.hi[2] / r};
    const int x = (P.lo[0] - 2 + gx) / r, y = (P.lo[1] - 2 + gy) / r, z = (P.lo[2] - 2 + gz) / r;
    const int near = near_boxes(boxes, n, lo, hi, list, &count);
    for (int k = 0; k < (near < 0 ? n : near); ++k) {
      const PatchDesc& B = boxes[near < 0 ? k : __builtin_amdgcn_readfirstlane(list[k])];
      if (valid && from == nullptr && x >= B.lo[0] && x <= B.hi[0] && y >= B.lo[1] && y <= B.hi[1] && z >= B.lo[2] &&
          z <= B.hi[2]) {
        from = state + B.at(x - B.lo[0] + 2, y - B.lo[1] + 2, z - B.lo[2] + 2);
        stride = B.qs;
      }
    }
  };
  look(old_patches, nold, fold, 1);
  if constexpr (PC) {
    look(cpatches, ncoarse, cnow, ratio);
  } else if (valid && from == nullptr) {
    const int x = (P.lo[0] - 2 + gx) / ratio, y = (P.lo[1] - 2 + gy) / ratio, z = (P.lo[2] - 2 + gz) / ratio;
    from = cnow + clat.at(0, y * clat.nx + x, z);
    stride = clat.ps;
  }
  if (from == nullptr) return;
  const long long to = P.at(gx, gy, gz);
#pragma unroll
  for (int q = 0; q < NV; ++q) fnew[to + q * P.qs] = from[q * stride];
}

// Valid cells of one patch <-> packed FP64 f [15][nz][ny][nx].
template <int OP, typename S>  // 0 pack, 1 unpack
__global__ __launch_bounds__(256) void k_patch_io(S* __restrict__ f, const PatchDesc* __restrict__ patches, int b,
                                                  double* __restrict__ a, double rho0) {
  static_assert(OP == 0 || OP == 1);
  const PatchDesc P = patches[b];
  const int nx = P.hi[0] - P.lo[0] + 1, ny = P.hi[1] - P.lo[1] + 1, nz = P.hi[2] - P.lo[2] + 1;
  const int n = nx * ny * nz;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int x = i % nx, t = i / nx, y = t % ny, z = t / ny;
  const long long li = P.at(x + 2, y + 2, z + 2);
  if (OP == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) a[(long long)q * n + i] = to_f64(f[li + q * P.qs], q, rho0);
  } else {
#pragma unroll
    for (int q = 0; q < NV; ++q) f[li + q * P.qs] = from_f64<S>(a[(long long)q * n + i], q, rho0);
  }
}

// Density and velocity of the valid cells of every patch (blockIdx.y) in one
// launch.
template <typename S>
__global__ __launch_bounds__(256) void k_patch_hydro(const S* __restrict__ f, const PatchDesc* __restrict__ patches,
                                                     int first_box, int nbox, double* __restrict__ rho,
                                                     double* __restrict__ u, double rho0) {
  for (int b = blockIdx.y; b < nbox; b += gridDim.y) {
    const PatchDesc& P = patches[first_box + b];
    const int n0 = P.hi[0] - P.lo[0] + 1, n1 = P.hi[1] - P.lo[1] + 1, n = n0 * n1 * (P.hi[2] - P.lo[2] + 1);
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) continue;
    const int t = i / n0, x = i - t * n0, z = t / n1, y = t - z * n1;
    const long long li = P.at(x + 2, y + 2, z + 2);
    double g[NV], r, u0, u1, u2;
#pragma unroll
    for (int q = 0; q < NV; ++q) g[q] = to_f64(f[li + q * P.qs], q, rho0);
    hydro_f64(g, r, u0, u1, u2);
    const long long at = P.first - patches[first_box].first;
    rho[at + i] = r;
    u[3 * at + i] = u0;
    u[3 * at + n + i] = u1;
    u[3 * at + 2ll * n + i] = u2;
  }
}

template <typename S>
hipError_t patch_io(int op, S* f, const PatchDesc* patches, int b, int valid_cells, double* a, double rho0,
                    hipStream_t st) {
  const int blocks = (valid_cells + 255) / 256;
  if (op == 0)
    k_patch_io<0, S><<<blocks, 256, 0, st>>>(f, patches, b, a, rho0);
  else
    k_patch_io<1, S><<<blocks, 256, 0, st>>>(f, patches, b, a, rho0);
  return hipGetLastError();
}

}  // namespace

template <typename S>
hipError_t fill_collide(const S* fnow, S* fnext, const S* cnow, const Lattice& clat, const PatchDesc* cpatches,
                        const PatchDesc* patches, const PatchDesc* own, int first, const long long* fill,
                        const unsigned char* mask, const Relax& r, dim3 grid, hipStream_t st) {
  if (cpatches && mask)
    k_fine_fill_collide<S, true, true><<<grid, 256, 0, st>>>(fnow, fnext, cnow, clat, cpatches, patches, own, first,
                                                             fill, mask, r);
  else if (cpatches)
    k_fine_fill_collide<S, true, false><<<grid, 256, 0, st>>>(fnow, fnext, cnow, clat, cpatches, patches, own,
                                                              first, fill, mask, r);
  else if (mask)
    k_fine_fill_collide<S, false, true><<<grid, 256, 0, st>>>(fnow, fnext, cnow, clat, cpatches, patches, own,
                                                              first, fill, mask, r);
  else
    k_fine_fill_collide<S, false, false><<<grid, 256, 0, st>>>(fnow, fnext, cnow, clat, cpatches, patches, own,
                                                               first, fill, mask, r);
  return hipGetLastError();
}

hipError_t launch_fine_fill_collide(int precision, const void* fnow, void* fnext, const void* cnow,
                                    const Lattice& clat, const PatchDesc* cpatches, const PatchDesc* patches,
                                    const PatchDesc* own, int first, int npatch, int max_cells,
                                    const long long* fill, const unsigned char* mask, const Relax& r,
                                    hipStream_t st) {
  // A multiple of 8 workgroups per patch, so that xcd_chunk() gives each XCD
  // the same slab of every patch: the rows whose first or last two cells an
  // x-neighbour's ghost fill reads (and the rows a y-neighbour's reads) are
  // then fetched into that XCD's L2 by both patches' workgroups at about the
  // same time.  The extra workgroups exit at once.
  const dim3 grid(((max_cells + 255) / 256 + 7) / 8 * 8, npatch);
  if (precision == 0)
    return fill_collide((const double*)fnow, (double*)fnext, (const double*)cnow, clat, cpatches, patches, own,
                        first, fill, mask, r, grid, st);
  return fill_collide((const float*)fnow, (float*)fnext, (const float*)cnow, clat, cpatches, patches, own, first,
                      fill, mask, r, grid, st);
}

hipError_t launch_fine_stream_zero(int precision, const void* in, void* out, const PatchDesc* patches, int first,
                                   int npatch, int max_cells, double rho0, const long long* spans,
                                   const double* avg, long long avg_stride, const int* contrib, hipStream_t st) {
  const dim3 grid(((max_cells + 255) / 256 + 7) / 8 * 8, npatch);  // for xcd_chunk()
  if (precision == 0)
    k_fine_stream_zero<double><<<grid, 256, 0, st>>>((const double*)in, (double*)out, patches, first, rho0, spans,
                                                     avg, avg_stride, contrib);
  else
    k_fine_stream_zero<float><<<grid, 256, 0, st>>>((const float*)in, (float*)out, patches, first, rho0, spans, avg,
                                                    avg_stride, contrib);
  return hipGetLastError();
}

template <typename S, bool FINEST, bool AVG, int CELLS>
static hipError_t fine_step(const FineStep& a, hipStream_t st) {
  k_fine_step<S, FINEST, !FINEST, !FINEST, AVG, CELLS><<<(a.ntiles + 7) / 8 * 8, CELLS, 0, st>>>(
      (const S*)a.now, (S*)a.next, (const S*)a.parent, a.own, a.tiles, a.ntiles, a.fill, a.strides, a.parent_stride,
      a.mask, a.relax, a.avg, a.avg_stride, a.spans, a.cavg, a.cavg_stride, a.contrib);
  return hipGetLastError();
}

template <typename S, int CELLS>
static hipError_t fine_step(const FineStep& a, hipStream_t st) {
  if (a.finest) return fine_step<S, true, true, CELLS>(a, st);
  return a.avg ? fine_step<S, false, true, CELLS>(a, st) : fine_step<S, false, false, CELLS>(a, st);
}

hipError_t launch_fine_step(int precision, const FineStep& a, hipStream_t st) {
  if (a.cells == kFineSmall)
    return precision == 0 ? fine_step<double, kFineSmall>(a, st) : fine_step<float, kFineSmall>(a, st);
  if (a.finest)
    return precision == 0 ? fine_step<double, true, true, fine_tile_cells(8, true)>(a, st)
                          : fine_step<float, true, true, fine_tile_cells(4, true)>(a, st);
  if (precision == 0) return hipErrorInvalidValue;
  return a.avg ? fine_step<float, false, true, fine_tile_cells(4, false)>(a, st)
               : fine_step<float, false, false, fine_tile_cells(4, false)>(a, st);
}

hipError_t launch_fine_stream_collide(int precision, const void* in, void* out,
                                      const PatchDesc* patches, int first, int npatch, int max_cells, const Relax& r,
                                      hipStream_t st, bool inner) {
  const dim3 grid(((max_cells + 255) / 256 + 7) / 8 * 8, npatch);  // for xcd_chunk()
  if (precision == 0 && inner)
    k_fine_stream_collide<double, true><<<grid, 256, 0, st>>>((const double*)in, (double*)out, patches, first, r);
  else if (precision == 0)
    k_fine_stream_collide<double><<<grid, 256, 0, st>>>((const double*)in, (double*)out, patches, first, r);
  else if (inner)
    k_fine_stream_collide<float, true><<<grid, 256, 0, st>>>((const float*)in, (float*)out, patches, first, r);
  else
    k_fine_stream_collide<float><<<grid, 256, 0, st>>>((const float*)in, (float*)out, patches, first, r);
  return hipGetLastError();
}

hipError_t launch_coarse_push(int precision, const void* cnow, void* cnext, const Lattice& L,
                              const unsigned char* flags, const Relax& r, LaunchShape sh, hipStream_t st) {
  const dim3 grid((L.nx + sh.bx - 1) / sh.bx, (L.ny + sh.by - 1) / sh.by, L.nz);
  const dim3 block(sh.bx, sh.by, 1);
  if (precision == 0)
    k_coarse_push<double><<<grid, block, sh.lds_bytes, st>>>((const double*)cnow, (double*)cnext, L, flags, r);
  else
    k_coarse_push<float><<<grid, block, sh.lds_bytes, st>>>((const float*)cnow, (float*)cnext, L, flags, r);
  return hipGetLastError();
}

hipError_t launch_sum_apply(int precision, const double* avg, long long avg_stride, void* cnext, const Lattice& L,
                            const long long* cell, const int* start, const int* contrib, int ncell, double rho0,
                            hipStream_t st) {
  if (ncell <= 0) return hipSuccess;
  const int blocks = ((ncell + 255) / 256 + 7) / 8 * 8;  // for xcd_chunk()
  if (precision == 0)
    k_sum_apply<double><<<blocks, 256, 0, st>>>(avg, avg_stride, (double*)cnext, L, cell, start, contrib, ncell,
                                                rho0);
  else
    k_sum_apply<float><<<blocks, 256, 0, st>>>(avg, avg_stride, (float*)cnext, L, cell, start, contrib, ncell,
                                               rho0);
  return hipGetLastError();
}

hipError_t launch_fine_from_coarse(int precision, void* fnow, const void* cnow, const Lattice& clat,
                                   const PatchDesc* patches, int npatch, int max_cells, int ratio,
                                   hipStream_t st) {
  const dim3 grid((max_cells + 255) / 256, npatch);
  if (precision == 0)
    k_fine_from_coarse<double><<<grid, 256, 0, st>>>((double*)fnow, (const double*)cnow, clat, patches, ratio);
  else
    k_fine_from_coarse<float><<<grid, 256, 0, st>>>((float*)fnow, (const float*)cnow, clat, patches, ratio);
  return hipGetLastError();
}

hipError_t launch_fine_stream_valid(int precision, const void* in, void* out, const PatchDesc* patches, int first,
                                    int npatch, int max_cells, double rho0, hipStream_t st) {
  const dim3 grid((max_cells + 255) / 256, npatch);
  if (precision == 0)
    k_fine_stream_valid<double><<<grid, 256, 0, st>>>((const double*)in, (double*)out, patches, first, rho0);
  else
    k_fine_stream_valid<float><<<grid, 256, 0, st>>>((const float*)in, (float*)out, patches, first, rho0);
  return hipGetLastError();
}

hipError_t launch_fine_avg_valid(int precision, const void* f, double* avg, long long avg_stride,
                                 const PatchDesc* patches, int first, int npatch, int max_blocks, int ratio,
                                 double rho0, hipStream_t st) {
  const dim3 grid((max_blocks + 255) / 256, npatch, NV);
  if (precision == 0 && ratio == 3)
    k_fine_avg_valid<double, 3><<<grid, 256, 0, st>>>((const double*)f, avg, avg_stride, patches, first, rho0);
  else if (precision == 0)
    k_fine_avg_valid<double, 4><<<grid, 256, 0, st>>>((const double*)f, avg, avg_stride, patches, first, rho0);
  else if (ratio == 3)
    k_fine_avg_valid<float, 3><<<grid, 256, 0, st>>>((const float*)f, avg, avg_stride, patches, first, rho0);
  else
    k_fine_avg_valid<float, 4><<<grid, 256, 0, st>>>((const float*)f, avg, avg_stride, patches, first, rho0);
  return hipGetLastError();
}

hipError_t launch_fine_remake(int precision, void* fnew, const void* fold, const void* cnow, const Lattice& clat,
                              const PatchDesc* cpatches, int ncoarse, const PatchDesc* patches, int npatch,
                              int max_cells, const PatchDesc* old_patches, int nold, int ratio, hipStream_t st) {
  const dim3 grid((max_cells + 255) / 256, npatch);
  if (precision == 0 && cpatches)
    k_fine_remake<double, true><<<grid, 256, 0, st>>>((double*)fnew, (const double*)fold, (const double*)cnow, clat,
                                                      cpatches, ncoarse, patches, old_patches, nold, ratio);
  else if (precision == 0)
    k_fine_remake<double, false><<<grid, 256, 0, st>>>((double*)fnew, (const double*)fold, (const double*)cnow, clat,
                                                       cpatches, ncoarse, patches, old_patches, nold, ratio);
  else if (cpatches)
    k_fine_remake<float, true><<<grid, 256, 0, st>>>((float*)fnew, (const float*)fold, (const float*)cnow, clat,
                                                     cpatches, ncoarse, patches, old_patches, nold, ratio);
  else
    k_fine_remake<float, false><<<grid, 256, 0, st>>>((float*)fnew, (const float*)fold, (const float*)cnow, clat,
                                                      cpatches, ncoarse, patches, old_patches, nold, ratio);
  return hipGetLastError();
}

hipError_t launch_patch_io(int precision, int op, void* f, const PatchDesc* patches, int b, int valid_cells,
                           double* a, double rho0, hipStream_t st) {
  if (precision == 0) return patch_io(op, (double*)f, patches, b, valid_cells, a, rho0, st);
  return patch_io(op, (float*)f, patches, b, valid_cells, a, rho0, st);
}

hipError_t launch_patch_hydro(int precision, const void* f, const PatchDesc* patches, int first_box, int nbox,
                              long long max_cells, double* rho, double* u, double rho0, hipStream_t st) {
  const dim3 grid((unsigned)((max_cells + 255) / 256), nbox < 65535 ? nbox : 65535);
  if (precision == 0)
    k_patch_hydro<double><<<grid, 256, 0, st>>>((const double*)f, patches, first_box, nbox, rho, u, rho0);
  else
    k_patch_hydro<float><<<grid, 256, 0, st>>>((const float*)f, patches, first_box, nbox, rho, u, rho0);
  return hipGetLastError();
}

}  // namespace lbx
