// lbx_serve.hip -- kernels of the batched serving path.
//
// Every admitted run is an independent periodic lattice (nx, ny, nz) in the
// serving arena.  One launch advances every active run by one pass over the
// patch list (the work items of all runs: one item = 256 consecutive cells,
// x fastest, of one run, so every lane has a cell whatever the run's shape).
// The launch normally has one workgroup per item, with resident workgroups
// per CU capped as for the stream-collide kernels; the loop below walks
// further items with a static stride when the grid is smaller than the list,
// so every workgroup ends after a bounded number of items.  A run of n steps
// takes n + 1 passes: collide-only, n - 1 fused pull + collide, stream-only
// (the same S (C S)^(n-1) C association as lbx_iterate); a launch of two steps
// (k_serve_pair) takes two of them at once.  The per-cell arithmetic does not
// depend on which other runs share the launch nor on how passes are paired, so
// a run's result is the same alone and in any mix, bit for bit.
#include <hip/hip_runtime.h>

#include "d3q15.h"
#include "lbx_internal.h"

#pragma clang fp contract(off)

namespace lbx {
namespace {

template <typename S>
__device__ __forceinline__ void serve_cell(const ServeRun& R, int kind, const S* __restrict__ src,
                                           S* __restrict__ dst, int x, int y, int z) {
  const int nx = R.n[0], ny = R.n[1], nz = R.n[2];
  const long long zst = NV * R.ps;
  const long long selfz = z * zst;
  const int selfp = y * nx + x;
  int xs[3], ys[3];
  long long zs[3];
  xs[0] = (x == nx - 1) ? 0 : x + 1;
  xs[1] = x;
  xs[2] = (x == 0) ? nx - 1 : x - 1;
  ys[0] = ((y == ny - 1) ? 0 : y + 1) * nx;
  ys[1] = y * nx;
  ys[2] = ((y == 0) ? ny - 1 : y - 1) * nx;
  zs[0] = ((z == nz - 1) ? 0 : z + 1) * zst;
  zs[1] = selfz;
  zs[2] = ((z == 0) ? nz - 1 : z - 1) * zst;
  S f[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const long long off =
        (kind == STEP_COLLIDE) ? selfz + selfp : (zs[1 + kC[q][2]] + ys[1 + kC[q][1]] + xs[1 + kC[q][0]]);
    f[q] = src[off + q * R.ps];  // cached: small runs stay in the 256 MB MALL between steps
  }
  if (kind != STEP_STREAM) {
    if constexpr (sizeof(S) == 8)
      collide_f64(f, R.omega_s, R.omega_b);
    else
      collide_f32_shifted(f, float(R.rho0), float(R.omega_s), float(R.omega_b));
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) __builtin_nontemporal_store(f[q], dst + selfz + q * R.ps + selfp);
}

// The run holding a work item: the last r with item_begin <= item.
__device__ __forceinline__ int run_of(const ServeBatch& B, int item) {
  int lo = 0, hi = B.nruns - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (B.run[mid].item_begin <= item) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <typename S>
__global__ __launch_bounds__(256) void k_serve_step(ServeBatch B) {
  for (int item = blockIdx.x; item < B.total_items; item += gridDim.x) {
    const ServeRun& R = B.run[run_of(B, item)];
    const S* src = (const S*)R.src;
    S* dst = (S*)R.dst;
    const int plane = R.n[0] * R.n[1];
    const long long c = (long long)(item - R.item_begin) * 256 + threadIdx.x;
    if (c < (long long)plane * R.n[2]) {
      const int z = int(c / plane), r = int(c - (long long)z * plane);
      const int y = r / R.n[0], x = r - y * R.n[0];
      serve_cell<S>(R, R.kind, src, dst, x, y, z);
    }
  }
}

// Two passes of every run in one pass over its state, as k_step_pair does for
// one lattice: a work item is a column of cells and the ring around it, walked
// through `depth` planes of z, the first pass of a plane handed over in LDS to
// the second pass of the plane below.  The column is the run's own (rows of 32
// cells and 16 of them on cubes of 32, 64, 96 and 128; 48 x 10 on 48^3), so a
// small run wastes few lanes.  Bound like k_step_pair: by the collisions (the
// ring repeats a fifth of the first ones) with one workgroup of 10 waves per CU
// in FP64, by the reads and writes beside them in FP32 with two.  30 runs of
// 32^3 to 128^3, us per step: FP32 414 -> 305, FP64 823 -> 543; 8 runs of 64^3
// 48 -> 36 and 88 -> 62.
template <typename S>
__global__ __launch_bounds__(kServePairCells, sizeof(S) == 4 ? 5 : 3) void k_serve_pair(ServeBatch B) {
  __shared__ S ring[2][NV][kServePairCells];
  const int w = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // an XCD takes neighbouring columns
  if (w >= B.total_items) return;
  const ServeRun& R = B.run[run_of(B, w)];
  const int nx = R.n[0], ny = R.n[1], nz = R.n[2], bx = R.bx, by = R.by, kind = R.kind;
  const int item = w - R.item_begin, tx = (nx + bx - 1) / bx, ty = (ny + by - 1) / by;
  const int x0 = item % tx * bx, y0 = item / tx % ty * by, z0 = item / (tx * ty) * R.depth;
  const int z1 = min(z0 + R.depth, nz);
  const int wx = bx + 2, t = threadIdx.x;
  const S* __restrict__ src = (const S*)R.src;
  S* __restrict__ dst = (S*)R.dst;
  const long long ps = R.ps, zst = NV * ps;
  const bool pull = kind & PAIR_PULL;

  // first pass: cell t of the ring, its periodic image in the domain, and
  // where its populations come from
  const bool first = t < wx * (by + 2);
  const int rx = (x0 - 1 + (first ? t % wx : 0) + nx) % nx, ry = (y0 - 1 + (first ? t / wx : 0) + ny) % ny;
  unsigned xs[3], ys[3];
  xs[1] = rx;
  xs[0] = !pull ? rx : rx == nx - 1 ? 0 : rx + 1;
  xs[2] = !pull ? rx : rx == 0 ? nx - 1 : rx - 1;
  ys[1] = ry * nx;
  ys[0] = (!pull ? ry : ry == ny - 1 ? 0 : ry + 1) * nx;
  ys[2] = (!pull ? ry : ry == 0 ? ny - 1 : ry - 1) * nx;
  // second pass: a cell of the column
  const int cx = t % bx, cy = t / bx, ox = x0 + cx, oy = y0 + cy;
  const bool second = cy < by && ox < nx && oy < ny;
  const int self = oy * nx + ox, mid = second ? (cy + 1) * wx + cx + 1 : wx + 1;

  auto load = [&](int z, S* f) {
    z = z < 0 ? z + nz : z >= nz ? z - nz : z;
    const S* zs[3] = {src + (!pull ? z : z == nz - 1 ? 0 : z + 1) * zst, src + z * zst,
                      src + (!pull ? z : z == 0 ? nz - 1 : z - 1) * zst};
#pragma unroll
    for (int q = 0; q < NV; ++q) f[q] = (zs[1 + kC[q][2]] + q * ps)[ys[1 + kC[q][1]] + xs[1 + kC[q][0]]];
  };
  auto collide = [&](S* f) {
    if constexpr (sizeof(S) == 8)
      collide_f64(f, R.omega_s, R.omega_b);
    else
      collide_f32_shifted(f, float(R.rho0), float(R.omega_s), float(R.omega_b));
  };

  S next[NV], keep1[NV], keep2[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) next[q] = keep1[q] = keep2[q] = S(0);
  // as in k_step_pair, every lane loads and pulls
  auto arrived = [&] {
#pragma unroll
    for (int q = 0; q < NV; ++q) asm volatile("" : "+v"(next[q]));
  };
  load(z0 - 1, next);
  arrived();
  auto walk = [&](int z, bool more) {
    S(*plane)[kServePairCells] = ring[z & 1];
    S f[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) f[q] = next[q];
    if (more) load(z + 1, next);
    if (kind & PAIR_COLLIDE1) collide(f);
    if (first) {
#pragma unroll
      for (int q = 0; q < NV; ++q) plane[q][t] = f[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const S v = plane[q][mid - kC[q][1] * wx - kC[q][0]];
      if (kC[q][2] < 0) {
        f[q] = v;
      } else {
        f[q] = keep1[q];
        keep1[q] = kC[q][2] == 0 ? v : keep2[q];
        if (kC[q][2] > 0) keep2[q] = v;
      }
    }
    const bool out = second && z > z0;
    if (out && (kind & PAIR_COLLIDE2)) collide(f);
    if (more) arrived();
    if (out) {
      S* to = dst + (z - 1) * zst + self;
#pragma unroll
      for (int q = 0; q < NV; ++q) __builtin_nontemporal_store(f[q], to + q * ps);
    }
  };
  for (int z = z0 - 1; z < z1; ++z) walk(z, true);
  walk(z1, false);
}

// Equilibrium of a plane pulse (rho = 1 + amplitude on one plane normal to
// `axis`, 1 elsewhere, u = 0), the reference's operation order, into the
// run's buffer 0.
template <typename S>
__global__ __launch_bounds__(256) void k_serve_init_pulse(S* __restrict__ f, Lattice L, int axis, int plane,
                                                         double amplitude, double rho0) {
  const int nx = L.nx, ny = L.ny;
  const long long n = (long long)nx * ny * L.nz;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int x = int(i % nx), y = int((i / nx) % ny), z = int(i / ((long long)nx * ny));
  const long long self = L.at(0, y * nx + x, z);
  const int c = axis == 0 ? x : (axis == 1 ? y : z);
  const double rho = (c == plane) ? 1.0 + amplitude : 1.0;
  double fe[NV];
  equilibrium_f64(rho, 0.0, 0.0, 0.0, fe);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    if constexpr (sizeof(S) == 8)
      f[self + q * L.ps] = fe[q];
    else
      f[self + q * L.ps] = float(fe[q] - kT.W[q] * rho0);
  }
}

}  // namespace

hipError_t launch_serve_step(int precision, const ServeBatch& b, int grid, hipStream_t st) {
  if (b.total_items <= 0) return hipSuccess;
  const int blocks = b.total_items < grid ? b.total_items : grid;
  // resident workgroups per CU capped like the stream-collide launches
  const int lds = lds_bytes_for_cap(precision == 0 ? 3 : 4);
  if (precision == 0)
    k_serve_step<double><<<blocks, 256, lds > 0 ? lds : 0, st>>>(b);
  else
    k_serve_step<float><<<blocks, 256, lds > 0 ? lds : 0, st>>>(b);
  return hipGetLastError();
}

hipError_t launch_serve_pair(int precision, const ServeBatch& b, hipStream_t st) {
  if (b.total_items <= 0) return hipSuccess;
  const int blocks = (b.total_items + 7) / 8 * 8;
  if (precision == 0)
    k_serve_pair<double><<<blocks, kServePairCells, 0, st>>>(b);
  else
    k_serve_pair<float><<<blocks, kServePairCells, 0, st>>>(b);
  return hipGetLastError();
}

hipError_t launch_serve_init_pulse(int precision, void* f, const Lattice& L, int axis, int plane,
                                   double amplitude, double rho0, hipStream_t st) {
  const long long cells = (long long)L.nx * L.ny * L.nz;
  const int blocks = int((cells + 255) / 256);
  if (precision == 0)
    k_serve_init_pulse<double><<<blocks, 256, 0, st>>>((double*)f, L, axis, plane, amplitude, rho0);
  else
    k_serve_init_pulse<float><<<blocks, 256, 0, st>>>((float*)f, L, axis, plane, amplitude, rho0);
  return hipGetLastError();
}

}  // namespace lbx
