// lbx_lattice.hip -- stream-collide and field kernels on periodic lattices
// (gfx950).
//
// The reference step (src/AmrSim.cpp:124-135, 109-122; include/AmrSim.h:89-94)
// is: copy now -> next with ghosts, collide valid cells, refill ghosts,
// pull-stream valid+1 ghost layer into a fresh array, swap.  That is four
// passes over 15 populations per step.  Here one pass does pull + collide:
// h'(x) = C(S(h))(x), reading population q of the upstream cell x - c_q and
// writing the collided populations of x.  Each z-plane stores its 15
// population planes in turn (x fastest), so every load and store of a
// wavefront is a contiguous 64-element run (shifted by at most one element
// for c_x = +-1).
//
// Bandwidth bound: 15 loads + 15 stores per lattice update and ~430 FP64
// add/mul (+5 divisions).  No MFMA: there is no dense contraction here.
#include <hip/hip_runtime.h>

#include "d3q15.h"
#include "lbx_internal.h"

#pragma clang fp contract(off)

namespace lbx {
namespace {

// Source offsets of the 15 populations of cell (x, y, z) on a periodic
// lattice.  xs/ys/zo are indexed by 1 + c: the upstream coordinate of
// x is x - c, so index 0 (c = -1) holds x+1, 1 holds x, 2 (c = +1) holds x-1.
struct Upstream {
  int xs[3], ys[3];
  long long zo[3];
};

__device__ __forceinline__ Upstream upstream(int x, int y, int z, const Lattice& L) {
  Upstream u;
  const int row = L.nx;
  u.xs[0] = (x == L.nx - 1) ? 0 : x + 1;
  u.xs[1] = x;
  u.xs[2] = (x == 0) ? L.nx - 1 : x - 1;
  u.ys[0] = ((y == L.ny - 1) ? 0 : y + 1) * row;
  u.ys[1] = y * row;
  u.ys[2] = ((y == 0) ? L.ny - 1 : y - 1) * row;
  u.zo[0] = ((z == L.nz - 1) ? 0 : z + 1) * L.zs;
  u.zo[1] = z * L.zs;
  u.zo[2] = ((z == 0) ? L.nz - 1 : z - 1) * L.zs;
  return u;
}

// self: (z*zs, y*nx + x) of the cell itself
template <typename S, bool STREAM>
__device__ __forceinline__ void load_cell(const S* __restrict__ src, const Lattice& L, long long selfz,
                                          int selfp, const Upstream& u, S* f) {
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const long long off = STREAM ? (u.zo[1 + kC[q][2]] + u.ys[1 + kC[q][1]] + u.xs[1 + kC[q][0]])
                                 : selfz + selfp;
    f[q] = __builtin_nontemporal_load(src + off + q * L.ps);
  }
}

// Index of the population opposite to q (c_opp = -c_q).
__device__ constexpr int opposite(int q) {
  int o = 0;
  for (int p = 0; p < NV; ++p)
    if (kC[p][0] == -kC[q][0] && kC[p][1] == -kC[q][1] && kC[p][2] == -kC[q][2]) o = p;
  return o;
}

// Pull with halfway bounce-back: population q of cell (x, y, z) comes from
// x - c_q, unless that crosses a wall face (an axis with its bit in
// L.walls), where the cell's own opposite population, which left towards
// the wall, returns instead.  Periodic axes wrap as in load_cell.
template <typename S>
__device__ __forceinline__ void load_cell_walls(const S* __restrict__ src, const Lattice& L, int x, int y,
                                                int z, long long selfz, int selfp, const Upstream& u, S* f) {
  const bool wx = L.walls & 1u, wy = L.walls & 2u, wz = L.walls & 4u;
  const bool lo_x = wx && x == 0, hi_x = wx && x == L.nx - 1;
  const bool lo_y = wy && y == 0, hi_y = wy && y == L.ny - 1;
  const bool lo_z = wz && z == 0, hi_z = wz && z == L.nz - 1;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const bool bounce = (kC[q][0] > 0 && lo_x) || (kC[q][0] < 0 && hi_x) || (kC[q][1] > 0 && lo_y) ||
                        (kC[q][1] < 0 && hi_y) || (kC[q][2] > 0 && lo_z) || (kC[q][2] < 0 && hi_z);
    const long long off = bounce ? selfz + opposite(q) * L.ps + selfp
                                 : u.zo[1 + kC[q][2]] + q * L.ps + u.ys[1 + kC[q][1]] + u.xs[1 + kC[q][0]];
    f[q] = __builtin_nontemporal_load(src + off);
  }
}

template <typename S>
__device__ __forceinline__ void store_cell(S* __restrict__ dst, const Lattice& L, long long selfz, int selfp,
                                           const S* f) {
#pragma unroll
  for (int q = 0; q < NV; ++q) __builtin_nontemporal_store(f[q], dst + selfz + q * L.ps + selfp);
}

// Resident workgroups per CU are capped at launch time by reserving
// dynamic LDS (LaunchShape::lds_bytes); the kernels do not use it.  With 30
// streams per cell, fewer resident wavefronts contend less for DRAM: at
// 256^3 one 512-lane workgroup per CU (FP64) and four 256-lane workgroups
// per CU (FP32) run ~8% and ~7% faster than uncapped launches.  Every
// element is loaded once per pass (the x+-1 neighbours of a wavefront are
// in the lines its own row fetches), so loads are non-temporal too.
template <int KIND, bool WALLS>
__global__ __launch_bounds__(512) void k_step_f64(const double* __restrict__ src,
                                                  double* __restrict__ dst, Lattice L, Relax r) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= L.nx || y >= L.ny) return;
  const long long selfz = (long long)z * L.zs;
  const int selfp = y * L.nx + x;
  double f[NV];
  if (KIND == STEP_COLLIDE) {
    load_cell<double, false>(src, L, selfz, selfp, Upstream{}, f);
  } else if (WALLS) {
    load_cell_walls<double>(src, L, x, y, z, selfz, selfp, upstream(x, y, z, L), f);
  } else {
    const Upstream u = upstream(x, y, z, L);
    load_cell<double, true>(src, L, selfz, selfp, u, f);
  }
  if (KIND != STEP_STREAM) collide_f64(f, r.omega_s, r.omega_b);
  store_cell<double>(dst, L, selfz, selfp, f);
}

template <int KIND, bool WALLS>
__global__ __launch_bounds__(512) void k_step_f32s(const float* __restrict__ src,
                                                   float* __restrict__ dst, Lattice L, Relax r) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= L.nx || y >= L.ny) return;
  const long long selfz = (long long)z * L.zs;
  const int selfp = y * L.nx + x;
  float f[NV];
  if (KIND == STEP_COLLIDE) {
    load_cell<float, false>(src, L, selfz, selfp, Upstream{}, f);
  } else if (WALLS) {
    load_cell_walls<float>(src, L, x, y, z, selfz, selfp, upstream(x, y, z, L), f);
  } else {
    const Upstream u = upstream(x, y, z, L);
    load_cell<float, true>(src, L, selfz, selfp, u, f);
  }
  if (KIND != STEP_STREAM)
    collide_f32_shifted(f, float(r.rho0), float(r.omega_s), float(r.omega_b));
  store_cell<float>(dst, L, selfz, selfp, f);
}

// Two fused steps in one pass over the state: h'' = C(S(C(S(h)))).  One step
// alone moves 240 B (FP64) per update and runs at the copy rate (256^3 FP64:
// 652 us a step), so only a pass that keeps the state between two steps on
// the chip is faster.  A workgroup owns a BX x BY column of cells and walks
// its z-planes: it computes the first step of each plane over the column and
// a ring of one cell (redundantly with its neighbours), hands the plane over
// in LDS, and forms the second step of the plane below, whose populations
// with c_z = -1 come from this plane, those with c_z = 0 and +1 from the two
// planes before (carried in registers).  Two LDS planes alternate, so a
// plane costs one barrier; the loads of the next plane are in flight while
// this one is collided.  Each cell's arithmetic is that of two single
// passes, so the results are the same bits.
//
// Bound: what the ring adds (64 x 8: 1.29 x the first-step collisions, but
// only 1.07 x the reads beyond L2, the rest hits there since each XCD takes
// a contiguous range of columns) and, with one workgroup of 11 waves per CU
// (LDS, and ~150 VGPRs in FP64), the part of the collisions that the loads
// do not cover; in FP32 the vector units are busy 90 % of the time.
// Measured (us per step, single pass -> pair): 256^3 FP64 652 -> 389, FP32
// 328 -> 206 (5.2 and 4.9 TB/s, of a copy's 6.5); 128^3 FP64 88 -> 57, FP32
// 42.5 -> 29.  FP64 408 and FP32 216 with the next plane's loads waited for
// before the second step.  Slower: 32 x 8 and 64 x 4 columns with two
// workgroups per CU, separate waves for the two steps, non-temporal loads (the
// ring misses L2); in FP32 32 x 16 (221), 64 x 12 (229), 128 x 5 (226) and 64 x
// 7 with two workgroups (238).
constexpr int pair_cells(int bx, int by) { return bx ? (bx + 2) * (by + 2) : kPairCells; }
constexpr int pair_threads(int bx, int by) { return (pair_cells(bx, by) + 63) / 64 * 64; }

template <typename S>
__device__ __forceinline__ void collide_any(S* f, const Relax& r) {
  if constexpr (sizeof(S) == 8)
    collide_f64(f, r.omega_s, r.omega_b);
  else
    collide_f32_shifted(f, float(r.rho0), float(r.omega_s), float(r.omega_b));
}

// The faces (x low, x high, y low, ...: bits 0 to 5) through which population
// q can enter a cell.
__device__ constexpr unsigned wall_faces(int q) {
  unsigned m = 0;
  for (int d = 0; d < 3; ++d) m |= kC[q][d] > 0 ? 1u << 2 * d : kC[q][d] < 0 ? 2u << 2 * d : 0u;
  return m;
}

// The x and y faces with walls that cell (x, y, .) touches.
__device__ __forceinline__ unsigned lateral_faces(int x, int y, const Lattice& L) {
  unsigned m = 0;
  if (L.walls & 1u) m |= (x == 0 ? 1u : 0u) | (x == L.nx - 1 ? 2u : 0u);
  if (L.walls & 2u) m |= (y == 0 ? 4u : 0u) | (y == L.ny - 1 ? 8u : 0u);
  return m;
}

// BX = 0: columns of p.bx x p.by cells (1 % slower than the same known here)
template <typename S, int BX, int BY, bool WALLS>
__global__ __launch_bounds__(pair_threads(BX, BY)) void k_step_pair(const S* __restrict__ src,
                                                                    S* __restrict__ dst, Lattice L, Relax r,
                                                                    PairShape p) {
  constexpr int NC = pair_cells(BX, BY);
  __shared__ S ring[2][NV][NC];
  const int bx = BX ? BX : p.bx, by = BX ? BY : p.by, wx = bx + 2;
  // XCD k takes the k-th eighth of the columns (consecutive workgroups go
  // to the 8 XCDs in turn; the grid is a multiple of 8)
  const int w = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (w >= p.tx * p.ty * p.tz) return;
  const int x0 = (w % p.tx) * bx, y0 = (w / p.tx % p.ty) * by, z0 = w / (p.tx * p.ty) * p.depth;
  const int z1 = min(z0 + p.depth, L.nz);
  const int t = threadIdx.x;

  // first step: cell t of the ring, its periodic image in the domain
  const bool first = t < wx * (by + 2);
  const int rx = (x0 - 1 + (first ? t % wx : 0) + L.nx) % L.nx, ry = (y0 - 1 + (first ? t / wx : 0) + L.ny) % L.ny;
  const Upstream u = upstream(rx, ry, 0, L);
  // second step: cell (ox, oy) of the column
  const int cx = t % bx, cy = t / bx, ox = x0 + cx, oy = y0 + cy;
  const bool second = cy < by && ox < L.nx && oy < L.ny;
  const int self = oy * L.nx + ox;
  const int mid = WALLS || cy < by ? (cy + 1) * wx + cx + 1 : wx + 1;

  // wall faces that a cell touches in x and y, and those that plane z lies on,
  // as a mask of wall_faces(); a population that comes from behind one of
  // them is the cell's own opposite population
  const unsigned first_faces = WALLS ? lateral_faces(rx, ry, L) : 0;
  const unsigned second_faces = WALLS ? lateral_faces(ox, oy, L) : 0;
  auto z_faces = [&](int z) { return (L.walls & 4u) ? (z == 0 ? 16u : 0u) | (z == L.nz - 1 ? 32u : 0u) : 0u; };

  auto load = [&](int z, S* f) {
    z = z < 0 ? z + L.nz : z >= L.nz ? z - L.nz : z;
    const S* zs[3] = {src + (z == L.nz - 1 ? 0 : z + 1) * L.zs, src + z * L.zs,
                      src + (z == 0 ? L.nz - 1 : z - 1) * L.zs};
    const unsigned faces = WALLS ? first_faces | z_faces(z) : 0;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const S* from = zs[1 + kC[q][2]] + q * L.ps;
      unsigned at = u.ys[1 + kC[q][1]] + u.xs[1 + kC[q][0]];
      if (WALLS && (faces & wall_faces(q))) {
        from = zs[1] + opposite(q) * L.ps;
        at = u.ys[1] + u.xs[1];
      }
      f[q] = from[at];
    }
  };

  S next[NV];   // first step's populations of the coming plane
  S keep1[NV];  // second step of the coming plane: c_z = 0 and +1
  S keep2[NV];  // ... of the plane after it: c_z = +1
  S back[NV];   // walls: what the coming plane's c_z = -1 populations bounce to
#pragma unroll
  for (int q = 0; q < NV; ++q) next[q] = keep1[q] = keep2[q] = back[q] = S(0);
  auto pull = [&](const S(*plane)[NC], S* f) {
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
  };
  auto store = [&](int z, const S* f) {
    S* out = dst + z * L.zs + self;
#pragma unroll
    for (int q = 0; q < NV; ++q) __builtin_nontemporal_store(f[q], out + q * L.ps);
  };
  if constexpr (WALLS) {
    if (first) load(z0 - 1, next);
    for (int z = z0 - 1; z <= z1; ++z) {
      S(*plane)[NC] = ring[z & 1];
      if (first) {
        S f[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) f[q] = next[q];
        if (z < z1) load(z + 1, next);
        collide_any(f, r);
#pragma unroll
        for (int q = 0; q < NV; ++q) plane[q][t] = f[q];
      }
      __syncthreads();
      if (second) {
        S f[NV];
        pull(plane, f);
        // the plane just formed is the own plane of the next second step:
        // its bounced populations return from this cell
#pragma unroll
        for (int q = 0; q < NV; ++q) {
          if (kC[q][2] < 0) {
            if ((second_faces | z_faces(z - 1)) & wall_faces(q)) f[q] = back[q];
            back[q] = plane[opposite(q)][mid];
          } else if ((second_faces | z_faces(z)) & wall_faces(q)) {
            keep1[q] = plane[opposite(q)][mid];
          }
        }
        if (z > z0) {
          collide_any(f, r);
          store(z - 1, f);
        }
      }
    }
  } else {
    // Every lane loads and pulls (one without a cell, another's): behind a
    // branch, as with walls, the loaded values are copied where it joins and
    // so waited for there, before the second step.  They are waited for after
    // it, but before the stores are issued, or the wait would be for those as
    // well.  (With walls the registers do not suffice for this in FP64, and it
    // gained nothing in FP32.)
    auto arrived = [&] {
#pragma unroll
      for (int q = 0; q < NV; ++q) asm volatile("" : "+v"(next[q]));
    };
    load(z0 - 1, next);
    arrived();
    auto walk = [&](int z, bool more) {
      S(*plane)[NC] = ring[z & 1];
      S f[NV];
#pragma unroll
      for (int q = 0; q < NV; ++q) f[q] = next[q];
      if (more) load(z + 1, next);
      collide_any(f, r);
      if (first) {
#pragma unroll
        for (int q = 0; q < NV; ++q) plane[q][t] = f[q];
      }
      __syncthreads();
      pull(plane, f);
      const bool out = second && z > z0;
      if (out) collide_any(f, r);
      if (more) arrived();
      if (out) store(z - 1, f);
    };
    for (int z = z0 - 1; z < z1; ++z) walk(z, true);
    walk(z1, false);
  }
}

// T fused steps of a small lattice in one pass.  Such a lattice leaves a pass
// nothing to do but wait: a launch, the loads' way to memory and back and one
// collision take 4 us whether it has 500 cells or 10000.  A workgroup takes a
// block of cells and a ring of T - 1 around it, a cell per lane: every lane
// takes its cell's first step, the lanes one in from the edge the second, and
// so on, the populations between them in LDS (one at rest stays in its lane).
// The ring repeats work (4x4x4 cells of 3 steps: 8 x the first collision), on
// CUs that have nothing else to do as long as the blocks fit them in one
// round.  Us per step, one pass a step -> so: 10x10x50 FP64 4.1 -> 2.75, FP32
// 4.0 -> 2.3; 32^3 5.2 -> 3.6 and 4.0 -> 2.9; 40^3 5.7 -> 5.0 and 5.0 -> 3.9.
template <typename S, bool WALLS, int T>
__global__ __launch_bounds__(kBlockCells) void k_step_block(const S* __restrict__ src, S* __restrict__ dst, Lattice L,
                                                            Relax r, BlockShape b) {
  __shared__ S moved[NV - 1][kBlockCells];
  const int w = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // an XCD takes neighbouring blocks
  if (w >= b.n[0] * b.n[1] * b.n[2]) return;
  constexpr int R = T - 1;
  const int ex = b.b[0] + 2 * R, ey = b.b[1] + 2 * R, ez = b.b[2] + 2 * R, t = threadIdx.x;
  const int lx = t % ex, ly = t / ex % ey, lz = t / (ex * ey);
  const bool on = lz < ez;
  const int x = w % b.n[0] * b.b[0] + lx - R, y = w / b.n[0] % b.n[1] * b.b[1] + ly - R;
  const int z = w / (b.n[0] * b.n[1]) * b.b[2] + lz - R;
  auto wrapped = [](int v, int n) { return (v % n + n) % n; };
  const int wx = wrapped(x, L.nx), wy = wrapped(y, L.ny), wz = on ? wrapped(z, L.nz) : 0;
  unsigned faces = 0;
  if (WALLS) {
    faces = lateral_faces(wx, wy, L);
    if (L.walls & 4u) faces |= (wz == 0 ? 16u : 0u) | (wz == L.nz - 1 ? 32u : 0u);
  }
  S f[NV];
  if (on) {
    const Upstream u = upstream(wx, wy, wz, L);
    const long long own = L.at(0, wy * L.nx + wx, wz);
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      long long at = u.zo[1 + kC[q][2]] + u.ys[1 + kC[q][1]] + u.xs[1 + kC[q][0]] + q * L.ps;
      if (WALLS && (faces & wall_faces(q))) at = own + opposite(q) * L.ps;
      f[q] = src[at];
    }
    collide_any(f, r);
  }
#pragma unroll
  for (int s = 1; s < T; ++s) {
    if (s > 1) __syncthreads();
    if (on) {
#pragma unroll
      for (int q = 1; q < NV; ++q) moved[q - 1][t] = f[q];
    }
    __syncthreads();
    if (lx >= s && lx < ex - s && ly >= s && ly < ey - s && lz >= s && lz < ez - s) {
#pragma unroll
      for (int q = 1; q < NV; ++q) {
        if (WALLS && (faces & wall_faces(q)))
          f[q] = moved[opposite(q) - 1][t];
        else
          f[q] = moved[q - 1][t - (kC[q][2] * ey + kC[q][1]) * ex - kC[q][0]];
      }
      collide_any(f, r);
    }
  }
  if (lx >= R && lx < ex - R && ly >= R && ly < ey - R && lz >= R && lz < ez - R && x < L.nx && y < L.ny && z < L.nz) {
    const long long own = L.at(0, y * L.nx + x, z);
#pragma unroll
    for (int q = 0; q < NV; ++q) dst[own + q * L.ps] = f[q];
  }
}

dim3 grid_of(const Lattice& L, LaunchShape s) {
  return dim3((L.nx + s.bx - 1) / s.bx, (L.ny + s.by - 1) / s.by, L.nz);
}

// ------------------------------------------------------------ field kernels

__device__ __forceinline__ int region_cell(const Region& R, int i, int& x, int& y, int& z) {
  const int n0 = R.n[0], n1 = R.n[1];
  const int a = i % n0;
  const int t = i / n0;
  const int b = t % n1;
  const int c = t / n1;
  x = R.lo[0] + a;
  y = R.lo[1] + b;
  z = R.lo[2] + c;
  return i;
}

template <typename S>
__global__ __launch_bounds__(256) void k_equilibrium(S* __restrict__ f, Lattice L, Region R,
                                                     const double* __restrict__ rho,
                                                     const double* __restrict__ u, double rho0) {
  const int n = R.n[0] * R.n[1] * R.n[2];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int x, y, z;
  region_cell(R, i, x, y, z);
  const long long selfz = (long long)z * L.zs;
  const int selfp = y * L.nx + x;
  double fe[NV];
  equilibrium_f64(rho[i], u[i], u[n + i], u[2 * n + i], fe);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    if constexpr (sizeof(S) == 8)
      f[selfz + q * L.ps + selfp] = fe[q];
    else
      f[selfz + q * L.ps + selfp] = float(fe[q] - kT.W[q] * rho0);
  }
}

// FP64 populations of cell (x, y, z).  Without PULL they are stored at the
// cell.  With PULL the lattice holds the post-collision state g of the
// previous step and f = S(g) is gathered from the upstream cells exactly as
// the stream-only pass would (periodic wrap or bounce-back walls), so a
// reader sees the same bits as after that pass.
template <typename S, bool PULL>
__device__ __forceinline__ void cell_at(const S* __restrict__ f, const Lattice& L, int x, int y, int z,
                                        double rho0, double* g) {
  const long long selfz = (long long)z * L.zs;
  const int selfp = y * L.nx + x;
  S v[NV];
  if (!PULL)
    load_cell<S, false>(f, L, selfz, selfp, Upstream{}, v);
  else if (L.walls)
    load_cell_walls<S>(f, L, x, y, z, selfz, selfp, upstream(x, y, z, L), v);
  else
    load_cell<S, true>(f, L, selfz, selfp, upstream(x, y, z, L), v);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    if constexpr (sizeof(S) == 8)
      g[q] = v[q];
    else
      g[q] = kT.W[q] * rho0 + double(v[q]);
  }
}

template <typename S, bool PULL>
__global__ __launch_bounds__(256) void k_pack(const S* __restrict__ f, Lattice L, Region R,
                                              double* __restrict__ out, double rho0) {
  const int n = R.n[0] * R.n[1] * R.n[2];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int x, y, z;
  region_cell(R, i, x, y, z);
  double g[NV];
  cell_at<S, PULL>(f, L, x, y, z, rho0, g);
#pragma unroll
  for (int q = 0; q < NV; ++q) out[q * (long long)n + i] = g[q];
}

template <typename S>
__global__ __launch_bounds__(256) void k_unpack(S* __restrict__ f, Lattice L, Region R,
                                                const double* __restrict__ in, double rho0) {
  const int n = R.n[0] * R.n[1] * R.n[2];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int x, y, z;
  region_cell(R, i, x, y, z);
  const long long self = L.at(0, y * L.nx + x, z);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    if constexpr (sizeof(S) == 8)
      f[self + q * L.ps] = in[q * (long long)n + i];
    else
      f[self + q * L.ps] = float(in[q * (long long)n + i] - kT.W[q] * rho0);
  }
}

template <typename S, bool PULL>
__global__ __launch_bounds__(256) void k_hydro(const S* __restrict__ f, Lattice L, Region R,
                                               double* __restrict__ rho, double* __restrict__ u,
                                               double rho0) {
  const int n = R.n[0] * R.n[1] * R.n[2];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int x, y, z;
  region_cell(R, i, x, y, z);
  double g[NV];
  cell_at<S, PULL>(f, L, x, y, z, rho0, g);
  double r, u0, u1, u2;
  hydro_f64(g, r, u0, u1, u2);
  rho[i] = r;
  u[i] = u0;
  u[n + i] = u1;
  u[2 * n + i] = u2;
}

// k_hydro for every box of a level (blockIdx.y): a launch per box is 4 us, more
// than most boxes take.
template <typename S, bool PULL>
__global__ __launch_bounds__(256) void k_hydro_boxes(const S* __restrict__ f, Lattice L,
                                                     const PatchDesc* __restrict__ boxes, int first_box, int nbox,
                                                     double* __restrict__ rho, double* __restrict__ u, double rho0) {
  for (int b = blockIdx.y; b < nbox; b += gridDim.y) {
    const PatchDesc& B = boxes[first_box + b];
    const int n0 = B.hi[0] - B.lo[0] + 1, n1 = B.hi[1] - B.lo[1] + 1, n = n0 * n1 * (B.hi[2] - B.lo[2] + 1);
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) continue;
    const int t = i / n0, x = i - t * n0, z = t / n1, y = t - z * n1;
    double g[NV], r, u0, u1, u2;
    cell_at<S, PULL>(f, L, B.lo[0] + x, B.lo[1] + y, B.lo[2] + z, rho0, g);
    hydro_f64(g, r, u0, u1, u2);
    const long long at = B.first - boxes[first_box].first;
    rho[at + i] = r;
    u[3 * at + i] = u0;
    u[3 * at + n + i] = u1;
    u[3 * at + 2ll * n + i] = u2;
  }
}

constexpr int kTagX = 32, kTagY = 16;  // k_tag_gradient's tile
constexpr int kTagGroups = 1024;       // and the workgroups it cuts z for
// Cells from which a tile pays: k_tag against it, 32^3 6.4 and 8.8 us (FP32
// 6.8 and 8.2), 48^3 13.4 and 10.7 (9.7 and 8.2).
constexpr long long kTagTiled = 64000;
// ... and its lanes per cell, rings and idle ones counted, up to which it does.
// Whole calls, k_tag against the tiles, in us: 192x160x128 (1.5) 2.8 times the
// kernel's time; 64^3 (3.8) 57 and 55, 4 rows of 1000x1000 (4.6) 667 and 554
// (FP32 499 and 460), 32x32x400 (6) 80 and 72 (61 and 62), 8x256x256 (7) 92 and
// 91 (76 and 78), 3x600x600 (13) 209 and 275, 4x1000x1000 (10) 614 and 1350,
// 1x256x256 (57) 35 and 59.
constexpr int kTagLanes = 6;

// ErrorEst on device data: tag[c] = 1 (c = (z*ny + y)*nx + x) where
// CRIT 0: |grad rho|^2 > thr2, central differences with periodic wrap;
// CRIT 1: |u|^2 > thr2.  rho and u are exactly what k_hydro returns.
template <typename S, int CRIT, bool PULL>
__global__ __launch_bounds__(256) void k_tag(const S* __restrict__ f, Lattice L, double rho0, double thr2,
                                             unsigned char* __restrict__ tag) {
  const long long n = (long long)L.nx * L.ny * L.nz;
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  const int x = int(c % L.nx), y = int((c / L.nx) % L.ny), z = int(c / ((long long)L.nx * L.ny));
  auto hydro_at = [&](int xx, int yy, int zz, double& r, double& u0, double& u1, double& u2) {
    double g[NV];
    cell_at<S, PULL>(f, L, xx, yy, zz, rho0, g);
    hydro_f64(g, r, u0, u1, u2);
  };
  double s;
  if (CRIT == 0) {
    double rp, rm, u0, u1, u2;
    hydro_at(x == L.nx - 1 ? 0 : x + 1, y, z, rp, u0, u1, u2);
    hydro_at(x == 0 ? L.nx - 1 : x - 1, y, z, rm, u0, u1, u2);
    const double gx = (rp - rm) * 0.5;
    hydro_at(x, y == L.ny - 1 ? 0 : y + 1, z, rp, u0, u1, u2);
    hydro_at(x, y == 0 ? L.ny - 1 : y - 1, z, rm, u0, u1, u2);
    const double gy = (rp - rm) * 0.5;
    hydro_at(x, y, z == L.nz - 1 ? 0 : z + 1, rp, u0, u1, u2);
    hydro_at(x, y, z == 0 ? L.nz - 1 : z - 1, rm, u0, u1, u2);
    const double gz = (rp - rm) * 0.5;
    s = gx * gx + gy * gy + gz * gz;
  } else {
    double r, u0, u1, u2;
    hydro_at(x, y, z, r, u0, u1, u2);
    s = u0 * u0 + u1 * u1 + u2 * u2;
  }
  tag[c] = s > thr2 ? 1 : 0;
}

// k_tag's criterion 0 with each density formed once per tile instead of six
// times: a workgroup marches a tile of kTagX x kTagY cells, its outer ring
// included, through `depth` planes of z; the densities of the plane below and
// above are the lane's own, those beside it come through LDS.  Bound by the
// cells' one read: 192x160x128 after a step 354 -> 123 us (FP32 190 -> 90),
// 256^3 1495 -> 605 us (788 -> 370); 178 us with the tiles dealt to the XCDs in
// turn, 156 and 149 us with tiles of 64x16 and 64x8.
template <typename S, bool PULL>
__global__ __launch_bounds__(kTagX* kTagY) void k_tag_gradient(const S* __restrict__ f, Lattice L, double rho0,
                                                               double thr2, int tx, int ty,
                                                               int groups, int depth,
                                                               unsigned char* __restrict__ tag) {
  __shared__ double plane[2][kTagY][kTagX];
  const int lx = threadIdx.x, ly = threadIdx.y;
  const int w = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // an XCD takes neighbouring tiles
  if (w >= groups) return;
  const int x = (w % tx) * (kTagX - 2) + lx - 1, y = (w / tx % ty) * (kTagY - 2) + ly - 1;
  const int z0 = w / (tx * ty) * depth, z1 = min(z0 + depth, L.nz);
  const bool on = x <= L.nx && y <= L.ny;
  const bool inner = lx > 0 && lx < kTagX - 1 && ly > 0 && ly < kTagY - 1 && x < L.nx && y < L.ny;
  const int wx = x < 0 ? L.nx - 1 : x == L.nx ? 0 : x, wy = y < 0 ? L.ny - 1 : y == L.ny ? 0 : y;
  auto density = [&](int z) {
    double g[NV], r, u0, u1, u2;
    cell_at<S, PULL>(f, L, wx, wy, z < 0 ? L.nz - 1 : z == L.nz ? 0 : z, rho0, g);
    hydro_f64(g, r, u0, u1, u2);
    return r;
  };
  double below = 0.0, here = 0.0, above = 0.0;
  if (on) {
    below = density(z0 - 1);
    here = density(z0);
    plane[z0 & 1][ly][lx] = here;
  }
  for (int z = z0; z < z1; ++z) {
    __syncthreads();  // plane z is there, and the one it replaces has been read
    if (on) {
      above = density(z + 1);
      plane[(z + 1) & 1][ly][lx] = above;
    }
    if (inner) {
      const double(&p)[kTagY][kTagX] = plane[z & 1];
      const double gx = (p[ly][lx + 1] - p[ly][lx - 1]) * 0.5;
      const double gy = (p[ly + 1][lx] - p[ly - 1][lx]) * 0.5;
      const double gz = (above - below) * 0.5;
      const double s = gx * gx + gy * gy + gz * gz;
      tag[((long long)z * L.ny + y) * L.nx + x] = s > thr2 ? 1 : 0;
    }
    below = here;
    here = above;
  }
}

// Block sum of 4 doubles in a fixed order: wavefront butterfly, then the
// wavefront partials in index order.
__device__ __forceinline__ void block_sum4(double v[4], double* out) {
  __shared__ double part[4][4];  // [wave][component], 256 threads = 4 waves
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    double s = v[c];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    v[c] = s;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0)
    for (int c = 0; c < 4; ++c) part[wave][c] = v[c];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int c = 0; c < 4; ++c) out[c] = ((part[0][c] + part[1][c]) + part[2][c]) + part[3][c];
}

template <typename S, bool PULL>
__global__ __launch_bounds__(256) void k_conservation(const S* __restrict__ f, Lattice L,
                                                      double rho0, double* __restrict__ partials) {
  const long long n = (long long)L.nx * L.ny * L.nz;
  const long long plane = (long long)L.nx * L.ny;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    double g[NV];
    const long long pc = i % plane;
    cell_at<S, PULL>(f, L, int(pc % L.nx), int(pc / L.nx), int(i / plane), rho0, g);
    acc[0] += mode_of<0>(g, std::make_integer_sequence<int, NV>{});
    acc[1] += mode_of<1>(g, std::make_integer_sequence<int, NV>{});
    acc[2] += mode_of<2>(g, std::make_integer_sequence<int, NV>{});
    acc[3] += mode_of<3>(g, std::make_integer_sequence<int, NV>{});
  }
  block_sum4(acc, partials + 4 * blockIdx.x);
}

// The same sums over the valid cells of patched boxes (2 ghost layers, see
// PatchDesc), every patch in one launch: workgroup (c, b) of the grid
// (chunks, npatch) adds the c-th strided share of patch b's valid cells, x
// fastest, into partials[4 * (b * chunks + c)].
template <typename S>
__global__ __launch_bounds__(256) void k_patch_conservation(const S* __restrict__ f,
                                                            const PatchDesc* __restrict__ patches, double rho0,
                                                            double* __restrict__ partials) {
  const PatchDesc& P = patches[blockIdx.y];
  const int nx = P.hi[0] - P.lo[0] + 1, ny = P.hi[1] - P.lo[1] + 1, nz = P.hi[2] - P.lo[2] + 1;
  const int n = nx * ny * nz;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int x = i % nx, t = i / nx, y = t % ny, z = t / ny;
    const long long li = P.at(x + 2, y + 2, z + 2);
    double g[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      if constexpr (sizeof(S) == 8)
        g[q] = f[li + q * P.qs];
      else
        g[q] = kT.W[q] * rho0 + double(f[li + q * P.qs]);
    }
    acc[0] += mode_of<0>(g, std::make_integer_sequence<int, NV>{});
    acc[1] += mode_of<1>(g, std::make_integer_sequence<int, NV>{});
    acc[2] += mode_of<2>(g, std::make_integer_sequence<int, NV>{});
    acc[3] += mode_of<3>(g, std::make_integer_sequence<int, NV>{});
  }
  block_sum4(acc, partials + 4 * ((long long)blockIdx.y * gridDim.x + blockIdx.x));
}

__global__ __launch_bounds__(256) void k_reduce_partials(const double* __restrict__ partials,
                                                         int nblocks, double* __restrict__ out) {
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int b = threadIdx.x; b < nblocks; b += 256)
    for (int c = 0; c < 4; ++c) acc[c] += partials[4 * b + c];
  __shared__ double res[4];
  block_sum4(acc, res);
  __syncthreads();
  if (threadIdx.x < 4) out[threadIdx.x] = res[threadIdx.x];
}

int blocks_for(long long n) { return int((n + 255) / 256); }

// Plain streaming copy (one read + one write per element): the achievable
// read+write bandwidth ceiling, and the calibration kernel for counter-based
// traffic measurements.  16-byte elements, one per lane, non-temporal on both
// sides: the fastest plain copy shape measured on gfx950.
typedef double copy_vec __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(256) void k_copy(const copy_vec* __restrict__ a, copy_vec* __restrict__ b,
                                              long long n) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) __builtin_nontemporal_store(__builtin_nontemporal_load(a + i), b + i);
}

}  // namespace

int lds_bytes_for_cap(int cap) {
  static int per_cu = -1, per_block = -1;
  if (per_cu < 0) {
    int dev = 0;
    per_cu = 64 * 1024;
    per_block = 64 * 1024;
    if (hipGetDevice(&dev) == hipSuccess) {
      (void)hipDeviceGetAttribute(&per_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev);
      (void)hipDeviceGetAttribute(&per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    }
  }
  if (cap <= 0) return 0;
  const int bytes = per_cu / cap - 512;
  return (bytes > 0 && bytes <= per_block) ? bytes : -1;
}

LaunchShape default_shape(const Lattice& L, int precision) {
  LaunchShape s;
  const int lanes = precision == 0 ? 512 : 256;
  s.bx = L.nx < 256 ? L.nx : 256;
  s.by = lanes / s.bx;
  if (s.by > L.ny) s.by = L.ny;
  if (s.by < 1) s.by = 1;
  s.cap = precision == 0 ? 1 : 4;
  s.lds_bytes = lds_bytes_for_cap(s.cap);
  if (s.lds_bytes < 0) {
    s.cap = 0;
    s.lds_bytes = 0;
  }
  return s;
}

#define LBX_STEP_LAUNCH(KERNEL, SRC, DST)                                                          \
  do {                                                                                          \
    const dim3 grid = grid_of(L, s), block(s.bx, s.by, 1);                                      \
    const bool w = L.walls != 0;                                                                \
    switch (kind) {                                                                             \
      case STEP_FUSED:                                                                          \
        if (w) KERNEL<STEP_FUSED, true><<<grid, block, s.lds_bytes, st>>>(SRC, DST, L, r);      \
        else KERNEL<STEP_FUSED, false><<<grid, block, s.lds_bytes, st>>>(SRC, DST, L, r);       \
        break;                                                                                  \
      case STEP_COLLIDE:                                                                        \
        KERNEL<STEP_COLLIDE, false><<<grid, block, s.lds_bytes, st>>>(SRC, DST, L, r);          \
        break;                                                                                  \
      case STEP_STREAM:                                                                         \
        if (w) KERNEL<STEP_STREAM, true><<<grid, block, s.lds_bytes, st>>>(SRC, DST, L, r);     \
        else KERNEL<STEP_STREAM, false><<<grid, block, s.lds_bytes, st>>>(SRC, DST, L, r);      \
        break;                                                                                  \
    }                                                                                           \
    return hipGetLastError();                                                                   \
  } while (0)

hipError_t launch_step_f64(StepKind kind, const double* src, double* dst, const Lattice& L,
                           const Relax& r, LaunchShape s, hipStream_t st) {
  LBX_STEP_LAUNCH(k_step_f64, src, dst);
}

hipError_t launch_step_f32s(StepKind kind, const float* src, float* dst, const Lattice& L,
                            const Relax& r, LaunchShape s, hipStream_t st) {
  LBX_STEP_LAUNCH(k_step_f32s, src, dst);
}

static int compute_units() {
  static const int cus = [] {
    int dev = 0, n = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    return n < 1 ? 256 : n;
  }();
  return cus;
}

// Blocks of k_step_block for a lattice, or none (steps = 0): the first of
// three shapes whose blocks fit the CUs in one round.  In one round a launch
// takes 7 to 10 us (FP64) whatever the lattice; a second round loses what the
// fused steps save (48^3 FP64 6.8 to 7.5 us a step in two rounds, 6.2 in
// single passes).  Of 15 shapes swept at 16^3 to 40^3 and 10x10x50 these are
// the fastest: 4x4x4 of 3 steps at 24^3 (3.15 us, the 2-step blocks 3.2 and
// more), 8x4x4 of 2 at 32^3 (3.6; 4x4x8 of 3 steps 4.0), 8x8x4 at 40^3.  In FP32
// two blocks of 6x6x6 may share a CU, which then takes 4.7 us a step whatever the
// lattice, and 0.5 more with walls: from 90000 cells on less than single passes or
// the same (48^3 5.1 and 4.7 us, with walls 5.2 and 5.2, 36x36x72 5.0 and 4.6,
// 60x60x30 4.9 and 5.0), below more (64x36x36 4.5 and 4.9, 199x15x30 4.8 and 5.4,
// 90x15x63 between walls 4.9 and 5.4).  One to a CU 103x10x41 4.2 and 4.1,
// 11x369x11 4.2 and 3.6.
constexpr long long kBlockShared = 90000;
BlockShape block_shape(const Lattice& L, int precision) {
  // steps, cells of a block, blocks per CU at most
  static constexpr int kShapes[4][5] = {{3, 4, 4, 4, 1}, {2, 8, 4, 4, 1}, {2, 8, 8, 4, 1}, {2, 6, 6, 6, 2}};
  const long long n[3] = {L.nx, L.ny, L.nz};
  for (const int(&c)[5] : kShapes) {
    if (c[4] > 1 && precision == 0) continue;
    const long long room = (n[0] * n[1] * n[2] < kBlockShared ? 1 : c[4]) * (long long)compute_units();
    BlockShape b{};
    b.steps = c[0];
    long long blocks = 1;
    for (int d = 0; d < 3; ++d) {
      b.b[d] = c[1 + d];
      b.n[d] = int((n[d] + c[1 + d] - 1) / c[1 + d]);
      blocks = blocks > room ? blocks : blocks * b.n[d];
    }
    if (blocks <= room) return b;
  }
  return BlockShape{};
}

// Shape of the two-step pass for a lattice, or none (tx = 0) where two single
// passes are the faster.  Every workgroup count that fills the device for one
// or more rounds is a candidate: rounds x (planes of a workgroup + 2 of the
// ring + 1 to start) x the time of a plane, taken as 6.8 us (FP64) and 4.1 us
// (FP32), and 4.4 and 2.8 us where both buffers stay in the 256 MB MALL.  A
// single pass is taken at 5.3 TB/s.  These place the line between the two and
// are no figures of the kernel, which takes 5.9 and 3.1 us a plane at 256^3 and
// 128^3 alike: of 150 drawn lattices of each type none that takes the pair is
// the slower for it.  At 64^3 the rule takes the pair
// in FP64 (10.2 against 12.4 us a step) and not in FP32 (6.9 against 5.9); at
// 48^3 in neither (7.1 against 6.4, 5.6 against 4.7); at 96x80x72 in both (18.5
// against 25.7, 12.2 against 12.9).
// Columns are 64 x 8 or 32 x 16 cells, or, where that wastes enough of them at
// the lattice's edges, an even part of a row (or all of it) with as many rows
// as the ring has room for.  Their rows cross the lines that a wave's lanes
// share, which is dearer: 1.2 x the time of a plane (1.35 x below 32 cells) and
// 1.5 x beyond the MALL cover what was measured.  Us per step, with the two
// and so: 72^3 FP64 18.6 and 14.4, 100^3 FP64 37.5 and 32.4 (FP32 23.3 and
// 20.2), 48x48x256 21.7 and 18.6 (15.4 and 11.9), 10x256x256 33.0 and 24.4;
// taken there too it would be slower at 250^3 (405 and 478, 229 and 310) and
// 161x130x97 (70 and 71, 40.5 and 42).
PairShape pair_shape(const Lattice& L, int precision) {
  const int cus = compute_units();
  PairShape best{};
  const double bytes = double(L.elems()) * (precision == 0 ? 8 : 4);
  const bool mall = 2 * bytes <= 256e6;
  const double plane_us = precision == 0 ? (mall ? 4.4 : 6.8) : (mall ? 2.8 : 4.1);
  double best_us = 2 * (2 * bytes / 5.3e6);  // two single passes
  auto consider = [&](int bx, int by, double factor) {
    const long long tx = (L.nx + bx - 1) / bx, ty = (L.ny + by - 1) / by;
    if (tx * ty > (1 << 20)) return;
    for (int chunks = 1; 2 * chunks <= L.nz || chunks == 1; ++chunks) {
      const int depth = (L.nz + chunks - 1) / chunks;
      const long long n = tx * ty * ((L.nz + depth - 1) / depth);
      const long long rounds = (n + cus - 1) / cus;
      const double us = double(rounds) * (depth + 3) * plane_us * factor;
      if (us < best_us) {
        best_us = us;
        best = PairShape{bx, by, (int)tx, (int)ty, (L.nz + depth - 1) / depth, depth};
      }
      if (rounds > 16) break;  // deeper splits only add ring planes
    }
  };
  consider(kPairWide[0], kPairWide[1], 1.0);
  consider(kPairSquare[0], kPairSquare[1], 1.0);
  for (int parts = 1; parts <= L.nx; ++parts) {
    const int bx = (L.nx + parts - 1) / parts, rows = kPairCells / (bx + 2) - 2;
    if (rows < 1) continue;
    if (bx < 16 && parts > 1) break;
    const int pieces = (L.ny + rows - 1) / rows;
    consider(bx, (L.ny + pieces - 1) / pieces, !mall ? 1.5 : bx < 32 && parts > 1 ? 1.35 : 1.2);
  }
  return best;
}

template <typename S>
static hipError_t step_pair(const S* src, S* dst, const Lattice& L, const Relax& r, const PairShape& p,
                            hipStream_t st) {
  constexpr int wx = kPairWide[0], wy = kPairWide[1], qx = kPairSquare[0], qy = kPairSquare[1];
  const unsigned grid = unsigned(((long long)p.tx * p.ty * p.tz + 7) / 8 * 8);
  const bool walls = L.walls != 0, wide = p.bx == wx && p.by == wy, square = p.bx == qx && p.by == qy;
  if (wide && walls)
    k_step_pair<S, wx, wy, true><<<grid, pair_threads(wx, wy), 0, st>>>(src, dst, L, r, p);
  else if (wide)
    k_step_pair<S, wx, wy, false><<<grid, pair_threads(wx, wy), 0, st>>>(src, dst, L, r, p);
  else if (square && walls)
    k_step_pair<S, qx, qy, true><<<grid, pair_threads(qx, qy), 0, st>>>(src, dst, L, r, p);
  else if (square)
    k_step_pair<S, qx, qy, false><<<grid, pair_threads(qx, qy), 0, st>>>(src, dst, L, r, p);
  else if (walls)
    k_step_pair<S, 0, 0, true><<<grid, pair_threads(0, 0), 0, st>>>(src, dst, L, r, p);
  else
    k_step_pair<S, 0, 0, false><<<grid, pair_threads(0, 0), 0, st>>>(src, dst, L, r, p);
  return hipGetLastError();
}

template <typename S>
static hipError_t step_block(const S* src, S* dst, const Lattice& L, const Relax& r, const BlockShape& b, int steps,
                             hipStream_t st) {
  const int grid = (b.n[0] * b.n[1] * b.n[2] + 7) / 8 * 8, ring = 2 * (steps - 1);
  const int threads = ((b.b[0] + ring) * (b.b[1] + ring) * (b.b[2] + ring) + 63) / 64 * 64;
  if (steps == 3 && L.walls)
    k_step_block<S, true, 3><<<grid, threads, 0, st>>>(src, dst, L, r, b);
  else if (steps == 3)
    k_step_block<S, false, 3><<<grid, threads, 0, st>>>(src, dst, L, r, b);
  else if (L.walls)
    k_step_block<S, true, 2><<<grid, threads, 0, st>>>(src, dst, L, r, b);
  else
    k_step_block<S, false, 2><<<grid, threads, 0, st>>>(src, dst, L, r, b);
  return hipGetLastError();
}

hipError_t launch_step_block(int precision, const void* src, void* dst, const Lattice& L, const Relax& r,
                             const BlockShape& b, int steps, hipStream_t st) {
  if (steps < 2 || steps > b.steps) return hipErrorInvalidValue;
  if (precision == 0) return step_block((const double*)src, (double*)dst, L, r, b, steps, st);
  return step_block((const float*)src, (float*)dst, L, r, b, steps, st);
}

hipError_t launch_step_pair(int precision, const void* src, void* dst, const Lattice& L, const Relax& r,
                            const PairShape& p, hipStream_t st) {
  if (p.tx < 1) return hipErrorInvalidValue;
  if (precision == 0) return step_pair((const double*)src, (double*)dst, L, r, p, st);
  return step_pair((const float*)src, (float*)dst, L, r, p, st);
}

hipError_t launch_equilibrium(int precision, void* f, const Lattice& L, const Region& R,
                              const double* rho, const double* u, double rho0, hipStream_t st) {
  const long long n = (long long)R.n[0] * R.n[1] * R.n[2];
  if (precision == 0)
    k_equilibrium<double><<<blocks_for(n), 256, 0, st>>>((double*)f, L, R, rho, u, rho0);
  else
    k_equilibrium<float><<<blocks_for(n), 256, 0, st>>>((float*)f, L, R, rho, u, rho0);
  return hipGetLastError();
}

// Launch KERNEL<S, ..., PULL> for the storage precision and the pull flag.
#define LBX_PULL_LAUNCH(KERNEL, GRID, ...)                                                              \
  do {                                                                                                \
    if (precision == 0 && pull)                                                                       \
      KERNEL<double, true><<<GRID, 256, 0, st>>>((const double*)f, __VA_ARGS__);                      \
    else if (precision == 0)                                                                          \
      KERNEL<double, false><<<GRID, 256, 0, st>>>((const double*)f, __VA_ARGS__);                     \
    else if (pull)                                                                                    \
      KERNEL<float, true><<<GRID, 256, 0, st>>>((const float*)f, __VA_ARGS__);                        \
    else                                                                                              \
      KERNEL<float, false><<<GRID, 256, 0, st>>>((const float*)f, __VA_ARGS__);                       \
  } while (0)

hipError_t launch_pack_f(int precision, bool pull, const void* f, const Lattice& L, const Region& R,
                         double* out, double rho0, hipStream_t st) {
  const long long n = (long long)R.n[0] * R.n[1] * R.n[2];
  LBX_PULL_LAUNCH(k_pack, blocks_for(n), L, R, out, rho0);
  return hipGetLastError();
}

hipError_t launch_unpack_f(int precision, void* f, const Lattice& L, const Region& R,
                           const double* in, double rho0, hipStream_t st) {
  const long long n = (long long)R.n[0] * R.n[1] * R.n[2];
  if (precision == 0)
    k_unpack<double><<<blocks_for(n), 256, 0, st>>>((double*)f, L, R, in, rho0);
  else
    k_unpack<float><<<blocks_for(n), 256, 0, st>>>((float*)f, L, R, in, rho0);
  return hipGetLastError();
}

hipError_t launch_hydro(int precision, bool pull, const void* f, const Lattice& L, const Region& R,
                        double* rho, double* u, double rho0, hipStream_t st) {
  const long long n = (long long)R.n[0] * R.n[1] * R.n[2];
  LBX_PULL_LAUNCH(k_hydro, blocks_for(n), L, R, rho, u, rho0);
  return hipGetLastError();
}

hipError_t launch_hydro_boxes(int precision, bool pull, const void* f, const Lattice& L, const PatchDesc* boxes,
                              int first_box, int nbox, long long max_cells, double* rho, double* u, double rho0,
                              hipStream_t st) {
  const dim3 grid(blocks_for(max_cells), nbox < 65535 ? nbox : 65535);
  LBX_PULL_LAUNCH(k_hydro_boxes, grid, L, boxes, first_box, nbox, rho, u, rho0);
  return hipGetLastError();
}

template <typename S, bool PULL>
static void tag_launch(int criterion, const S* f, const Lattice& L, double rho0, double thr2, unsigned char* tag,
                int blocks, hipStream_t st) {
  if (criterion == 1)
    return k_tag<S, 1, PULL><<<blocks, 256, 0, st>>>(f, L, rho0, thr2, tag);
  const long long cells = (long long)L.nx * L.ny * L.nz;
  const int tx = (L.nx + kTagX - 3) / (kTagX - 2), ty = (L.ny + kTagY - 3) / (kTagY - 2);
  const long long columns = (long long)tx * ty;
  const long long want = columns * L.nz / kTagGroups;  // planes per workgroup that leave kTagGroups of them
  const int depth = want < 2 ? 2 : want > 32 ? 32 : (int)want;
  const long long tz = (L.nz + depth - 1) / depth;
  if (cells < kTagTiled || columns * (L.nz + 2 * tz) * (kTagX * kTagY) > kTagLanes * cells)
    return k_tag<S, 0, PULL><<<blocks, 256, 0, st>>>(f, L, rho0, thr2, tag);
  const int groups = int(columns * tz);
  k_tag_gradient<S, PULL><<<(groups + 7) / 8 * 8, dim3(kTagX, kTagY), 0, st>>>(f, L, rho0, thr2, tx, ty, groups, depth,
                                                                              tag);
}

hipError_t launch_tag(int precision, bool pull, int criterion, const void* f, const Lattice& L, double rho0,
                      double thr2, unsigned char* tag, hipStream_t st) {
  const long long n = (long long)L.nx * L.ny * L.nz;
  const int blocks = int((n + 255) / 256);
  if (precision == 0 && pull)
    tag_launch<double, true>(criterion, (const double*)f, L, rho0, thr2, tag, blocks, st);
  else if (precision == 0)
    tag_launch<double, false>(criterion, (const double*)f, L, rho0, thr2, tag, blocks, st);
  else if (pull)
    tag_launch<float, true>(criterion, (const float*)f, L, rho0, thr2, tag, blocks, st);
  else
    tag_launch<float, false>(criterion, (const float*)f, L, rho0, thr2, tag, blocks, st);
  return hipGetLastError();
}

hipError_t launch_conservation(int precision, bool pull, const void* f, const Lattice& L, double rho0,
                               double* partials, int nblocks, double* out, hipStream_t st) {
  LBX_PULL_LAUNCH(k_conservation, nblocks, L, rho0, partials);
  k_reduce_partials<<<1, 256, 0, st>>>(partials, nblocks, out);
  return hipGetLastError();
}

hipError_t launch_patch_conservation(int precision, const void* f, const PatchDesc* patches, int npatch,
                                     int chunks, double rho0, double* partials, double* out, hipStream_t st) {
  const dim3 grid(chunks, npatch);
  if (precision == 0)
    k_patch_conservation<double><<<grid, 256, 0, st>>>((const double*)f, patches, rho0, partials);
  else
    k_patch_conservation<float><<<grid, 256, 0, st>>>((const float*)f, patches, rho0, partials);
  k_reduce_partials<<<1, 256, 0, st>>>(partials, chunks * npatch, out);
  return hipGetLastError();
}

hipError_t launch_copy(const double* a, double* b, long long n, hipStream_t st) {
  const long long nv = n / 2;  // whole 16-byte elements; callers pass even n
  k_copy<<<(unsigned)((nv + 255) / 256), 256, 0, st>>>((const copy_vec*)a, (copy_vec*)b, nv);
  return hipGetLastError();
}

}  // namespace lbx
