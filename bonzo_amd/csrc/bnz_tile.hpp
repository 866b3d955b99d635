// bnz_tile.hpp -- pieces shared by the fused stage kernels (bnz_tile64.hpp,
// bnz_tile32.hpp), which form a stage's fluxes, EMFs and update in one pass
// over a tile: the dt of the step, the CFL maximum of a workgroup, and the
// ghost images of an active cell.
#pragma once
#include "bnz_common.hpp"

namespace bnz {

// The dt of a step, by every workgroup of its first launch (dt_reduce_block's
// rule): each reduces the partials itself, so that the launch that needs dt
// can also be the one that finds it; workgroup 0 records it.  In two halves,
// so that the fluxes, which do not need dt, run while the partials come in:
// load at the start of the kernel, value() (every thread of the NT) where dt
// is first needed.
template <int NT>
struct StepDt {
  double m = 0., tnow = 0., tmax = 0.;
  __device__ __forceinline__ StepDt(const DtFold &f, const double *dev) {
    if (f.npart == 0) {
      m = dev[0];
      return;
    }
    double p[4] = {0., 0., 0., 0.};
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if ((int)threadIdx.x + u * NT < f.npart) p[u] = f.part[threadIdx.x + u * NT];
    for (int q = threadIdx.x + 4 * NT; q < f.npart; q += NT) p[0] = fmax(p[0], f.part[q]);
    m = fmax(fmax(p[0], p[1]), fmax(p[2], p[3]));
    tnow = dev[1];
    tmax = dev[2];
  }
  // a step past t_max, known before dt (step_past_tmax)
  __device__ __forceinline__ bool past(const DtFold &f) const {
    if (f.npart == 0) return m == 0.;
    if (f.use_fixed) return f.fixed_dt == 0.;
    return tmax >= 0. && !(tnow < tmax);
  }
  __device__ __forceinline__ double value(const DtFold &f, double *dev) const {
    if (f.npart == 0) return m;
    __shared__ double red[NT / 64];
    const double mm = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mm;
    __syncthreads();
    double x = red[0];
#pragma unroll
    for (int r = 1; r < NT / 64; ++r) x = fmax(x, red[r]);
    double dt = f.use_fixed ? f.fixed_dt : f.cour / x;
    if (!f.use_fixed && tmax >= 0.) {
      if (!(tnow < tmax))
        dt = 0.;
      else if (tnow + dt > tmax)
        dt = tmax - tnow;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      dev[0] = dt;
      if (dt != 0.) dev[7] = dt;
    }
    return dt;
  }
};

// Maximum over a workgroup of NT threads, valid in thread 0.
template <int NT>
__device__ __forceinline__ double block_max_nt(double v) {
  __shared__ double red[NT / 64];
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = red[0];
#pragma unroll
  for (int q = 1; q < NT / 64; ++q) m = fmax(m, red[q]);
  return m;
}

// The value of the lane to the left (right) in a row of 16 lanes (a DPP row);
// the row's first (last) lane gets its own `end`.  Every lane must be active.
template <int CTRL>
__device__ __forceinline__ int dpp_mov(int end, int v) {
  return __builtin_amdgcn_update_dpp(end, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double end, double v) {
  const int lo = dpp_mov<CTRL>(__double2loint(end), __double2loint(v));
  const int hi = dpp_mov<CTRL>(__double2hiint(end), __double2hiint(v));
  return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float end, float v) {
  return __int_as_float(dpp_mov<CTRL>(__float_as_int(end), __float_as_int(v)));
}
template <int TX, typename T>
__device__ __forceinline__ T from_left(T v, T end = T(0)) {  // row_shr:1
  static_assert(TX == 16, "a row of the tile is a DPP row");
  return dpp_mov<0x111>(end, v);
}
template <int TX, typename T>
__device__ __forceinline__ T from_right(T v, T end = T(0)) {  // row_shl:1
  static_assert(TX == 16, "a row of the tile is a DPP row");
  return dpp_mov<0x101>(end, v);
}
// The same in rows of TX lanes, TX any divisor of 64 from 16 up (wave_shr:1,
// wave_shl:1 and the rows' ends put in by hand); first, last: whether the lane
// is its row's.
template <int TX, typename T>
__device__ __forceinline__ T row_left(T v, T end, bool first) {
  if (TX == 16) return dpp_mov<0x111>(end, v);
  const T x = dpp_mov<0x138>(end, v);
  return first ? end : x;
}
template <int TX, typename T>
__device__ __forceinline__ T row_right(T v, T end, bool last) {
  if (TX == 16) return dpp_mov<0x101>(end, v);
  const T x = dpp_mov<0x130>(end, v);
  return last ? end : x;
}

// Value of array a (a uniform address) at byte offset o: with a 32-bit offset
// the load takes its base from scalar registers and one vector register
// serves every variable of a cell.
template <typename T>
__device__ __forceinline__ T at(const T *a, unsigned o) {
  return *(const T *)((const char *)a + o);
}
template <typename T>
__device__ __forceinline__ void put(T *a, unsigned o, T v) {
  *(T *)((char *)a + o) = v;
}

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ double uniform(double v) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
  const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
  return __hiloint2double(hi, lo);
}

// dt over a cell's volume and faces, and the face areas, as the updates form
// them.  On a uniform grid they are the same for every cell and wait in
// scalar registers.
template <bool UG>
struct ColGeo {
  double dt, dlx, dly;
  __device__ __forceinline__ ColGeo(double t, double x, double y, double) : dt(t), dlx(x), dly(y) {}
  __device__ __forceinline__ double tv(double z) const { return dt / (dlx * dly * z); }
  __device__ __forceinline__ double tyz(double z) const { return dt / (dly * z); }
  __device__ __forceinline__ double txz(double z) const { return dt / (dlx * z); }
  __device__ __forceinline__ double txy() const { return dt / (dlx * dly); }
  __device__ __forceinline__ double ayz(double z) const { return dly * z; }
  __device__ __forceinline__ double axz(double z) const { return dlx * z; }
  __device__ __forceinline__ double axy() const { return dlx * dly; }
};
template <>
struct ColGeo<true> {
  double v, yz, xz, xy, a_yz, a_xz, a_xy;
  __device__ __forceinline__ ColGeo(double t, double x, double y, double z)
      : v(uniform(t / (x * y * z))), yz(uniform(t / (y * z))), xz(uniform(t / (x * z))),
        xy(uniform(t / (x * y))), a_yz(uniform(y * z)), a_xz(uniform(x * z)),
        a_xy(uniform(x * y)) {}
  __device__ __forceinline__ double tv(double) const { return v; }
  __device__ __forceinline__ double tyz(double) const { return yz; }
  __device__ __forceinline__ double txz(double) const { return xz; }
  __device__ __forceinline__ double txy() const { return xy; }
  __device__ __forceinline__ double ayz(double) const { return a_yz; }
  __device__ __forceinline__ double axz(double) const { return a_xz; }
  __device__ __forceinline__ double axy() const { return a_xy; }
};

// The boundaries of a grid, for the kernels that write the ghost cells along
// with the active cells they copy (build_ghosts composes per-axis maps, so
// the ghosts of an active cell are the products of its images per axis).
enum { END_NONE = 0, END_WALL = 1, END_FACE = 2 };  // END_FACE: the image's bit
struct Bnd {
  int a1[3], a2[3];  // first and last active index
  int flag[6];       // BNZ_BC_PERIODIC, _OUTFLOW or _REFLECT per side
  int ng, dims;
  int plain;         // no reflecting side
  int end[3];        // END_*, see close
  // The low ghosts of an axis can mirror a face past its active cells: with a
  // reflecting low side and just ng cells, ghost face a1 - ng mirrors face
  // a2 + 1, which the high side sets.  It then mirrors what that side copies
  // there: face a2 with outflow, else a wall face, 0 (build_ghosts does the
  // same).  Worked out here, once, to keep the kernels short.
  void close() {
    plain = 1;
    for (int a = 0; a < 3; ++a) {
      end[a] = END_NONE;
      if (a >= dims) continue;
      if (flag[2 * a] == BNZ_BC_REFLECT || flag[2 * a + 1] == BNZ_BC_REFLECT) plain = 0;
      if (flag[2 * a] == BNZ_BC_REFLECT && a2[a] - a1[a] + 1 == ng)
        end[a] = flag[2 * a + 1] == BNZ_BC_OUTFLOW ? END_FACE : END_WALL;
    }
  }
};

// Images of index x along one axis, bit 0 x itself, bit 1 + g the low ghost
// a1 - ng + g, bit 1 + ng + g the high ghost a2 + 1 + g.  FACE: the images of
// a face index of the axis's own normal field (mirrored about the wall face).
template <bool FACE>
__host__ __device__ __forceinline__ unsigned images(const Bnd &b, int axis, int x) {
  unsigned m = 1u;
  if (axis >= b.dims) return m;
  const int a1 = b.a1[axis], a2 = b.a2[axis], ng = b.ng, n = a2 - a1 + 1;
  const int lo = b.flag[2 * axis], hi = b.flag[2 * axis + 1];
  if (lo == BNZ_BC_OUTFLOW) {
    if (x == a1) m |= ((1u << ng) - 1) << 1;
  } else {
    const int q = lo == BNZ_BC_PERIODIC ? x - n : FACE ? 2 * a1 - x : 2 * a1 - 1 - x;
    if (q >= a1 - ng && q < a1) m |= 1u << (1 + q - (a1 - ng));
  }
  if (hi == BNZ_BC_OUTFLOW) {
    if (x == a2) m |= ((1u << ng) - 1) << (1 + ng);
    if (FACE && x == a2) m |= b.end[axis];
  } else {
    const int q = hi == BNZ_BC_PERIODIC ? x + n : FACE ? 2 * a2 + 2 - x : 2 * a2 + 1 - x;
    const int q0 = (FACE && hi == BNZ_BC_REFLECT) ? a2 + 2 : a2 + 1;
    if (q >= q0 && q <= a2 + ng) m |= 1u << (1 + ng + q - (a2 + 1));
  }
  return m;
}

// Index of image bit s of x, and whether that side mirrors it.
__host__ __device__ __forceinline__ int image_at(const Bnd &b, int axis, int s, int x,
                                                 bool &flip) {
  flip = false;
  if (s == 0) return x;
  const int g = s - 1;
  flip = b.flag[2 * axis + (g < b.ng ? 0 : 1)] == BNZ_BC_REFLECT;
  return g < b.ng ? b.a1[axis] - b.ng + g : b.a2[axis] + 1 + (g - b.ng);
}

// f(cell index, flips) for every combination of images but the cell itself;
// bit a of flips: mirrored along axis a.
template <class F>
__host__ __device__ __forceinline__ void each_image(const Bnd &b, const Geo &g,
                                                    const unsigned m[3], int i, int j, int k,
                                                    const F &f) {
  for (unsigned mz = m[2]; mz; mz &= mz - 1) {
    bool fz, fy, fx;
    const int kk = image_at(b, 2, __builtin_ctz(mz), k, fz);
    for (unsigned my = m[1]; my; my &= my - 1) {
      const int jj = image_at(b, 1, __builtin_ctz(my), j, fy);
      for (unsigned mx = m[0]; mx; mx &= mx - 1) {
        const int ii = image_at(b, 0, __builtin_ctz(mx), i, fx);
        if (((mx | my | mz) & 1u) && ii == i && jj == j && kk == k) continue;
        f(((long)kk * g.nt[1] + jj) * g.nt[0] + ii,
          (unsigned)fx | ((unsigned)fy << 1) | ((unsigned)fz << 2));
      }
    }
  }
}

// Whether active cell (i, j, k) has images, or a wall face of its own.
__host__ __device__ __forceinline__ bool near_side(const Bnd &b, int i, int j, int k) {
  const int x[3] = {i, j, k};
  bool any = false;
  for (int a = 0; a < 3; ++a)
    if (a < b.dims)
      any = any || x[a] <= b.a1[a] + b.ng || x[a] >= b.a2[a] - b.ng;
  return any;
}

// The ghosts of active cell (i, j, k) after its update: cells(dst, flips)
// copies its cell variables to cell dst, face(a, dst, flip) its face a,
// wall(a, dst) zeroes face a of dst (the wall face of a reflecting side).
// Together over the active cells this writes every ghost cell as build_ghosts
// and the ghost fill do; each target has one source.
template <class CELLS, class FACE, class WALL>
__host__ __device__ __forceinline__ void scatter_ghosts(const Bnd &b, const Geo &g, int i, int j,
                                                        int k, const CELLS &cells,
                                                        const FACE &face, const WALL &wall) {
  const unsigned m[3] = {images<false>(b, 0, i), images<false>(b, 1, j), images<false>(b, 2, k)};
  each_image(b, g, m, i, j, k, cells);
  const int x[3] = {i, j, k};
  for (int a = 0; a < 3; ++a) {
    if (a >= b.dims) {
      each_image(b, g, m, i, j, k, [&](long dst, unsigned) { face(a, dst, false); });
      continue;
    }
    unsigned f[3] = {m[0], m[1], m[2]};
    f[a] = a == 0 ? images<true>(b, 0, i) : a == 1 ? images<true>(b, 1, j) : images<true>(b, 2, k);
    each_image(b, g, f, i, j, k,
               [&](long dst, unsigned flips) { face(a, dst, ((flips >> a) & 1u) != 0); });
    // wall faces, bit 0 the cell's own, bit 1 its upper one, bit 2 the mirror
    // image past the low ghosts, and their images along the other axes
    unsigned walls = b.flag[2 * a] == BNZ_BC_REFLECT && x[a] == b.a1[a] ? 1u : 0u;
    if (x[a] == b.a2[a]) {
      if (b.flag[2 * a + 1] == BNZ_BC_REFLECT) walls |= 2u;
      if (b.end[a] == END_WALL) walls |= 4u;
    }
    unsigned o[3] = {m[0], m[1], m[2]};
    o[a] = 1u;
    const long step = a == 0 ? 1 : a == 1 ? g.sy : g.sz;
    const long self = ((long)k * g.nt[1] + j) * g.nt[0] + i;
#pragma unroll 1
    for (; walls; walls &= walls - 1) {
      const int q = __builtin_ctz(walls);
      const long off = q == 0 ? 0 : q == 1 ? step : -(b.a2[a] - b.a1[a] + b.ng) * step;
      wall(a, self + off);
      each_image(b, g, o, i, j, k, [&](long dst, unsigned) { wall(a, dst + off); });
    }
  }
}

// --------------------------------------------------------------------------
// Host side

inline Bnd bnd_of(const bnz_ctx *c) {
  Bnd b;
  const int lo[3] = {c->i1, c->j1, c->k1}, hi[3] = {c->i2, c->j2, c->k2};
  for (int a = 0; a < 3; ++a) {
    b.a1[a] = lo[a];
    b.a2[a] = hi[a];
  }
  for (int q = 0; q < 6; ++q) b.flag[q] = c->p.bc[q];
  b.ng = c->ng;
  b.dims = c->dims;
  b.close();
  return b;
}

// A launch of tiles with an own range of `span` cells per axis: the tiles'
// counts and origin.  pred: the whole grid (cells outside the limits are
// copied); else the cells of flux3_box(L), whose faces a stage solves.
struct Tiling {
  int o[2], n[2];
  int blocks() const { return n[0] * n[1]; }
};
inline Tiling tiling2(const int *nt, const Lims &L, bool pred, int ex, int ey) {
  Tiling t;
  const int e[2] = {ex, ey};
  for (int a = 0; a < 2; ++a) {
    const int lo = pred ? 0 : L.lo[a] - 1, hi = pred ? nt[a] - 1 : L.hi[a] + 1;
    t.o[a] = lo;
    t.n[a] = (hi - lo + e[a]) / e[a];
  }
  return t;
}

// Workgroups of a 3D stage that a CU holds: 256 threads each, compiled for up
// to 256 registers, with 39 LDS doubles a thread (FP64) or fewer (FP32C).
// FP32C fits three or four, which measured no faster (256^3: 3.24 ms a step
// with two, 3.76 with three, 3.27 with four).
constexpr int STAGE3_PER_CU = 2;

// Cells from which the 3D stages take their workgroups in run_block order
// (256^3: 4.24 -> 4.17 ms a step; 200x144x168 and below are slower so).
constexpr long STAGE3_RUN_CELLS = 1L << 23;

// Columns of a 3D stage (stage3_column): tiles in x and y as tiling2, cut in
// z into runs of nz planes each of which pays two planes of x and y faces
// more.  The runs are chosen so that the workgroups fill the CUs in as few
// and as short rounds as possible (STAGE3_PER_CU workgroups per CU and round).
struct Tiling3 {
  int o[3], n[3], nz, top;  // origin, tiles per axis, planes per run, last plane
  int runs;                 // workgroups in run_block order
  long cost;                // planes walked one after the other, over the rounds
  int blocks() const { return n[0] * n[1] * n[2]; }
};
inline Tiling3 tiling3(const bnz_ctx *c, const Lims &L, bool pred, bool active, int ex,
                       int ey) {
  Tiling3 t;
  t.runs = c->ncell >= STAGE3_RUN_CELLS;
  const int e[2] = {ex, ey};
  const int lo[3] = {c->i1, c->j1, c->k1}, hi[3] = {c->i2, c->j2, c->k2};
  for (int a = 0; a < 3; ++a) {
    const int x0 = pred ? 0 : active ? lo[a] : L.lo[a] - 1;
    const int x1 = pred ? c->nt[a] - 1 : active ? hi[a] : L.hi[a] + 1;
    t.o[a] = x0;
    if (a < 2) {
      t.n[a] = (x1 - x0 + e[a]) / e[a];
    } else {
      t.top = x1;
      const int planes = x1 - x0 + 1;
      const long cols = (long)t.n[0] * t.n[1], slots = (long)STAGE3_PER_CU * c->ncu;
      long best = 0;
      for (int q = 1; q <= planes; ++q) {
        const int run = (planes + q - 1) / q, runs = (planes + run - 1) / run;
        const long cost = (cols * runs + slots - 1) / slots * (run + 2);
        if (!best || cost < best) {
          best = t.cost = cost;
          t.nz = run;
          t.n[2] = runs;
        }
      }
    }
  }
  return t;
}

// The 3D stages address a variable's plane with 32-bit byte offsets.  Below
// the lower bounds a column has too few planes to fill the chip, and the
// separate kernels are faster (us per step, separate -> columns: FP64 64^3
// 151 -> 155, 128^3 862 -> 732; FP32C 64^3 92 -> 104, 128^3 590 -> 530).
constexpr long STAGE3_MAX_CELLS = 1L << 29;
constexpr long STAGE3_MIN_CELLS64 = 400000, STAGE3_MIN_CELLS32 = 1L << 20;

constexpr int TILE3[2] = {16, 16};

// Whether a 3D grid's stages run as columns.  Columns take as long as the planes
// their rounds walk (Tiling3::cost), the separate kernels as long as the grid
// has cells: columns pay where the cells are at least the given share of the
// cells that the walked planes have room for.  Thin sides, which leave most of
// a tile idle, and grids whose last round is nearly empty fall below it.  Over 101
// shapes of 3 to 30000 cells a side no shape is more than 6 % slower than with the
// better of the two.  us per step, separate / columns, at that share: FP64 0.40
// (3x3x30000) 979 / 1454, 0.59 (30x30x1000) 524 / 516, 0.64 (200x16x200) 351 / 359,
// 0.66 (200x8x300) 326 / 283, 0.84 (128^3) 943 / 732; FMA 0.53 0.93 times as fast,
// 0.59 1.02; FP32C 0.62 (1000x3x1000) 1984 / 2612, 0.64 (5x320x300) 277 / 324, 0.71
// (96^3) 244 / 256, 0.73 (322x337x33) 1039 / 965, 0.74 (112^3) 406 / 408, 0.83
// (104^3) 320 / 277.
inline bool columns_pay(const bnz_ctx *c) {
  if (c->ncell > STAGE3_MAX_CELLS ||
      c->ncell < (c->f32 ? STAGE3_MIN_CELLS32 : STAGE3_MIN_CELLS64))
    return false;
  const int ex = TILE3[0] - 2, ey = TILE3[1] - 2;
  const long cost = tiling3(c, integr_lims(c, 0), true, !c->f32, ex, ey).cost +
                    tiling3(c, integr_lims(c, c->order), false, !c->f32, ex, ey).cost;
  const double room = (double)ex * ey * STAGE3_PER_CU * c->ncu * (double)cost;
  const double share = c->f32 ? 0.725 : c->p.precision == BNZ_PREC_FP64_FMA ? 0.55 : 0.63;
  return 2. * (double)c->ncell >= share * room;
}

// Whether a 2D grid is too thin for tiles: long grids some ten cells across
// with their ghosts, where a tile's row or column is mostly idle.  us per step,
// separate / tiles: FP64 200000x3 514 / 542, 3x200000 601 / 561, 4x150000 472 /
// 424 (FMA 200000x3 504 / 517); FP32C 3x22222 61 / 66, 4x20000 58 / 60, 5x18181
// 59 / 58, 22222x3 55 / 37 (its tile is wider than high).  Short grids are bound
// by their launches, of which tiles have fewer (FP32C 3x2000 27 / 22).
inline bool thin2(const bnz_ctx *c) {
  if (c->f32) return c->nt[0] <= 10 && c->ncell > 1L << 17;
  return c->nt[1] <= 9 && c->ncell > 1L << 20 && c->p.precision == BNZ_PREC_FP64;
}

// Grids whose stages run as fused passes: 2D and 3D Van-Leer steps in the
// default placement (bnz_set_tuning 0, 0, 0) of grids that fill their tiles.
// The upwind EMF, characteristic limiting and user boundaries keep the separate
// kernels.
inline bool fused_stages(const bnz_ctx *c) {
  return c->dims >= 2 && !(c->dims == 3 ? !c->columns : thin2(c)) && !c->p.tintegr &&
         !c->p.ct_upwind && !c->p.char_proj && c->npass == 0 && c->flux_chunk == 0 &&
         c->emf_chunk == 0 && c->update_chunk == 0;
}

// Cells up to which a 2D stage takes its small tile (16 x 8: more workgroups
// on an idle chip; 128^2 18.7 us a step).
constexpr long TILE2_SMALL_CELLS = 1L << 16;

// Own cells of the tiles, and the partials their launches can leave.  Beyond
// the small tile FP64 takes 16 x 16 threads, whose 256 registers hold the
// stencils loaded up front (1024^2 FMA 178 us a step; 32 x 16 threads with the
// 128 registers that two workgroups a CU leave them 406, one a CU 232, 16 x 16
// with 168 registers 224), FP32C 32 x 16, which fit there (24 blasts 138 us a
// step with either; fewer rim cells, 32 x 32 is slower).
constexpr int TILE2_BIG64[2] = {16, 16}, TILE2_BIG32[2] = {32, 16}, TILE2_SMALL[2] = {16, 8};

// Threads of a launch of tiles of e[0] x e[1] threads.
inline long tile_threads(const int *nt, const Lims &L, bool pred, const int *e) {
  return (long)tiling2(nt, L, pred, e[0] - 2, e[1] - 2).blocks() * e[0] * e[1];
}

// Whether an FP64 2D grid takes the small tile: its workgroups find a CU each,
// or neither tile's do and the grid is below TILE2_SMALL_CELLS or covered with
// four fifths of the threads (a thin grid of 12 rows: 18 with ghosts are 3
// rows of small tiles, 2 of big).  us per step, FP64, small / big tile (256
// CUs): 128^2 (230 / 100 workgroups) 18.5 / 20.3, 160^2 (336 / 144) 25.1 / 20.5,
// 200^2 (525 / 225) 25.7 / 21.1, 300x190 (726 / 308) 26.9 / 28.1, 250^2 (836 /
// 361) 28.0 / 28.0, 11111x12 63 / 77, 83333x12 345 / 495 (separate kernels 449).
inline bool tile_small64(const bnz_ctx *c, const Lims &L, bool pred) {
  const auto fits = [&](const int *e) {
    return tiling2(c->nt, L, pred, e[0] - 2, e[1] - 2).blocks() <= c->ncu;
  };
  if (fits(TILE2_SMALL)) return true;
  if (fits(TILE2_BIG64)) return false;
  return c->ncell <= TILE2_SMALL_CELLS ||
         5 * tile_threads(c->nt, L, pred, TILE2_SMALL) <=
             4 * tile_threads(c->nt, L, pred, TILE2_BIG64);
}

// Whether an FP32C one does, which holds more waves a CU: by cells (200^2 20.9 /
// 23.4, 250^2 22.5 / 22.6), or where it takes nine tenths of the threads, as on
// grids that use little of the big tile's rows of 32 (8x14285 45 / 56, 8x107142
// 202 / 343, separate 305; 10x93750 223 / 295, 12x83333 278 / 283).
inline bool tile_small32(const bnz_ctx *c, const Lims &L, bool pred) {
  return c->ncell <= TILE2_SMALL_CELLS ||
         10 * tile_threads(c->nt, L, pred, TILE2_SMALL) <=
             9 * tile_threads(c->nt, L, pred, TILE2_BIG32);
}

// Partials that the launches of a grid's stages can leave, whatever the tile.
inline long tile_parts(const bnz_ctx *c) {
  long n = 0;
  for (const bool pred : {true, false}) {
    const Lims L = integr_lims(c, pred ? 0 : c->order);
    if (c->dims == 3) {
      n = std::max<long>(n, tiling3(c, L, pred, !c->f32, TILE3[0] - 2, TILE3[1] - 2).blocks());
      continue;
    }
    for (const int *e : {TILE2_BIG64, TILE2_BIG32, TILE2_SMALL})
      n = std::max<long>(n, tiling2(c->nt, L, pred, e[0] - 2, e[1] - 2).blocks());
  }
  return n;
}

// A pending dt over more partials than this is reduced by a launch of its own,
// not by every workgroup of the stage: on the first step after an upload of a
// large grid (k_dt_partial leaves one per 256 cells), and on every step of a 2D
// grid of more tiles than that (FP64 from about 900^2 on: 1024^2 leaves 5476),
// which then is three launches (k_dt_final takes 5 us there).
constexpr int DT_PARTS_IN_STAGE = 4096;

}  // namespace bnz
