// bnz_tile64.hpp -- one stage of the FP64 VL step on a tile, in one pass:
// fluxes into LDS, edge EMFs from them, the update of the tile's cells from
// both, so that neither fluxes nor EMFs go through HBM.  The per-face, per-
// edge and per-cell arithmetic is that of the separate kernels
// (bnz_kern64.hpp); single grids and batches share these bodies.
#pragma once
#include "bnz_kern64.hpp"
#include "bnz_tile.hpp"

namespace bnz {

// Slots of a face in LDS: the six hydro fluxes and the two tangential field
// fluxes, in the order RHO..PSC, then the fields of an x face (BY, BZ) or of
// a y face (BX, BZ).
constexpr int NSLOT = 8;

// A 2D tile of TX x TY threads: thread t = ty * TX + tx stands on cell
// (i0 + tx - 1, j0 + ty - 1), computes that cell's lower x and y faces and
// corner EMF, and updates the cell unless it lies on the tile's rim (one
// cell wide on each side, which the neighbouring tiles own).
template <int NT>
struct Tile2Flux {
  const double *sx, *sy;
  int t, tx_stride;
  __device__ __forceinline__ double x(int n, long off) const { return sx[n * NT + t + (int)off]; }
  __device__ __forceinline__ double y(int n, long off) const {
    return sy[n * NT + t + (off ? tx_stride : 0)];
  }
  __device__ __forceinline__ double z(int, long) const { return 0.; }
};
template <int NT>
struct Tile2Emf {  // ex = -F_y[Bz], ey = F_x[Bz] (emf_edge_d<2>), ez from its array
  const double *sx, *sy, *se;
  int t, tx_stride;
  long sy_stride;
  __device__ __forceinline__ double operator()(int comp, long off) const {
    const int o = off >= sy_stride ? tx_stride + (int)(off - sy_stride) : (int)off;
    if (comp == 0) return -sy[7 * NT + t + o];
    if (comp == 1) return sx[7 * NT + t + o];
    return se[t + o];
  }
};

// The ghosts of an updated active cell: its new prim wn and lower faces f.
__device__ __forceinline__ void copy_ghosts64(const Bnd &b, const Geo &g, int i, int j, int k,
                                              const double *wn, const double *f, double *w1,
                                              double *b1) {
  const long sv = g.sv;
  if (b.plain) {  // nothing mirrored: cells and faces have the same images
    const unsigned m[3] = {images<false>(b, 0, i), images<false>(b, 1, j), images<false>(b, 2, k)};
    each_image(b, g, m, i, j, k, [&](long dst, unsigned) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n) w1[n * sv + dst] = wn[n];
#pragma unroll
      for (int a = 0; a < 3; ++a) b1[a * sv + dst] = f[a];
    });
    return;
  }
  scatter_ghosts(
      b, g, i, j, k,
      [&](long dst, unsigned flips) {
#pragma unroll
        for (int n = 0; n < NMODE; ++n) {
          const int a = n >= VX && n <= VZ ? n - VX : n >= BX ? n - BX : 3;
          w1[n * sv + dst] = ((flips >> a) & 1u) ? -wn[n] : wn[n];
        }
      },
      [&](int a, long dst, bool flip) {
        const double v = a == 0 ? f[0] : a == 1 ? f[1] : f[2];
        b1[a * sv + dst] = flip ? -v : v;
      },
      [&](int a, long dst) { b1[a * sv + dst] = 0.; });
}

// LDS doubles of a 2D tile: two faces, the cell EMF and the corner EMF
template <int NT>
constexpr int tile2_lds() {
  return (2 * NSLOT + 2) * NT;
}

// One stage over one tile; every thread must call it.  wf, bf: the stage's
// prim and faces (fluxes, EMFs); w0, b0: the state that is updated.  PRED
// writes prim and faces of every cell it owns (cells outside L keep w0); the
// corrector (DTRED) updates the active cells only, writes their ghosts too
// and returns the CFL speed.  No call writes what another tile's call reads:
// the corrector's faces b1 are neither bf nor b0, its prim w1 may be w0,
// which is read at the thread's own cell alone.  A face whose solver matches
// no region (non-finite speeds) has flux 0.
//   A thread loads its stencil once, up front, and takes its x neighbours and
// their half slopes from the lanes beside it; along y both faces form the half
// slopes, which costs less than another barrier.  Against loading each face's
// stencil for itself (82 loads a thread, slopes of both faces; us per step):
// 1024^2 FMA 207 -> 178, 128^2 FP64 20.3 -> 18.7, 24 FP64 blasts of side 64 ..
// 320 (292 as separate kernels) 219; FP32C, 24 blasts, 140 -> 138.
template <bool PRED, int ORDER, int RS, int TX, int TY, class DT>
__device__ __forceinline__ double stage2_tile(const Geo &g, const double *__restrict__ wf,
                                              const double *__restrict__ bf, const double *w0,
                                              const double *b0, double *w1, double *b1,
                                              const Lims &L, const DT &step_dt, const Box &act,
                                              const Bnd &bnd, int fms_ref, int i0, int j0,
                                              double *lds) {
  constexpr int NT = TX * TY;
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int i = i0 + tx - 1, j = j0 + ty - 1;
  const long sv = g.sv;
  double *sx = lds, *sy = lds + NSLOT * NT, *sc = lds + 2 * NSLOT * NT, *se = sc + NT;
  const bool in = i >= 0 && i < g.nt[0] && j >= 0 && j < g.nt[1];
  const bool reach = in && i >= L.lo[0] - 1 && i <= L.hi[0] + 1 && j >= L.lo[1] - 1 &&
                     j <= L.hi[1] + 1;
  bool gx = false, gy = false;
  // Threads off the grid stand on cell (0, 0), neighbours past the grid's end
  // are the cell itself: what they give is not used.
  const int ic = in ? i : 0, jc = in ? j : 0;
  const long c = (long)jc * g.nt[0] + ic;
  const bool first = tx == 0, last = tx == TX - 1;
  const int oxe = first && ic > 0 ? -1 : last && ic < g.nt[0] - 1 ? 1 : 0;
  const int oyl = jc > 0 ? -g.sy : 0, oyl2 = jc > 1 ? -2 * g.sy : oyl;
  const int oyr = jc < g.nt[1] - 1 ? g.sy : 0;
  double wc[NMODE], wl[NMODE], wr[NMODE], f[NMODE];
  double ym2[NMODE], ym[NMODE], yp[NMODE], xe[NMODE];
#pragma unroll
  for (int n = 0; n < NMODE; ++n) {
    const double *p = wf + n * sv + c;
    wc[n] = p[0];
    if (ORDER == 1 && n != BX) xe[n] = p[oxe];
  }
  const double bnx = bf[c], bny = bf[sv + c];
#pragma unroll
  for (int n = 0; n < NMODE; ++n)
    if (n != BY) {
      const double *p = wf + n * sv + c;
      ym[n] = p[oyl];
      if (ORDER == 1) {
        ym2[n] = p[oyl2];
        yp[n] = p[oyr];
      }
    }
  // x face: a cell's half slope is formed once and passed to the next lane
#pragma unroll
  for (int n = 0; n < NMODE; ++n) {
    if (n == BX) continue;
    if (ORDER == 0) {
      wl[n] = row_left<TX>(wc[n], 0., first);
      wr[n] = wc[n];
    } else {
      const double d = vl_half(wc[n] - row_left<TX>(wc[n], xe[n], first),
                            row_right<TX>(wc[n], xe[n], last) - wc[n]);
      wl[n] = row_left<TX>(wc[n] + d, 0., first);
      wr[n] = wc[n] - d;
    }
  }
  wl[BX] = wr[BX] = bnx;
  if (reach && tx > 0 && i >= L.lo[0])
    if (solve_face<RS>(f, wl, wr, g.gam, g.gamm1i)) {
#pragma unroll
      for (int n = 0; n < 6; ++n) sx[n * NT + t] = f[n];
      sx[6 * NT + t] = f[BY];
      sx[7 * NT + t] = f[BZ];
      gx = true;
    }
  // y face: both cells' half slopes here
#pragma unroll
  for (int n = 0; n < NMODE; ++n) {  // local slot n is variable perm<1>(n)
    if (n == BX) continue;
    const int v = perm<1>(n);
    if (ORDER == 0) {
      wl[n] = ym[v];
      wr[n] = wc[v];
    } else {
      const double dm = wc[v] - ym[v];
      wl[n] = ym[v] + vl_half(ym[v] - ym2[v], dm);
      wr[n] = wc[v] - vl_half(dm, yp[v] - wc[v]);
    }
  }
  wl[BX] = wr[BX] = bny;
  if (reach && ty > 0 && j >= L.lo[1])
    if (solve_face<RS>(f, wl, wr, g.gam, g.gamm1i)) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n) {
        if (n == BX) continue;
        const int v = perm<1>(n);
        sy[(v < 6 ? v : v == BX ? 6 : 7) * NT + t] = f[n];
      }
      gy = true;
    }
  if (!gx)
    for (int n = 0; n < NSLOT; ++n) sx[n * NT + t] = 0.;
  if (!gy)
    for (int n = 0; n < NSLOT; ++n) sy[n * NT + t] = 0.;
  sc[t] = -(wc[VX] * wc[BY] - wc[VY] * wc[BX]);  // ec_comp
  const double dt = step_dt();  // the fluxes did not need it
  __syncthreads();
  // corner EMF of the cell's lower edges (emf_edge_d<2>)
  if (tx > 0 && ty > 0)
    se[t] = (0.5 * (-sx[6 * NT + t - TX] - sx[6 * NT + t] + sy[6 * NT + t - 1] +
                    sy[6 * NT + t]) -
             0.25 * (sc[t - 1] + sc[t] + sc[t - TX - 1] + sc[t - TX]));
  __syncthreads();
  const bool own = in && tx > 0 && tx < TX - 1 && ty > 0 && ty < TY - 1;
  const Tile2Flux<NT> fl{sx, sy, t, TX};
  const Tile2Emf<NT> em{sx, sy, se, t, TX, (long)g.sy};
  if (PRED) {
    if (own)
      update_cell_e<2, true, false>(g, GeoArr{g}, w0, fl, em, b0, b1, w1, L, &dt, act, fms_ref, i,
                                    j, 0);
    return 0.;
  }
  double cds = 0.;
  if (own && i >= act.lo[0] && i < act.lo[0] + act.n[0] && j >= act.lo[1] &&
      j < act.lo[1] + act.n[1]) {
    const auto ghosts = [&](const double *wn, double bx, double by, double bz) {
      if (!near_side(bnd, i, j, 0)) return;
      const double f[3] = {bx, by, bz};
      copy_ghosts64(bnd, g, i, j, 0, wn, f, w1, b1);
    };
    cds = update_cell_e<2, false, true, decltype(em), GeoArr, decltype(fl),
                        decltype(ghosts)>(g, GeoArr{g}, w0, fl, em, b0, b1, w1, L, &dt, act,
                                          fms_ref, i, j, 0, ghosts);
  }
  return cds;
}

// LDS slots per thread of a 3D column.  Shared with the neighbouring rows:
// the plane's y fluxes and what its edges need (X.), its edge EMFs (E.), the
// new By of the plane below (BYU).  Private, here to spare registers while
// the solvers run (P.): the z states of the column and the cell half updated.
enum {
  XFY = 0,                   // hydro fluxes of the y face
  XFB = 6, XZB, XE0, XE2,    // F_x[By], F_z[By], cell EMFs x and z
  EX = 10, EZ,
  BYU = 12,
  PWP = 13,                  // upper z state of the cell below
  PDM = 21,                  // the cell's lower z differences
  PU = 29,                   // conserved, x and y fluxes applied
  PFX = 35, PFY, PBX, PBY,   // F_x[Bz], F_y[Bz]; faces with the Ez terms applied
  NSLOT3 = 39
};

// One stage of a column of a 3D grid: 16 x TY threads stand on the cells
// (i0 + tx - 1, j0 + ty - 1) of a plane and walk the planes kb - 1 .. ke + 1.
// At plane k a thread solves its cell's lower faces and edges; the cell of
// plane k - 1, whose upper faces and edges that completes, is then updated.
// A half slope along x is formed once, by its own cell, and passes to the
// next lane (a row of the tile is one DPP row of 16 lanes), along z to the
// next plane; along y both faces form it.  The plane above is loaded while
// the x and y faces are solved.  Ownership, arguments and arithmetic are
// those of stage2_tile, except that no ghosts are written; every thread must
// call it.
//   Bound by FP64 VALU issue: the separate kernels move about 35 GB per 256^3
// step (24 flux words a cell and stage), this 16.4 (7.4 + 9.0, reads that the
// MALL serves included) and leaves the solves, 1.46 times those of the grid (rims,
// and the two planes more of each run).  The SIMDs issue VALU work 0.64 (predictor)
// and 0.73 (corrector) of the time, the rest being load and barrier waits of two
// waves per SIMD, at 1917 and 2360 us a launch (FMA, 256^3; IEEE 0.72 and 0.79 at
// 2141 and 2742).
// How it got there (FMA, one after another on one card; us per launch): separate
// kernels 3330 / 3760; one 32 x 16 workgroup a CU with every face's stencil
// loaded 2560 / 3740, two of 16 x 16 2410 / 3000 (a workgroup's barrier waits
// then overlap the other's solves), plane above loaded ahead and half slopes
// shared 2100 / 2620, carried values in LDS instead of registers and scratch
// 1940 / 2340, no branches around the solves 1850 / 2260.  Compiled for three
// workgroups a CU it spills (4900 for the corrector); rows of 32 lanes and
// 16 x 32 threads gained nothing; ghosts written from here cost 400.
template <bool PRED, int ORDER, int RS, class GM, int TX, int TY>
__device__ __forceinline__ double stage3_column(const Geo &g, const double *__restrict__ wf,
                                                const double *__restrict__ bf, const double *w0,
                                                const double *__restrict__ b0, double *w1,
                                                double *b1, const Lims &L, const double step_dt,
                                                const Box &act, int fms_ref, int i0, int j0,
                                                int kb, int ke, double *lds) {
  constexpr int NT = TX * TY;
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int i = i0 + tx - 1, j = j0 + ty - 1;
  const long sv = g.sv;
  const GM gm{g};
  const double dt = PRED ? 0.5 * step_dt : step_dt;
  double *s = lds + t;  // slot n of this thread: s[n * NT]
  const int dn = ty > 0 ? -TX : 0, up = ty < TY - 1 ? TX : 0;
  const bool in = i >= 0 && i < g.nt[0] && j >= 0 && j < g.nt[1];
  const bool inI = in && i >= L.lo[0] && i <= L.hi[0], inJ = in && j >= L.lo[1] && j <= L.hi[1];
  const bool upI = in && i >= L.lo[0] && i <= L.hi[0] + 1;
  const bool upJ = in && j >= L.lo[1] && j <= L.hi[1] + 1;
  bool own = in && tx > 0 && tx < TX - 1 && ty > 0 && ty < TY - 1;
  if (!PRED)
    own = own && i >= act.lo[0] && i < act.lo[0] + act.n[0] && j >= act.lo[1] &&
          j < act.lo[1] + act.n[1];
  // Threads off the grid stand on cell (0, 0); neighbours past the grid's end
  // are the cell itself.  What they compute is not used.
  const int ic = in ? i : 0, jc = in ? j : 0;
  const double dlx = gm.dlf(0, ic), dly = gm.dlf(1, jc);
  const ColGeo<std::is_same<GM, GeoUni>::value> ge(dt, dlx, dly, gm.dlf(2, 0));
  const unsigned row = 8u * (unsigned)g.sy, plane = 8u * (unsigned)g.sz;
  const unsigned oxe = tx == 0 && ic > 0 ? -8u : tx == TX - 1 && ic < g.nt[0] - 1 ? 8u : 0u;
  const unsigned oyl = jc > 0 ? row : 0u, oyl2 = jc > 1 ? 2 * row : oyl;
  const unsigned oyr = jc < g.nt[1] - 1 ? row : 0u;
  const unsigned oxy = 8u * (unsigned)(jc * g.nt[0] + ic);

  // carried from plane to plane (of plane k - 1 at the top of iteration k),
  // beside the P. slots and this thread's own XE0 and EX
  double fzl[6];              // lower z flux
  double bzl = 0., eyl = 0.;  // new lower z face; lower edge EMF along y
  double e0y = 0., e1 = 0.;   // cell EMFs: x of (j - 1), y
#pragma unroll
  for (int n = 0; n < 6; ++n) fzl[n] = 0.;
  double cds = 0.;

  const auto solve = [&](double *f, const double *wl, const double *wr) {
#pragma unroll
    for (int n = 0; n < NMODE; ++n) f[n] = 0.;  // left so if no region matches
    solve_face<RS>(f, wl, wr, g.gam, g.gamm1i);
  };
  // the cell's prim, and that of the plane above (loaded an iteration ahead)
  double wc[NMODE], wu[NMODE], bc[3];  // (bc: the cell's lower faces)
  const auto clamp_k = [&](int k) { return (unsigned)min(max(k, 0), g.nt[2] - 1); };
  {
    const unsigned o = oxy + clamp_k(kb - 1) * plane, ob = oxy + clamp_k(kb - 2) * plane;
    const unsigned ou = oxy + clamp_k(kb) * plane;
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      wc[n] = at(wf + n * sv, o);
      wu[n] = at(wf + n * sv, ou);
      if (ORDER == 1 && n != BZ) s[(PDM + n) * NT] = wc[n] - at(wf + n * sv, ob);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) bc[a] = at(bf + a * sv, o);
  }
  for (int k = kb - 1; k <= ke + 1; ++k) {
    const unsigned o = oxy + clamp_k(k) * plane;
    const int km = k - 1;  // the plane being completed
    const bool done = km >= kb;
    const double dlz = gm.dlf(2, (int)clamp_k(k)), dlzm = gm.dlf(2, (int)clamp_k(km));
    double wl[NMODE], wr[NMODE], f[NMODE];
    // The three faces are solved without branches, also where they are
    // outside the stage's range: no cell or edge inside it reads those.

    // ---- z face
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      if (n == BX) continue;
      const int v = perm<2>(n);
      wl[n] = s[(PWP + v) * NT];
      if (ORDER == 0) {
        wr[n] = wc[v];
        s[(PWP + v) * NT] = wc[v];
      } else {
        const double du = wu[v] - wc[v];
        const double d = vl_half(s[(PDM + v) * NT], du);
        wr[n] = wc[v] - d;
        s[(PWP + v) * NT] = wc[v] + d;
        s[(PDM + v) * NT] = du;
      }
    }
    wl[BX] = wr[BX] = bc[2];
    double xe[NMODE];  // the cell beyond the row's end, for the end lanes
    if (ORDER == 1) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) xe[n] = at(wf + n * sv, o + oxe);
    }
    solve(f, wl, wr);
    double fzbx = 0.;  // F_z[Bx]
    {
      const double dtdv = ge.tv(dlzm), az = ge.axy();
#pragma unroll
      for (int n = 0; n < NMODE; ++n) {
        const int v = perm<2>(n);
        if (v < 6) {  // the conserved state of plane k - 1 is complete
          s[(PU + v) * NT] -= dtdv * (az * f[n] - az * fzl[v]);
          fzl[v] = f[n];
        }
        if (v == BX) fzbx = f[n];
        if (v == BY) s[XZB * NT] = f[n];
      }
    }

    // ---- x face
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      if (n == BX) continue;
      if (ORDER == 0) {
        wl[n] = from_left<TX>(wc[n]);
        wr[n] = wc[n];
      } else {
        const double d = vl_half(wc[n] - from_left<TX>(wc[n], xe[n]),
                                 from_right<TX>(wc[n], xe[n]) - wc[n]);
        wl[n] = from_left<TX>(wc[n] + d);
        wr[n] = wc[n] - d;
      }
    }
    wl[BX] = wr[BX] = bc[0];
    solve(f, wl, wr);
    double xd[6];  // the x fluxes of the update
    const double ax = ge.ayz(dlz);
#pragma unroll
    for (int n = 0; n < 6; ++n) xd[n] = ax * from_right<TX>(f[n]) - ax * f[n];
    s[XFB * NT] = f[BY];
    const double fxzn = f[BZ];  // F_x[Bz]

    // ---- y face
    double ym2[NMODE], ym[NMODE], yp[NMODE];
#pragma unroll
    for (int n = 0; n < NMODE; ++n)
      if (n != BY) {
        const double *p = wf + n * sv;
        ym[n] = at(p, o - oyl);
        if (ORDER == 1) {
          ym2[n] = at(p, o - oyl2);
          yp[n] = at(p, o + oyr);
        }
      }
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      if (n == BX) continue;
      const int v = perm<1>(n);
      if (ORDER == 0) {
        wl[n] = ym[v];
        wr[n] = wc[v];
      } else {
        const double dm = wc[v] - ym[v];
        wl[n] = ym[v] + vl_half(ym[v] - ym2[v], dm);
        wr[n] = wc[v] - vl_half(dm, yp[v] - wc[v]);
      }
    }
    wl[BX] = wr[BX] = bc[1];
    solve(f, wl, wr);
    double fybx = 0., fyzn = 0.;  // F_y[Bx], F_y[Bz]
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      const int v = perm<1>(n);
      if (v < 6) s[(XFY + v) * NT] = f[n];
      if (v == BX) fybx = f[n];
      if (v == BZ) fyzn = f[n];
    }

    // ---- cell EMFs
    const double e0n = -(wc[VY] * wc[BZ] - wc[VZ] * wc[BY]);
    const double e1n = (wc[VX] * wc[BZ] - wc[VZ] * wc[BX]);
    const double e2n = -(wc[VX] * wc[BY] - wc[VY] * wc[BX]);
    const double e0 = s[XE0 * NT], fxz = s[PFX * NT], fyz = s[PFY * NT];
    s[XE0 * NT] = e0n;
    s[XE2 * NT] = e2n;
    s[PFX * NT] = fxzn;
    s[PFY * NT] = fyzn;
    // what the rest of the iteration and the next one read from memory
    const double bx0 = PRED ? bc[0] : at(b0, o), by0 = PRED ? bc[1] : at(b0 + sv, o),
                 bz0 = PRED ? bc[2] : at(b0 + 2 * sv, o);
    double wv[NMODE], wn2[NMODE];
    const unsigned ou2 = oxy + clamp_k(k + 2) * plane;
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      wv[n] = PRED ? wc[n] : at(w0 + n * sv, o);
      wn2[n] = at(wf + n * sv, ou2);
    }
    const unsigned on = oxy + clamp_k(k + 1) * plane;
    const double bnx = at(bf, on), bny = at(bf + sv, on), bnz = at(bf + 2 * sv, on);
    __syncthreads();

    // ---- edge EMFs of the cell's lower edges (emf_edge_d<3>); the rows and
    // lanes on the tile's lower rim have no use for theirs
    const double e0yn = s[XE0 * NT + dn], e1xn = from_left<TX>(e1n);
    const double e2y = s[XE2 * NT + dn];
    const double ex = (0.5 * (-fyz - fyzn + s[XZB * NT + dn] + s[XZB * NT]) -
                       0.25 * (e0yn + e0n + e0y + e0));
    const double ey = (0.5 * (-from_left<TX>(fzbx) - fzbx + fxz + fxzn) -
                       0.25 * (e1xn + e1n + from_left<TX>(e1) + e1));
    const double ez = (0.5 * (-s[XFB * NT + dn] - s[XFB * NT] + from_left<TX>(fybx) + fybx) -
                       0.25 * (from_left<TX>(e2n) + e2n + from_left<TX>(e2y) + e2y));
    const double exl = s[EX * NT];
    s[EX * NT] = ex;
    s[EZ * NT] = ez;
    e0y = e0yn;
    e1 = e1n;
    double yd[6];  // the y fluxes of the update
    const double ay = ge.axz(dlz);
#pragma unroll
    for (int n = 0; n < 6; ++n) yd[n] = ay * s[(XFY + n) * NT + up] - ay * s[(XFY + n) * NT];
    __syncthreads();

    // ---- faces (advance_b): those of plane k - 1 get their Ex, Ey terms,
    // those of plane k their Ez terms, the z face all of its own
    double bxl = s[PBX * NT], byl = s[PBY * NT], bzu;
    bxl += ge.tyz(dlzm) * (dly * ey - dly * eyl);
    byl -= ge.txz(dlzm) * (dlx * ex - dlx * exl);
    s[PBX * NT] = bx0 - ge.tyz(dlz) * (dlz * s[EZ * NT + up] - dlz * ez);
    s[PBY * NT] = by0 + ge.txz(dlz) * (dlz * from_right<TX>(ez) - dlz * ez);
    bzu = bz0 - ge.txy() * (dly * from_right<TX>(ey) - dly * ey);
    bzu += ge.txy() * (dlx * s[EX * NT + up] - dlx * ex);
    eyl = ey;
    s[BYU * NT] = byl;
    const double bxr = from_right<TX>(bxl);
    __syncthreads();

    // ---- the cell of plane k - 1 (interp_bc, cons2prim)
    if (done && own) {
      const bool inK = km >= L.lo[2] && km <= L.hi[2];
      const bool upK = km >= L.lo[2] && km <= L.hi[2] + 1;
      const unsigned om = oxy + (unsigned)km * plane;
      if (upI && inJ && inK) put(b1, om, bxl);
      if (inI && upJ && inK) put(b1 + sv, om, byl);
      if (inI && inJ && upK) put(b1 + 2 * sv, om, bzl);
      if (inI && inJ && inK) {
        double uv[NMODE], wn[NMODE];
#pragma unroll
        for (int n = 0; n < 6; ++n) uv[n] = s[(PU + n) * NT];
        uv[BX] = (gm.icm(0, i) * bxl + gm.icp(0, i) * bxr) * gm.dlfi(0, i);
        uv[BY] = (gm.icm(1, j) * byl + gm.icp(1, j) * s[BYU * NT + TX]) * gm.dlfi(1, j);
        uv[BZ] = (gm.icm(2, km) * bzl + gm.icp(2, km) * bzu) * gm.dlfi(2, km);
        cons2prim(wn, uv, g.gam);
#pragma unroll
        for (int n = 0; n < NMODE; ++n) put(w1 + n * sv, om, wn[n]);
        if (!PRED) cds = fmax(cds, cds_cell_g(gm, g, wn, fms_ref, i, j, km));
      } else if (PRED) {
#pragma unroll
        for (int n = 0; n < NMODE; ++n) put(w1 + n * sv, om, at(w0 + n * sv, om));
      }
    }
    bzl = bzu;
    {
      // plane k's conserved state with its x and y fluxes applied
      double uv[NMODE];
      prim2cons(uv, wv, g.gamm1i);
      const double dtdv = ge.tv(dlz);
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        double v = uv[n] - dtdv * xd[n];
        v -= dtdv * yd[n];
        s[(PU + n) * NT] = v;
      }
    }
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      wc[n] = wu[n];
      wu[n] = wn2[n];
    }
    bc[0] = bnx;
    bc[1] = bny;
    bc[2] = bnz;
  }
  return cds;
}

}  // namespace bnz
