// bnz_tile32.hpp -- one stage of the FP32-compensated VL step on a tile in
// one pass, as bnz_tile64.hpp does for FP64, from the bodies of
// bnz_kern32.hpp.
#pragma once
#include "bnz_kern32.hpp"
#include "bnz_tile.hpp"

namespace bnz {

// The ghosts of an updated active cell: its hi words uh, FP32 prim w and
// lower faces f (the low words have none, see Ghost32).
__device__ __forceinline__ void copy_ghosts32(const Bnd &b, const Geo &g, const Corr32 &a, int i,
                                              int j, int k, const float *uh, const double *w,
                                              const double *f) {
  const long sv = g.sv;
  if (b.plain) {  // nothing mirrored: cells and faces have the same images
    const unsigned m[3] = {images<false>(b, 0, i), images<false>(b, 1, j), images<false>(b, 2, k)};
    each_image(b, g, m, i, j, k, [&](long dst, unsigned) {
#pragma unroll
      for (int n = 0; n < 6; ++n) a.uh[n * sv + dst] = uh[n];
#pragma unroll
      for (int n = 0; n < NMODE; ++n) a.w32[n * sv + dst] = (float)w[n];
#pragma unroll
      for (int q = 0; q < 3; ++q) a.b1[q * sv + dst] = f[q];
    });
    return;
  }
  scatter_ghosts(
      b, g, i, j, k,
      [&](long dst, unsigned flips) {
#pragma unroll
        for (int n = 0; n < 6; ++n) {
          const int x = n >= MX && n <= MZ ? n - MX : 3;
          a.uh[n * sv + dst] = ((flips >> x) & 1u) ? -uh[n] : uh[n];
        }
#pragma unroll
        for (int n = 0; n < NMODE; ++n) {
          const float v = (float)w[n];
          const int x = n >= VX && n <= VZ ? n - VX : n >= BX ? n - BX : 3;
          a.w32[n * sv + dst] = ((flips >> x) & 1u) ? -v : v;
        }
      },
      [&](int q, long dst, bool flip) {
        const double v = q == 0 ? f[0] : q == 1 ? f[1] : f[2];
        a.b1[q * sv + dst] = flip ? -v : v;
      },
      [&](int q, long dst) { a.b1[q * sv + dst] = 0.; });
}

// The Riemann solver RS on one FP32 face.
template <int RS>
__device__ __forceinline__ int solve_face32(float *f, const float *wl, const float *wr, float gam,
                                            float gm1i, int &ng) {
  return RS == BNZ_RS_HLLD ? flux_hlld(f, wl, wr, gam, gm1i, &ng) : flux_hll(f, wl, wr, gam, gm1i);
}

template <int NT>
struct Tile2Flux32 {
  const float *sx, *sy;
  int t, tx_stride;
  __device__ __forceinline__ float x(int n, long off) const { return sx[n * NT + t + (int)off]; }
  __device__ __forceinline__ float y(int n, long off) const {
    return sy[n * NT + t + (off ? tx_stride : 0)];
  }
  __device__ __forceinline__ float z(int, long) const { return 0.f; }
};
template <int NT>
struct Tile2Emf32 {  // emf32_edge<2>: zero in a reflecting wall plane
  const float *sx, *sy, *se;
  int t, tx_stride;
  long sy_stride;
  int i, j;
  Walls wl;
  __device__ __forceinline__ float operator()(int comp, long off) const {
    const int up = off >= sy_stride ? 1 : 0, ri = (int)(up ? off - sy_stride : off);
    const int o = up * tx_stride + ri;
    const bool wx = i + ri == wl.at[0] || i + ri == wl.at[1];
    const bool wy = j + up == wl.at[2] || j + up == wl.at[3];
    if (comp == 0) return wy ? 0.f : -sy[7 * NT + t + o];
    if (comp == 1) return wx ? 0.f : sx[7 * NT + t + o];
    return se[t + o];
  }
};

template <int NT>
constexpr int tile2_lds32() {
  return (2 * 8 + 2) * NT;
}

// One FP32C stage over one 2D tile (stage2_tile).  The fluxes come from the
// stage's FP32 prim wf and faces bf; ap / ac as in the separate updates.  Like
// the FP64 tile's, the corrector updates the active cells only and writes their
// ghosts: it reads the words of its own active cells, which no other tile
// writes, and wf, bf and ac.b, which no corrector writes.  ng counts the guarded
// faces of the cells the tile owns.
template <bool PRED, int ORDER, int RS, int TX, int TY, typename BF, class DT>
__device__ __forceinline__ double stage2_tile32(const Geo &g, const float *__restrict__ wf,
                                                const BF *__restrict__ bf, const Pred32 &ap,
                                                const Corr32 &ac, const Lims &L, const DT &step_dt,
                                                const Box &act, const Bnd &bnd, const Walls &walls,
                                                int fms_ref, int i0, int j0, float *lds, int &ng) {
  constexpr int NT = TX * TY;
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int i = i0 + tx - 1, j = j0 + ty - 1;
  const long sv = g.sv;
  float *sx = lds, *sy = lds + 8 * NT, *sc = lds + 16 * NT, *se = sc + NT;
  const bool in = i >= 0 && i < g.nt[0] && j >= 0 && j < g.nt[1];
  const bool own = in && tx > 0 && tx < TX - 1 && ty > 0 && ty < TY - 1;
  const bool reach = in && i >= L.lo[0] - 1 && i <= L.hi[0] + 1 && j >= L.lo[1] - 1 &&
                     j <= L.hi[1] + 1;
  bool gx = false, gy = false;
  int guarded = 0;
  // Threads off the grid stand on cell (0, 0), neighbours past the grid's end
  // are the cell itself: what they give is not used.
  const int ic = in ? i : 0, jc = in ? j : 0;
  const long c = (long)jc * g.nt[0] + ic;
  const bool first = tx == 0, last = tx == TX - 1;
  const int oxe = first && ic > 0 ? -1 : last && ic < g.nt[0] - 1 ? 1 : 0;
  const int oyl = jc > 0 ? -g.sy : 0, oyl2 = jc > 1 ? -2 * g.sy : oyl;
  const int oyr = jc < g.nt[1] - 1 ? g.sy : 0;
  float wc[NMODE], wl[NMODE], wr[NMODE], f[NMODE];
  float ym2[NMODE], ym[NMODE], yp[NMODE], xe[NMODE];
#pragma unroll
  for (int n = 0; n < NMODE; ++n) {
    const float *p = wf + n * sv + c;
    wc[n] = p[0];
    if (ORDER == 1 && n != BX) xe[n] = p[oxe];
  }
  const BF bnx = bf[c], bny = bf[sv + c];
#pragma unroll
  for (int n = 0; n < NMODE; ++n)
    if (n != BY) {
      const float *p = wf + n * sv + c;
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
      wl[n] = row_left<TX>(wc[n], 0.f, first);
      wr[n] = wc[n];
    } else {
      const float d = vl_half(wc[n] - row_left<TX>(wc[n], xe[n], first),
                            row_right<TX>(wc[n], xe[n], last) - wc[n]);
      wl[n] = row_left<TX>(wc[n] + d, 0.f, first);
      wr[n] = wc[n] - d;
    }
  }
  wl[BX] = wr[BX] = (float)bnx;
  if (reach && tx > 0 && i >= L.lo[0])
    if (solve_face32<RS>(f, wl, wr, (float)g.gam, (float)g.gamm1i, guarded)) {
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
      const float dm = wc[v] - ym[v];
      wl[n] = ym[v] + vl_half(ym[v] - ym2[v], dm);
      wr[n] = wc[v] - vl_half(dm, yp[v] - wc[v]);
    }
  }
  wl[BX] = wr[BX] = (float)bny;
  if (reach && ty > 0 && j >= L.lo[1])
    if (solve_face32<RS>(f, wl, wr, (float)g.gam, (float)g.gamm1i, guarded)) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n) {
        if (n == BX) continue;
        const int v = perm<1>(n);
        sy[(v < 6 ? v : v == BX ? 6 : 7) * NT + t] = f[n];
      }
      gy = true;
    }
  if (own) ng += guarded;
  if (!gx)
    for (int n = 0; n < 8; ++n) sx[n * NT + t] = 0.f;
  if (!gy)
    for (int n = 0; n < 8; ++n) sy[n * NT + t] = 0.f;
  sc[t] = -(wc[VX] * wc[BY] - wc[VY] * wc[BX]);  // ec32
  const double dt = step_dt();  // the fluxes did not need it
  __syncthreads();
  if (tx > 0 && ty > 0) {
    const float ez = 0.5f * (-sx[6 * NT + t - TX] - sx[6 * NT + t] + sy[6 * NT + t - 1] +
                             sy[6 * NT + t]) -
                     0.25f * (sc[t - 1] + sc[t] + sc[t - TX - 1] + sc[t - TX]);
    const bool wx = i == walls.at[0] || i == walls.at[1], wy = j == walls.at[2] || j == walls.at[3];
    se[t] = (wx || wy) ? 0.f : ez;
  }
  __syncthreads();
  const Tile2Flux32<NT> fl{sx, sy, t, TX};
  const Tile2Emf32<NT> em{sx, sy, se, t, TX, (long)g.sy, i, j, walls};
  if (PRED) {
    if (own) update32_pred_e<2, GeoArr>(g, ap, L, &dt, fl, em, i, j, 0);
    return 0.;
  }
  double cds = 0.;
  if (own && i >= act.lo[0] && i < act.lo[0] + act.n[0] && j >= act.lo[1] &&
      j < act.lo[1] + act.n[1]) {
    const auto ghosts = [&](const float *uh, const double *w, const double *f) {
      if (near_side(bnd, i, j, 0)) copy_ghosts32(bnd, g, ac, i, j, 0, uh, w, f);
    };
    cds = update32_corr_e<2, GeoArr, decltype(fl), decltype(em), false, decltype(ghosts)>(
        g, ac, L, &dt, act, fms_ref, fl, em, i, j, 0, nullptr, nullptr, ghosts);
  }
  return cds;
}

// LDS floats per thread of a 3D column (as the FP64 slots), beside R words of
// the half-updated cell and its faces (U.).
enum {
  YFY = 0, YFB = 6, YZB, YE0, YE2, YEX = 10, YEZ, YWP = 12, YDM = 20, YFX = 28, YFYZ,
  NSLOT3_32 = 30
};
enum { UC = 0, UBX = 6, UBY, UBYU, NSLOT3_U = 9 };

// One FP32C stage of a column of a 3D grid, as the FP64 stage3_column; the
// updates are those of update32_pred_e (R = float: hi words and faces of the
// half step) and update32_corr_e (R = double: hi + lo words, FP64 faces).
// ng counts the guarded faces of the cells the column owns.
template <bool PRED, int ORDER, int RS, class GM, int TX, int TY, typename BF>
__device__ __forceinline__ double stage3_column32(const Geo &g, const float *__restrict__ wf,
                                                  const BF *__restrict__ bf, const Pred32 &ap,
                                                  const Corr32 &ac, const Lims &L,
                                                  const double step_dt, const Box &act,
                                                  const Walls &walls, int fms_ref, int i0, int j0,
                                                  int kb, int ke, float *lds,
                                                  typename std::conditional<PRED, float, double>::type
                                                      *ldu,
                                                  int &ng) {
  using R = typename std::conditional<PRED, float, double>::type;
  constexpr int NT = TX * TY;
  const int t = threadIdx.x, tx = t % TX, ty = t / TX;
  const int i = i0 + tx - 1, j = j0 + ty - 1;
  const long sv = g.sv;
  const GM gm{g};
  const double dt = PRED ? 0.5 * step_dt : step_dt;
  float *s = lds + t;
  R *su = ldu + t;
  const int dn = ty > 0 ? -TX : 0, up = ty < TY - 1 ? TX : 0;
  const bool in = i >= 0 && i < g.nt[0] && j >= 0 && j < g.nt[1];
  const bool reach = in && i >= L.lo[0] - 1 && i <= L.hi[0] + 1 && j >= L.lo[1] - 1 &&
                     j <= L.hi[1] + 1;
  const bool inI = in && i >= L.lo[0] && i <= L.hi[0], inJ = in && j >= L.lo[1] && j <= L.hi[1];
  const bool upI = in && i >= L.lo[0] && i <= L.hi[0] + 1;
  const bool upJ = in && j >= L.lo[1] && j <= L.hi[1] + 1;
  const bool own = in && tx > 0 && tx < TX - 1 && ty > 0 && ty < TY - 1;
  const bool actij = i >= act.lo[0] && i < act.lo[0] + act.n[0] && j >= act.lo[1] &&
                     j < act.lo[1] + act.n[1];
  const bool wx = i == walls.at[0] || i == walls.at[1], wy = j == walls.at[2] || j == walls.at[3];
  const int ic = in ? i : 0, jc = in ? j : 0;
  const double dlx = gm.dlf(0, ic), dly = gm.dlf(1, jc);
  const ColGeo<std::is_same<GM, GeoUni>::value> ge(dt, dlx, dly, gm.dlf(2, 0));
  const float gam = (float)g.gam, gm1i = (float)g.gamm1i;
  // cell offsets; bytes are 4 or 8 times these
  const unsigned row = (unsigned)g.sy, plane = (unsigned)g.sz;
  const unsigned oxe = tx == 0 && ic > 0 ? -1u : tx == TX - 1 && ic < g.nt[0] - 1 ? 1u : 0u;
  const unsigned oyl = jc > 0 ? row : 0u, oyl2 = jc > 1 ? 2 * row : oyl;
  const unsigned oyr = jc < g.nt[1] - 1 ? row : 0u;
  const unsigned oxy = (unsigned)(jc * g.nt[0] + ic);
  constexpr unsigned BB = sizeof(BF);

  float fzl[6];
  R bzl = R(0);
  float eyl = 0.f, e0y = 0.f, e1 = 0.f;
#pragma unroll
  for (int n = 0; n < 6; ++n) fzl[n] = 0.f;
  double cds = 0.;
  const auto solve = [&](float *f, const float *wl, const float *wr, bool count) {
#pragma unroll
    for (int n = 0; n < NMODE; ++n) f[n] = 0.f;
    int q = 0;
    solve_face32<RS>(f, wl, wr, gam, gm1i, q);
    if (count) ng += q;
  };

  float wc[NMODE], wu[NMODE];
  BF bc[3];
  const auto clamp_k = [&](int k) { return (unsigned)min(max(k, 0), g.nt[2] - 1); };
  {
    const unsigned o = oxy + clamp_k(kb - 1) * plane, ob = oxy + clamp_k(kb - 2) * plane;
    const unsigned ou = oxy + clamp_k(kb) * plane;
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      wc[n] = at(wf + n * sv, 4u * o);
      wu[n] = at(wf + n * sv, 4u * ou);
      if (ORDER == 1 && n != BZ) s[(YDM + n) * NT] = wc[n] - at(wf + n * sv, 4u * ob);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) bc[a] = at(bf + a * sv, BB * o);
  }
  for (int k = kb - 1; k <= ke + 1; ++k) {
    const unsigned o = oxy + clamp_k(k) * plane;
    const int km = k - 1;
    const bool done = km >= kb;
    const bool counted = own && reach && k >= kb && k <= ke && k >= L.lo[2] - 1 &&
                         k <= L.hi[2] + 1;
    const double dlz = gm.dlf(2, (int)clamp_k(k)), dlzm = gm.dlf(2, (int)clamp_k(km));
    float wl[NMODE], wr[NMODE], f[NMODE];

    // ---- z face
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      if (n == BX) continue;
      const int v = perm<2>(n);
      wl[n] = s[(YWP + v) * NT];
      if (ORDER == 0) {
        wr[n] = wc[v];
        s[(YWP + v) * NT] = wc[v];
      } else {
        const float du = wu[v] - wc[v];
        const float d = vl_half(s[(YDM + v) * NT], du);
        wr[n] = wc[v] - d;
        s[(YWP + v) * NT] = wc[v] + d;
        s[(YDM + v) * NT] = du;
      }
    }
    wl[BX] = wr[BX] = (float)bc[2];
    float xe[NMODE];
    if (ORDER == 1) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) xe[n] = at(wf + n * sv, 4u * (o + oxe));
    }
    solve(f, wl, wr, counted && k >= L.lo[2]);
    float fzbx = 0.f;
    {
      const R dtdv = (R)ge.tv(dlzm);
      const R az = PRED ? (R)((float)dlx * (float)dly) : (R)ge.axy();
#pragma unroll
      for (int n = 0; n < NMODE; ++n) {
        const int v = perm<2>(n);
        if (v < 6) {
          su[(UC + v) * NT] -= dtdv * (az * (R)f[n] - az * (R)fzl[v]);
          fzl[v] = f[n];
        }
        if (v == BX) fzbx = f[n];
        if (v == BY) s[YZB * NT] = f[n];
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
        const float d = vl_half(wc[n] - from_left<TX>(wc[n], xe[n]),
                                from_right<TX>(wc[n], xe[n]) - wc[n]);
        const float wp = wc[n] + d;
        wl[n] = from_left<TX>(wp);
        wr[n] = wc[n] - d;
      }
    }
    wl[BX] = wr[BX] = (float)bc[0];
    solve(f, wl, wr, counted && i >= L.lo[0]);
    R xd[6];
    {
      const R ax = PRED ? (R)((float)dly * (float)dlz) : (R)ge.ayz(dlz);
#pragma unroll
      for (int n = 0; n < 6; ++n) xd[n] = ax * (R)from_right<TX>(f[n]) - ax * (R)f[n];
    }
    s[YFB * NT] = f[BY];
    const float fxzn = f[BZ];

    // ---- y face
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      if (n == BX) continue;
      const int v = perm<1>(n);
      const float *p = wf + v * sv;
      const float ym = at(p, 4u * (o - oyl));
      if (ORDER == 0) {
        wl[n] = ym;
        wr[n] = wc[v];
      } else {
        const float ym2 = at(p, 4u * (o - oyl2)), yp = at(p, 4u * (o + oyr));
        const float dm = wc[v] - ym;
        wl[n] = ym + vl_half(ym - ym2, dm);
        wr[n] = wc[v] - vl_half(dm, yp - wc[v]);
      }
    }
    wl[BX] = wr[BX] = (float)bc[1];
    solve(f, wl, wr, counted && j >= L.lo[1]);
    float fybx = 0.f, fyzn = 0.f;
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      const int v = perm<1>(n);
      if (v < 6) s[(YFY + v) * NT] = f[n];
      if (v == BX) fybx = f[n];
      if (v == BZ) fyzn = f[n];
    }

    // ---- cell EMFs (ec32)
    const float e0n = -(wc[VY] * wc[BZ] - wc[VZ] * wc[BY]);
    const float e1n = (wc[VX] * wc[BZ] - wc[VZ] * wc[BX]);
    const float e2n = -(wc[VX] * wc[BY] - wc[VY] * wc[BX]);
    const float e0 = s[YE0 * NT], fxz = s[YFX * NT], fyz = s[YFYZ * NT];
    s[YE0 * NT] = e0n;
    s[YE2 * NT] = e2n;
    s[YFX * NT] = fxzn;
    s[YFYZ * NT] = fyzn;
    R b0[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) b0[a] = PRED ? (R)bc[a] : (R)at(ac.b + a * sv, 8u * o);
    float uh[6], ul[6], wn2[NMODE];
    BF bn[3];
    const unsigned ou2 = oxy + clamp_k(k + 2) * plane, on = oxy + clamp_k(k + 1) * plane;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      uh[n] = at((PRED ? ap.uh : ac.uh) + n * sv, 4u * o);
      ul[n] = PRED ? 0.f : at(ac.ul + n * sv, 4u * o);
    }
#pragma unroll
    for (int n = 0; n < NMODE; ++n) wn2[n] = at(wf + n * sv, 4u * ou2);
#pragma unroll
    for (int a = 0; a < 3; ++a) bn[a] = at(bf + a * sv, BB * on);
    __syncthreads();

    // ---- edge EMFs (emf32_edge<3>), zero in the reflecting wall planes
    const bool wz = k == walls.at[4] || k == walls.at[5];
    const float e0yn = s[YE0 * NT + dn], e1xn = from_left<TX>(e1n);
    const float e2y = s[YE2 * NT + dn];
    const float zbx = from_left<TX>(fzbx), ybx = from_left<TX>(fybx), e1x = from_left<TX>(e1);
    const float e2x = from_left<TX>(e2n), e2xy = from_left<TX>(e2y);
    float ex = 0.5f * (-fyz - fyzn + s[YZB * NT + dn] + s[YZB * NT]) -
               0.25f * (e0yn + e0n + e0y + e0);
    float ey = 0.5f * (-zbx - fzbx + fxz + fxzn) - 0.25f * (e1xn + e1n + e1x + e1);
    float ez = 0.5f * (-s[YFB * NT + dn] - s[YFB * NT] + ybx + fybx) -
               0.25f * (e2x + e2n + e2xy + e2y);
    if (wy || wz) ex = 0.f;
    if (wx || wz) ey = 0.f;
    if (wx || wy) ez = 0.f;
    const float exl = s[YEX * NT];
    s[YEX * NT] = ex;
    s[YEZ * NT] = ez;
    e0y = e0yn;
    e1 = e1n;
    R yd[6];
    {
      const R ay = PRED ? (R)((float)dlx * (float)dlz) : (R)ge.axz(dlz);
#pragma unroll
      for (int n = 0; n < 6; ++n)
        yd[n] = ay * (R)s[(YFY + n) * NT + up] - ay * (R)s[(YFY + n) * NT];
    }
    __syncthreads();

    // ---- faces (faces_d in working type R)
    R bxl = su[UBX * NT], byl = su[UBY * NT], bzu;
    {
      const R tyzm = (R)ge.tyz(dlzm), txzm = (R)ge.txz(dlzm), tyz = (R)ge.tyz(dlz),
              txz = (R)ge.txz(dlz), txy = (R)ge.txy();
      const R dx = (R)dlx, dy = (R)dly, dz = (R)dlz;
      const R rex = (R)ex, rey = (R)ey, rez = (R)ez, rexl = (R)exl, reyl = (R)eyl;
      bxl += tyzm * (dy * rey - dy * reyl);
      byl -= txzm * (dx * rex - dx * rexl);
      R v = b0[0];
      const R ezu = (R)s[YEZ * NT + up], ezr = (R)from_right<TX>(ez);
      const R eyr = (R)from_right<TX>(ey), exu = (R)s[YEX * NT + up];
      v -= tyz * (dz * ezu - dz * rez);
      su[UBX * NT] = v;
      v = b0[1] + txz * (dz * ezr - dz * rez);
      su[UBY * NT] = v;
      bzu = b0[2] - txy * (dy * eyr - dy * rey);
      bzu += txy * (dx * exu - dx * rex);
    }
    eyl = ey;
    su[UBYU * NT] = byl;
    const R bxr = from_right<TX>(bxl);
    __syncthreads();

    // ---- the cell of plane k - 1
    if (done && own) {
      const bool active = PRED || (actij && km >= act.lo[2] && km < act.lo[2] + act.n[2]);
      const bool inK = km >= L.lo[2] && km <= L.hi[2];
      const bool upK = km >= L.lo[2] && km <= L.hi[2] + 1;
      const unsigned om = oxy + (unsigned)km * plane;
      if constexpr (PRED) {
        if (upI && inJ && inK) put(ap.bs, 4u * om, bxl);
        if (inI && upJ && inK) put(ap.bs + sv, 4u * om, byl);
        if (inI && inJ && upK) put(ap.bs + 2 * sv, 4u * om, bzl);
      } else if (active) {
        put(ac.b1, 8u * om, bxl);
        put(ac.b1 + sv, 8u * om, byl);
        put(ac.b1 + 2 * sv, 8u * om, bzl);
      }
      if (inI && inJ && inK) {
        double uv[NMODE], wv[NMODE];
        const R byu = su[UBYU * NT + TX];
#pragma unroll
        for (int n = 0; n < 6; ++n) uv[n] = su[(UC + n) * NT];
        uv[BX] = ((R)gm.icm(0, i) * bxl + (R)gm.icp(0, i) * bxr) * (R)gm.dlfi(0, i);
        uv[BY] = ((R)gm.icm(1, j) * byl + (R)gm.icp(1, j) * byu) * (R)gm.dlfi(1, j);
        uv[BZ] = ((R)gm.icm(2, km) * bzl + (R)gm.icp(2, km) * bzu) * (R)gm.dlfi(2, km);
        cons2prim(wv, uv, g.gam);
        if (!PRED) {
#pragma unroll
          for (int n = 0; n < 6; ++n) {
            float h, l;
            split(uv[n], h, l);
            if (active) {
              put(ac.uh + n * sv, 4u * om, h);
              put(ac.ul + n * sv, 4u * om, l);
            }
          }
        }
        float *wo = PRED ? ap.ws : ac.w32;
        if (active) {
#pragma unroll
          for (int n = 0; n < NMODE; ++n) put(wo + n * sv, 4u * om, (float)wv[n]);
        }
        if (!PRED && active) cds = fmax(cds, cds_cell_g(gm, g, wv, fms_ref, i, j, km));
      } else if (PRED) {
#pragma unroll
        for (int n = 0; n < NMODE; ++n)
          put(ap.ws + n * sv, 4u * om, at(ap.w32 + n * sv, 4u * om));
      }
    }
    bzl = bzu;
    {
      const R dtdv = (R)ge.tv(dlz);
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        R v;
        if constexpr (PRED) v = uh[n] - dtdv * xd[n];
        else v = join(uh[n], ul[n]) - dtdv * xd[n];
        v -= dtdv * yd[n];
        su[(UC + n) * NT] = v;
      }
    }
#pragma unroll
    for (int n = 0; n < NMODE; ++n) {
      wc[n] = wu[n];
      wu[n] = wn2[n];
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) bc[a] = bn[a];
  }
  return cds;
}

}  // namespace bnz
