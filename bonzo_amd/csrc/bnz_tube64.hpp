// bnz_tube64.hpp -- many FP64 VL steps of a short 1D grid in one launch: the
// whole grid in one workgroup, its state in registers and LDS from step to
// step.  Single grids and batches share this body.
#pragma once
#include "bnz_kern64.hpp"
#include "bnz_tile.hpp"

namespace bnz {

// Cells (ghosts included) up to which a 1D grid runs so, one thread a cell.
// A step is bound by the FP64 issue of the one CU's four SIMDs: us per step,
// FP64 (FMA), against launches of single steps: 128 cells 5.1 (4.4) for 11.0
// (10.5), 256 5.5 (4.7) for 12.5 (11.6), 512 8.7 (7.2) for 12.7 (11.8).  With
// 576 threads a third wave on one SIMD makes it 12.0, and 1024 threads, whose
// 128 registers spill, 26.
constexpr int TUBE_CELLS = 512;
// Steps of one launch (some 2 ms), after which the host looks at the time.
constexpr int TUBE_STEPS = 256;

// LDS doubles per thread: the prims, the fluxes but the normal field's, and
// the normal field of the faces.
constexpr int TUBE_SLOTS = 2 * NMODE;

// Threads a kernel is compiled for (the stride of its LDS rows): fewer leave
// each more registers, and small tubes several to a CU.
constexpr int TUBE_NT[2] = {256, TUBE_CELLS};
inline int tube_threads(int nt) { return (nt + 63) / 64 * 64; }
inline int tube_class(int nt) { return nt <= TUBE_NT[0] ? 0 : 1; }

// Single grids whose steps run so: short 1D VL grids in FP64, in the default
// placement (bnz_set_tuning 0, 0, 0); characteristic limiting and user
// boundaries keep the launches of single steps.
inline bool tube_grid(const bnz_ctx *c) {
  return c->dims == 1 && c->nt[0] <= TUBE_CELLS && !c->f32 && !c->p.tintegr && !c->p.char_proj &&
         c->npass == 0 && c->flux_chunk == 0 && c->emf_chunk == 0 && c->update_chunk == 0;
}

// Where a tube stands between steps: time, end (clip false: none), the CFL
// maximum m of its state and the dt of its next step.
struct TubeClock {
  double t, tmax, m, dt, cour;
  bool clip;
  __device__ __forceinline__ bool past() const { return clip && !(t < tmax); }
  __device__ __forceinline__ void next_dt() {  // dt_reduce_block's rule
    dt = cour / m;
    if (clip && t + dt > tmax) dt = tmax - t;
  }
};

// Up to nsteps steps of the 1D grid g by a workgroup of tube_threads(nt)
// threads, or of more up to NT: thread t stands on cell t and its lower face.  Reads
// and leaves the state in w and b (in 1D the x faces never change, and the
// cell's By and Bz are its faces', so b is only written), ghosts included.
// A step is step1_block's, with the same arithmetic; fx_old as there.
// zero_stops: a step whose dt is 0 is not taken (a single grid's rule).
// Returns the steps taken; ck ends where the next step begins (dt is then
// that of the last step taken, ck.m the new maximum), last is their last dt.
template <int ORDER, int RS, int NT>
__device__ __forceinline__ int tube_run(const Geo &g, const Bnd &bnd, double *w, double *b,
                                        const double *__restrict__ fx_old, int fms_ref, int nsteps,
                                        bool zero_stops, TubeClock &ck, double &last, double *lds) {
  __shared__ double red[NT / 64];
  const int i = threadIdx.x, nt = g.nt[0], nw = blockDim.x / 64;
  const int a1 = bnd.a1[0], a2 = bnd.a2[0];
  const long sv = g.sv;
  double *sw = lds, *sf = lds + NMODE * NT, *sb = sf + (NMODE - 1) * NT;
  const bool in = i < nt, act = i >= a1 && i <= a2;
  // cells whose predicted state the corrector's faces read, and their faces
  const bool pc = i >= a1 - 1 - ORDER && i <= a2 + 1 + ORDER;
  const bool pf = i >= a1 - 1 - ORDER && i <= a2 + 2 + ORDER;
  const bool cf = i >= a1 && i <= a2 + 1;
  const int c = in ? i : 0;
  // the active cell a ghost copies, and whether a wall mirrors it
  int src = c;
  bool flip = false;
  if (in && !act) {
    const int flag = bnd.flag[i < a1 ? 0 : 1], n = a2 - a1 + 1;
    if (flag == BNZ_BC_PERIODIC) src = i < a1 ? i + n : i - n;
    else if (flag == BNZ_BC_OUTFLOW) src = i < a1 ? a1 : a2;
    else src = i < a1 ? 2 * a1 - 1 - i : 2 * a2 + 1 - i;
    flip = flag == BNZ_BC_REFLECT;
  }
  const double dlx = g.dlf[0][c], dly = g.dlf[1][0], dlz = g.dlf[2][0];
  const double icm = g.icm[0][c], icp = g.icp[0][c], dlfi = g.dlfi[0][c];
  const double ax = dly * dlz;
  Geo gl = g;  // the LDS rows: variable stride NT
  gl.sv = NT;

  double wv[NMODE];
#pragma unroll
  for (int n = 0; n < NMODE; ++n) wv[n] = w[n * sv + c];
  const double bx = b[c], bxu = b[in && i < nt - 1 ? c + 1 : c];
  sb[i] = bx;
#pragma unroll
  for (int n = 0; n < NMODE; ++n)
    if (n != BX) sw[n * NT + i] = wv[n];
  __syncthreads();

  const auto row = [](int n) { return n < BX ? n : n - 1; };  // of a flux slot
  const auto flux = [&](auto order) {
    bool got = false;
    flux_face_to<0, decltype(order)::value, RS>(gl, sw, sb, i, 0, 0, [&](const double *f, long) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) sf[row(n) * NT + i] = f[n];
      got = true;
    });
    if (!got)  // no region matched: as step1_block
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) sf[row(n) * NT + i] = fx_old[n * sv + i];
  };
  // the cell updated by dt (update_cell_e<1>)
  const auto update = [&](double *wn, double dt) {
    double u[NMODE];
    prim2cons(u, wv, g.gamm1i);
    const double dtdv = dt / (dlx * dly * dlz);
#pragma unroll
    for (int n = 0; n < NMODE - 3; ++n)
      u[n] = u[n] - dtdv * (ax * sf[n * NT + i + 1] - ax * sf[n * NT + i]);
    u[BX] = (icm * bx + icp * bxu) * dlfi;
    const double ez0 = -sf[row(BY) * NT + i], ez1 = -sf[row(BY) * NT + i + 1];
    const double ey0 = sf[row(BZ) * NT + i], ey1 = sf[row(BZ) * NT + i + 1];
    u[BY] = wv[BY] + dt / (dlx * dlz) * (dlz * ez1 - dlz * ez0);
    u[BZ] = wv[BZ] - dt / (dlx * dly) * (dly * ey1 - dly * ey0);
    cons2prim(wn, u, g.gam);
  };

  int taken = 0;
  while (taken < nsteps && !ck.past() && !(zero_stops && ck.dt == 0.)) {
    const double dt = ck.dt;
    // predictor (donor cell, dt/2)
    if (pf) flux(std::integral_constant<int, 0>());
    __syncthreads();
    double wn[NMODE];
    if (pc) {
      update(wn, 0.5 * dt);
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) sw[n * NT + i] = wn[n];
    }
    __syncthreads();
    // corrector
    if (cf) flux(std::integral_constant<int, ORDER>());
    __syncthreads();
    double cds = 0.;
    if (act) {
      update(wn, dt);
#pragma unroll
      for (int n = 0; n < NMODE; ++n) {
        wv[n] = wn[n];
        if (n != BX) sw[n * NT + i] = wn[n];
      }
      cds = cds_cell_g(GeoArr{g}, g, wn, fms_ref, i, 0, 0);
    }
    cds = wave_max(cds);
    if ((i & 63) == 0) red[i >> 6] = cds;
    __syncthreads();
    // its ghosts and the next dt
    if (in && !act) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) {
          const double v = sw[n * NT + src];
          wv[n] = flip && n == VX ? -v : v;
          sw[n * NT + i] = wv[n];
        }
    }
    double m = red[0];
    for (int q = 1; q < nw; ++q) m = fmax(m, red[q]);
    ++taken;
    last = dt;
    ck.t += dt;
    ck.m = m;
    ck.next_dt();
    __syncthreads();
  }
  if (taken && in) {
#pragma unroll
    for (int n = 0; n < NMODE; ++n) w[n * sv + i] = wv[n];
    b[sv + i] = wv[BY];
    b[2 * sv + i] = wv[BZ];
  }
  return taken;
}

}  // namespace bnz
