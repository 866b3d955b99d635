// bnz_tube64.hpp -- FP64 VL steps of 1D grids: a step's cells in one pass, and
// many steps of a short grid in one launch, the whole grid in one workgroup,
// its state in registers and LDS from step to step.  Single grids and batches
// share these bodies.
#pragma once
#include "bnz_tile64.hpp"

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

// A run of cells of a 1D grid, one per thread of a workgroup (slot = thread),
// for the two stages of a step.  A thread's cell stays in its registers,
// loaded once, all of it at once; LDS holds what neighbours read: the prims of
// the stage, the normal field, the fluxes.  In 1D the x faces never change,
// and the cell's By and Bz are its faces'.  The arithmetic is that of
// flux_face_to and update_cell_e<1>.
template <int RS, bool CP, int NT>
struct TubeLine {
  const Geo &g;
  Geo gl;  // the LDS rows: variable stride NT
  const double *fx_old;
  double *sw, *sf, *sb;
  int i, t;
  double wv[NMODE], bx, bxu, dlx, dly, dlz, icm, icp, dlfi;

  static __device__ __forceinline__ int row(int n) { return n < BX ? n : n - 1; }
  __device__ __forceinline__ void publish(const double *v) {
#pragma unroll
    for (int n = 0; n < NMODE; ++n)
      if (CP || n != BX) sw[n * NT + t] = v[n];
  }
  // cell i of prim w and faces b (a cell outside the grid stands on its end)
  __device__ __forceinline__ TubeLine(const Geo &geo, const double *w, const double *b,
                                      const double *fx, int cell, double *lds)
      : g(geo), gl(geo), fx_old(fx), sw(lds), sf(lds + NMODE * NT),
        sb(lds + (2 * NMODE - 1) * NT), i(cell), t(threadIdx.x) {
    gl.sv = NT;
    const int c = min(max(i, 0), g.nt[0] - 1);
#pragma unroll
    for (int n = 0; n < NMODE; ++n) wv[n] = w[n * g.sv + c];
    bx = b[c];
    bxu = b[min(c + 1, g.nt[0] - 1)];
    dlx = g.dlf[0][c];
    dly = g.dlf[1][0];
    dlz = g.dlf[2][0];
    icm = g.icm[0][c];
    icp = g.icp[0][c];
    dlfi = g.dlfi[0][c];
    sb[t] = bx;
    publish(wv);
  }
  // flux of the cell's lower face into sf; a face whose solver matches no
  // region (non-finite speeds) takes the old row of fx_old, which a fused pass
  // never writes
  template <int ORDER>
  __device__ __forceinline__ void flux() {
    bool got = false;
    const auto sink = [&](const double *f, long) {
#pragma unroll
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) sf[row(n) * NT + t] = f[n];
      got = true;
    };
    flux_face_to<0, ORDER, RS, decltype(sink), CP>(gl, sw, sb, t, 0, 0, sink);
    if (!got)
      for (int n = 0; n < NMODE; ++n)
        if (n != BX) sf[row(n) * NT + t] = fx_old[n * g.sv + i];
  }
  // the cell wv updated by dt
  __device__ __forceinline__ void update(double *wn, double dt) const {
    const double ax = dly * dlz;
    double u[NMODE];
    prim2cons(u, wv, g.gamm1i);
    const double dtdv = dt / (dlx * dly * dlz);
#pragma unroll
    for (int n = 0; n < NMODE - 3; ++n)
      u[n] = u[n] - dtdv * (ax * sf[n * NT + t + 1] - ax * sf[n * NT + t]);
    u[BX] = (icm * bx + icp * bxu) * dlfi;
    const double ez0 = -sf[row(BY) * NT + t], ez1 = -sf[row(BY) * NT + t + 1];
    const double ey0 = sf[row(BZ) * NT + t], ey1 = sf[row(BZ) * NT + t + 1];
    u[BY] = wv[BY] + dt / (dlx * dlz) * (dlz * ez1 - dlz * ez0);
    u[BZ] = wv[BZ] - dt / (dlx * dly) * (dly * ey1 - dly * ey0);
    cons2prim(wn, u, g.gam);
  }
};

// A whole VL step of a 1D grid for a workgroup of BLK threads that owns the
// STEP1_CELLS active cells from i0: thread t stands on cell i0 - 3 + t, the
// cells beside the owned ones are predicted by the neighbouring workgroups
// too.  Reads the step's prim w and faces b only and writes the new ones of
// the active cells and their ghosts to wout and bout, so no read races a
// write; ghosts(i) false: the caller fills them.  step_dt() gives the dt
// where it is first needed, after the predictor's fluxes; with zero_stops and
// dt = 0 nothing is written and the result is -1.  Every thread must call it;
// returns the CFL speed of the thread's cell.
template <int ORDER, int RS, bool CP, class DT>
__device__ __forceinline__ double step1_block(const Geo &g, const double *w, const double *b,
                                              double *wout, double *bout,
                                              const double *__restrict__ fx_old, const Bnd &bnd,
                                              bool ghosts, const DT &step_dt, bool zero_stops,
                                              int fms_ref, int i0, double *lds) {
  constexpr int LO = 3, HI = BLK - 4;  // slots of the owned cells
  static_assert(HI - LO + 1 == STEP1_CELLS, "owned cells");
  const int a1 = bnd.a1[0], a2 = bnd.a2[0];
  TubeLine<RS, CP, BLK> ln(g, w, b, fx_old, i0 - LO + (int)threadIdx.x, lds);
  const int i = ln.i, t = ln.t;
  __syncthreads();
  if (t >= 1 && i >= a1 - 1 - ORDER && i <= a2 + 2 + ORDER) ln.template flux<0>();
  const double dt = step_dt();
  if (zero_stops && dt == 0.) return -1.;  // alike in every thread
  __syncthreads();
  double wn[NMODE];
  if (t >= 1 && t <= BLK - 2 && i >= a1 - 1 - ORDER && i <= a2 + 1 + ORDER) {
    ln.update(wn, 0.5 * dt);
    ln.publish(wn);
  }
  __syncthreads();
  if (t >= LO && t <= HI + 1 && i >= a1 && i <= a2 + 1) ln.template flux<ORDER>();
  __syncthreads();
  if (t < LO || t > HI || i < a1 || i > a2) return 0.;
  ln.update(wn, dt);
  const long sv = g.sv;
#pragma unroll
  for (int n = 0; n < NMODE; ++n) wout[n * sv + i] = wn[n];
  const double f[3] = {ln.bx, wn[BY], wn[BZ]};
#pragma unroll
  for (int a = 0; a < 3; ++a) bout[a * sv + i] = f[a];
  if (ghosts && near_side(bnd, i, 0, 0)) copy_ghosts64(bnd, g, i, 0, 0, wn, f, wout, bout);
  return cds_cell_g(GeoArr{g}, g, wn, fms_ref, i, 0, 0);
}

// Up to nsteps steps of the 1D grid g by a workgroup of tube_threads(nt)
// threads, or of more up to NT: thread t stands on cell t and its lower face.
// Reads and leaves the state in w and b, ghosts included.  A step is
// step1_block's.  zero_stops: a step whose dt is 0 is not taken (a single
// grid's rule).  Returns the steps taken; ck ends where the next step begins
// (ck.m the new maximum), last is the dt of the last step taken.
template <int ORDER, int RS, int NT>
__device__ __forceinline__ int tube_run(const Geo &g, const Bnd &bnd, double *w, double *b,
                                        const double *__restrict__ fx_old, int fms_ref, int nsteps,
                                        bool zero_stops, TubeClock &ck, double &last, double *lds) {
  __shared__ double red[NT / 64];
  const int nt = g.nt[0], nw = blockDim.x / 64;
  const int a1 = bnd.a1[0], a2 = bnd.a2[0];
  const long sv = g.sv;
  TubeLine<RS, false, NT> ln(g, w, b, fx_old, threadIdx.x, lds);
  const int i = ln.i;
  const bool in = i < nt, act = i >= a1 && i <= a2;
  // the active cell a ghost copies, and whether a wall mirrors it
  int src = i;
  bool flip = false;
  if (in && !act) {
    const int flag = bnd.flag[i < a1 ? 0 : 1], n = a2 - a1 + 1;
    if (flag == BNZ_BC_PERIODIC) src = i < a1 ? i + n : i - n;
    else if (flag == BNZ_BC_OUTFLOW) src = i < a1 ? a1 : a2;
    else src = i < a1 ? 2 * a1 - 1 - i : 2 * a2 + 1 - i;
    flip = flag == BNZ_BC_REFLECT;
  }
  __syncthreads();
  int taken = 0;
  while (taken < nsteps && !ck.past() && !(zero_stops && ck.dt == 0.)) {
    const double dt = ck.dt;
    // predictor (donor cell, dt/2), where the corrector's faces read it
    if (i >= a1 - 1 - ORDER && i <= a2 + 2 + ORDER) ln.template flux<0>();
    __syncthreads();
    double wn[NMODE];
    if (i >= a1 - 1 - ORDER && i <= a2 + 1 + ORDER) {
      ln.update(wn, 0.5 * dt);
      ln.publish(wn);
    }
    __syncthreads();
    // corrector
    if (i >= a1 && i <= a2 + 1) ln.template flux<ORDER>();
    __syncthreads();
    double cds = 0.;
    if (act) {
      ln.update(wn, dt);
#pragma unroll
      for (int n = 0; n < NMODE; ++n) ln.wv[n] = wn[n];
      ln.publish(wn);
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
          const double v = ln.sw[n * NT + src];
          ln.wv[n] = flip && n == VX ? -v : v;
        }
      ln.publish(ln.wv);
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
    for (int n = 0; n < NMODE; ++n) w[n * sv + i] = ln.wv[n];
    b[sv + i] = ln.wv[BY];
    b[2 * sv + i] = ln.wv[BZ];
  }
  return taken;
}

}  // namespace bnz
