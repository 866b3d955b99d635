// Host check of the ghosts that the fused stages write with the active cells
// (scatter_ghosts, images) against the lists of the ghost fill (build_ghosts):
// every boundary of every side, 1D to 3D, from the smallest axis up.  Prints
// each difference (at most 20) and returns their number, capped at 99.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

#include "../bonzo_amd/csrc/bnz_tile.hpp"

using namespace bnz;

static long bad = 0, grids = 0;

static void check(const int n[3], int dims, int ng, const int bc[6]) {
  Bnd b{};
  Geo g{};
  int nt[3];
  b.ng = ng;
  b.dims = dims;
  for (int a = 0; a < 3; ++a) {
    nt[a] = g.nt[a] = a < dims ? n[a] + 2 * ng : 1;
    b.a1[a] = a < dims ? ng : 0;
    b.a2[a] = a < dims ? n[a] + ng - 1 : 0;
  }
  for (int q = 0; q < 6; ++q) b.flag[q] = bc[q];
  b.close();
  g.dims = dims;
  g.sy = nt[0];
  g.sz = nt[0] * nt[1];
  g.sv = (long)nt[0] * nt[1] * nt[2];
  const long sv = g.sv;
  ++grids;
  // nine cell variables and three faces, each value its own; the ghosts hold
  // values of their own too, which none may keep
  std::vector<double> from(12 * sv), fill, scat;
  for (long q = 0; q < 12 * sv; ++q) from[q] = 1. + q;
  fill = scat = from;
  // the cell whose thread wrote it (a thread's own writes are in order)
  std::vector<long> writer(12 * sv, -1);
  long me = -1, shared = 0;
  const auto put = [&](long q, double v) {
    scat[q] = v;
    shared += writer[q] >= 0 && writer[q] != me;
    writer[q] = me;
  };
  std::vector<int2> pairs;
  std::vector<GhostOp> ops;
  build_ghosts(nt, dims, ng, bc, 0, pairs, ops);
  for (const int2 &p : pairs)
    for (int v = 0; v < 12; ++v) fill[v * sv + p.x] = from[v * sv + p.y];
  for (const GhostOp &o : ops) {
    if (!(o.bits & (1u << 15)))
      for (int v = 0; v < 9; ++v)
        fill[v * sv + o.dst] = ((o.bits >> v) & 1u ? -1. : 1.) * from[v * sv + o.src];
    for (int a = 0; a < 3; ++a)
      fill[(9 + a) * sv + o.dst] = (o.bits >> (12 + a)) & 1u ? 0.
                                   : ((o.bits >> (9 + a)) & 1u ? -1. : 1.) *
                                         from[(9 + a) * sv + o.srcf[a]];
  }
  for (int k = b.a1[2]; k <= b.a2[2]; ++k)
    for (int j = b.a1[1]; j <= b.a2[1]; ++j)
      for (int i = b.a1[0]; i <= b.a2[0]; ++i) {
        if (!near_side(b, i, j, k)) continue;
        const long c = me = ((long)k * nt[1] + j) * nt[0] + i;
        if (b.plain) {  // copy_ghosts64's short form
          const unsigned m[3] = {images<false>(b, 0, i), images<false>(b, 1, j),
                                 images<false>(b, 2, k)};
          each_image(b, g, m, i, j, k, [&](long dst, unsigned) {
            for (int v = 0; v < 12; ++v) put(v * sv + dst, from[v * sv + c]);
          });
          continue;
        }
        scatter_ghosts(
            b, g, i, j, k,
            [&](long dst, unsigned flips) {
              for (int v = 0; v < 9; ++v) {
                const int a = v >= VX && v <= VZ ? v - VX : v >= BX ? v - BX : 3;
                put(v * sv + dst, ((flips >> a) & 1u ? -1. : 1.) * from[v * sv + c]);
              }
            },
            [&](int a, long dst, bool flip) {
              put((9 + a) * sv + dst, (flip ? -1. : 1.) * from[(9 + a) * sv + c]);
            },
            [&](int a, long dst) { put((9 + a) * sv + dst, 0.); });
      }
  const auto say = [&](const char *what, long q, double x, double y) {
    if (bad++ < 20)
      printf("%dx%dx%d ng %d bc %d%d%d%d%d%d: %s, variable %ld cell %ld: %g, fill %g\n", n[0], n[1],
             n[2], ng, bc[0], bc[1], bc[2], bc[3], bc[4], bc[5], what, q / sv, q % sv, x, y);
  };
  for (long q = 0; q < 12 * sv; ++q)
    if (scat[q] != fill[q]) say("value", q, scat[q], fill[q]);
  if (shared) say("two writers", 0, (double)shared, 0.);
}

int main() {
  for (int ng = 2; ng <= 3; ++ng)
    for (int dims = 1; dims <= 3; ++dims) {
      int pairs = 1;
      for (int a = 0; a < dims; ++a) pairs *= 9;
      for (int q = 0; q < pairs; ++q) {
        int bc[6] = {0, 0, 0, 0, 0, 0};
        for (int a = 0, r = q; a < dims; ++a, r /= 9) {
          bc[2 * a] = r % 9 / 3;
          bc[2 * a + 1] = r % 3;
        }
        // outflow axes go down to one cell (ng on one in 3D, to save time)
        int lo[3], hi[3];
        for (int a = 0; a < 3; ++a) {
          const bool out = bc[2 * a] == BNZ_BC_OUTFLOW && bc[2 * a + 1] == BNZ_BC_OUTFLOW;
          lo[a] = a >= dims ? 1 : out && dims < 3 ? 1 : ng;
          hi[a] = a >= dims ? 1 : dims < 3 ? 2 * ng + 2 : ng + 1;
        }
        int n[3];
        for (n[2] = lo[2]; n[2] <= hi[2]; ++n[2])
          for (n[1] = lo[1]; n[1] <= hi[1]; ++n[1])
            for (n[0] = lo[0]; n[0] <= hi[0]; ++n[0]) check(n, dims, ng, bc);
      }
    }
  printf("%ld grids, %ld differences\n", grids, bad);
  return bad > 99 ? 99 : (int)bad;
}
