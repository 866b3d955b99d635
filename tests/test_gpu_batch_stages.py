"""The 2D stages of a batch, a tile per workgroup, against single grids bit for
bit: boxes of one tile, whole tiles and remainders, both tile sizes, every
boundary, beside 1D and 3D boxes."""
import numpy as np
import pytest

from tests.test_gpu_batch import check_against_single, say
from tests.test_gpu_fused_stages import _state
from bonzo_amd import problems as P

pytestmark = pytest.mark.gpu

SIDES = [(0,) * 6, (1, 2, 0, 0, 0, 0), (2, 2, 1, 1, 0, 0), (0, 0, 2, 2, 0, 0)]


@pytest.mark.parametrize("precision,rsolver,reconstr,mixed", [
    ("fp64", "hlld", "linear", False), ("fp64", "hll", "const", True),
    ("fp64", "hllt", "linear", False), ("fp32c", "hlld", "linear", True),
    ("fp32c", "hll", "const", False)])
@pytest.mark.parametrize("sizes", [[(4, 4), (14, 6), (29, 43), (60, 28)],
                                   [(5, 300), (250, 251), (3, 3), (64, 64), (61, 15)]])
def test_batch_2d_stages_bitwise_vs_single(sizes, precision, rsolver, reconstr, mixed):
    say(f"case: 2D boxes {sizes} {precision} {rsolver} {reconstr} mixed {mixed}")
    ng = 2 if reconstr == "const" else 3
    cases = []
    for q, (nx, ny) in enumerate(sizes):
        cases.append((_state(nx, ny, 1, ng, 70 + q), SIDES[q % 4], (0.004, 0.002, 0.006)[q % 3]))
    if mixed:
        rng = np.random.Generator(np.random.PCG64(71))
        cases.insert(1, (P.riemann_tube(90, rng, ng=ng), (1,) * 6, 0.01))
        cases.append((_state(17, 9, 12, ng, 72), (2, 1, 0, 0, 1, 2), 0.005))
    check_against_single(cases, rsolver, reconstr, precision=precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("n,extra", [((3, 900), False), ((3, 900), True), ((900, 3), False),
                                     ((12, 500), True), ((10, 600), False)])
def test_thin_boxes(n, extra, precision):
    """Many thin boxes: in FP32C some run separate kernels, beside boxes of
    every other kind, in FP64 the tile goes by the threads it takes."""
    say(f"case: 20 boxes of {n}, extra {extra}, {precision}")
    cases = []
    for q in range(20):
        bc = SIDES[q % 4]
        s, prim, bfld = _state(n[0], n[1] + q, 1, 3, 200 + q)
        for a in (0, 1):
            if 2 in bc[2 * a:2 * a + 2]:
                bfld[a][:] = 0.0  # no field through a wall
        cases.append(((s, prim, bfld), bc, (4e-4, 1e-4, 3e-4)[q % 3]))
    if extra:
        cases[3:3] = [(_state(70, 60, 1, 3, 231), (0,) * 6, 1e-3),
                      (_state(90, 1, 1, 3, 232), (1,) * 6, 1e-3),
                      (_state(12, 11, 10, 3, 233), (0,) * 6, 1e-3)]
    check_against_single(cases, precision=precision)
