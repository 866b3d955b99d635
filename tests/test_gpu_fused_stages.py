"""The fused stage kernels (2D tiles, 3D columns) against the oracle and the
separate kernels, at the sizes where tiles, columns and runs of planes end.

FP64 (IEEE) and FP32C results are the separate kernels' bit for bit, FP64 is
the oracle's; the FMA build is held to its bar, 1e-12 relative L1."""
import numpy as np
import pytest

from bonzo_amd import problems as P

pytestmark = pytest.mark.gpu


def _state(nx, ny, nz, ng, seed):
    """Smooth state with every variable and field component at work; the face
    fields depend on the other axes' indices only, so div B = 0."""
    s = P.GridShape(nx, ny, nz, ng)
    prim, bfld = s.empty()
    rng = np.random.Generator(np.random.PCG64(seed))
    x = [(np.arange(n) + 0.5) / n for n in (nx, ny, nz)]
    Z, Y, X = np.meshgrid(x[2], x[1], x[0], indexing="ij")

    def wave(axes):
        arg = sum(rng.integers(1, 4) * (X, Y, Z)[a] for a in axes)
        return np.sin(2 * np.pi * arg + rng.uniform(0, 6))

    act = s.active()
    prim[0][act] = 1.0 + 0.2 * wave((0, 1, 2))
    for v in (1, 2, 3):
        prim[v][act] = 0.4 * wave((0, 1, 2))
    prim[4][act] = 0.7 + 0.2 * wave((0, 1, 2))
    prim[5][act] = 0.5 + 0.3 * wave((0, 1, 2))
    for a in range(3):
        bfld[a][act] = 0.2 + 0.2 * wave([q for q in range(3) if q != a])
    return s, prim, bfld


def _run(s, prim, bfld, steps, tune=None, **kw):
    from bonzo_amd._lib import Context
    g = Context(s.nx, s.ny, s.nz, **kw)
    if tune:
        g.set_tuning(*tune)
    g.upload(prim, bfld)
    g.init_state()
    g.run_steps(steps)
    t, n, dt = g.time()
    # on to a t_max that clips a step, and steps past it that change nothing
    g.advance(t + 1.5 * dt)
    g.run_steps(0)
    g.set_time(*g.time()[:2])
    out = g.download() + (g.time(), g.diag())
    g.close()
    return out


# 2D: one tile, whole tiles and their neighbours (own cells 14 x 6 and 30 x
# 14), both sides of the size where the tile grows; thin grids
SIZES_2D = [(4, 4), (14, 6), (15, 7), (61, 29), (250, 250), (251, 257), (900, 3), (5, 600)]


@pytest.mark.parametrize("prec", ["fp64", "fp64fma", "fp32c"])
@pytest.mark.parametrize("nx,ny", SIZES_2D)
def test_tiles_2d(nx, ny, prec):
    k = SIZES_2D.index((nx, ny))
    bc = [(0,) * 6, (1, 2, 0, 0, 0, 0), (2, 2, 1, 1, 0, 0), (0, 0, 2, 2, 0, 0)][k % 4]
    rs, rc = ("hlld", "hll")[k % 2], ("linear", "linear", "const")[k % 3]
    print(f"case: {nx}x{ny} {prec} {rs} {rc} bc {bc}", flush=True)
    s, prim, bfld = _state(nx, ny, 1, 2 if rc == "const" else 3, 31 + k)
    kw = dict(precision=prec, rsolver=rs, reconstr=rc, bc=bc)
    a = _run(s, prim, bfld, 4, **kw)
    b = _run(s, prim, bfld, 4, tune=(0, 1, 0), **kw)
    _same(a, b, prec)


# 3D: rows, columns and runs of planes that end inside, at and past a tile
# (own cells 14 x 14), grids of few planes and of few rows
SIZES_3D = [(79, 83, 71), (98, 98, 98), (99, 113, 85), (400, 400, 4), (5, 320, 300)]


@pytest.mark.parametrize("prec", ["fp64", "fp64fma", "fp32c"])
@pytest.mark.parametrize("nx,ny,nz", SIZES_3D)
def test_columns_3d(nx, ny, nz, prec):
    if prec == "fp32c" and (nx, ny, nz) == SIZES_3D[0]:
        pytest.skip("below the FP32C column size")
    k = SIZES_3D.index((nx, ny, nz))
    bc = [(0,) * 6, (1, 2, 0, 0, 2, 1), (2, 2, 1, 1, 0, 0), (0, 0, 2, 2, 1, 1)][k % 4]
    rs, rc = ("hlld", "hll")[k % 2], ("linear", "linear", "const")[k % 3]
    print(f"case: {nx}x{ny}x{nz} {prec} {rs} {rc} bc {bc}", flush=True)
    s, prim, bfld = _state(nx, ny, nz, 2 if rc == "const" else 3, 41 + k)
    kw = dict(precision=prec, rsolver=rs, reconstr=rc, bc=bc)
    a = _run(s, prim, bfld, 3, **kw)
    b = _run(s, prim, bfld, 3, tune=(0, 0, 1), **kw)
    _same(a, b, prec)


def _same(a, b, prec):
    assert a[2] == b[2] or prec == "fp64fma"
    assert a[2][1] == b[2][1]
    assert a[3]["hlld_guards"] == b[3]["hlld_guards"]
    assert np.isfinite(a[0]).all()
    for x, y in zip(a[:2], b[:2]):
        if prec == "fp64fma":
            for v in range(x.shape[0]):
                den = max(np.abs(y[v]).sum(), 1e-9 * np.abs(b[0][0]).sum())
                assert np.abs(x[v] - y[v]).sum() <= 1e-12 * den, v
        else:
            assert np.array_equal(x, y)  # ghosts included


@pytest.mark.parametrize("n,rs,kw", [
    ((45, 31, 1), "hllt", {}), ((270, 260, 1), "hlld", {"dt_fms_ref": False}),
    ((33, 20, 1), "hllc", {"hydro": True}), ((75, 80, 77), "hlld", {"dt_fms_ref": False}),
    ((80, 75, 76), "hllt", {})])
def test_fused_matches_the_oracle(n, rs, kw):
    from bonzo_amd._lib import Context
    from oracle.oracle import OracleSim
    print(f"case: {n} {rs} {kw}", flush=True)
    s, prim, bfld = _state(*n, 3, 57)
    if kw.get("hydro"):
        bfld[:] = 0.0
    o = OracleSim(*n, rsolver=rs, **kw)
    o.prim[:] = prim
    o.bfld[:] = bfld
    o.init()
    o.advance_steps(3)
    g = Context(*n, rsolver=rs, **kw)
    g.upload(prim, bfld)
    g.init_state()
    g.run_steps(3)
    gp, gb = g.download()
    g.close()
    act = (slice(None),) + s.active()
    assert np.array_equal(gp[act], o.prim[act])
    assert np.array_equal(gb[act], o.bfld[act])
    o.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
@pytest.mark.parametrize("hi", [1, 2])
@pytest.mark.parametrize("n,axis", [((3, 1, 1), 0), ((3, 40, 1), 0), ((40, 3, 1), 1)])
def test_ghosts_of_the_shortest_walled_axis(n, axis, hi, prec):
    """A reflecting low side on an axis of just ng cells: its outermost ghost
    face mirrors a face that the high side fills, on every route."""
    from bonzo_amd._lib import Batch
    from tests.test_gpu_batch import box_desc
    print(f"case: {n} axis {axis} hi {hi} {prec}", flush=True)
    bc = [0] * 6
    bc[2 * axis], bc[2 * axis + 1] = 2, hi
    s, prim, bfld = _state(*n, 3, 71)
    outs = []
    for tune in ((0, 0, 0), (1, 1, 1)):
        outs.append(_run(s, prim, bfld, 4, tune=tune, bc=tuple(bc), precision=prec)[:2])
    if prec == "fp64" and n[1] == 1:
        out = outs[1]  # one launch a step (k_step1), and in a batch beside a long box
        s2, prim2, bfld2 = _state(600, 1, 1, 3, 72)
        b = Batch([box_desc(s, tuple(bc), 1e9), box_desc(s2, (0,) * 6, 1e9)])
        b.upload(1, prim2, bfld2)
    else:
        out = outs[0]
        b = Batch([box_desc(s, tuple(bc), 1e9)], precision=prec)
    b.upload(0, prim, bfld)
    b.init_state()
    b.advance(max_steps=3, use_graph=False)
    outs.append(b.download(0))
    b.close()
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])
    for _, face in outs:
        f = np.moveaxis(face[axis], 2 - axis, 0)  # the axis first
        other = [slice(3, -3) if m > 1 else slice(None) for m in f.shape[1:]]
        last = f[5] if hi == 1 else 0.0 * f[5]
        assert np.array_equal(f[0], -last)
        assert np.abs(f[5][tuple(other)]).min() > 0.0


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
@pytest.mark.parametrize("n,fused", [
    ((128, 128, 128), "both"), ((98, 98, 98), "both"), ((96, 96, 96), "fp64"),
    ((5, 320, 300), "fp64"), ((72, 72, 72), ""),
    ((1000, 3, 200), ""), ((400, 400, 4), "both"), ((3, 30000, 1), "fp64"),
    ((30000, 3, 1), "both"), ((3, 900, 1), "both")])
def test_thin_grids_keep_the_separate_kernels(n, fused, prec):
    """Tiles and columns run where they are the faster route."""
    from bonzo_amd._lib import Context
    print(f"case: {n} {prec}", flush=True)
    s, prim, bfld = _state(*n, 3, 61)
    out = []
    for tune in ((0, 0, 0), (0, 1, 1)):
        g = Context(*n, precision=prec)
        g.set_tuning(*tune)
        g.upload(prim, bfld)
        g.init_state()
        g.set_kernel_timing(True)
        g.run_steps(2)
        g.set_kernel_timing(False)
        names = set(g.kernel_timing())
        stage = any(name.startswith("stage") for name in names)
        assert stage == (fused in ("both", prec) and tune == (0, 0, 0)), names
        assert stage != any(name.startswith("flux") for name in names), names
        out.append(g.download())
        g.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
@pytest.mark.parametrize("nx,ny", [(11111, 12), (8, 14285), (12, 9000)])
def test_tiles_of_long_thin_grids(nx, ny, prec):
    print(f"case: {nx}x{ny} {prec}", flush=True)
    s, prim, bfld = _state(nx, ny, 1, 3, 62)
    a = _run(s, prim, bfld, 2, precision=prec)
    b = _run(s, prim, bfld, 2, tune=(0, 1, 0), precision=prec)
    _same(a, b, prec)


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
@pytest.mark.parametrize("n", [(150, 140, 1), (104, 98, 112)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -1.0])
def test_a_bad_cell_stays_where_it_is(n, value, prec):
    """A cell that is not finite, or of negative density: a face whose solver
    matches no region has flux 0 in a fused stage.  Cells that a step's stages
    do not reach from it are the separate kernels' bit for bit, and finite."""
    from bonzo_amd._lib import Context
    print(f"case: {n} {value} {prec}", flush=True)
    s, prim, bfld = _state(*n, 3, 63)
    at = [3 + m // 2 if m > 1 else 0 for m in n]
    prim[0][at[2], at[1], at[0]] = value
    out = []
    for tune in ((0, 0, 0), (0, 0, 1) if n[2] > 1 else (0, 1, 0)):
        g = Context(*n, precision=prec)
        g.set_tuning(*tune)
        g.upload(prim, bfld)
        g.init_state()
        assert g.diag()["bad_ijk"] == tuple(at)
        g.vl_step(1e-4)
        out.append(g.download())
        g.close()
    far = np.ones(prim.shape[1:], bool)  # outside the cells the two stages reach
    far[tuple(slice(max(0, x - 6), x + 7) for x in reversed(at))] = False
    for x, y in zip(*out):
        assert np.isfinite(x[:, far]).all()
        assert np.array_equal(x[:, far], y[:, far])


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
def test_columns_beyond_256_cubed(prec):
    """Columns against the separate kernels on a grid larger than any other here,
    of sides that end inside a tile and a run of planes."""
    n = (272, 261, 285)
    print(f"case: {n} {prec}", flush=True)
    s, prim, bfld = _state(8, 9, 10, 3, 64)  # a small state, repeated over the grid
    big = P.GridShape(*n, 3)
    w, b = big.empty()
    act = big.active()
    for dst, src in ((w, prim), (b, bfld)):
        for v in range(dst.shape[0]):
            tile = src[v][s.active()]
            reps = [-(-m // t) for m, t in zip(reversed(n), tile.shape)]
            dst[v][act] = np.tile(tile, reps)[:n[2], :n[1], :n[0]]
    bc = (0, 0, 1, 2, 0, 0)
    a = _run(big, w, b, 1, bc=bc, precision=prec)
    c = _run(big, w, b, 1, tune=(0, 0, 1), bc=bc, precision=prec)
    _same(a, c, prec)
