"""Many steps of a short 1D grid in one launch against the launches of single
steps, bit for bit (FP64 IEEE), at the sizes where the workgroup's threads end, and
around t_max, save and load."""
import numpy as np
import pytest

from tests.test_gpu_batch import check_against_single, say
from tests.test_gpu_fused_stages import _state
from bonzo_amd import problems as P

pytestmark = pytest.mark.gpu

SIDES = [(0,) * 6, (1, 1, 0, 0, 0, 0), (2, 1, 0, 0, 0, 0), (1, 2, 0, 0, 0, 0), (2, 2, 0, 0, 0, 0)]
# active cells + 6 ghosts: a wave, the compiled classes (256, 512) and one past
# them, which runs single steps
SIZES = [3, 58, 59, 250, 251, 400, 506, 507]


def _run(s, prim, bfld, steps, tune=None, **kw):
    from bonzo_amd._lib import Context
    g = Context(s.nx, rsolver=kw.pop("rsolver", "hlld"), **kw)
    if tune:
        g.set_tuning(*tune)
    g.upload(prim, bfld)
    g.init_state()
    g.run_steps(steps)
    t, n, dt = g.time()
    g.vl_step(0.5 * dt)
    blob = g.save_state()
    n1 = g.advance(t + 3.3 * dt)
    n2 = g.advance(t + 9.0 * dt, 2)
    g.run_steps(1)
    out = g.download() + (g.time(), n1, n2)
    g.load_state(blob)
    g.advance(1e9, 3)
    out += g.download() + (g.time(),)
    g.close()
    return out


@pytest.mark.parametrize("nx", SIZES)
def test_tube_matches_single_steps(nx):
    k = SIZES.index(nx)
    rs, rc = ("hlld", "hll", "hllt")[k % 3], ("linear", "const")[k % 2]
    if rc == "const":
        nx += 2  # the same cells with two ghosts a side
    bc = SIDES[k % 5]
    print(f"case: {nx} {rs} {rc} bc {bc}", flush=True)
    s, prim, bfld = _state(nx, 1, 1, 2 if rc == "const" else 3, 81 + k)
    bfld[0][:] = 0.0 if 2 in bc else 0.3  # no field through a wall
    kw = dict(rsolver=rs, reconstr=rc, bc=bc)
    a = _run(s, prim, bfld, 300, **kw)
    b = _run(s, prim, bfld, 300, tune=(1, 1, 1), **kw)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("nx", SIZES)
def test_tube_fma_within_its_bar(nx):
    """The FMA unit's two routes contract differently: 1e-12 relative L1 after
    a few steps, as its other routes are held to."""
    from bonzo_amd._lib import Context
    print(f"case: {nx} fp64fma", flush=True)
    s, prim, bfld = _state(nx, 1, 1, 3, 101 + nx)
    bfld[0][:] = 0.3
    out = []
    for tune in ((0, 0, 0), (1, 1, 1)):
        g = Context(nx, precision="fp64fma")
        g.set_tuning(*tune)
        g.upload(prim, bfld)
        g.init_state()
        g.run_steps(4)
        out.append(g.download())
        g.close()
    for x, y in zip(*out):
        for v in range(x.shape[0]):
            den = max(np.abs(y[v]).sum(), 1e-9 * np.abs(out[1][0][0]).sum())
            assert np.abs(x[v] - y[v]).sum() <= 1e-12 * den, v


@pytest.mark.parametrize("rsolver,reconstr", [("hlld", "linear"), ("hll", "const"),
                                              ("hllt", "linear")])
@pytest.mark.parametrize("sizes", [[250, 30, 64, 3], [506, 128, 251, 64, 400],
                                   [500, 59], [507, 64]])
def test_batch_of_tubes_bitwise_vs_single(sizes, rsolver, reconstr):
    say(f"case: tubes {sizes} {rsolver} {reconstr}")
    ng = 2 if reconstr == "const" else 3
    cases = []
    for q, n in enumerate(sizes):
        s, prim, bfld = _state(n, 1, 1, ng, 90 + q)
        bc = SIDES[q % 5]
        bfld[0][:] = 0.0 if 2 in bc else 0.3  # no field through a wall
        cases.append(((s, prim, bfld), bc, (0.05, 0.02, 0.03)[q % 3]))
    check_against_single(cases, rsolver, reconstr)


def test_batch_tubes_pieces_match_one_run():
    from bonzo_amd._lib import Batch
    from tests.test_gpu_batch import box_desc
    rng = np.random.Generator(np.random.PCG64(95))
    cases = [(P.riemann_tube(n, rng), (1,) * 6, tm)
             for n, tm in ((80, 0.05), (450, 0.03), (300, 0.04), (506, 0.02), (64, 0.0))]
    outs = []
    for pieces in (False, True):
        b = Batch([box_desc(c[0][0], c[1], c[2]) for c in cases])
        for q, ((s, prim, bfld), _, _) in enumerate(cases):
            b.upload(q, prim, bfld)
        b.init_state()
        if pieces:
            assert b.advance(max_steps=5, use_graph=False) == 5
            assert list(b.times()[1][:4]) == [5] * 4
            b.advance(max_steps=7)
            assert list(b.times()[1][:4]) == [13] * 4
        b.advance(use_graph=not pieces)
        outs.append(([b.download(q) for q in range(len(cases))], b.times()))
        b.close()
    (da, ta), (db, tb) = outs
    assert np.array_equal(ta[0], tb[0]) and np.array_equal(ta[1], tb[1])
    for x, y in zip(da, db):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])


@pytest.mark.parametrize("precision,char_proj", [("fp64", False), ("fp64", True),
                                                 ("fp64fma", False)])
@pytest.mark.parametrize("nx", [508, 747, 748, 2503])
def test_one_launch_steps_against_the_oracle(nx, precision, char_proj):
    """Steps of one launch at the sizes where its workgroups end (251 cells
    each), every boundary: IEEE bit for bit, FMA to 1e-12 relative L1."""
    from bonzo_amd._lib import Context
    from oracle.oracle import OracleSim
    bc = SIDES[nx % 5]
    print(f"case: {nx} {precision} char {char_proj} bc {bc}", flush=True)
    s, prim, bfld = _state(nx, 1, 1, 3, 120 + nx)
    bfld[0][:] = 0.0 if 2 in bc else 0.3
    o = OracleSim(nx, bc=bc, char_proj=char_proj)
    o.prim[:] = prim
    o.bfld[:] = bfld
    o.init()
    o.advance_steps(9)
    g = Context(nx, bc=bc, precision=precision, char_proj=char_proj)
    for graph in (False, True):
        g.set_step_graph(graph)
        g.upload(prim, bfld)
        g.init_state()
        assert g.advance(1e9, 9) == 9
        gp, gb = g.download()
        for x, y in ((gp, o.prim), (gb, o.bfld)):
            x, y = x[..., 3:-3], y[..., 3:-3]
            if precision == "fp64":
                assert np.array_equal(x, y)
            else:
                for v in range(x.shape[0]):
                    den = max(np.abs(y[v]).sum(), 1e-9 * np.abs(prim[0]).sum())
                    assert np.abs(x[v] - y[v]).sum() <= 1e-12 * den, v
        t, n, dt = g.time()
        assert g.advance(t + 0.4 * dt) == 1 and g.time()[0] == t + 0.4 * dt
    g.close()
    o.close()


@pytest.mark.parametrize("precision", ["fp64", "fp64fma"])
@pytest.mark.parametrize("nx", [744, 745, 743, 994])
def test_one_launch_steps_at_the_ends_of_workgroups(nx, precision):
    """Grids whose last workgroup (250 cells each, ghosts included) is just full,
    holds one cell, lacks one, or is full again: IEEE bit for bit, FMA to 1e-12
    relative L1."""
    from bonzo_amd._lib import Context
    from oracle.oracle import OracleSim
    bc = SIDES[nx % 5]
    print(f"case: {nx} {precision} bc {bc}", flush=True)
    s, prim, bfld = _state(nx, 1, 1, 3, 140 + nx)
    bfld[0][:] = 0.0 if 2 in bc else 0.3
    o = OracleSim(nx, bc=bc)
    o.prim[:] = prim
    o.bfld[:] = bfld
    o.init()
    o.advance_steps(7)
    g = Context(nx, bc=bc, precision=precision)
    g.upload(prim, bfld)
    g.init_state()
    g.run_steps(7)
    gp, gb = g.download()
    g.close()
    for x, y in ((gp, o.prim), (gb, o.bfld)):
        x, y = x[..., 3:-3], y[..., 3:-3]
        if precision == "fp64":
            assert np.array_equal(x, y)
        else:
            for v in range(x.shape[0]):
                den = max(np.abs(y[v]).sum(), 1e-9 * np.abs(prim[0]).sum())
                assert np.abs(x[v] - y[v]).sum() <= 1e-12 * den, v
    o.close()


@pytest.mark.parametrize("reconstr", ["linear", "const"])
def test_batch_steps_at_the_ends_of_workgroups(reconstr):
    say(f"case: boxes of 744, 745, 743, 994 cells {reconstr}")
    ng = 2 if reconstr == "const" else 3
    cases = []
    for q, n in enumerate((744, 745, 743, 994)):
        s, prim, bfld = _state(n + 6 - 2 * ng, 1, 1, ng, 150 + q)
        bc = SIDES[q % 5]
        bfld[0][:] = 0.0 if 2 in bc else 0.3  # no field through a wall
        cases.append(((s, prim, bfld), bc, 0.004))
    check_against_single(cases, "hlld", reconstr)
