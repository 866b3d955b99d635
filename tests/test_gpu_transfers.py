"""Uploads and downloads through the pinned buffer: what goes in comes out, for
transfers of one launch, of several chunks and with a short last one, for many
uploads in flight, and with the caller's array reused right after the call."""
import threading

import numpy as np
import pytest

from bonzo_amd import problems as P

pytestmark = pytest.mark.gpu

CHUNK = (2 << 20) // 96  # cells (12 doubles each) of one chunk


def _arrays(shape, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.standard_normal((9,) + shape), rng.standard_normal((3,) + shape)


@pytest.mark.parametrize("cells", [10, CHUNK, 2 * CHUNK, 2 * CHUNK + 1, 8 * CHUNK + 1, 300000])
def test_context_round_trip(cells):
    from bonzo_amd._lib import Context
    print(f"case: {cells} cells", flush=True)
    g = Context(cells - 6, bc=(1,) * 6)
    for seed in range(2):
        w, b = _arrays((1, 1, cells), seed)
        w0, b0 = w.copy(), b.copy()
        g.upload(w, b)
        w[:] = 0.0
        b[:] = 0.0
        w1, b1 = g.download()
        assert np.array_equal(w1, w0) and np.array_equal(b1, b0)
    g.close()


def test_batch_round_trip_many_boxes():
    from bonzo_amd._lib import Batch
    sizes = [1, 7, 256, 2 * CHUNK - 6, 2 * CHUNK - 5, 3, 130000] + [CHUNK - 100] * 14
    print(f"case: boxes {sizes}", flush=True)
    b = Batch([dict(nx=n, bc=(1,) * 6, tmax=0.1) for n in sizes])
    data = [_arrays((1, 1, n + 6), 10 + q) for q, n in enumerate(sizes)]
    for q, (w, f) in enumerate(data):
        tw, tf = w.copy(), f.copy()
        b.upload(q, tw, tf)
        tw[:] = 0.0
        tf[:] = 0.0
    for q in reversed(range(len(sizes))):
        w, f = b.download(q)
        assert np.array_equal(w, data[q][0]) and np.array_equal(f, data[q][1]), q
    b.close()


def test_download_from_several_threads():
    from bonzo_amd._lib import Batch
    sizes = [40, 3 * CHUNK, 500, 50]
    b = Batch([dict(nx=n, bc=(1,) * 6, tmax=0.1) for n in sizes])
    data = [_arrays((1, 1, n + 6), 30 + q) for q, n in enumerate(sizes)]
    for q, (w, f) in enumerate(data):
        b.upload(q, w, f)
    bad = []

    def take(q):
        for _ in range(5):
            w, f = b.download(q)
            if not (np.array_equal(w, data[q][0]) and np.array_equal(f, data[q][1])):
                bad.append(q)

    pool = [threading.Thread(target=take, args=(q,)) for q in range(len(sizes))]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    assert not bad
    b.close()


def test_run_between_transfers_matches_one_run():
    from bonzo_amd._lib import Context
    s, prim, bfld = P.turbulence(80)
    a, c = Context(80, 80, 80), Context(80, 80, 80)
    for g in (a, c):
        g.upload(prim, bfld)
        g.init_state()
    a.run_steps(4)
    for _ in range(4):
        c.run_steps(1)
        c.download()
    for x, y in zip(a.download(), c.download()):
        assert np.array_equal(x, y)
    a.close()
    c.close()


@pytest.mark.parametrize("n", [20, 128, 300])
def test_upload_waits_for_the_queued_work(n):
    """Plain, one-launch and chunked uploads alike return when the steps queued
    before them have ended."""
    import time
    from bonzo_amd._lib import Context
    print(f"case: {n}^2", flush=True)
    s, prim, bfld = P.orszag_tang(n)
    g = Context(n, n)
    g.upload(prim, bfld)
    g.init_state()
    g.run_steps(50)
    g.synchronize()
    g.run_steps(4000)  # some 80 ms
    t0 = time.perf_counter()
    g.upload(prim, bfld)
    t1 = time.perf_counter()
    g.synchronize()
    t2 = time.perf_counter()
    g.close()
    # what is left of the queue: an idle stream's wait, not thousands of steps
    assert t2 - t1 < 0.25 * (t1 - t0) + 1e-3, (t1 - t0, t2 - t1)
