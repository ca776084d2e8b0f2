"""SEM2D meshes that take several steps per launch, against the one-step kernel
(an explicit number of rows per wavefront), bit for bit: every order, meshes
of one and of several tiles with ragged last ones, runs shorter than, equal to
and past whole launches (odd and even numbers of them), sources on edges,
corners and in the interior, receivers on the source and past the number the
multi-step launch samples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MESHES = [(2, 2, 1), (60, 33, 1), (9, 40, 2), (30, 31, 2), (65, 20, 3), (13, 14, 3), (20, 11, 4), (3, 30, 5), (14, 9, 5)]


@pytest.mark.parametrize("ex,ez,order", MESHES)
def test_multi_step_launches_equal_single_steps(gpu, ex, ez, order):
    print("\n[sem2d-multi] %d x %d order %d" % (ex, ez, order), flush=True)
    rng = np.random.default_rng(ex * 100 + ez)
    model = rng.uniform(1500, 3000, ex * ez).astype(np.float32)
    for se in (0, (ez // 2) * ex + ex // 2, ex * ez - 1):
        kw = dict(ex=ex, ez=ez, lx=20.0 * ex, lz=20.0 * ez, order=order, dt=4e-4, f0=60.0, nsamples=80, model=model,
                  src_element=se)
        a, b = gpu.Sem2dSolver(**kw), gpu.Sem2dSolver(chunk=3, **kw)
        cur, prev = (rng.normal(0, 1, a.nn).astype(np.float32) for _ in range(2))
        nodes = rng.integers(0, a.nn, 150)
        nodes[3] = a.src_node
        for s in (a, b):
            s.set_field(s.i2, cur)
            s.set_field(s.i1, prev)
            s.set_receivers(nodes)
        for n in (1, 3, 8, 4, 8, 12, 17, 5, 16):
            (sa, ra), (sb, rb) = a.run(n), b.run(n)
            assert np.array_equal(sa, sb) and np.array_equal(ra, rb), n
            assert np.array_equal(a.current(), b.current()) and np.array_equal(a.previous(), b.previous()), n
        assert np.isfinite(a.current()).all() and np.abs(a.current()).max() > 0
        a.close()
        b.close()


def test_receiver_counts_and_steps_between_runs(gpu):
    print("\n[sem2d-multi] receivers", flush=True)
    kw = dict(ex=40, ez=41, lx=800.0, lz=820.0, order=2, dt=4e-4, f0=60.0, nsamples=60, src_element=40 * 20 + 7)
    a, b = gpu.Sem2dSolver(**kw), gpu.Sem2dSolver(chunk=5, **kw)
    rng = np.random.default_rng(8)
    for nrec in (1, 1025, 2048, 2049):
        nodes = rng.integers(0, a.nn, nrec)
        for s in (a, b):
            s.set_receivers(nodes)
        (sa, ra), (sb, rb) = a.run(9), b.run(9)
        assert np.array_equal(sa, sb) and np.array_equal(ra, rb), nrec
        a.step()
        b.step()
        assert np.array_equal(a.current(), b.current()) and np.array_equal(a.previous(), b.previous())
    a.set_timing(True)  # event-bracketed launches
    for n in (11, 8):
        (sa, ra), (sb, rb) = a.run(n), b.run(n)
        assert np.array_equal(sa, sb) and np.array_equal(ra, rb)
        assert np.array_equal(a.current(), b.current()) and np.array_equal(a.previous(), b.previous())
    a.close()
    b.close()


def test_timed_runs_time_the_launches_that_runs_make(gpu):
    """A timed run takes the same launches as an untimed one: on a mesh that
    takes several steps per launch its time per step is well under a single
    step's (2.5 of 6 us)."""
    print("\n[sem2d-multi] timing", flush=True)
    ms = {}
    for chunk in (0, 4):
        s = gpu.Sem2dSolver(ex=65, nsamples=400, chunk=chunk)
        s.run(80)
        s.set_timing(True)
        s.run(200)
        ms[chunk] = s.last_kernel_ms()
        s.close()
    print("[sem2d-multi] ms per step", ms, flush=True)
    assert ms[0] < 0.8 * ms[4]
