"""SEM2D runs of several steps per launch, against the one-step kernel (an
explicit number of rows per wavefront), bit for bit: every kernel (order, steps
per launch, rows per wavefront) on a mesh of several tiles with ragged last
ones and on one of 2 x 2 elements, and the shapes that create chooses on its own;
runs shorter than, equal to and past whole launches (odd and even numbers of
them), sources on edges, corners and in the interior, receivers on the source
and past the number the multi-step launch samples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (order, steps per launch, rows per wavefront): the tile, 64 columns by 16
# wavefronts' rows less order x steps on each side, is at least 16 x 8 nodes
SHAPES = [(p, t, r) for p in range(1, 6) for t in (4, 8) for r in (2, 3, 4)
          if 2 * p * t + 16 <= 64 and 2 * p * t + 8 <= 16 * r]
# meshes, and whether create chooses several steps per launch for them (256 CUs)
PLANNED = [(2, 2, 1, True), (60, 33, 1, True), (9, 40, 2, True), (30, 31, 2, True), (65, 20, 3, True),
           (13, 14, 3, True), (20, 11, 4, True), (26, 26, 5, True), (3, 30, 5, False), (14, 9, 5, False)]


def check_equal(gpu, ex, ez, order, shape=None, multi=True):
    rng = np.random.default_rng(ex * 100 + ez)
    model = rng.uniform(1500, 3000, ex * ez).astype(np.float32)
    for se in (0, (ez // 2) * ex + ex // 2, ex * ez - 1):
        kw = dict(ex=ex, ez=ez, lx=20.0 * ex, lz=20.0 * ez, order=order, dt=4e-4, f0=60.0, nsamples=80, model=model,
                  src_element=se)
        a, b = gpu.Sem2dSolver(**kw), gpu.Sem2dSolver(chunk=3, **kw)
        if shape:
            a.set_steps_per_launch(*shape)
            assert a.steps_per_launch() == shape
        assert (a.steps_per_launch()[0] > 0) == multi and b.steps_per_launch() == (0, 0)
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


@pytest.mark.parametrize("order,steps,rows", SHAPES)
def test_every_kernel_equals_single_steps(gpu, order, steps, rows):
    print("\n[sem2d-multi] order %d, %d steps, %d rows" % (order, steps, rows), flush=True)
    tx, tz = 64 - 2 * order * steps, 16 * rows - 2 * order * steps
    check_equal(gpu, (2 * tx + 7) // order + 1, (3 * tz + 5) // order + 1, order, (steps, rows))
    check_equal(gpu, 2, 2, order, (steps, rows))


@pytest.mark.parametrize("ex,ez,order,multi", PLANNED)
def test_planned_launches_equal_single_steps(gpu, ex, ez, order, multi):
    print("\n[sem2d-multi] %d x %d order %d" % (ex, ez, order), flush=True)
    check_equal(gpu, ex, ez, order, multi=multi)


def test_choosing_steps_between_runs(gpu):
    """The choice changes between runs (levels in either pair of buffers); what
    has no kernel is refused and leaves the choice."""
    print("\n[sem2d-multi] choosing", flush=True)
    kw = dict(ex=30, ez=31, lx=600.0, lz=620.0, order=2, dt=4e-4, f0=60.0, nsamples=80, src_element=400)
    a, b = gpu.Sem2dSolver(chunk=4, **kw), gpu.Sem2dSolver(chunk=4, **kw)
    for shape, n in (((8, 3), 9), ((4, 2), 5), ((0, 0), 3), ((4, 4), 13), ((8, 4), 8)):
        a.set_steps_per_launch(*shape)
        for bad in ((8, 2), (3, 2), (14, 2), (-6, 2), (4, 5), (4, 0), (0, 2)):
            with pytest.raises(gpu.PhcError):
                a.set_steps_per_launch(*bad)
        assert a.steps_per_launch() == shape
        (sa, _), (sb, _) = a.run(n), b.run(n)
        assert np.array_equal(sa, sb)
        assert np.array_equal(a.current(), b.current()) and np.array_equal(a.previous(), b.previous()), shape
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


def test_autotune_drops_a_slower_choice_and_keeps_a_faster_one(gpu):
    """2001^2 nodes of order 5 with 4 steps per launch: some 100 us per step
    against 20 in single steps; 196^2 nodes of order 3: 1.6 against 2.9."""
    print("\n[sem2d-multi] autotune", flush=True)
    for kw, shape, want in ((dict(ex=400, ez=400, order=5, lx=8000.0, src_element=80200), (4, 3), (0, 0)),
                            (dict(ex=65, ez=65, order=3, lx=2600.0, src_element=2000), (4, 2), (4, 2))):
        a, b = (gpu.Sem2dSolver(dt=4e-4, f0=60.0, nsamples=40, **kw) for _ in range(2))
        a.set_steps_per_launch(*shape)
        b.set_steps_per_launch(0, 0)
        for s in (a, b):
            s.run(12)
        state = a.current(), a.previous()
        assert a.autotune(steps_per_trial=20) >= 1
        assert a.steps_per_launch() == want
        assert np.array_equal(a.current(), state[0]) and np.array_equal(a.previous(), state[1])
        assert np.array_equal(a.run(13)[0], b.run(13)[0])
        assert np.array_equal(a.current(), b.current()) and np.array_equal(a.previous(), b.previous())
        a.close()
        b.close()
