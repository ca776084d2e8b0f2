"""Fused runs in chunks: a captured chunk is replayed for later samples (its
nodes name no sample), chunks of other lengths and both level parities are
captured beside it, and each step's receivers are sampled by the next launch.
A run cut into chunks gives the uncut run's traces and levels bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one step; the same length three times (replays), an odd length (the other
# level parity) twice, then the first length again from that parity
CHUNKS = [1, 8, 8, 8, 5, 8, 5, 8]
NSTEPS = sum(CHUNKS)


def fd(gpu, pml):
    s = gpu.FdSetup(nx=40, ny=37, nz=70, xs=20, ys=18, zs=33, f0=25.0, nsamples=NSTEPS, sponge_width=0 if pml else 6)
    sol = gpu.FdSolver(s, arith=gpu.ARITH_FP32)
    if pml:
        sol.set_pml(ndamp=6)
    rng = np.random.default_rng(3)
    # more receivers than one sampling block's 1024 threads, one on the source
    ijk = np.stack([rng.integers(0, n, 1100) for n in (40, 37, 70)], 1)
    ijk[7] = (20, 18, 33)
    sol.set_receivers(ijk)
    return sol, lambda it, n: sol.run(it, n)


def sem(gpu, order, face):
    # face: the source element's first node lies on the boundary (never updated)
    kw = dict(ex=6, ey=5, ez=12, lx=120.0, ly=100.0, lz=240.0, order=order, dt=0.0005, f0=40.0, nsamples=NSTEPS,
              src_point=(1.0, 41.0, 121.0) if face else (61.0, 41.0, 121.0))
    sol = gpu.SemSolver(**kw)
    nodes = np.random.default_rng(4).integers(0, sol.nn, 1100)
    sol.set_receivers(nodes)

    def run(it, n):
        sol.it = it
        return sol.run(n)
    return sol, run


def sem2d(gpu):
    sol = gpu.Sem2dSolver(ex=20, ez=17, lx=400.0, lz=340.0, order=3, dt=0.0005, f0=40.0, nsamples=NSTEPS,
                          src_element=20 * 8 + 9)
    nodes = np.random.default_rng(5).integers(0, sol.nn, 600)
    nodes[11] = sol.src_node
    sol.set_receivers(nodes)

    def run(it, n):
        sol.it = it
        return sol.run(n)
    return sol, run


CASES = {"fd sponge": lambda g: fd(g, False), "fd pml": lambda g: fd(g, True), "sem p2": lambda g: sem(g, 2, False),
         "sem p4": lambda g: sem(g, 4, False), "sem p3, source on the boundary": lambda g: sem(g, 3, True),
         "sem2d": sem2d}


@pytest.mark.parametrize("case", list(CASES))
def test_chunks_equal_one_run(gpu, case):
    print("\n[run-chunks] " + case, flush=True)
    whole, run_whole = CASES[case](gpu)
    cut, run_cut = CASES[case](gpu)
    src, rec = run_whole(0, NSTEPS)
    assert np.abs(src).max() > 0 and np.abs(rec).max() > 0
    it, parts = 0, []
    for n in CHUNKS:
        parts.append(run_cut(it, n))
        cut.synchronize()
        it += n
    assert np.array_equal(np.concatenate([p[0] for p in parts]), src)
    assert np.array_equal(np.concatenate([p[1] for p in parts], axis=1), rec)
    assert np.array_equal(cut.current(), whole.current())
    assert np.array_equal(cut.previous(), whole.previous())
    whole.close()
    cut.close()
