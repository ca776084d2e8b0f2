"""What calls do when the HIP runtime refuses them something, and how much
device memory they ask for.  Runs whose graph cannot be instantiated: the call
returns an error and the state is as before it, so the same call succeeds
afterwards with the values of a run that never failed.  Fields read and written
without device memory for the packing: the same values.  The scratch memory of
the packing: bounded, and none held before a field is read.  A learned layer's
loss and gradient: no device memory asked for.  Runs that alternate between two
lengths: no graph instantiated twice.  A shim between
libphc.so and the HIP runtime (tests/cpp/hip_faults.c) refuses and counts; it
has to be loaded first, so each test runs in a process of its own."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
NEVER = ctypes.c_size_t(-1).value


def fd(phc, **kw):
    return phc.FdSolver(phc.FdSetup(40, 30, 70, sponge_width=6, f0=25.0, nsamples=64), **kw)


def sem(phc, **kw):
    return phc.SemSolver(ex=6, lx=240.0, order=2, dt=0.002, f0=20.0, nsamples=64, src_point=(121.0, 121.0, 121.0), **kw)


def sem2d(phc, **kw):
    return phc.Sem2dSolver(ex=30, ez=31, lx=600.0, lz=620.0, order=2, dt=4e-4, f0=60.0, nsamples=64, src_element=400, **kw)


def batch(phc, **kw):
    return phc.FdBatch([phc.FdSetup(*g, sponge_width=6, f0=25.0, nsamples=64) for g in ((30, 40, 50), (20, 17, 70))], **kw)


def state(sol):
    if hasattr(sol, "dims"):
        return [sol.field(s, c) for s in range(len(sol.dims)) for c in (True, False)]
    return [sol.current(), sol.previous()]


def run(sol, it, n):
    if hasattr(sol, "i2") and hasattr(sol, "add_rhs"):
        return sol.run(it, n)[0]
    return np.asarray(sol.run(n)[0])


def check_failed_run(phc, faults, make):
    a, b = make(phc), make(phc)
    for it, n in ((0, 9), (9, 10), (19, 9)):  # the captured chunk's length changes, so each run captures anew
        want = run(a, it, n)
        faults.hip_faults_set(NEVER, 1)
        for _ in range(2):
            try:
                run(b, it, n)
                raise SystemExit("the run did not fail")
            except phc.PhcError:
                pass
        assert faults.hip_faults_refused() == 2
        faults.hip_faults_set(NEVER, 0)
        got = run(b, it, n)
        assert np.array_equal(want, got), (it, n)
        for x, y in zip(state(a), state(b)):
            assert np.array_equal(x, y), (it, n)
    assert np.abs(state(a)[0]).max() > 0


def check_graphs_kept(phc, faults):
    """Runs of two lengths in turn from one sample instantiate each graph once."""
    for make in (fd, sem, sem2d, batch):
        a = make(phc)
        for k in range(24):
            if k == 8:
                faults.hip_faults_set(NEVER, 0)
            if hasattr(a, "it"):
                a.it = 0
            run(a, 0, (10, 7)[k % 2])
        assert faults.hip_faults_graphs() == 0, make.__name__
        if hasattr(a, "it"):
            a.it = 0
        run(a, 0, 5)
        assert faults.hip_faults_graphs() == 1, make.__name__


def fd_fields(phc, faults, dims, lh, refuse):
    """Set, step (the previous level then owes its sponge product), read."""
    nx, ny, nz = dims
    sol = phc.FdSolver(phc.FdSetup(nx, ny, nz, L=lh[0], ly=lh[1], lz=lh[2], sponge_width=2, f0=25.0, nsamples=10))
    rng = np.random.default_rng(nx)
    faults.hip_faults_set(0 if refuse else NEVER, 0)
    shape = [n + 2 * l for n, l in zip(dims, lh)]
    for level in (0, 1):
        sol.set_field(level, rng.normal(0, 1, shape).astype(np.float32))
    out = [sol.field(0), sol.field(1)]
    refused = faults.hip_faults_refused()
    faults.hip_faults_set(NEVER, 0)  # the first step uploads its schedule
    sol.step(0)
    faults.hip_faults_set(0 if refuse else NEVER, 0)
    out += [sol.field(0), sol.field(1)] + [sol.slice_xz(lv, j) for lv in (0, 1) for j in (0, ny - 1)]
    refused += faults.hip_faults_refused()
    faults.hip_faults_set(NEVER, 0)
    sol.close()
    return out, refused


def check_no_scratch(phc, faults):
    for dims, lh in (((5, 7, 3), (4, 4, 4)), ((60, 50, 66), (4, 3, 2)), ((6, 11, 130), (1, 4, 2)), ((3, 5, 65), (6, 6, 6))):
        (want, _), (got, refused) = (fd_fields(phc, faults, dims, lh, r) for r in (False, True))
        assert refused >= 10  # every read and write went without scratch
        for a, b in zip(want, got):
            assert np.array_equal(a, b), (dims, lh)
    rng = np.random.default_rng(3)
    for make in (sem, sem2d):
        sol = make(phc)
        f = [rng.normal(0, 1, sol.nn).astype(np.float32) for _ in range(2)]
        faults.hip_faults_set(0, 0)
        for level in (0, 1):
            sol.set_field(level, f[level])
        for level in (0, 1):
            assert np.array_equal(sol.field(level), f[level])
        assert faults.hip_faults_refused() >= 2
        faults.hip_faults_set(NEVER, 0)
        sol.close()


def check_scratch_size(phc, faults):
    """Fields of 84 and 71 MB (a 2D field is one plane), a slice of 35 MB."""
    piece = 32 << 20
    big = (phc.FdSolver(phc.FdSetup(268, 268, 268, sponge_width=0, nsamples=2)),
           phc.Sem2dSolver(ex=2100, ez=2100, lx=42e3, lz=42e3, order=2, nsamples=2, src_element=50))
    for sol in big:
        shape = sol.nn if hasattr(sol, "nn") else (276, 276, 276)
        f = np.random.default_rng(2).normal(0, 1, shape).astype(np.float32)
        assert f.nbytes > 64 << 20
        held = faults.hip_faults_live()
        faults.hip_faults_set(NEVER, 0)
        sol.set_field(1, f)
        assert np.array_equal(sol.field(1), f)
        assert 0 < faults.hip_faults_peak() <= piece
        assert 0 < faults.hip_faults_live() - held <= piece
        sol.close()
    sol = phc.FdSolver(phc.FdSetup(2600, 1, 3400, L=1, sponge_width=0, nsamples=2, model="homogeneous"))
    faults.hip_faults_set(NEVER, 0)
    sol.slice_xz(0, 0)
    assert 0 < faults.hip_faults_peak() <= piece
    sol.close()


def check_eval_allocates_nothing(phc, faults):
    rng = np.random.default_rng(5)
    lb = phc.LearnedBoundary(seed=3)
    lb.set_capacity(300)
    for f in range(phc.LB_FACES):
        lb.add_samples(f, rng.uniform(0, 1, (300, phc.LB_SAMPLE)).astype(np.float32))
    want = lb.eval()
    faults.hip_faults_set(0, 0)
    got = lb.eval()
    faults.hip_faults_set(NEVER, 0)
    # float atomics: sums of 1800 terms in any order
    assert abs(got[0] - want[0]) <= 1e-5 * want[0]
    assert np.allclose(got[1], want[1], rtol=1e-4, atol=1e-5 * np.abs(want[1]).max())


CASES = {
    "graphs_kept": check_graphs_kept,
    "eval_allocates_nothing": check_eval_allocates_nothing,
    "no_scratch": check_no_scratch,
    "scratch_size": check_scratch_size,
    "failed_run_fd": lambda phc, f: check_failed_run(phc, f, fd),
    "failed_run_sem": lambda phc, f: check_failed_run(phc, f, sem),
    "failed_run_sem2d": lambda phc, f: check_failed_run(phc, f, sem2d),
    "failed_run_batch": lambda phc, f: check_failed_run(phc, f, batch),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_refused_calls(gpu, case):
    print("\n[failed-calls] %s" % case, flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), case], cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "ok " + case in r.stdout, r.stdout + r.stderr


if __name__ == "__main__":
    shim = ctypes.CDLL(os.path.join(HERE, "cpp", "libhip_faults.so"), mode=ctypes.RTLD_GLOBAL)
    shim.hip_faults_set.argtypes = [ctypes.c_size_t, ctypes.c_int]
    shim.hip_faults_peak.restype = shim.hip_faults_live.restype = ctypes.c_size_t
    sys.path.insert(0, os.path.join(ROOT, "proxy-geos-hc_amd"))
    import phc
    CASES[sys.argv[1]](phc, shim)
    print("ok", sys.argv[1])
