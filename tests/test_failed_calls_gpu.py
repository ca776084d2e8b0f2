"""Runs whose graph cannot be instantiated: the call returns an error and the
state is as before it, so the same call succeeds afterwards with the values of
a run that never failed.  The failures are refusals by a shim between
libphc.so and the HIP runtime (tests/cpp/hip_faults.c), which has to be loaded
first: each test runs in a process of its own."""
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


CASES = {
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
