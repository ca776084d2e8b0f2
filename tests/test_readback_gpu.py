"""Fields read back through the device-packed path: rows shorter, equal and
longer than a wavefront, unequal half widths, a level that owes its sponge
product, fields of several 32 MiB pieces, and the x-z slice, against the same
values through single-point reads and the field itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,lh", [((5, 7, 3), (4, 4, 4)), ((60, 50, 66), (4, 3, 2)), ((9, 4, 64), (2, 1, 3)), ((6, 11, 130), (1, 4, 2)),
                                     ((3, 5, 65), (6, 6, 6))])
def test_set_get_round_trip_and_points(gpu, dims, lh):
    print("\n[readback] %s %s" % (dims, lh), flush=True)
    nx, ny, nz = dims
    s = gpu.FdSetup(nx, ny, nz, L=lh[0], ly=lh[1], lz=lh[2], sponge_width=2, f0=25.0, nsamples=10)
    sol = gpu.FdSolver(s)
    rng = np.random.default_rng(1)
    shape = tuple(n + 2 * l for n, l in zip(dims, lh))
    for level in (0, 1):
        f = rng.normal(0, 1, shape).astype(np.float32)
        sol.set_field(level, f)
        assert np.array_equal(sol.field(level), f)
    sol.step(0)  # the previous level now owes its sponge product
    for level in (0, 1):
        f = sol.field(level)
        for _ in range(25):
            p = [int(rng.integers(-l, n + l)) for n, l in zip(dims, lh)]
            assert sol.read_point(level, *p) == f[p[0] + lh[0], p[1] + lh[1], p[2] + lh[2]]
        inner = f[lh[0]:lh[0] + nx, lh[1]:lh[1] + ny, lh[2]:lh[2] + nz]
        for j in (0, ny - 1):
            assert np.array_equal(sol.slice_xz(level, j), inner[:, j, :].T)
    sol.close()


def test_field_of_several_pieces(gpu):
    """276^3 values with the halo: 84 MB, three pieces."""
    print("\n[readback] pieces", flush=True)
    s = gpu.FdSetup(268, 268, 268, sponge_width=0, nsamples=2)
    sol = gpu.FdSolver(s)
    f = np.random.default_rng(2).normal(0, 1, (276, 276, 276)).astype(np.float32)
    sol.set_field(1, f)
    assert np.array_equal(sol.field(1), f)
    sol.close()


def test_sem_fields(gpu):
    print("\n[readback] sem", flush=True)
    rng = np.random.default_rng(3)
    a = gpu.SemSolver(ex=3, ey=4, ez=23, lx=60.0, ly=80.0, lz=460.0, order=3, nsamples=2, src_point=(25.0, 25.0, 25.0))
    b = gpu.Sem2dSolver(ex=40, ez=9, lx=800.0, lz=180.0, order=2, nsamples=2, src_element=50)
    for sol in (a, b):
        for level in (0, 1):
            f = rng.normal(0, 1, sol.nn).astype(np.float32)
            sol.set_field(level, f)
            assert np.array_equal(sol.field(level), f)
        sol.close()


def test_slice_of_a_long_axis(gpu):
    """More points along x than 4 x 65536, and a slice of two pieces."""
    print("\n[readback] long slices", flush=True)
    rng = np.random.default_rng(4)
    for nx, nz in ((262500, 2), (2600, 3400)):
        s = gpu.FdSetup(nx, 1, nz, L=1, sponge_width=0, nsamples=2, model="homogeneous")
        sol = gpu.FdSolver(s)
        f = rng.normal(0, 1, (nx + 2, 3, nz + 2)).astype(np.float32)
        sol.set_field(0, f)
        assert np.array_equal(sol.slice_xz(0, 0), f[1:-1, 1, 1:-1].T)
        sol.close()
