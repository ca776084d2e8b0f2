"""The four-points-per-lane FD shapes (4 rows per wavefront) against the
one-point tile, bit for bit: rows that end inside a quad, tiles with one row
or one quad, grids narrower than the sponge or the PML slabs, sources in the
last point of a quad, both offset widths, halos that hold arbitrary values
(a quad that ends beyond the grid must leave them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(9, 17, 61), (14, 16, 62), (11, 33, 63), (10, 31, 64), (13, 1, 65), (12, 15, 67), (7, 40, 1), (1, 5, 6),
         (25, 36, 130), (3, 2, 3)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("boundary", ["none", "sponge", "pml"])
def test_quad_shapes_equal_the_one_point_tile(gpu, grid, boundary):
    print("\n[fd-quad] %s %s" % (grid, boundary), flush=True)
    nx, ny, nz = grid
    rng = np.random.default_rng(nx * 1000 + nz)
    s = gpu.FdSetup(nx, ny, nz, L=4, f0=25.0, sponge_width=5 if boundary == "sponge" else 0,
                    model=rng.uniform(0.5, 2.0, nx * ny * nz).astype(np.float32), nsamples=20,
                    xs=nx // 2, ys=ny // 2, zs=nz - 1)
    fields = rng.normal(0, 1, (2, nx + 8, ny + 8, nz + 8)).astype(np.float32)
    rec = np.stack([rng.integers(0, n, 9) for n in grid], 1)
    nd = min(4, min(grid) // 2)

    def run(**kw):
        sol = gpu.FdSolver(s, **kw)
        if boundary == "pml" and nd > 0:
            sol.set_pml(ndamp=nd)
        sol.set_field(0, fields[0])
        sol.set_field(1, fields[1])
        sol.set_receivers(rec)
        out = list(sol.run(0, 7)) + [sol.current(), sol.previous()]
        sol.step(7)
        out += [sol.current(), sol.previous()]
        sol.close()
        return out
    for arith in (gpu.ARITH_REF, gpu.ARITH_FP32):
        want = run(arith=arith, tile_j=8, block_waves=8, chunk_i=4)
        assert all(np.isfinite(w).all() for w in want)
        for kw in (dict(tile_j=16, block_waves=4, chunk_i=3), dict(tile_j=32, block_waves=8, chunk_i=-1),
                   dict(tile_j=16, block_waves=4, chunk_i=-3, index64=True), dict(tile_j=32, block_waves=8, k_remainder=1),
                   dict()):
            for w, g in zip(want, run(arith=arith, **kw)):
                assert np.array_equal(w, g), (arith, kw)


@pytest.mark.parametrize("boundary", ["sponge", "pml"])
def test_streaming_quad_shapes_equal_the_one_point_tile(gpu, boundary):
    """Arrays past the memory-side cache (three of them above 300 MB) take
    non-temporal accesses, with 32-bit offsets."""
    nx, ny, nz = 40, 803, 790
    pitch = (32 + nz + 4 + 31) // 32 * 32
    assert 12 * pitch * (ny + 8) * (nx + 8) > 300e6
    print("\n[fd-quad] streaming %s" % boundary, flush=True)
    rng = np.random.default_rng(11)
    s = gpu.FdSetup(nx, ny, nz, L=4, f0=25.0, sponge_width=5 if boundary == "sponge" else 0,
                    model=rng.uniform(0.5, 2.0, nx * ny * nz).astype(np.float32), nsamples=6, zs=nz - 1)
    fields = rng.normal(0, 1, (2, nx + 8, ny + 8, nz + 8)).astype(np.float32)

    def run(**kw):
        sol = gpu.FdSolver(s, **kw)
        if boundary == "pml":
            sol.set_pml(ndamp=6)
        for level in (0, 1):
            sol.set_field(level, fields[level])
        out = [sol.run(0, 3)[0], sol.current(), sol.previous()]
        sol.close()
        return out
    for arith in (gpu.ARITH_REF, gpu.ARITH_FP32):
        want = run(arith=arith, tile_j=8, block_waves=8, chunk_i=20)
        assert all(np.isfinite(w).all() for w in want)
        for kw in (dict(tile_j=16, block_waves=4, chunk_i=13), dict(tile_j=32, block_waves=8, chunk_i=-2)):
            for w, g in zip(want, run(arith=arith, **kw)):
                assert np.array_equal(w, g), (arith, kw)
