"""The four-nodes-per-lane SEM shapes (4 rows per wavefront) against the
one-node tile, bit for bit: rows that end inside a quad, one element per axis,
an x remainder, sources in an interior node and on the boundary, both offset
widths, per-XCD schedules and plane chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MESHES = [(1, 1, 1), (3, 2, 4), (13, 3, 2), (16, 5, 4), (17, 4, 3), (22, 2, 5), (33, 3, 7)]


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("mesh", MESHES)
def test_quad_shapes_equal_the_one_node_tile(gpu, mesh, order):
    print("\n[sem-quad] %s order %d" % (mesh, order), flush=True)
    ex, ey, ez = mesh
    rng = np.random.default_rng(100 * ex + order)
    kw = dict(ex=ex, ey=ey, ez=ez, lx=100.0 * ex, ly=100.0 * ey, lz=100.0 * ez, order=order, dt=0.001 / order ** 2,
              model=rng.uniform(1000, 2000, ex * ey * ez), rhs=rng.normal(0, 1e3, 20).astype(np.float32))
    nn = (ex * order + 1) * (ey * order + 1) * (ez * order + 1)
    f = rng.normal(0, 1, (2, nn)).astype(np.float32)
    rec = rng.integers(0, nn, 9)

    def run(pt, **sh):
        s = gpu.SemSolver(src_point=pt, **kw, **sh)
        s.set_field(0, f[0])
        s.set_field(1, f[1])
        s.set_receivers(rec)
        out = list(s.run(7)) + [s.field(0), s.field(1)]
        s.close()
        return out
    for pt in ((0.0, 0.0, 0.0), (100.0 * (ex - 1) + 1, 100.0 * (ey // 2) + 1, 100.0 * (ez // 2) + 1)):
        want = run(pt, block_waves=8, tile_j=8, chunk_i=1 << 20)
        assert all(np.isfinite(w).all() for w in want)
        for sh in (dict(block_waves=4, tile_j=16, chunk_i=4), dict(block_waves=8, tile_j=32, chunk_i=-1),
                   dict(block_waves=4, tile_j=16, chunk_i=-3, index64=True),
                   dict(block_waves=8, tile_j=32, chunk_i=-2, k_remainder=1),
                   dict(block_waves=4, tile_j=16, chunk_i=-2, k_remainder=-1), dict()):
            for w, g in zip(want, run(pt, **sh)):
                assert np.array_equal(w, g), sh


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
def test_streaming_quad_shapes_equal_the_one_node_tile(gpu, order):
    """Arrays past the memory-side cache (three of them above 300 MB) take
    non-temporal accesses, with 32-bit offsets."""
    ex, ez, ey = 790 // order, 803 // order, 40 // order
    nx, ny, nz = (e * order + 1 for e in (ex, ey, ez))
    pitch = (32 + nx + order + 31) // 32 * 32
    assert 12 * pitch * (nz + 2 * order) * (ny + 2 * order) > 300e6
    print("\n[sem-quad] streaming order %d" % order, flush=True)
    rng = np.random.default_rng(order)
    f = rng.normal(0, 1, (2, nx * ny * nz)).astype(np.float32)
    kw = dict(ex=ex, ey=ey, ez=ez, lx=20.0 * ex, ly=20.0 * ey, lz=20.0 * ez, order=order, dt=0.001 / order ** 2,
              model=rng.uniform(1000, 2000, ex * ey * ez), rhs=rng.normal(0, 1e3, 6).astype(np.float32),
              src_point=(20.0 * (ex - 1) + 1, 20.0 * (ey // 2) + 1, 20.0 * (ez // 2) + 1))

    def run(**sh):
        s = gpu.SemSolver(**kw, **sh)
        for level in (0, 1):
            s.set_field(level, f[level])
        out = [s.run(3)[0], s.field(0), s.field(1)]
        s.close()
        return out
    want = run(block_waves=8, tile_j=8, chunk_i=20)
    assert all(np.isfinite(w).all() for w in want)
    for sh in (dict(block_waves=4, tile_j=16, chunk_i=8), dict(block_waves=8, tile_j=32, chunk_i=-2)):
        for w, g in zip(want, run(**sh)):
            assert np.array_equal(w, g), sh


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("planes", [6, 25, 30, 60, 66])
def test_default_shapes_of_flat_meshes_equal_the_one_node_tile(gpu, order, planes):
    """Few planes along the march axis under a plane of at least 25,000 nodes
    (fewer than 26, than 64, more): the shapes that create chooses."""
    print("\n[sem-quad] flat order %d, %d planes" % (order, planes), flush=True)
    ex, ey, ez = 190 // order, planes // order, 150 // order
    assert (ex * order + 1) * (ez * order + 1) >= 25000
    rng = np.random.default_rng(planes)
    kw = dict(ex=ex, ey=ey, ez=ez, lx=100.0 * ex, ly=100.0 * ey, lz=100.0 * ez, order=order, dt=0.001 / order ** 2,
              model=rng.uniform(1000, 2000, ex * ey * ez), rhs=rng.normal(0, 1e3, 6).astype(np.float32),
              src_point=(100.0 * (ex - 1) + 1, 100.0 * (ey // 2) + 1, 100.0 * (ez // 2) + 1))
    nn = (ex * order + 1) * (ey * order + 1) * (ez * order + 1)
    f = rng.normal(0, 1, (2, nn)).astype(np.float32)

    def run(**sh):
        s = gpu.SemSolver(**kw, **sh)
        for level in (0, 1):
            s.set_field(level, f[level])
        out = [s.run(4)[0], s.field(0), s.field(1)]
        s.close()
        return out
    want = run(block_waves=8, tile_j=8, chunk_i=1 << 20)
    assert all(np.isfinite(w).all() for w in want)
    for w, g in zip(want, run()):
        assert np.array_equal(w, g)
