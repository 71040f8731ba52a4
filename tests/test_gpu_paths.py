"""Edges of the launch rules: scene extents, lane-team walks, sort routes, read-backs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1, 0, 257, 5000, 3], [3] * 1100, [70001]])
def test_scene_extents_measured_on_the_device(sphk, sizes):
    # The extents of scenes whose state was replaced are measured on the device in one launch
    # (parts of a scene folded on the host): scenes of one particle, none, only non-finite
    # ones, more scenes than workgroups, one scene over many parts.  A particle outside its
    # measured grid would be reported by the read-back; the step equals the scene alone.
    rng = np.random.default_rng(7)
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(offs[-1])
    centre = np.repeat(rng.uniform(-3, 3, (len(sizes), 3)), sizes, axis=0)
    pos = (centre + rng.uniform(-0.2, 0.2, (n, 3))).astype(np.float32)
    if len(sizes) > 4:
        a, b = int(offs[4]), int(offs[5])
        pos[a:b] = np.nan
        pos[int(offs[2])] = np.inf
    p = sphk.default_params(xmin=-4, xmax=4, ymin=-4, ymax=4, zmin=-4, zmax=4, formulation=1)
    e = sphk.Engine(n, p)
    e.upload(pos)
    e.set_scenes(offs)
    e.snapshot_save()
    for _ in range(2):
        e.snapshot_restore()
        e.step(1e-4)
    got = e.positions()
    for k in [0, 2, 3, 4, len(sizes) - 1]:
        if k >= len(sizes) or sizes[k] == 0:
            continue
        a, b = int(offs[k]), int(offs[k + 1])
        one = sphk.Engine(b - a, p)
        one.upload(pos[a:b])
        one.step(1e-4)
        np.testing.assert_array_equal(got[a:b], one.positions())


@pytest.mark.parametrize("n", [1, 2, 255, 32767, 32768, 32769, 70000])
def test_uploads_and_downloads_return_the_rows(sphk, n):
    # Rows go up and come back through work arrays and two pinned halves of 32,768 rows: every
    # read-back returns the uploaded bits, non-finite ones included, also after a second
    # upload behind the first, and a refused upload leaves the state as it was.
    rng = np.random.default_rng(n)
    pos = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    vel = rng.normal(0, 1, (n, 3)).astype(np.float32)
    mass = rng.uniform(1, 2, n).astype(np.float32)
    pos[n // 2, 1] = np.nan
    pos[n - 1, 2] = -np.inf
    e = sphk.Engine(n + 300, sphk.default_params())
    e.upload(pos, vel, mass)
    far = pos[:1].repeat(300, 0)
    far[:] = 0.25
    far[7] = far[11] = 1e9
    with pytest.raises(sphk.SphkError, match=f"particle {n + 7} "):
        e.upload(far, offset=n)
    assert e.size() == n
    np.testing.assert_array_equal(e.positions(), pos)
    np.testing.assert_array_equal(e.velocities(), vel)
    np.testing.assert_array_equal(e.masses(), mass)
    e.upload(pos[:300], offset=n)  # no velocities, default mass
    m = min(n, 300)
    np.testing.assert_array_equal(e.positions(), np.concatenate([pos, pos[:m]]))
    np.testing.assert_array_equal(e.velocities()[n:], np.zeros((m, 3), np.float32))
    np.testing.assert_array_equal(e.masses()[n:],
                                  np.full(m, sphk.default_params().particle_mass, np.float32))
    assert e.densities().shape == (n + 300,)


@pytest.mark.parametrize("scenes", [1, 2])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 4097, 12287, 12288, 12289])
def test_small_build_equals_the_launches_it_replaces(sphk, n, scenes):
    # Up to 12,288 particles on up to 8,190 cells are sorted, tabled and listed by one workgroup.
    # The same particles in wider bounds have more cells and take the radix sort: from the second
    # step on (the grid then covers the bounds) the two engines build differently, and
    # walk the same pairs in the same order.  A pile-up of one cell, empty columns, particles
    # with a NaN coordinate (their own bin, stepped by the gather) and two scenes.
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.12, 0.28, (n, 3)).astype(np.float32)
    pos[: n // 3] = rng.uniform(0.20, 0.24, (n // 3, 3))
    pos[n // 2 + 1 : n // 2 + 4, 1] = np.nan
    vel = rng.normal(0, 0.1, (n, 3)).astype(np.float32)
    out = []
    for hi in (0.4, 2.0):
        p = sphk.default_params(xmin=0, xmax=hi, ymin=0, ymax=hi, zmin=0, zmax=hi, formulation=1)
        e = sphk.Engine(n, p)
        e.upload(pos, vel)
        if scenes == 2:
            e.set_scenes(np.array([0, n // 2, n], np.uint64))
        for _ in range(3):
            e.step(1e-6)
        offs, idx = e.neighbors()
        cells = e.grid()[2]
        assert (cells <= 8190) == (hi == 0.4), cells
        out.append((e.positions(), e.velocities(), e.densities()[:n], e.accelerations(), offs,
                    idx))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("shape", ["seg32_waves4_split", "seg24_waves4", "pp16_waves4"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 33, 1000, 1025])
def test_every_particle_its_own_chunk(sphk, n, shape):
    # The walks' launches provide for at most n chunks: here every particle is alone in its
    # (x, y) column, so there are exactly n.  Each has only itself as a neighbour: density
    # m W(0), which the force rows and the integration then use.
    side = 40
    k = np.random.default_rng(n).permutation(side * side)[:n]
    pos = np.stack([0.1 * (k // side) + 0.02, 0.1 * (k % side) + 0.02, 0.001 * (k % 7)], 1)
    p = sphk.default_params(xmin=-1, xmax=5, ymin=-1, ymax=5, zmin=-1, zmax=1)
    e = sphk.Engine(n, p)
    e.upload(pos.astype(np.float32))
    v = sphk.walk_shape_names().index(shape)
    e.set_walk_shapes(v, v)
    e.step(1e-4)
    assert len(e.walk_words()[0]) == n
    h, m = float(np.float32(p.smoothing_length)), float(np.float32(p.particle_mass))
    w0 = m * (2.0 / 3.0) / (np.pi * h**3)
    # one FP32 product each for sigma, W(0) and m W(0), and the spline's own two roundings
    np.testing.assert_allclose(e.densities()[:n], w0, rtol=8 * 2.0**-24)
    np.testing.assert_allclose(e.accelerations()[:, 1], -9.81, rtol=4 * 2.0**-24)


def test_wide_grid_stores_words_for_its_particles_only(sphk):
    # A chunk holds at least one particle, so 2,000 of them have at most 2,000 chunks, however many
    # columns their grid has (a million here): the word buffers stay at 2,000 x 64 KiB and all
    # 256 words of a chunk are stored.
    import ctypes

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert e.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n = 2000
    rng = np.random.default_rng(3)
    pos = rng.uniform([0, 0, 0], [40, 40, 0.4], (n, 3)).astype(np.float32)
    p = sphk.default_params(xmin=0, xmax=40, ymin=0, ymax=40, zmin=0, zmax=1)
    e = sphk.Engine(n, p)
    e.upload(pos)
    before = free_bytes()
    items, _, wj0, _ = e.walk_words()
    dims = e.grid()[1]
    assert int(dims[0]) * int(dims[1]) > 900000 and len(items) <= n
    assert wj0.shape[1] == 256
    # (the sort, scan and cell table of ten million cells among it)
    assert before - free_bytes() < 1 << 30


@pytest.mark.parametrize("n", [1, 7, 8, 9, 1000])
def test_surrogate_of_particles_alone_in_their_columns(sphk, n):
    # The surrogate's launches provide for as many chunks as there are particles: here there are
    # exactly that many, each particle without a neighbour, and so with the same prediction.
    side = 40
    k = np.random.default_rng(n).permutation(side * side)[:n]
    pos = np.stack([0.1 * (k // side) + 0.02, 0.1 * (k % side) + 0.02, 0.001 * (k % 7)], 1)
    p = sphk.default_params(xmin=-1, xmax=5, ymin=-1, ymax=5, zmin=-1, zmax=1, formulation=1)
    e = sphk.Engine(n, p)
    e.upload(pos.astype(np.float32))
    e.surrogate_init(seed=1)
    w = e.surrogate_params()
    w[-3:] = [1.0, -2.0, 3.0]  # the output bias
    e.surrogate_set_params(w)
    assert len(e.walk_words()[0]) == n
    out = e.surrogate_predict()
    assert np.abs(out).min() > 0.0
    np.testing.assert_array_equal(out, np.broadcast_to(out[0], out.shape))
    e.surrogate_macro_step(1e-4)
    np.testing.assert_array_equal(e.accelerations(), np.broadcast_to(e.accelerations()[0], out.shape))
    np.testing.assert_allclose(e.accelerations(), out, rtol=1e-5)


@pytest.mark.parametrize("radius", [0.04, 0.03, 0.0123, 0.9])
def test_pairs_two_cells_apart_are_listed(sphk, oracle, radius):
    # Pairs whose rounding puts them two cells apart and yet within the radius, a few ulps from a
    # cell edge, along each axis and in both directions: the walks look two cells out only
    # for chunks with a particle that the quick test lets through.
    f = np.float32
    R = f(radius)
    inv, r2 = f(1) / R, R * R
    rng = np.random.default_rng(5)
    x = np.concatenate([-R * 10.0 ** rng.uniform(-30, -6, 60),
                        [np.nextafter(k * R, f(-np.inf)) for k in range(-40, 40)]]).astype(f)
    c = np.floor(x * inv)
    b = x + R
    for _ in range(6):
        b = np.nextafter(b, f(-np.inf))
    pairs = []
    for _ in range(13):
        d = b - x
        pairs += [(x[i], b[i]) for i in np.nonzero((np.floor(b * inv) == c + 2) & (d * d <= r2))[0]]
        b = np.nextafter(b, f(np.inf))
    assert pairs
    pairs = pairs[:: max(1, len(pairs) // 40)]
    pos = []
    for k, (lo, hi) in enumerate(pairs):
        p = np.full((2, 3), 2.5 * R * (k // 3 + 1), f)  # pairs apart from each other
        p[:, k % 3] = (lo, hi) if k % 2 else (hi, lo)
        p[:, (k + 1) % 3] *= -1
        pos.append(p)
    pos = np.concatenate(pos)
    w = float(200 * R)
    e = sphk.Engine(len(pos), sphk.default_params(xmin=-w, xmax=w, ymin=-w, ymax=w, zmin=-w, zmax=w,
                                                  neighbor_search_radius=float(R),
                                                  smoothing_length=float(R) / 2))
    e.upload(pos)
    offs, idx = e.neighbors()
    boffs, bidx = oracle.brute_neighbors(pos, r2)
    for i in range(len(pos)):
        got = sorted(idx[offs[i]:offs[i + 1]].tolist())
        assert got == bidx[boffs[i]:boffs[i + 1]].tolist() and i ^ 1 in got


@pytest.mark.parametrize("rows", [9, 2054, 2055, 2056, 5000])
def test_refused_uploads_on_both_routes(sphk, rows):
    # Up to 2,048 rows are checked on the host, more on the device: either way the first row
    # beyond the cell range is named and the state stays as it was, and what is accepted sets the
    # same extent (the next step finds every particle inside its grid).
    rng = np.random.default_rng(rows)
    pos = rng.uniform(-1, 1, (100, 3)).astype(np.float32)
    more = rng.uniform(2, 3, (rows, 3)).astype(np.float32)
    p = sphk.default_params(xmin=-4, xmax=4, ymin=-4, ymax=4, zmin=-4, zmax=4, formulation=1)
    e = sphk.Engine(100 + rows - 7, p)  # the last seven rows do not fit
    e.upload(pos)
    before = e.neighbors()
    far = more.copy()
    far[rows - 9] = far[rows - 8, 2] = 1e9
    with pytest.raises(sphk.SphkError, match=f"particle {100 + rows - 9} "):
        e.upload(far, offset=100)
    assert e.size() == 100
    for a, b in zip(before, e.neighbors()):
        np.testing.assert_array_equal(a, b)
    more[5, 1] = np.nan
    more[rows - 3] = 1e9  # beyond the capacity: dropped, not checked
    with pytest.raises(sphk.SphkError, match="capacity"):
        e.upload(more, offset=100)
    assert e.size() == 100 + rows - 7
    np.testing.assert_array_equal(e.positions(), np.concatenate([pos, more[:-7]]))
    e.step(1e-5)
    e.positions()  # (would report a particle outside its grid)


@pytest.mark.parametrize("cut,graph", [(False, False), (False, True), (True, False)])
def test_corner_pile_ups_step_alike_in_every_shape(sphk, cut, graph):
    # The reference formulas pile a block up in its box's corners within a few steps: most chunks
    # then have more words than are stored, nearly all of one column, and in the team shapes every
    # wavefront goes over to a chunk of its own (1,100 chunks and more), and back to teams when
    # the block is uploaded again.  Bits and neighbour statistics are those of the other shapes.
    names = sphk.walk_shape_names()
    n = 80000
    s = n ** (1 / 3) * 0.01
    pos = np.random.default_rng(1).uniform(0, s, (n, 3)).astype(np.float32)
    p = sphk.default_params(xmin=0, xmax=2.5 * s, ymin=0, ymax=1.5 * s, zmin=0, zmax=1.2 * s,
                            smoothing_length=0.025 if cut else 0.02)
    out = []
    for d, f in ((None, None), ("seg16_waves4_split",) * 2, ("seg24_waves4", "pp16_waves4")):
        e = sphk.Engine(n, p)
        e.upload(pos)
        e.set_graph(graph)
        if d:
            e.set_walk_shapes(names.index(d), names.index(f))
        got = []
        for steps in (5, 1, 1):
            for _ in range(steps):
                e.step(1e-3)
            st = e.stats()
            got += [e.positions(), e.velocities(), e.densities()[:n], e.accelerations(),
                    np.array([st.max_neighbors, st.total_neighbors])]
        if d is None:
            items, nwords, _, _ = e.walk_words()
            assert len(items) >= 1100 and np.mean(nwords > 256) > 0.5
        for _ in range(2):
            e.upload(pos)
            e.step(1e-3)
            got += [e.positions(), e.velocities()]
        out.append(got)
    for other in out[1:]:
        for a, b in zip(out[0], other):
            np.testing.assert_array_equal(a, b)
