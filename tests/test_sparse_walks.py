"""Walks of sparse scenes, whose chunks span many z cells: the stored candidate words against the
integer test, and particles with non-finite values that reach no one beyond the radius."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = np.float32
RADIUS = F32(0.04)


def _column_scene(per_cell, seed):
    """A tall, sparsely filled block of 4 x 4 x 125 cells, a dense block in some of its columns and,
    well above it, a layer that shares words with what lies below."""
    rng = np.random.default_rng(seed)
    n = int(4 * 4 * 125 * per_cell)
    return np.concatenate([
        rng.uniform([0.01, 0.01, -2.0], [0.17, 0.17, 3.0], size=(n, 3)),
        rng.uniform(0.02, 0.10, size=(700, 3)),
        rng.uniform([0.01, 0.01, 4.5], [0.17, 0.17, 4.55], size=(100, 3))]).astype(F32)


def _params(sphk, **kw):
    return sphk.default_params(xmin=0, xmax=1, ymin=0, ymax=1, zmin=-3, zmax=6, **kw)


def _integer_test(pos):
    """Coordinates and threshold of the candidate test: 256 units a cell, a pair passes when its
    squared distance in units is at most T (the radius plus the rounding of both ends)."""
    inv = F32(1) / RADIUS
    scale = 256.0 * float(inv)
    x = np.floor(pos.astype(np.float64) * scale).astype(np.int64)
    reach = np.sqrt(float(RADIUS * RADIUS)) * (1 + 1e-6) * scale + np.sqrt(3.0) * 1.001
    return x, int(np.floor(reach * reach))


def _check_words(sphk, pos, params, shape):
    """Every stored bit against the integer test; the stored pairs and those within the radius."""
    n = len(pos)
    e = sphk.Engine(n, params)
    e.upload(pos)
    names = sphk.walk_shape_names()
    e.set_walk_shapes(names.index(shape), names.index("seg32_waves4"))
    items, nwords, wj0, mask = e.walk_words()
    order, cells = e.sorted_order()
    nz = int(e.grid()[1][2])
    x, T = _integer_test(pos[order])
    col = cells // nz
    pairs, near, wide = 0, 0, 0
    for c in range(len(items)):
        a, nw = int(items[c]), int(nwords[c])
        assert nw <= wj0.shape[1]
        tgt = np.arange(a, min(a + 64, n))
        tgt = tgt[col[tgt] == col[a]]
        wide += int(cells[tgt[-1]] - cells[tgt[0]] > 4)
        # a word ends after 32 slots or with its column's candidate range: bits beyond are zero,
        # so every slot whose bit is set is a candidate, and the rest are compared up to the
        # last slot of the word's column
        slots = wj0[c, :nw, None].astype(np.int64) + np.arange(32)
        inside = slots < n
        slots = np.minimum(slots, n - 1)
        inside &= col[slots] == col[slots[:, :1]]
        d = x[slots][:, :, None, :] - x[tgt][None, None, :, :]
        d2 = (d * d).sum(3)
        want = (d2 <= T) & inside[:, :, None]
        bits = (mask[c, :nw, None, : len(tgt)] >> (31 - np.arange(32))[None, :, None]) & 1
        got = bits.astype(bool)
        assert not (got & ~want).any(), "a pair beyond the integer test is stored"
        # a passing pair past the word's end belongs to the next word of its column
        ends = np.array([np.count_nonzero(g) for g in inside])
        full = ends == 32
        assert (got == want)[full].all(), "a pair of the integer test is missing"
        assert not mask[c, :nw, len(tgt):].any()
        pairs += int(got.sum())
        near += int((d2[got] <= 256 * 256).sum())
    assert wide > 0
    return pairs, near


@pytest.mark.parametrize("shape", ["seg24_waves4", "seg16_waves4_split", "seg32_waves4_split",
                                   "pp12_waves4"])
@pytest.mark.parametrize("per_cell", [0.3, 1.0, 3.0, 6.0, 12.0])
def test_words_of_sparse_columns_equal_the_integer_test(sphk, per_cell, shape):
    # The matrix cores take a word whose candidates lie within some z cells, the VALU any
    # other: bit by bit both are the integer test, so no pair beyond it is walked (its row, if
    # not finite, would reach the sums) and the order of a target's pairs does not depend on
    # which unit tested them.
    pairs, near = _check_words(sphk, _column_scene(per_cell, int(10 * per_cell)), _params(sphk),
                               shape)
    assert pairs <= 1.06 * near, (pairs, near)


@pytest.mark.parametrize("shape", ["seg24_waves4", "seg32_waves4_split"])
@pytest.mark.parametrize("cells", [300, 65536])
def test_words_of_tall_columns_equal_the_integer_test(sphk, cells, shape):
    # Candidates so far apart that the square of their distance passes 2^31 units, or the
    # distance itself 2^24: neither may wrap around into the radius.
    rng = np.random.default_rng(cells)
    top = cells * 0.04
    ends = [rng.uniform([0.01, 0.01, z], [0.17, 0.17, z + 0.08], size=(400, 3)) for z in (0.0, top)]
    between = rng.uniform([0.01, 0.01, 0.0], [0.17, 0.17, top], size=(1200, 3))
    pos = np.concatenate(ends + [between]).astype(F32)
    p = sphk.default_params(xmin=0, xmax=1, ymin=0, ymax=1, zmin=-1, zmax=top + 1)
    _check_words(sphk, pos, p, shape)


@pytest.mark.parametrize("shape", ["seg24_waves4", "seg32_waves4_split", "pp16_waves4"])
def test_far_particles_reach_no_one(sphk, shape):
    # Particles of a sparse column with a NaN velocity, an infinite one or an infinite mass, and
    # a massless one without neighbours (density 0, mass over density not a number): every
    # particle beyond the radius steps to the same bits as beside ordinary ones.
    pos = _column_scene(0.5, 3)
    n = len(pos)
    rng = np.random.default_rng(4)
    vel = rng.normal(0, 0.1, (n, 3)).astype(F32)
    mass = np.full(n, 1e-3, F32)
    from scipy.spatial import cKDTree
    tree = cKDTree(pos.astype(np.float64))
    alone = np.array([i for i in range(1000) if len(tree.query_ball_point(pos[i], 0.041)) == 1])
    odd = alone[:: max(1, len(alone) // 40)][:40]
    assert len(odd) >= 30
    vel2, mass2 = vel.copy(), mass.copy()
    vel2[odd[0::4]] = np.nan
    vel2[odd[1::4], 1] = np.inf
    mass2[odd[2::4]] = np.inf
    mass2[odd[3::4]] = 0.0
    out = []
    for v, m in ((vel, mass), (vel2, mass2)):
        e = sphk.Engine(n, _params(sphk, formulation=1))
        e.upload(pos, v, m)
        k = sphk.walk_shape_names().index(shape)
        e.set_walk_shapes(k, k)
        e.step(1e-5)
        out.append((e.densities()[:n], e.accelerations(), e.velocities(), e.positions()))
    rest = np.setdiff1d(np.arange(n), odd)
    for a, b in zip(*out):
        assert np.isfinite(a[rest]).all()
        np.testing.assert_array_equal(a[rest], b[rest])


@pytest.mark.parametrize("radius_cut", [False, True])
@pytest.mark.parametrize("shape", ["seg32_waves4_split", "seg24_waves4", "pp16_waves4"])
def test_tall_grids_step_like_low_ones(sphk, shape, radius_cut):
    # Grids of more than 180 z cells take walk kernels of their own.  The same particles, a pile
    # with more words than are stored (tested again by the force walk) among them, in low and in
    # tall bounds: from the second step on, when the grid covers the bounds, one engine takes the
    # one, the other the other, and every bit agrees.
    rng = np.random.default_rng(9)
    pos = np.concatenate([rng.uniform(0.1, 0.5, (3000, 3)),
                          rng.uniform([0.22, 0.22, 0.22], [0.26, 0.26, 0.30], (9000, 3))]).astype(F32)
    vel = rng.normal(0, 0.1, pos.shape).astype(F32)
    k = sphk.walk_shape_names().index(shape)
    out = []
    for top in (0.6, 12.0):
        p = sphk.default_params(xmin=0, xmax=0.6, ymin=0, ymax=0.6, zmin=0, zmax=top, formulation=1,
                                particle_mass=1e-5, smoothing_length=0.025 if radius_cut else 0.02)
        e = sphk.Engine(len(pos), p)
        e.upload(pos, vel)
        e.set_walk_shapes(k, k)
        for graph in (False, False, True, True):
            e.set_graph(graph)
            e.step(1e-6)
        assert (int(e.grid()[1][2]) > 180) == (top > 1)
        assert e.walk_words()[1].max() > 256
        out.append((e.positions(), e.velocities(), e.densities()[:len(pos)], e.accelerations()))
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
