"""The walks skip the exact two-cells-apart test for particles well inside their cell: the skip
rule against the exact flags, in FP32 arithmetic on the CPU."""
import numpy as np
import pytest

F = np.float32


def exact_flags(x, inv, r2):
    """Can x have a neighbour two cells up or down: the nearest float of that cell, tested with
    the reference's rounded arithmetic (found by stepping from the cell's edge)."""
    c = np.floor(x * inv)
    up = ((c + F(2)) / inv).astype(F)
    lo = ((c - F(1)) / inv).astype(F)
    for _ in range(8):  # smallest float with fl(b inv) >= c + 2; largest with fl(b inv) < c - 1
        up = np.where(up * inv >= c + F(2), up, np.nextafter(up, F(np.inf)))
        lo = np.where(lo * inv < c - F(1), lo, np.nextafter(lo, F(-np.inf)))
    for _ in range(8):
        d = np.nextafter(up, F(-np.inf))
        up = np.where(d * inv >= c + F(2), d, up)
        d = np.nextafter(lo, F(np.inf))
        lo = np.where(d * inv < c - F(1), d, lo)
    du, dl = up - x, x - lo
    return (du * du <= r2) | (dl * dl <= r2)


def near(x, inv):
    t = x * inv
    c = np.floor(t)
    m = (np.abs(c) + F(3)) * F(2.0 ** -19)
    f = t - c
    return ~((f > m) & (f < F(1) - m))


@pytest.mark.parametrize("radius", [0.04, 0.05, 1.0, 0.0123, 3.7, 1e-3])
def test_skipped_particles_have_no_neighbour_two_cells_away(radius):
    R = F(radius)
    inv, r2 = F(1) / R, R * R
    rng = np.random.default_rng(1)
    k = np.concatenate([np.arange(-300, 300), rng.integers(-(1 << 22), 1 << 22, 4000)])
    edge = (k.astype(np.float64) * float(R)).astype(F)
    xs = [(rng.uniform(-5, 5, 200000) * radius).astype(F), edge]
    for ulps in (1, 2, 3, 5, 9, 17, 40, 200):  # floats around every cell edge
        up = edge.copy()
        for _ in range(min(ulps, 40)):
            up = np.nextafter(up, F(np.inf))
        xs += [up, -up, edge + F(ulps * 1e-7) * np.abs(edge), edge - F(ulps * 1e-7) * R]
    x = np.concatenate(xs)
    flags = exact_flags(x, inv, r2)
    assert flags.any()
    assert not (flags & ~near(x, inv)).any()
    # and the rule does skip: almost no particle of a random scene is near an edge
    y = (rng.uniform(0, 100, 200000) * radius).astype(F)
    assert near(y, inv).mean() < 2e-3
