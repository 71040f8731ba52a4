"""The walks' two-cells-apart rule itself (csrc/sphk_edge_rule.h, built for the host): the exact flags
against partners found by trying floats, and the quick test against the exact flags."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

F = np.float32
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    so = str(tmp_path_factory.mktemp("edge") / "edge_rule.so")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared",
                        "-fPIC", "-o", so, os.path.join(HERE, "native", "edge_rule.cpp")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lib = C.CDLL(so)
    pf, pi = C.POINTER(C.c_float), C.POINTER(C.c_int)
    lib.edge_rule.argtypes = [pf, C.c_size_t, C.c_float, C.c_float, pi, pi]

    def run(x, inv, r2):
        x = np.ascontiguousarray(x, F)
        flags, near = np.empty(len(x), np.int32), np.empty(len(x), np.int32)
        lib.edge_rule(x.ctypes.data_as(pf), len(x), inv, r2, flags.ctypes.data_as(pi),
                      near.ctypes.data_as(pi))
        return flags, near.astype(bool)

    return run


def _samples(R):
    rng = np.random.default_rng(1)
    k = np.concatenate([np.arange(-300, 300), rng.integers(-(1 << 22), 1 << 22, 4000)])
    edge = (k.astype(np.float64) * float(R)).astype(F)
    xs = [(rng.uniform(-5, 5, 200000) * R).astype(F), edge,
          (-R * 10.0 ** rng.uniform(-30, -6, 2000)).astype(F)]
    up = down = edge
    for ulps in range(1, 41):  # floats around every cell edge
        up, down = np.nextafter(up, F(np.inf)), np.nextafter(down, F(-np.inf))
        xs += [up, down]
        xs += [edge + F(ulps * 1e-7) * np.abs(edge), edge - F(ulps * 1e-7) * R]
    return np.concatenate(xs)


@pytest.mark.parametrize("radius", [0.04, 0.05, 1.0, 0.0123, 3.7, 1e-3])
def test_every_partner_two_cells_away_is_flagged(rule, radius):
    R = F(radius)
    inv, r2 = F(1) / R, R * R
    x = _samples(R)
    flags, near = rule(x, inv, r2)
    c = np.floor(x * inv)
    found = 0
    for sign, bit in ((F(1), 2), (F(-1), 1)):
        b = x + sign * R
        for _ in range(6):
            b = np.nextafter(b, -sign * F(np.inf))
        for _ in range(13):  # the floats around x +- R: the reference's cell and distance tests
            d = b - x
            partner = (np.floor(b * inv) == c + 2 * sign) & (d * d <= r2)
            assert not (partner & ((flags & bit) == 0)).any()
            found += int(partner.sum())
            b = np.nextafter(b, sign * F(np.inf))
    assert found > 0
    assert not ((flags != 0) & ~near).any(), "the quick test skips a flagged particle"
    # and it does skip: almost no particle of a random scene is near an edge
    y = (np.random.default_rng(2).uniform(0, 100, 200000) * radius).astype(F)
    assert rule(y, inv, r2)[1].mean() < 2e-3
