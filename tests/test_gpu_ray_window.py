"""Solid fill of triangle soups whose rays' hits depend on rounding: k_ray_slots
leaves out triangles by a window round them, which must not lose a hit that
the oracle's test of every triangle finds. Each kind has shapes at which u and
v of the ray test are inexact: slivers, triangles almost parallel to the rays,
tiny and huge ones, edges through cell centres, far from the grid."""
import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers

pytestmark = pytest.mark.gpu


def _soup(kind, rng, o, L, dl, n):
    a = o + rng.uniform(-0.1, 1.1, (n, 3)) * L
    if kind == "sliver":  # b and c almost in line with a
        d = rng.normal(size=(n, 3)) * 0.4 * L
        t = rng.uniform(0.2, 2.0, (n, 1))
        return a, a + d, a + d * t + rng.normal(size=(n, 3)) * L * 10.0 ** rng.uniform(-9, -3, (n, 1))
    if kind == "along":  # almost parallel to x
        d, e = rng.normal(size=(2, n, 3)) * 0.4 * L
        s = 10.0 ** rng.uniform(-7, -1, (2, n, 1))
        d[:, 1:] *= s[0]
        e[:, 1:] *= s[1]
        return a, a + d, a + e
    if kind == "tiny":
        s = dl * 10.0 ** rng.uniform(-4, 0, (n, 1))
        return a, a + rng.normal(size=(n, 3)) * s, a + rng.normal(size=(n, 3)) * s
    if kind == "huge":
        return tuple(o + rng.uniform(-40, 41, (n, 3)) * L for _ in range(3))
    # vertices on cell centres
    return tuple(o + (rng.integers(0, 24, (n, 3)) + 0.5) * dl for _ in range(3))


@pytest.mark.parametrize("shift", [0.0, 300.0])
@pytest.mark.parametrize("kind", ["sliver", "along", "tiny", "huge", "centres"])
def test_soup_equals_oracle(kind, shift):
    rng = np.random.default_rng(len(kind) + int(shift))
    dims, dl = (31, 27, 25), 0.02
    origin = tuple(float(np.float32(x + shift * dl)) for x in (-0.2, 0.1, 0.05))
    L, o = np.array(dims) * dl, np.array(origin)
    cells = 0
    for n in (8, 90, 700):
        v = np.stack(_soup(kind, rng, o, L, dl, n), 1).reshape(-1, 3).astype(np.float32)
        sc = scenes.Scene(*dims, None, dl=dl, origin=origin)
        sc.ops = [("mesh", v, np.arange(3 * n, dtype=np.int32).reshape(n, 3), (0.0, 0.0, 0.0), 3, True)]
        print(f"[window] {kind} {n} shift {shift}", flush=True)
        host = helpers.oracle_build(sc)
        with tlm.TlmDevice(*dims, dl) as dev:
            tlm.apply_ops(dev, sc)
            got = dev.mat_read()
        assert np.array_equal(got, host.mat)
        cells += int(host.mat.any())
    assert cells
