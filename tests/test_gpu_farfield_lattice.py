"""The far field of a context's Huygens box as sums over its lattice
(k_ff_lattice) and of plain face lists (k_ff_sums), with and without opposite
directions taken together (an odd or even number of phi samples).

Tolerance: that of test_gpu_ntff.py, 2e-5 of U_max against sums in double
(numpy's here, over some of the directions; over all of them the two device
paths are held to each other, to twice that): float
products and sums of at most some 1e4 terms a direction, random
rounding errors of 6e-8 each, of which the peak takes about sqrt(1e4) * 6e-8 =
6e-6."""
import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from oracle import oracle_tlm as ot

pytestmark = pytest.mark.gpu
GRID = (91, 181)  # directions enough for the lattice


def _accumulated(dims, offset, keep=None, pec=None, listed=False, V0=None):
    """A context after some steps, its faces and accumulators; keep picks
    faces (listed: set as a list), pec holes in the box."""
    nx, ny, nz = dims
    mat = np.zeros((nz, ny, nx), np.uint8)
    if pec:
        (x0, y0, z0), (x1, y1, z1) = pec
        mat[z0:z1, y0:y1, x0:x1] = 1
    sc = scenes.Scene(nx, ny, nz, mat.reshape(-1), total_steps=90, name="ff")
    sc.waveform, sc.f0 = scenes.WF_GAUSS_DERIV, 2e9
    sc.gd_width, sc.gd_delay = 8.0, 20.0
    sc.sources = [(sc.cell(nx // 2, ny // 2 - 1, nz // 2), 2, 1.0), (sc.cell(nx // 2 - 2, ny // 2, nz // 2), 0, 0.6)]
    sc.faces, sc.settle_steps = False, 0
    sc.V0 = V0
    dev = tlm.open_scene(sc)
    if listed:
        cells, axes = tlm.huygens_faces(nx, ny, nz, sc.mat, offset)[:2]
        k = np.ones(len(cells), bool) if keep is None else keep(cells, axes)
        dev.set_huygens(cells[k], axes[k])
    else:
        dev.huygens_mat(offset)
    dev.run(0, sc.total_steps)
    dev.sync()
    return sc, dev


def _far64(pos, axes, sg, d8, f0, nt, nph, d):
    """Intensity from face currents in directions d of the grid, in doubles."""
    e = np.asarray(d8, np.float64).reshape(-1, 4, 2) @ np.array([1, 1j])  # E1, E2, eta0 H1, eta0 H2
    S = np.zeros((len(e), 6), complex)
    for a, (t1, t2) in enumerate(((1, 2), (0, 2), (0, 1))):
        w = np.nonzero(np.asarray(axes) == a)[0]
        s = sg[w] * (-1.0 if a == 1 else 1.0)
        for col, x in ((t2, e[w, 2]), (t1, -e[w, 3]), (3 + t2, -e[w, 0]), (3 + t1, e[w, 1])):
            S[w, col] = s * x
    th, ph = np.pi * (d // nph) / (nt - 1), 2 * np.pi * (d % nph) / (nph - 1)
    r = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], 1)
    V = np.exp(2j * np.pi * f0 / 299792458.0 * (r @ np.asarray(pos, np.float64).T)) @ S
    t = np.stack([np.cos(th) * np.cos(ph), np.cos(th) * np.sin(ph), -np.sin(th)], 1)
    p = np.stack([-np.sin(ph), np.cos(ph), 0 * ph], 1)
    Nt, Np, Lt, Lp = ((V[:, a:a + 3] * q).sum(1) for a, q in ((0, t), (0, p), (3, t), (3, p)))
    return np.abs(Lp + Nt) ** 2 + np.abs(Lt - Np) ** 2


def _check(got, plain, geometry, f0, grid):
    """Both results against doubles in the peak's and 400 other directions."""
    n = grid[0] * grid[1]
    d = np.unique(np.r_[0, n - 1, got.U.argmax(), plain.U.argmax(), np.random.default_rng(n).integers(0, n, 400)])
    U = _far64(*geometry, f0, *grid, d)
    for r in (got, plain):
        assert np.abs(r.U.reshape(-1)[d] - U).max() < 2e-5 * U.max()
        assert abs(r.u_max - U.max()) < 2e-5 * U.max()
    assert np.abs(got.U - plain.U).max() < 4e-5 * U.max()


@pytest.mark.parametrize("dims,offset,listed,pec", [
    ((34, 33, 47), 3, False, None),                    # even, odd, odd counts of cells in the box
    ((41, 36, 35), 2, True, None),                     # as a list
    ((40, 40, 40), 3, True, ((0, 10, 12), (9, 24, 30))),  # faces missing
    ((9, 60, 61), 2, False, None),                     # a side of 5 cells: fewer rows than a batch
    ((24, 22, 26), 2, False, None),                    # under the least number of faces: a plain list
])
@pytest.mark.parametrize("grid", [(121, 241), (120, 150), (5, 9), (2, 3)])  # the latter two: plain sums
def test_lattice_matches_doubles(dims, offset, listed, pec, grid):
    sc, dev = _accumulated(dims, offset, None, pec, listed)
    with dev:
        cells, axes = dev.read_huygens_faces()
        d8 = dev.read_huygens()
        assert np.abs(d8).max() > 0
        print(f"[lattice] {dims} offset {offset} {len(cells)} faces, {grid}", flush=True)
        got = tlm.far_field_ctx(dev, sc.origin, 1, sc.f0, *grid)
        again = tlm.far_field_ctx(dev, sc.origin, 1, sc.f0, *grid, noalloc=True)
        assert np.array_equal(got.U, again.U)
        pos, sg = ot.huygens_geometry(dims, sc.origin, sc.dl, cells, axes)
        plain = tlm.far_field(pos, axes, sg, d8, sc.f0, *grid)
        _check(got, plain, (pos, axes, sg, d8), sc.f0, grid)


def test_lists_that_are_no_box():
    """Faces listed twice, and a non-finite accumulator: the plain sums."""
    dims = (40, 38, 36)

    def half_twice(cells, axes):
        return np.r_[np.arange(len(cells)), np.arange(0, len(cells), 2)]

    sc, dev = _accumulated(dims, 3, half_twice, None, True)
    with dev:
        cells, axes = dev.read_huygens_faces()
        d8 = dev.read_huygens()
        pos, sg = ot.huygens_geometry(dims, sc.origin, sc.dl, cells, axes)
        got = tlm.far_field_ctx(dev, sc.origin, 1, sc.f0, *GRID)
        plain = tlm.far_field(pos, axes, sg, d8, sc.f0, *GRID)
        assert np.array_equal(got.U, plain.U)
        _check(got, plain, (pos, axes, sg, d8), sc.f0, GRID)


def test_infinite_field_takes_plain_sums():
    dims = (40, 38, 36)
    v = np.zeros((12, 36, 38, 40), np.float32)
    v[4, 18, 19, 20] = np.inf
    sc, dev = _accumulated(dims, 3, None, None, True, v.reshape(-1))
    with dev:
        cells, axes = dev.read_huygens_faces()
        d8 = dev.read_huygens()
        assert not np.isfinite(d8).all()
        pos, sg = ot.huygens_geometry(dims, sc.origin, sc.dl, cells, axes)
        got = tlm.far_field_ctx(dev, sc.origin, 1, sc.f0, *GRID)
        want = tlm.far_field(pos, axes, sg, d8, sc.f0, *GRID)
        assert np.array_equal(got.U, want.U, equal_nan=True)
