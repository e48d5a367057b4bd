"""Two steps a launch (k_step2) against the CPU restatement: the same bits as
single steps at the edges of its tiles (rows shorter and longer than a wave,
slabs of one tile or several, a last tile cut short, one and two blocks per
wave, one slab), with every monitor that a pair records, odd numbers of steps
and single steps in between. Energies agree to the tolerance of a sum in
another order (1e-12 relative), all else exactly."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers

pytestmark = pytest.mark.gpu


def _scene(nx, ny, nz, steps, rho=0.37, seed=0, diel=True, plane=-1, record=0):
    rng = np.random.default_rng([nx, ny, nz, seed])
    n = nx * ny * nz
    u = rng.random(n)
    mat = np.zeros(n, np.uint8)
    # a mix of materials in part of the grid, plain air in the rest
    m3 = mat.reshape(nz, ny, nx)
    u3 = u.reshape(nz, ny, nx)
    part = np.zeros((nz, ny, nx), bool)
    part[:, :(ny + 1) // 2, :(nx + 2) // 3] = True
    m3[part & (u3 < 0.08)] = scenes.MAT_PEC
    if diel:
        m3[part & (u3 >= 0.08) & (u3 < 0.4)] = 2
        m3[part & (u3 >= 0.4) & (u3 < 0.5)] = 4
    nd = 3 if diel else 0
    s = scenes.Scene(nx, ny, nz, mat, rng.uniform(1, 10, nd).astype(np.float32),
                     rng.uniform(0, 0.05, nd).astype(np.float32), rho=rho, total_steps=steps,
                     settle_steps=3, name=f"pairs_{nx}x{ny}x{nz}")
    ok = np.flatnonzero(mat != scenes.MAT_PEC)
    s.sources = [(int(ok[len(ok) // 2]), 2, 1.0), (int(ok[len(ok) // 2]), 0, 0.5), (int(ok[-1]), 1, -0.7)]
    s.probes = np.array(rng.choice(n, min(6, n), replace=False), np.int64)
    s.dft_freqs = np.array([1e8, 1e9])
    s.plane_axis, s.record_every = plane, record
    if min(nx, ny, nz) > 8:
        s.huy_offset = 2
        c = [s.cell(nx // 2, ny // 2, k) for k in (nz // 2, nz // 2 + 1)]
        mat[c] = scenes.MAT_AIR
        s.ports = [(c, 2, 0.6)]
    V0 = rng.standard_normal((n, 12)).astype(np.float32)
    V0[mat == scenes.MAT_PEC] = 0
    s.V0 = V0.reshape(-1)
    if diel:
        Vs0 = rng.standard_normal((n, 3)).astype(np.float32)
        Vs0[mat < 2] = 0
        s.Vs0 = Vs0.reshape(-1)
    return s


def _check(sc, block=256):
    print(f"[pairs] {sc.name} rho={sc.rho} steps={sc.total_steps} block={block}", flush=True)
    helpers.compare_results(tlm.run_scene(sc, block=block), helpers.oracle_run(sc), sc)


# nx, ny, nz: below a wave; a wave and one either side; a slab of one tile;
# several tiles with a short last one; rims of 2, 4 and 5+ blocks (two blocks
# per wave), the widest rim; one slab
SHAPES = [(1, 1, 1), (3, 40, 5), (63, 9, 4), (64, 9, 11), (65, 12, 10), (64, 64, 12), (130, 21, 9),
          (256, 11, 9), (257, 10, 9), (330, 13, 10), (768, 9, 9), (40, 40, 1), (100, 37, 19)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("rho", [0.37, -1.0])
def test_pairs_match_the_restatement(shape, rho):
    _check(_scene(*shape, steps=23 if shape[0] < 700 else 9, rho=rho))


def test_pairs_without_stubs():
    _check(_scene(70, 30, 14, steps=20, diel=False))


def test_wider_grids_keep_single_steps():
    _check(_scene(769, 5, 4, steps=6))


@pytest.mark.parametrize("plane,record,block", [(1, 0, 256), (2, 6, 256), (0, 5, 7), (-1, 3, 5), (-1, 0, 1)])
def test_pairs_between_single_steps(plane, record, block):
    """Steps whose plane, frame or energy comes second are single steps, and a
    block may end between the two of a pair."""
    _check(_scene(37, 26, 15, steps=31, plane=plane, record=record), block=block)


def test_two_blocks_per_wave_on_a_large_grid_equal_single_steps():
    """A grid large enough for two blocks per wave and several rounds of
    tiles: every record and the whole state against the same grid stepped one
    step a launch."""
    sc = scenes.dielectric_boxes(n=200, nboxes=8, steps=37, nprobes=8, nfreq=4, seed=9)
    sc.rho = 0.37
    sc.probes = np.array([sc.cell(100 + d, 100, 100 - d) for d in range(8)], np.int64)  # round the source
    a = tlm.run_scene(sc)
    with tlm.open_scene(sc) as dev:
        dev.set_tuning(fold=1)  # a launch shape of the caller's: single steps
        dev.run(0, 37)
        dev.sync()
        b = tlm.collect(dev, sc, 37)
    for f in ("probes", "js_inst", "js_dft4", "V", "Vs"):
        helpers.assert_bitexact(f, getattr(a, f), getattr(b, f))
    assert np.abs(a.probes).max() > 0
    assert np.array_equal(a.probe_dft[0], b.probe_dft[0])
    assert np.allclose(a.energy, b.energy, rtol=1e-12, atol=0)


def test_a_new_scene_in_the_same_context():
    """The second stub buffer holds nothing of the scene before."""
    one, two = _scene(48, 30, 14, steps=12, seed=1), _scene(48, 30, 14, steps=12, seed=2)
    m3 = two.mat.reshape(14, 30, 48)
    m3[7:] = np.where(m3[7:] >= 2, 0, m3[7:])  # dielectric only where `one` may have had none
    two = dataclasses.replace(two, Vs0=None)
    with tlm.open_scene(one) as dev:
        dev.run(0, 12)
        dev.sync()
        yh, gh = tlm.stub_admittances(two.epsr, two.sigma, two.dl)
        dev.upload(two.mat, yh, gh, two.V0)
        dev.set_sources([c for c, _, _ in two.sources], [p for _, p, _ in two.sources],
                        [a for _, _, a in two.sources])
        dev.run(0, 12)
        dev.sync()
        V, Vs = dev.read_state()
    ref = helpers.oracle_run(dataclasses.replace(two, ports=[]))
    helpers.assert_bitexact("V", V, ref.V)
    helpers.assert_bitexact("Vs", Vs, ref.Vs)


def test_timed_steps_count_both_steps_of_a_pair():
    sc = _scene(64, 20, 12, steps=40, diel=False)
    with tlm.open_scene(sc) as dev:
        total, per = dev.time_steps(0, 40, kernel_every=1)
    assert 0 < per * 40 <= total * 1.05
