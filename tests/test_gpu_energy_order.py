"""A step's energy is the same bits for every launch shape and every way the
run is cut into blocks: whether the step is the first of two in a launch or
alone, and which wave takes which cells."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers

pytestmark = pytest.mark.gpu


def _scene(nx, ny, nz, pulse="f32", seed=4):
    rng = np.random.default_rng(seed)
    mat = np.zeros((nz, ny, nx), np.uint8)
    mat[:, : ny // 2] = rng.choice([0, 1, 2], (nz, ny // 2, nx), p=[0.6, 0.1, 0.3])
    mat[nz // 2, ny // 2, nx // 2] = 0
    s = scenes.Scene(nx, ny, nz, mat.reshape(-1), np.array([4.0], np.float32), np.array([0.02], np.float32),
                     rho=0.37, total_steps=24, pulse=pulse, fp32_halo=2, name=f"energy_{nx}x{ny}x{nz}")
    s.sources = [(s.cell(nx // 2, ny // 2, nz // 2), 2, 1.0)]
    s.faces, s.energy_every = False, 3
    s.V0 = rng.standard_normal(12 * mat.size).astype(np.float32)
    s.V0.reshape(-1, 12)[s.mat == scenes.MAT_PEC] = 0
    return s


def _energy(sc, blocks, **tuning):
    with tlm.open_scene(sc) as dev:
        if tuning:
            dev.set_tuning(**tuning)
        n = 0
        while n < sc.total_steps:
            m = min(blocks[n % len(blocks)], sc.total_steps - n)
            dev.run(n, m)
            n += m
        dev.sync()
        return dev.read_energy()[1]


# one tile a slab and several, a short last block, one and two blocks a wave
@pytest.mark.parametrize("dims", [(13, 9, 5), (70, 41, 9), (130, 37, 18), (260, 33, 7), (200, 190, 180)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("pulse", ["f32", "f16"])
def test_energy_does_not_depend_on_the_launch(dims, pulse):
    sc = _scene(*dims, pulse=pulse)
    print(f"[energy] {sc.name} {pulse}", flush=True)
    first = _energy(sc, [24])
    assert first.size == 8 and first.min() > 0
    for blocks in ([1], [3], [2, 5, 1]):
        assert np.array_equal(_energy(sc, blocks), first), blocks
    for tuning in ({"fold": 1}, {"planes": 3}, {"planes": 2, "block_waves": 1}, {"grid_blocks": 16}):
        assert np.array_equal(_energy(sc, [24], **tuning), first), tuning


def test_energy_against_the_restatement():
    sc = dataclasses.replace(_scene(70, 41, 9), energy_every=16)  # the restatement's interval
    ref = helpers.oracle_run(sc)
    assert np.allclose(_energy(sc, [24]), ref.energy, rtol=1e-12, atol=0)
