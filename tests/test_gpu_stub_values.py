"""Stub values that a caller uploads in cells that are no dielectric: the step
leaves them alone (as the restatement does), whatever number of pairs of steps
ran, alone and in a batch."""
import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers

pytestmark = pytest.mark.gpu


def _scene(steps):
    """Rows of 70 cells; dielectric in a few cells only, so that most 32-cell
    halves of a block hold none, PEC among them, stub values everywhere."""
    nx, ny, nz = 70, 12, 9
    rng = np.random.default_rng(3)
    mat = np.zeros(nx * ny * nz, np.uint8)
    mat[rng.choice(mat.size, 40, replace=False)] = 2
    mat[rng.choice(mat.size, 40, replace=False)] = scenes.MAT_PEC
    s = scenes.Scene(nx, ny, nz, mat, np.array([3.0], np.float32), np.array([0.01], np.float32), rho=0.37,
                     total_steps=steps, name="stub_values")
    s.faces, s.energy_every = False, 0
    s.V0 = rng.standard_normal(12 * mat.size).astype(np.float32)
    s.V0.reshape(-1, 12)[mat == scenes.MAT_PEC] = 0
    s.Vs0 = rng.standard_normal(3 * mat.size).astype(np.float32)
    return s


@pytest.mark.parametrize("steps", [16, 18, 19])
@pytest.mark.parametrize("batch", [False, True])
def test_stubs_outside_dielectrics_stay(steps, batch):
    sc = _scene(steps)
    with tlm.open_scene(sc) as dev:
        if batch:
            with tlm.TlmBatch() as b:
                b.add(dev, steps)
                b.run(steps)
                b.remove(dev)
        else:
            dev.run(0, steps)
            dev.sync()
        assert dev.step_launches()[1] == steps // 2
        V, Vs = dev.read_state()
    ref = helpers.oracle_run(sc)
    helpers.assert_bitexact("V", V, ref.V)
    helpers.assert_bitexact("Vs", Vs, ref.Vs)
    out = sc.mat < 2
    assert np.array_equal(Vs.reshape(-1, 3)[out], sc.Vs0.reshape(-1, 3)[out])
