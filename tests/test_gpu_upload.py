"""tlm_upload makes codes and block flags on the device; the map passes through
an idle pulse plane, or through memory of its own where the context has a state.
Every bit of the state must be that of a fresh context."""
import numpy as np
import pytest

from emsolver_amd import scenes, tlm

pytestmark = pytest.mark.gpu


def _scene(dims, seed):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    mat = rng.choice([0, 0, 0, 1, 2, 3, 255], nx * ny * nz).astype(np.uint8)
    sc = scenes.Scene(nx, ny, nz, mat, rng.uniform(1, 8, 254).astype(np.float32), np.zeros(254, np.float32),
                      total_steps=12, name="upload")
    c = sc.cell(nx // 2, ny // 2, nz // 2)
    mat[-1], mat[c] = 255, 0
    sc.sources = [(c, 2, 1.0)]
    sc.faces = False
    return sc


@pytest.mark.parametrize("fmt", ["f32", "f16"])
@pytest.mark.parametrize("dims", [(1, 1, 3), (17, 9, 5), (64, 3, 4), (70, 33, 12)])
def test_second_upload_equals_fresh_context(dims, fmt):
    a, b = _scene(dims, 1), _scene(dims, 2)
    a.pulse = b.pulse = fmt
    print(f"[upload] {dims} {fmt}", flush=True)
    with tlm.open_scene(b) as dev:
        dev.run(0, 12)
        want = dev.read_state()
    with tlm.open_scene(a) as dev:
        dev.run(0, 12)
        yh, gh = tlm.stub_admittances(b.epsr, b.sigma, b.dl)
        with pytest.raises(tlm.TlmError, match="material id"):
            dev.upload(b.mat, yh[:3], gh[:3])
        dev.upload(b.mat, yh, gh)
        dev.run(0, 12)
        got = dev.read_state()
    for x, y in zip(got, want):
        assert np.array_equal(x, y)
