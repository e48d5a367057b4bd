"""tlm_upload's look at the material ids, on the host for maps of up to 262144
cells and on the device above: the largest id decides what is refused, wherever
it lies and whatever its value, and a map without dielectrics takes no stubs."""
import numpy as np
import pytest

from emsolver_amd import tlm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 7, 3), (64, 64, 64), (65, 64, 64)])
@pytest.mark.parametrize("where", [0, -1, 0.37])
def test_largest_id(dims, where):
    n = int(np.prod(dims))
    at = int(where * n) if isinstance(where, float) else where
    with tlm.TlmDevice(*dims, 0.01) as dev:
        for top in (0, 1, 2, 3, 255):
            mat = np.zeros(n, np.uint8)
            mat[at] = top
            y = np.ones(254, np.float32)
            need = max(0, top - 1)  # materials of ids up to top
            if need:
                with pytest.raises(tlm.TlmError, match="material id"):
                    dev.upload(mat, y[:need - 1], y[:need - 1])
            Vs = np.arange(3 * n, dtype=np.float32)
            dev.upload(mat, y[:need], y[:need], Vs=Vs)
            assert np.array_equal(dev.read_state()[1], Vs if need else np.zeros(3 * n, np.float32))
