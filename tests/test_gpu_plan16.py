"""16-bit storage: the scales planned between two steps of a run
(k_plan_inject, four slabs a workgroup) are those of steps run one by one
(k_slab_max, then k_inject), and so is every bit of state and record."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import tlm
from tests.test_gpu_parity import _random_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pulse", ["f16", "bf16"])
@pytest.mark.parametrize("dims", [(9, 7, 1), (20, 11, 3), (13, 9, 4), (40, 33, 5), (17, 5, 9), (150, 120, 18)])
def test_run_equals_single_steps(dims, pulse):
    steps = 11
    sc = dataclasses.replace(_random_scene(*dims, seed=3, rho=0.4, steps=steps), pulse=pulse, fp32_halo=1)
    print(f"[plan16] {dims} {pulse}", flush=True)
    out = []
    for block in (1, steps):
        with tlm.open_scene(sc) as dev:
            for n in range(0, steps, block):
                dev.run(n, block)
            dev.sync()
            out.append(dev.read_state() + tuple(dev.read_scales() or ()) + (dev.read_probes(0, steps),))
    assert len(out[0]) == len(out[1]) and np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
