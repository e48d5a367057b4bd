"""Grids of very many slabs: setting one up does not take longer with their
number than its memory does, and its steps are the restatement's."""
import time

import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers

pytestmark = pytest.mark.gpu


def test_choosing_the_launch_does_not_grow_with_the_slabs():
    """Looking at every number of slabs a tile took 11 ms here, the buffers
    take 1."""
    best = 1e9
    for _ in range(4):
        t = time.perf_counter()
        d = tlm.TlmDevice(8, 8, 4_000_000, 0.01)
        best = min(best, time.perf_counter() - t)
        d.close()
    print(f"[tall] create {best * 1e3:.2f} ms", flush=True)
    assert best < 5e-3


def test_tall_grid_matches_the_restatement():
    s = scenes.Scene(3, 5, 4001, np.zeros(3 * 5 * 4001, np.uint8), rho=-1.0, total_steps=24, name="tall")
    s.sources = [(s.cell(1, 2, 63), 2, 1.0), (s.cell(2, 4, 4000), 0, 0.5)]
    s.faces = False
    s.probes = np.array([s.cell(1, 1, k) for k in (0, 62, 65, 3999, 4000)], np.int64)
    helpers.compare_results(tlm.run_scene(s), helpers.oracle_run(s), s)
