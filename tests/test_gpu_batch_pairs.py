"""Batches whose FP32 members take two ticks in one launch: every member's
state and records are the bits of its run alone, whatever the blocks of ticks,
the parity of the members' ends, and who leaves or joins in between."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import scenes, tlm
from tests import helpers
from tests.test_gpu_batch import _compare, _oracle
from tests.test_gpu_parity import _random_scene

pytestmark = pytest.mark.gpu


def _members():
    """Tiles of one and of several a slab, one and two blocks a wave (nx > 192), one
    slab and many, with and without stubs, ends of both parities, a 16-bit
    member and one with more sources than a step adds itself."""
    out = []
    for q, (dims, steps, diel) in enumerate([((70, 41, 9), 33, True), ((64, 20, 40), 40, False), ((33, 35, 18), 7, True),
                                             ((5, 3, 1), 16, True), ((130, 17, 6), 25, False), ((9, 9, 35), 1, True),
                                             ((200, 30, 7), 18, True), ((259, 25, 5), 17, False)]):
        s = _random_scene(*dims, seed=20 + q, diel=diel, rho=(0.0, -1.0, 0.4)[q % 3], steps=steps)
        s.faces, s.energy_every = False, 0
        out.append(s)
    out.append(dataclasses.replace(out[2], pulse="f16", name="f16"))
    many = _random_scene(24, 18, 14, seed=40, steps=22)
    many.faces, many.energy_every = False, 0
    air = np.nonzero(np.asarray(many.mat).reshape(-1) == 0)[0][::7][:40]
    many.sources = [(int(c), k % 3, 0.5) for k, c in enumerate(air)]
    out.append(many)
    return out


@pytest.mark.parametrize("block,graph", [(1, 0), (2, 0), (5, 4), (64, 8), (64, 0)])
def test_members_equal_their_run_alone(block, graph):
    scs = _members()
    print(f"[batch pairs] blocks of {block}, graphs of {graph}", flush=True)
    res = tlm.run_scenes_batched(scs, tuning={"graph_ticks": graph}, block=block)
    for g, sc in zip(res, scs):
        _compare(g, _oracle(sc), sc)


@pytest.mark.parametrize("first", [4, 7])
def test_leave_run_alone_and_rejoin(first):
    scs = [s for s in _members() if s.pulse == "f32" and s.total_steps >= 16]
    devs = [tlm.open_scene(s) for s in scs]
    with tlm.TlmBatch() as b:
        for d, s in zip(devs, scs):
            b.add(d, s.total_steps)
        b.run(first)
        b.remove(devs[0])
        devs[0].run(first, 3)
        b.run(2)
        b.add(devs[0], scs[0].total_steps - first - 3)
        b.run(64)
        b.sync()
        for d in devs:
            b.remove(d)
    for d, s in zip(devs, scs):
        g = tlm.collect(d, s, s.total_steps)
        _compare(g, _oracle(s), s)
        d.close()
