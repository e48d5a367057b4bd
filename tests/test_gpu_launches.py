"""How many launches the steps of a context took (tlm_step_launches): two steps
a launch where the solver says so, and single steps where it says so."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import scenes, tlm

pytestmark = pytest.mark.gpu


def _scene(nx, ny, nz, steps, diel=True, sources=1, **kw):
    mat = np.zeros(nx * ny * nz, np.uint8)
    if diel:
        mat[:(mat.size + 1) // 2] = 2
    s = scenes.Scene(nx, ny, nz, mat, np.full(int(diel), 3.0, np.float32), np.zeros(int(diel), np.float32),
                     total_steps=steps, name=f"launches_{nx}x{ny}x{nz}", **kw)
    s.sources = [(int(c), 2, 1.0) for c in np.arange(sources)]
    s.faces, s.energy_every = False, 0
    s.probes = np.array([mat.size - 1], np.int64)
    return s


def _launches(sc, block=256, **tuning):
    with tlm.open_scene(sc) as dev:
        if tuning:
            dev.set_tuning(**tuning)
        for n in range(0, sc.total_steps, block):
            dev.run(n, min(block, sc.total_steps - n))
        dev.sync()
        return dev.step_launches()


@pytest.mark.parametrize("shape", [(1, 1, 1), (64, 9, 11), (65, 12, 10), (130, 21, 9), (257, 10, 9), (768, 9, 9),
                                   (192, 192, 192)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("diel", [False, True])
def test_fp32_steps_go_in_pairs(shape, diel):
    assert _launches(_scene(*shape, steps=41, diel=diel, sources=1)) == (21, 20)


def test_single_steps():
    """Wider than 768 cells, more sources than a step adds itself, a launch
    shape of the caller's, 16-bit pulses, blocks of one step."""
    sc = _scene(64, 9, 11, steps=40)
    assert _launches(_scene(769, 5, 4, steps=40)) == (40, 0)
    assert _launches(_scene(64, 9, 11, steps=40, sources=32)) == (20, 20)
    assert _launches(_scene(64, 9, 11, steps=40, sources=33)) == (40, 0)
    assert _launches(sc, fold=1) == (40, 0)
    assert _launches(dataclasses.replace(sc, pulse="f16")) == (40, 0)
    assert _launches(sc, block=1) == (40, 0)


def test_an_upload_counts_anew():
    sc = _scene(64, 9, 11, steps=40)
    with tlm.open_scene(sc) as dev:
        dev.run(0, 40)
        yh, gh = tlm.stub_admittances(sc.epsr, sc.sigma, sc.dl)
        dev.upload(sc.mat, yh, gh)
        assert dev.step_launches() == (0, 0)
        dev.run(0, 30)
        assert dev.step_launches() == (15, 15)


def test_batch_members():
    """Members count what they took part in: pairs while all have an even
    number of steps left or more than one, single ticks at an odd end."""
    scs = [_scene(64, 9, 11, steps=40), _scene(33, 20, 7, steps=31, diel=False),
           dataclasses.replace(_scene(20, 20, 20, steps=24), pulse="f16")]
    devs = [tlm.open_scene(s) for s in scs]
    devs[0].run(0, 4)
    first = devs[0].step_launches()
    with tlm.TlmBatch() as b:
        b.add(devs[0], 36)
        b.add(devs[1], 31)
        b.add(devs[2], 24)
        b.run(10)
        b.sync()
        assert [d.step_launches() for d in devs] == [(first[0] + 5, first[1] + 5), (5, 5), (10, 0)]
        b.set_tuning(graph_ticks=0)  # the tables are built again
        b.run(30)
        b.sync()
        # 10 pairs, the odd member's last step, 2 pairs, the last step of 35, none of the rest
        assert [d.step_launches() for d in devs] == [(first[0] + 19, first[1] + 17), (16, 15), (24, 0)]
        for d in devs:
            b.remove(d)
    for d in devs:
        d.close()


def _plates(n, every, probes=1):
    """PEC plates across z, one every so many slabs: n^2 faces on either side of each."""
    s = _scene(n, n, n, steps=20, diel=False)
    v = s.mat.reshape(n, n, n)
    if every:
        v[1:n - 1:every] = scenes.MAT_PEC
    s.faces = True
    s.probes = np.sort(np.random.default_rng(1).choice(n ** 3, probes, replace=False)).astype(np.int64)
    return s


@pytest.mark.parametrize("n,every,probes,huy,pairs", [
    (16, 2, 4096, 0, True),                           # a small grid full of them
    (64, 31, 0, 0, True), (64, 31, 1, 0, False),      # 16384 faces, and one record more
    (64, 0, 0, 4, True),                              # a Huygens box of 18816
    (96, 24, 0, 0, False),                            # 73728 faces: 0.08 a cell
    (96, 95, 10752, 0, True), (96, 95, 10753, 0, False)])
def test_many_records_take_single_steps(n, every, probes, huy, pairs):
    sc = _plates(n, every, probes)
    sc.huy_offset = huy
    assert _launches(sc) == ((10, 10) if pairs else (20, 0))


def test_many_probes_in_a_batch_take_single_steps():
    few, many = _scene(20, 20, 20, steps=20), _scene(20, 20, 20, steps=20)
    many.probes = np.arange(6827, dtype=np.int64)  # 12 each: above 81920
    devs = [tlm.open_scene(s) for s in (few, many)]
    with tlm.TlmBatch() as b:
        for d in devs:
            b.add(d, 20)
        b.run(20)
        b.sync()
        assert [d.step_launches() for d in devs] == [(10, 10), (20, 0)]
    for d in devs:
        d.close()


def test_an_upload_without_dielectrics_gives_both_stub_buffers_back():
    sc = _scene(128, 128, 128, steps=20)
    with tlm.open_scene(sc) as dev:
        dev.run(0, 20)
        dev.sync()
        before, _ = tlm.device_memory()
        dev.upload(np.zeros(sc.ncell, np.uint8))
        after, _ = tlm.device_memory()
        assert after - before >= 2 * 12 * sc.ncell - (4 << 20)


@pytest.mark.parametrize("short", [3, 4])
def test_autotune_times_pairs_as_pairs(short):
    """With windows of one tick too, and with a member that has one step left
    when the shape that takes pairs is timed."""
    scs = [_scene(40, 20, 20, steps=400), _scene(33, 20, 7, steps=400), _scene(20, 20, 20, steps=400)]
    devs = [tlm.open_scene(s) for s in scs]
    with tlm.TlmBatch() as b:
        default = b.get_tuning()
        b.add(devs[0], 400)
        b.add(devs[1], 399)
        b.add(devs[2], 8 * short + 1)  # ends while the candidates are timed
        b.autotune(1)
        b.sync()
        assert all(d.step_launches()[1] > 0 for d in devs[:2])
        b.set_tuning(**default)
        for d in devs:
            b.remove(d)
    for d in devs:
        d.close()


def test_timed_launches():
    """20 steps from step 5 with an energy record every 16: 15 cannot start a
    pair and 24 has no partner."""
    sc = _scene(64, 20, 12, steps=40)
    sc.energy_every = 16
    with tlm.open_scene(sc) as dev:
        dev.run(0, 5)
        total, per = dev.time_steps(5, 20, kernel_every=1)
        assert dev.timed_launches() == (11, 9)
        assert 0 < 20 * per <= 1.05 * total
        dev.time_steps(25, 10, kernel_every=7)  # steps 25 (a pair with 26) and 32 (a pair with 33)
        assert dev.timed_launches() == (2, 2)
        dev.time_steps(35, 4, kernel_every=0)
        assert dev.timed_launches() == (0, 0)


def test_pairs_begin_with_the_eighth_step():
    """A run of few steps of a small grid is not worth preparing for pairs."""
    sc = _scene(24, 20, 28, steps=40)
    with tlm.open_scene(sc) as dev:
        for n, m, want in ((0, 4, (4, 0)), (4, 3, (7, 0)), (7, 3, (9, 1)), (10, 30, (24, 16))):
            dev.run(n, m)
            assert dev.step_launches() == want
        dev.upload(sc.mat, *tlm.stub_admittances(sc.epsr, sc.sigma, sc.dl))
        dev.run(0, 7)
        assert dev.step_launches() == (7, 0)
    with tlm.open_scene(sc) as dev:
        dev.run(0, 8)
        assert dev.step_launches() == (4, 4)
    with tlm.open_scene(_scene(148, 148, 148, steps=40)) as dev:  # 3.2 M cells
        dev.run(0, 1)
        dev.run(1, 2)
        assert dev.step_launches() == (2, 1)
