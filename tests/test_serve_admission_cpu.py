"""Admission of the serving loop against free memory (host logic, no device):
stand-ins for the contexts and the batch take what the library takes, a context's
buffers when it is set up and the second stub buffer of an FP32 member with
dielectric cells at its first block of ticks."""
import dataclasses

import numpy as np
import pytest

from emsolver_amd import scenes, serve, tlm

MB = 1 << 20


class _Device:
    def __init__(self, mem, sc):
        self.mem, self.sc, self.nprobe, self.nport = mem, sc, 0, 0
        self.held = self.second = 0
        self.take(tlm.estimate_bytes(sc.nx, sc.ny, sc.nz, sc.pulse, sc.has_diel))

    def take(self, n):
        self.mem.free -= n
        self.held += n
        self.mem.least = min(self.mem.least, self.mem.free)

    def close(self):
        self.mem.free += self.held
        self.held = 0


class _Batch:
    def __init__(self, device):
        self.left = {}

    def add(self, dev, n):
        self.left[dev] = n

    def run(self, n):
        for d in self.left:
            s = d.sc
            if not d.second and s.pulse == "f32" and s.has_diel:
                d.second = (tlm.estimate_bytes(s.nx, s.ny, s.nz, s.pulse, True)
                            - tlm.estimate_bytes(s.nx, s.ny, s.nz, s.pulse, False))
                assert d.second >= 12 * s.ncell
                d.take(d.second)
            self.left[d] = max(0, self.left[d] - n)

    def remaining(self):
        return dict(self.left)

    def remove(self, dev):
        del self.left[dev]

    def sync(self):
        pass

    def get_tuning(self):
        return {}

    def close(self):
        pass


class _Memory:
    def __init__(self, free):
        self.free = self.least = free


@pytest.mark.parametrize("pulse,diel", [("f32", True), ("f32", False), ("f16", True)])
def test_the_reserve_stays_free(monkeypatch, pulse, diel):
    mem = _Memory(500 * MB)
    monkeypatch.setattr(serve.tlm, "TlmBatch", _Batch)
    monkeypatch.setattr(serve.tlm, "open_scene", lambda sc, device=0: _Device(mem, sc))
    monkeypatch.setattr(serve.tlm, "device_memory", lambda device=0: (mem.free, 500 * MB))
    n = 64
    sc = scenes.Scene(n, n, n, np.full(n ** 3, 2 if diel else 0, np.uint8), np.full(1, 2.0, np.float32),
                      np.zeros(1, np.float32), total_steps=40, pulse=pulse, fp32_halo=-1)
    reqs = [serve.Request(q, dataclasses.replace(sc), 0.0) for q in range(40)]
    srv = serve.TlmServer(block_ticks=16, hbm_reserve=100 * MB, keep_results=False)
    done = srv.serve(reqs, realtime=False)
    assert len(done) == 40 and mem.free == 500 * MB
    assert srv.stats["mean_members"] > 5   # as many as fit run together
    assert mem.least >= 100 * MB
