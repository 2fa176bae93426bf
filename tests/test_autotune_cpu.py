"""The autotuner's choice with an engine whose times are given: lists built by
the first step after a restore, then kept."""
import types

import pytest

from grains3dgpu_amd import autotune as T


class FakeEngine:
    """Staging mode 2: builds cost a quarter of mode 1's, steps a fifth more."""

    def __init__(self, held):
        self.held, self.now, self.mode, self.age = held, 0.0, 1, None

    def step(self, n, graph=False):
        for _ in range(n):
            if self.age is None or self.age >= self.held:
                self.now += {1: 2.0, 2: 0.5}[self.mode] * 1e-3
                self.age = 0
            self.now += {1: 0.30, 2: 0.36}[self.mode] * 1e-3
            self.age += 1

    def restore(self, blob):
        self.age = None

    def set_candidate_staging(self, mode):
        self.mode, self.age = mode, None

    def snapshot(self):
        return b""

    def nothing(self, *a):
        pass

    set_sims = set_launch = set_narrow_passes = close = nothing


@pytest.mark.parametrize("held,best", [(64, 1), (1, 2)])
@pytest.mark.parametrize("steps", [3, 10])
def test_builds_are_charged_to_the_steps_they_serve(held, best, steps, monkeypatch):
    eng = FakeEngine(held)
    monkeypatch.setattr(T, "load", lambda e, scene: eng)
    monkeypatch.setattr("grains3dgpu_amd.engine.Engine", lambda **kw: None)
    monkeypatch.setattr(T, "time", types.SimpleNamespace(perf_counter=lambda: eng.now))
    scene = types.SimpleNamespace(dt=1e-6, sims=[{}])
    out = T.autotune(scene, steps=steps, cell_factors=(1.0,), blocks=(256,), blocks_per_cu=(8,), narrow_passes=(2,))
    assert out["candidate_staging"] == best
    want = {1: 0.30 + 2.0 / 64, 2: 0.36 + 0.5}[best]
    assert out["ms_per_step"] == pytest.approx(want, rel=1e-9)
