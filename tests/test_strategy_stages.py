"""The template's first and last stage and its two entry points, for programs that replace them."""
import numpy as np
import pytest

from sph_amd.data_classes import SimulationState
from sph_amd.strategy import NaiveSPHStrategy


class Context:
    """The calls a strategy makes on its context; a step adds one to the positions."""

    n, generation = 4, 0

    def __init__(self):
        self.calls = []

    def upload(self, pos, vel):
        self.calls.append("upload")
        self.state = pos.numpy().copy(), vel.numpy().copy()

    def step(self, nsteps):
        self.calls.append(f"step {nsteps}")
        self.generation += 1
        self.state = self.state[0] + nsteps, self.state[1]

    def download(self, force=False):
        import torch

        self.calls.append("download")
        return [torch.from_numpy(a.copy()) for a in (*self.state, np.ones(self.n))]

    def advance_host(self, arrays, nsteps):
        self.calls.append(f"advance_host {nsteps}")
        self.generation += 1
        if arrays is not None:
            self.state = tuple(a.copy() for a in arrays)
        self.state = self.state[0] + nsteps, self.state[1]
        return (*(a.copy() for a in self.state), np.ones(self.n))


def strategy(cls):
    s = object.__new__(cls)
    s.ctx, s.device, s.keep_terms = Context(), "cpu", False
    s.old_state = s.new_state = None
    s._returned_generation = -1
    return s


def start():
    return SimulationState(np.zeros((4, 3)), np.zeros((4, 3)), np.zeros(4))


class First(NaiveSPHStrategy):
    def _initialize_computation(self):
        self.seen = self.old_state
        super()._initialize_computation()


class Last(NaiveSPHStrategy):
    frames = 0

    def _finalize_computation(self):
        super()._finalize_computation()
        self.frames += 1


def test_one_call_without_own_stages():
    s = strategy(NaiveSPHStrategy)
    assert np.array_equal(s.compute_next_state(start()).position, np.full((4, 3), 1.0))
    assert s.ctx.calls == ["advance_host 1"]


@pytest.mark.parametrize("cls", [First, Last])
def test_own_stages_are_called(cls):
    s, st = strategy(cls), start()
    a = s.compute_next_state(st)
    b = s.advance(a, 2)
    assert np.array_equal(b.position, np.full((4, 3), 3.0)) and not b.position.flags.writeable
    assert s.ctx.calls == ["upload", "step 1", "download", "step 2", "download"]
    assert s.seen is a if cls is First else s.frames == 2


def test_own_stage_of_one_object():
    s, seen = strategy(NaiveSPHStrategy), []
    s._finalize_computation = lambda: (seen.append(1), NaiveSPHStrategy._finalize_computation(s))
    s.compute_next_state(start())
    assert seen == [1] and s.ctx.calls == ["upload", "step 1", "download"]


def test_advance_by_single_frames():
    class Frames(NaiveSPHStrategy):
        def advance(self, state, nsteps):
            for _ in range(nsteps):
                state = self.compute_next_state(state)
            return state

    s = strategy(Frames)
    assert np.array_equal(s.advance(start(), 3).position, np.full((4, 3), 3.0))
    assert s.ctx.calls == ["advance_host 1"] * 3
