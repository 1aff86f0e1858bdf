"""A recording of a HIP graph runs without the garbage collector (no GPU needed: the recording itself is stood in for)."""
import contextlib
import gc

import pytest
import torch

from spec_mcts_amd import decode


class _InACycle:
    """An object that only a collection destroys, as a search's captured graphs are."""
    def __init__(self, log):
        self.me, self.log = self, log

    def __del__(self):
        self.log.append(gc.isenabled())


@pytest.mark.parametrize("enabled", [True, False])
@pytest.mark.parametrize("fails", [False, True])
def test_no_collection_falls_into_a_recording(monkeypatch, enabled, fails):
    inside, destroyed = [], []

    @contextlib.contextmanager
    def stand_in(graph):
        inside.append(graph)
        yield
        inside.pop()
    monkeypatch.setattr(torch.cuda, "graph", stand_in)
    was, threshold = gc.isenabled(), gc.get_threshold()
    try:
        (gc.enable if enabled else gc.disable)()
        gc.collect()
        gc.set_threshold(1, 1, 1)                     # (every second allocation collects, where anything does)
        with pytest.raises(RuntimeError) if fails else contextlib.nullcontext():
            with decode.recording("g"):
                assert inside == ["g"]
                for _ in range(50):
                    _InACycle(destroyed)
                assert not destroyed
                if fails:
                    raise RuntimeError
        assert gc.isenabled() == enabled
    finally:
        gc.set_threshold(*threshold)
        (gc.enable if was else gc.disable)()
        gc.collect()
    assert len(destroyed) == 50


@pytest.mark.parametrize("enabled", [True, False])
@pytest.mark.parametrize("first_out", [0, 1])
def test_recordings_of_several_threads_overlap(monkeypatch, enabled, first_out):
    """Each of two recordings that overlap keeps the collector off until both are over, whichever ends first; then it is as it was."""
    monkeypatch.setattr(torch.cuda, "graph", lambda graph: contextlib.nullcontext())
    was = gc.isenabled()
    try:
        (gc.enable if enabled else gc.disable)()
        stacks = [contextlib.ExitStack() for _ in range(2)]
        for s in stacks:
            s.enter_context(decode.recording("g"))
            assert not gc.isenabled()
        stacks[first_out].close()
        assert not gc.isenabled()
        stacks[1 - first_out].close()
        assert gc.isenabled() == enabled
    finally:
        (gc.enable if was else gc.disable)()
