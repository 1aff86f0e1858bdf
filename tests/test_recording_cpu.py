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
