"""Model._capture_warm against a stand-in for torch's graph objects (CPU): what
the capture brackets, and that no garbage is collected inside it (a collected
matrix or graph frees device memory, which a capturing stream does not allow;
torch.cuda.graph collects before it captures for this reason)."""
from __future__ import annotations

import contextlib
import gc
from types import SimpleNamespace

import pytest

from alpacca_amd.model import Model


class _Garbage:
    """A cycle whose collection is noted with the state of the capture."""

    def __init__(self, log, state):
        self.me, self.log, self.state = self, log, state

    def __del__(self):
        self.log.append(self.state["capturing"])


def _model(state):
    class Graph:
        def capture_begin(self):
            state["capturing"] = True

        def capture_end(self):
            state["capturing"] = False

    cuda = SimpleNamespace(CUDAGraph=Graph, stream=lambda s: contextlib.nullcontext())
    return SimpleNamespace(torch=SimpleNamespace(cuda=cuda), stream=None)


@pytest.mark.parametrize("fails", [False, True])
def test_capture_warm_collects_no_garbage(fails):
    state, log = {"capturing": False}, []
    threshold = gc.get_threshold()

    def fn():
        assert state["capturing"]
        _Garbage(log, state)
        keep = [[i] for i in range(2000)]  # far past the first threshold
        if fails:
            raise RuntimeError("launch")
        return keep

    gc.collect()
    gc.set_threshold(50, 1, 1)
    try:
        with (pytest.raises(RuntimeError) if fails else contextlib.nullcontext()):
            Model._capture_warm(_model(state), fn)
        assert gc.isenabled()
    finally:
        gc.set_threshold(*threshold)
    gc.collect()
    assert state["capturing"] is False and log == [False]


def test_capture_warm_leaves_collection_off():
    gc.disable()
    try:
        Model._capture_warm(_model({"capturing": False}), lambda: None)
        assert not gc.isenabled()
    finally:
        gc.enable()
