"""What render_chunks owes its caller around the library call, replayed on the host with stand-ins for the streams and the
library (no GPU): the library reads the current device for its launches, so the model's device is current during the call; and the
current stream is behind every side stream however the call ends, because the buffers go back to the allocator then."""
import contextlib
import types

import pytest
import torch

from landmark_amd import _lib as L
from landmark_amd import model as M


class _Stream:
    cuda_stream = 0

    def __init__(self, log, name):
        self.log, self.name = log, name

    def wait_event(self, e):
        self.log.append(("wait_event", self.name))

    def wait_stream(self, s):
        self.log.append(("wait_stream", self.name, s.name))


class _Torch:
    """The module's torch with the device side replaced: tensors on the host, a record of what is current when."""

    def __init__(self, log):
        self.log, self.current_device = log, 0
        outer = self

        @contextlib.contextmanager
        def device(d):
            before, outer.current_device = outer.current_device, d.index
            try:
                yield
            finally:
                outer.current_device = before

        stream = lambda s: device(torch.device("cuda:1"))  # a stream context makes the stream's device current
        current = _Stream(log, "current")
        self.cuda = types.SimpleNamespace(device=device, stream=stream, current_stream=lambda d=None: current,
                                          Event=lambda: types.SimpleNamespace(record=lambda s: None))

    def zeros(self, *a, device=None, **k):
        return torch.zeros(*a, **k)

    def __getattr__(self, name):
        return getattr(torch, name)


@pytest.fixture
def model(monkeypatch):
    log = []
    fake = _Torch(log)
    monkeypatch.setattr(M, "torch", fake)
    m = M.GridNeRFHIP.__new__(M.GridNeRFHIP)
    m.device = torch.device("cuda:1")
    m.counters = torch.zeros(L.LM_STAT_WORDS, dtype=torch.int32)
    ws = torch.zeros(64, dtype=torch.uint8)
    m._samples_for = lambda n: 8
    m._model_struct = lambda *a: L.LmModel()
    m.capacities = lambda n, S: (0, 0)
    m.workspace = lambda *a: ws
    m.side_streams = lambda n: [_Stream(log, f"side{i}") for i in range(n)]
    m.render_into = lambda *a, **k: log.append(("render_into", fake.current_device)) or (0, 0)
    m.lib = types.SimpleNamespace(lm_render_chunks=lambda *a: log.append(("lm_render_chunks", fake.current_device)) or 0)
    m.log = log
    return m


def _render(m, n=100, step=30, streams=3):
    return m.render_chunks(torch.zeros(n, 6), torch.zeros(n, 3), torch.zeros(n), step, streams=streams)


def test_the_models_device_is_current_during_the_library_call(model):
    assert _render(model) == 4
    assert ("lm_render_chunks", 1) in model.log and ("render_into", 1) in model.log
    assert M.torch.current_device == 0


@pytest.mark.parametrize("fails", ["library", "last chunk"])
def test_side_streams_are_waited_for_when_a_launch_fails(model, fails):
    if fails == "library":
        model.lib.lm_render_chunks = lambda *a: -4
    else:
        def render_into(*a, **k):
            raise L.LandmarkError("no room")
        model.render_into = render_into
    with pytest.raises(L.LandmarkError):
        _render(model)
    for i in range(2):
        assert ("wait_stream", "current", f"side{i}") in model.log
