"""Host side of `DecodeSession.step` without a GPU: the session's parts are stand-ins."""
import contextlib
from types import SimpleNamespace

import torch

from native_sparse_attention_pytorch_amd.decode_session import DecodeSession


def test_a_step_runs_on_the_session_s_device(monkeypatch):
    """Whatever device is current: the kernels of a direct step are launched on the session's, as a replayed graph is."""
    current = [0]

    @contextlib.contextmanager
    def device(dev):
        before, current[0] = current[0], dev.index
        yield
        current[0] = before

    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[0])
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    s = object.__new__(DecodeSession)
    s._graphs, s.direct, s.pos, s.nc, s.max_len, s.st, s.max_nc = [], True, 0, 0, 8, 4, 2
    s.K = SimpleNamespace(device=torch.device("cuda", 3))
    s._step_direct = lambda x: current[0]
    assert s.step(None) == 3 and current[0] == 0 and s.pos == 1
