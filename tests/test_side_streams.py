"""Work fanned out to side streams leaves every device's current stream and the current device
as they were: also where the model lives on another device than the current one, and where
a job raises.  Devices and streams are stand-ins that keep what torch keeps."""
from types import SimpleNamespace

import pytest
import torch

from hyperscalees_amd import kernels as K
from hyperscalees_amd import rwkv


class FakeStream:
    def __init__(self, device, name):
        self.device, self.name = torch.device("cuda", device), name

    def wait_event(self, event):
        pass

    def wait_stream(self, stream):
        pass


@pytest.mark.parametrize("device", [0, 1])
@pytest.mark.parametrize("fails", [False, True])
def test_streams_restored(monkeypatch, device, fails):
    now = {"device": 0, 0: FakeStream(0, "caller's"), 1: FakeStream(1, "the other device's")}
    before = dict(now)

    def set_stream(s):
        now[s.device.index] = s
        now["device"] = s.device.index

    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda d=None: now[now["device"] if d is None else torch.device(d).index])
    monkeypatch.setattr(torch.cuda, "Event", lambda: SimpleNamespace(record=lambda s: None))
    monkeypatch.setattr(K, "_set_stream", set_stream)
    sides = [FakeStream(device, f"side {i}") for i in range(4)]
    monkeypatch.setattr(rwkv, "_side_streams", lambda dev: sides)
    x = SimpleNamespace(shape=(3, 100, 100), device=torch.device("cuda", device), record_stream=lambda s: None)
    used = []

    def job(i):
        used.append(now[device].name)
        if fails and i == 5:
            raise ValueError("a job")
        return x

    jobs = {str(i): (lambda i=i: job(i)) for i in range(6)}
    if fails:
        with pytest.raises(ValueError):
            rwkv._fan_out(jobs, x)
    else:
        rwkv._fan_out(jobs, x)
    assert used == [f"side {i % 4}" for i in range(6)]
    assert now == before
