"""Which device a call runs on (no GPU): torch's device switch modelled with what it keeps per thread, the
runtime's device and the device it has still to switch to. torch.cuda.device leaves the switch
back to a device without a context pending: torch reports that device as the current one while
the runtime is on the other, so a launch must not go by the report."""

from __future__ import annotations

import pytest
import torch


class Devices:
    """The runtime's current device and torch's pending one (-1: none)."""

    def __init__(self, runtime, pending, contexts):
        self.runtime, self.pending, self.contexts = runtime, pending, contexts

    def current(self):
        return self.pending if self.pending >= 0 else self.runtime

    def exchange(self, to):
        before, self.pending, self.runtime = self.current(), -1, to
        return before

    def maybe_exchange(self, to):
        before = self.current()
        if to in self.contexts:
            self.pending, self.runtime = -1, to
        else:
            self.pending = to
        return before


@pytest.mark.parametrize("runtime,pending,contexts", [
    (0, -1, {0}), (1, -1, {0, 1}), (0, 1, {0}), (1, 0, {0, 1}), (1, 0, {1}), (1, -1, {1})])
def test_call_runs_on_the_tensors_device(monkeypatch, runtime, pending, contexts):
    from mambo_amd import _native
    devices = Devices(runtime, pending, contexts)
    monkeypatch.setattr(torch.cuda, "current_device", devices.current)
    monkeypatch.setattr(torch.cuda, "_exchange_device", devices.exchange)
    monkeypatch.setattr(torch.cuda, "_maybe_exchange_device", devices.maybe_exchange)
    before = devices.current()
    with _native.on_device(torch.device("cuda", 0)):
        assert devices.runtime == 0 and devices.current() == 0
    assert devices.current() == before


def test_a_host_tensor_has_no_device_to_run_on():
    from mambo_amd import _native
    with pytest.raises(ValueError):
        with _native.on_device(torch.device("cpu")):
            pass
