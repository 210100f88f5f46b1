"""The stream a launch goes to is torch's current one, whether or not torch has the call that says so without an object."""
import pytest
import torch

from axon_amd.kernels import lib


def test_without_the_short_call(monkeypatch):
    class Current:
        cuda_stream = 4321
    monkeypatch.setattr(lib, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: Current)
    assert lib._stream().value == 4321


@pytest.mark.gpu
def test_both_say_the_same(monkeypatch):
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        short = lib._stream().value
        monkeypatch.setattr(lib, "_raw_stream", None)
        assert short == lib._stream().value == side.cuda_stream
