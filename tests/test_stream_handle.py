"""stream_handle without torch's private raw-stream function falls back to current_stream() (CPU)."""
import torch

from rmagine_amd import simulation


class _Stream:
    cuda_stream = 0x1230


def test_current_stream_with_and_without_the_raw_function(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(simulation, "_raw_stream", lambda device: 0x4560 + device)
    assert simulation.stream_handle().value == 0x4563
    monkeypatch.setattr(simulation, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: _Stream)
    assert simulation.stream_handle().value == 0x1230
    assert simulation.stream_handle(_Stream).value == 0x1230
