"""The stream a call without one is queued on, on the CPU: the current device's current stream, by
torch's private raw-handle calls where they are there and by its public ones where they are not."""
import types

import pytest

torch = pytest.importorskip("torch")

from bigrig_amd import layer as ops  # noqa: E402

RAW, DEV = "_cuda_getCurrentRawStream", "_cuda_getDevice"


def test_given_stream_is_used():
    assert ops._stream(types.SimpleNamespace(cuda_stream=77)) == 77


def test_raw_handle_of_the_current_device(monkeypatch):
    monkeypatch.setattr(torch._C, DEV, lambda: 3, raising=False)
    monkeypatch.setattr(torch._C, RAW, lambda d: 1000 + d, raising=False)
    assert ops._stream() == 1003


@pytest.mark.parametrize("gone", [(RAW,), (DEV,), (RAW, DEV)])
def test_public_calls_where_the_private_ones_are_gone(monkeypatch, gone):
    for name in gone:
        monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=42))
    assert ops._stream() == 42
