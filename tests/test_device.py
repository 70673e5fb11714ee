"""Host-side helpers of localai_amd.device that need no GPU."""
from types import SimpleNamespace

import pytest

from localai_amd import device


def fake_torch(**private):
    cuda = SimpleNamespace(current_device=lambda: 3, current_stream=lambda: SimpleNamespace(cuda_stream=77))
    return SimpleNamespace(_C=SimpleNamespace(**private), cuda=cuda)


@pytest.mark.parametrize('private,want', [({}, 77), ({'_cuda_getCurrentRawStream': lambda dev: 100 + dev}, 103)])
def test_current_stream_with_and_without_the_raw_call(monkeypatch, private, want):
    """The current stream of the current device, through PyTorch's private call
    or, in a PyTorch without it, through current_stream()."""
    monkeypatch.setattr(device, '_TORCH', fake_torch(**private))
    assert device.stream_ptr() == want
    assert device.stream_ptr(SimpleNamespace(cuda_stream=5)) == 5
