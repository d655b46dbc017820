"""The stream that a launch goes to. A host tensor is refused before any launch: operators without a device check of their
own rely on it. CPU only."""
import pytest
import torch


def test_host_tensors_are_refused(monkeypatch):
    from mdx import _lib
    asked = []
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: asked.append(d) or 0, raising=False)
    monkeypatch.setattr(_lib, "_raw_stream", lambda d: asked.append(d) or 0, raising=False)
    with pytest.raises(RuntimeError, match="ROCm device"):
        _lib.stream_of(torch.zeros(4))
    assert not asked


class _OnDevice:
    """Stands in for a tensor on device 1."""
    device = "cuda:1"

    def get_device(self):
        return 1


@pytest.mark.parametrize("raw", [True, False])
def test_the_device_of_the_tensor_names_the_stream(monkeypatch, raw):
    from mdx import _lib

    class Stream:
        cuda_stream = 78

    monkeypatch.setattr(_lib, "_raw_stream", (lambda d: 77 if d == 1 else None) if raw else None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: Stream if d == 1 else None)
    assert _lib.stream_of(_OnDevice()) == (77 if raw else 78)
