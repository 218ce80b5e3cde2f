"""Host tensors do not reach a kernel: the stream lookup in front of every
launch refuses their device (torch.cuda.current_stream's ValueError)."""
import pytest
import torch

from tensormesh_amd import _native as nat


@pytest.fixture
def fake_stream(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 100 + index, raising=False)


def test_stream_of_refuses_other_devices(fake_stream):
    for name in ("cpu", "cpu:0", "meta"):
        with pytest.raises(ValueError, match="Expected a cuda device"):
            nat.stream_of(torch.device(name))
    assert nat.stream_of(torch.device("cuda")) == 100 and nat.stream_of(torch.device("cuda", 3)) == 103


def test_a_solver_on_host_tensors_is_refused(fake_stream):
    from tensormesh_amd.solve import BatchedPCG
    rp = torch.tensor([0, 1, 2])
    with pytest.raises(ValueError, match="Expected a cuda device"):
        BatchedPCG(rp, torch.tensor([0, 1]), torch.ones(2, dtype=torch.float64), [0, 2])
