"""The host side of a draw (tensorline_amd/sampling/sampler.py), without a GPU."""
import pytest
import torch

from tensorline_amd.ops import kernels
from tensorline_amd.sampling.sampler import Sampler


@pytest.mark.parametrize("capturing", [False, True])
def test_a_draws_numbers_are_pinned_except_under_capture(monkeypatch, capturing):
    """Outside a capture the numbers go to the device from pinned memory without waiting.  Under capture they take the waiting
    copy, which the capture refuses: a graph would read memory that has gone back to the pool."""
    class Logits:
        is_cuda, shape, device = True, (2, 10), "cpu"

    pinned, waits, real, real_to = [], [], torch.tensor, torch.Tensor.to
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    monkeypatch.setattr(torch, "tensor", lambda *a, pin_memory=False, **k: pinned.append(pin_memory) or real(*a, **k))
    monkeypatch.setattr(torch.Tensor, "to", lambda t, *a, non_blocking=False, **k: waits.append(not non_blocking) or real_to(t, *a, **k))
    monkeypatch.setattr(kernels, "sample", lambda logits, t, p, u, **k: (t.tolist(), p.tolist(), len(u)))
    got = Sampler("cpu").sample_device(Logits(), [0.5, 0.0], [1.0, 0.5], [3, 4], [0, 1])
    assert got == ([0.5, 0.0], [1.0, 0.5], 2) and pinned == [not capturing] and waits == [capturing]
