"""GPU: calls go to torch's current stream, with and without torch's private call for its raw handle."""
import pytest
import torch

import bonsai_vk_amd.cache as cache
from bonsai_vk_amd import KvCache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("private", [True, False])
def test_current_stream(private, monkeypatch):
    if not private:
        monkeypatch.setattr(cache, "_RAW_STREAM", None)
    assert KvCache._stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(torch.cuda.Stream()):
        assert KvCache._stream() == torch.cuda.current_stream().cuda_stream
    c = KvCache(n_layers=1, cap=8)
    c.append(0, 0, torch.ones(1, 4, 256, device="cuda"), torch.ones(1, 4, 256, device="cuda"))
    out, _ = c.decode(0, 1, torch.ones(16, 256, device="cuda"))
    assert torch.allclose(out, torch.ones_like(out), rtol=1e-3)
