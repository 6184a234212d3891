"""GPU: the split path's walk over batches of chunks (a batch: up to 256 chunks), with few and with so many
specials that the serial loop takes over, against the resident kernel's e and serial sums, bit
for bit, and past one batch against numpy's serial sum of the same e."""
import numpy as np
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_Q8_0, KvCache
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,grow", [(255, 0.0), (1025, 0.0), (20000, 0.0), (20000, 2e-3), (40961, 1e-3)])
def test_split_walk_batches(n, grow, monkeypatch):
    """grow: the scores rise along the keys by this much each, so the sum keeps doubling (many specials)."""
    say(f"split walk n={n} grow={grow}")
    monkeypatch.setenv("BKV_KEEP_INTERMEDIATES", "1")
    c = KvCache(n_layers=1, cap=n, k_fmt=BKV_Q8_0, v_fmt=BKV_Q8_0)
    k = torch.from_numpy(oracle.normal(n * 4 * 256, 3, 1).reshape(n, 4, 256)).cuda() * 0.2
    k[:, :, 0] += torch.arange(n, device="cuda")[:, None] * grow
    v = torch.from_numpy(oracle.normal(n * 4 * 256, 3, 2).reshape(n, 4, 256)).cuda()
    c.append(0, 0, k, v)
    q = torch.from_numpy(oracle.normal(16 * 256, 3, 4).reshape(16, 256)).cuda()
    q[:, 0] = 16.0
    got = {}
    for path in ("split", "resident"):
        monkeypatch.setenv("BKV_DECODE", path)
        c.workspace.zero_()                        # (bkv_workspace_init: the path changes)
        out, _ = c.decode(0, n, q)
        torch.cuda.synchronize()
        _, e, s, st = c.debug_intermediates(n)
        got[path] = (out, e, s)
        say(f"  {path}: walker status {st.tolist()}")
    assert torch.equal(got["split"][1], got["resident"][1])
    assert torch.equal(got["split"][2], got["resident"][2])
    # (an fp32 sum of products whose magnitudes sum to at most max |v|; the longest chain is 512 keys)
    assert float((got["split"][0] - got["resident"][0]).abs().max()) <= 1024 * 2.0 ** -24 * float(v.abs().max())


def test_split_walk_past_one_batch():
    n = 270001                                     # 264 chunks
    c = KvCache(n_layers=1, cap=n, k_fmt=BKV_Q8_0, v_fmt=BKV_Q8_0)
    g = torch.Generator(device="cuda").manual_seed(5)
    for s in range(0, n, 16384):
        m = min(16384, n - s)
        c.append(0, s, torch.randn(m, 4, 256, generator=g, device="cuda"), torch.randn(m, 4, 256, generator=g, device="cuda"))
    assert c.decode_path(n) == 0
    c.decode(0, n, torch.randn(16, 256, generator=g, device="cuda"))
    torch.cuda.synchronize()
    _, e, s, st = c.debug_intermediates(n)
    assert int(st.abs().sum()) == 0                # the walk, not its serial fallback
    want = np.cumsum(e.numpy(), axis=1, dtype=np.float32)[:, -1]   # (numpy accumulates one term at a time)
    assert np.array_equal(s.numpy(), want)
