"""GPU: the split path's walk over batches of chunks (a batch: up to 256 chunks), with few and with so many
specials that the serial loop takes over, against the resident kernel's e and serial sums, bit
for bit, and past one batch against numpy's serial sum of the same e."""
import numpy as np
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache
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


@pytest.mark.parametrize("ties,fallback", [(40, 0), (64, 0), (65, 1)])
def test_split_walk_specials_over_batches(ties, fallback, monkeypatch):
    """Exact ties in every chunk past 16384 keys, so that the walk takes them over several batches (512 specials
    each) up to a chunk's 64, and the serial loop at 65. Every key has e = 1 but `ties` per chunk with
    e = 1023/1024, which is an odd number of half ulps of a sum in [2^14, 2^15)."""
    monkeypatch.setenv("BKV_DECODE", "split")
    n, first = 33000, 17408                        # (the sum is past 2^14 from key 16385 on)
    say(f"split walk ties={ties}")
    c = KvCache(n_layers=1, cap=n, k_fmt=BKV_F16, v_fmt=BKV_Q8_0)
    x0 = np.float32(np.log(1023 / 1024))           # score * scale of the ties, within 2^-27 of it as q0 k0 + q1 k1
    k0 = -2.0 ** -6
    k1 = np.float16((x0 * 16.0 - k0) * 1024)
    k = torch.zeros(n, 4, 256)
    at = torch.cat([first + 1024 * b + torch.arange(ties) * (1024 // ties) + 3 for b in range(14)])
    k[at, :, 0], k[at, :, 1] = k0, float(k1)
    v = torch.from_numpy(oracle.normal(n * 4 * 256, 3, 2).reshape(n, 4, 256))
    c.append(0, 0, k.cuda(), v.cuda())
    q = torch.zeros(16, 256)
    q[:, 0], q[:, 1] = 1.0, 2.0 ** -10
    c.decode(0, n, q.cuda())
    torch.cuda.synchronize()
    _, e, s, st = c.debug_intermediates(n)
    e = e.numpy()
    assert np.all(e[:, at.numpy()] == np.float32(1023 / 1024)) and ties * 14 > 512
    run = np.cumsum(e[0], dtype=np.float32)        # (numpy accumulates one term at a time)
    assert 2 ** 14 < run[at[0] - 1] and run[at[-1]] < 2 ** 15
    assert st.tolist() == [fallback] * 16
    assert np.array_equal(s.numpy(), np.full(16, run[-1]))
