"""GPU: the error of the PV sum alone, given the fp16 probabilities, in short decodes and chunks of a few
queries: at most two roundings of the result (2^-23 in the 2-norm), as the longer decodes' sums have."""
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kf,vf", [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_F16)])
@pytest.mark.parametrize("pos0,n", [(299, 1), (379, 1), (300, 6), (500, 6), (1000, 6), (3000, 6), (16000, 12)])
def test_pv_error_given_p16(pos0, n, kf, vf, monkeypatch):
    monkeypatch.setenv("BKV_KEEP_INTERMEDIATES", "1")
    m = pos0 + n
    cache = KvCache(n_layers=1, cap=m, k_fmt=kf, v_fmt=vf)
    k, v = oracle.synth_kv(m, 4, 256, 11, 0, outliers=3)
    cache.append(0, 0, torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    q = torch.from_numpy(oracle.normal(n * 16 * 256, 11, 5).reshape(n, 16, 256)).cuda()
    out = cache.decode(0, m, q[0])[0].clone() if n == 1 else cache.prefill_chunk(0, pos0, q)[0][n - 1]
    cache.decode(0, m, q[n - 1].contiguous())      # the last row's e and sum
    torch.cuda.synchronize()
    _, e, s, _ = cache.debug_intermediates(m)
    p16 = (e / s[:, None]).half().double()
    if vf == BKV_F16:
        V = cache.v_data[0].view(torch.float16).view(m, 4, 256).cpu().double()
    else:
        b = cache.v_data[0].view(torch.int8).view(m, 4, 8, 32).cpu().double()
        V = (b * cache.v_scales[0].view(torch.float16).view(m, 4, 8, 1).cpu().double()).view(m, 4, 256)
    want = torch.stack([p16[h] @ V[:, h // 4].contiguous() for h in range(16)])
    err = float((out.cpu().double() - want).norm() / want.norm())
    say(f"PV error kf={kf} vf={vf} pos0={pos0} n={n}: {err:.2e}")
    assert err <= 2.0 ** -23
