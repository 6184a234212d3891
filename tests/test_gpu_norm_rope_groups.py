"""GPU: norm + rope + append for KV group counts that do not fill a workgroup's four: each group's rows
and cache bytes equal those of the same rows in a cache of that group alone (which the other tests hold to
the oracle)."""
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kf,vf", [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_Q8_0)])
@pytest.mark.parametrize("nkv", [1, 3, 4, 5, 9])
def test_group_counts(kf, vf, nkv):
    n, pos0 = 5, 70
    q = torch.from_numpy(oracle.normal(n * 4 * nkv * 256, nkv, 1).reshape(n, 4 * nkv, 256)).cuda()
    k = torch.from_numpy(oracle.normal(n * nkv * 256, nkv, 2).reshape(n, nkv, 256)).cuda()
    v = torch.from_numpy(oracle.normal(n * nkv * 256, nkv, 3).reshape(n, nkv, 256)).cuda()
    qw, kw = (torch.from_numpy(1 + 0.2 * oracle.normal(256, nkv, s)).float().cuda() for s in (4, 5))
    c = KvCache(n_layers=1, nh=4 * nkv, nkv=nkv, cap=pos0 + n, k_fmt=kf, v_fmt=vf)
    out = c.norm_rope_append(0, pos0, q, k, v, qw, kw)
    for g in range(nkv):
        one = KvCache(n_layers=1, nh=4, nkv=1, cap=pos0 + n, k_fmt=kf, v_fmt=vf)
        want = one.norm_rope_append(0, pos0, q[:, 4 * g:4 * g + 4], k[:, g:g + 1], v[:, g:g + 1], qw, kw)
        torch.cuda.synchronize()
        assert torch.equal(out[:, 4 * g:4 * g + 4], want), g
        for a, b in zip(c.host_arrays(), one.host_arrays()):
            if b is not None:
                row = b.shape[2]
                assert torch.equal(a[0, pos0:, g * row:(g + 1) * row], b[0, pos0:]), g
