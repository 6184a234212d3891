"""GPU: the exact prefill's e = exp(score * scale - max) and serial sums against the decode path's, bit for
bit (the decode's are checked against the oracle's in test_gpu_decode.py). The prefill keeps them in its
workspace: per unit of 4 queries [query][key][4 heads] fp32 past the decode arrays, then the sums."""
import ctypes

import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache, lib
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def slice_of(keys, n):
    """queries per slice: at least 512, more while their scores take at most 128 MiB, equal slices"""
    ld = -(-keys // 256) * 256 + 256
    most = max(512, min((128 << 20) // (4 * ld * 16) // 4 * 4, 4096))
    k = -(-n // min(n, most))
    return -(-(-(-n // k)) // 4) * 4


def queries(n, kind):
    """normal: two digits per q16, a third in a few rows; third: in every block; wide: the fp64 path; tiny:
    fp16 subnormals; mixed: blocks and rows of different ranges, an all-zero row, a row of one element."""
    q = torch.from_numpy(oracle.normal(n * 16 * 256, 5, 3).reshape(n, 16, 256).copy())
    if kind == "third":
        q[..., ::8] *= 1e-4
    elif kind == "wide":
        q[..., 5] *= 300
        q[..., 70], q[..., 200] = 1e-6, -3e-7
    elif kind == "tiny":
        q *= 1e-5
    elif kind == "mixed":
        q[:, :, 32:64] *= 1e-3
        q[:, 3] *= 40
        q[:, 7] = 0
        q[:, 9] = 0
        q[:, 9, 77] = 5.5
    return q.cuda()


# edges of the 64-key tiles, of the 64/128/256-query groups, one to four and more units, several key ranges
@pytest.mark.parametrize("kf,vf,pos0,n,kind", [
    (BKV_Q8_0, BKV_Q8_0, 560, 16, "normal"), (BKV_Q8_0, BKV_Q8_0, 687, 17, "normal"),
    (BKV_Q8_0, BKV_Q8_0, 940, 33, "normal"), (BKV_Q8_0, BKV_F16, 3000, 40, "third"),
    (BKV_Q8_0, BKV_Q8_0, 1000, 20, "wide"), (BKV_Q8_0, BKV_Q8_0, 700, 19, "tiny"),
    (BKV_Q8_0, BKV_Q8_0, 640, 18, "mixed"), (BKV_Q8_0, BKV_Q8_0, 2000, 513, "normal"),
    (BKV_Q8_0, BKV_Q8_0, 8000, 521, "normal"),
    (BKV_Q8_0, BKV_Q8_0, 1400, 3, "normal"), (BKV_Q8_0, BKV_F16, 1400, 7, "third"), (BKV_F16, BKV_Q8_0, 2100, 4, "normal"), (BKV_F16, BKV_Q8_0, 900, 21, "normal"),
    (BKV_F16, BKV_F16, 495, 130, "normal"), (BKV_F16, BKV_Q8_0, 0, 600, "normal")])
def test_prefill_e_and_sums_equal_decode(kf, vf, pos0, n, kind, monkeypatch):
    monkeypatch.setenv("BKV_KEEP_INTERMEDIATES", "1")
    say(f"prefill e: kf={kf} vf={vf} pos0={pos0} n={n} {kind}")
    cache = KvCache(n_layers=1, cap=pos0 + n, k_fmt=kf, v_fmt=vf)
    k, v = oracle.synth_kv(pos0 + n, 4, 256, 7, 0, outliers=3)
    cache.append(0, 0, torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    q = queries(n, kind)
    cache.prefill_chunk(0, pos0, q)
    torch.cuda.synchronize()
    step = slice_of(pos0 + n, n)
    last = (n - 1) // step * step                  # the workspace holds the last slice's
    m = n - last
    o = (ctypes.c_uint64 * 6)()
    assert lib().bkv_debug_layout(ctypes.byref(cache.desc), cache.max_positions, o) == 0
    base, ld = -(-int(o[5]) // 256) * 256, -(-(pos0 + n) // 256) * 256 + 256
    ws, nkv, units = cache._pws, cache.nkv, -(-m // 4)
    e = ws[base:base + nkv * units * 64 * ld].view(torch.float32).view(nkv, units, 4, ld, 4).clone()
    base += nkv * -(-step // 4) * 64 * ld          # (a multiple of 256)
    sums = ws[base:base + nkv * units * 64].view(torch.float32).view(nkv, units, 4, 4).clone()
    for i in sorted({0, 1, 2, 3, m // 2, m - 1} & set(range(m))):
        nfill = pos0 + last + i + 1
        cache.decode(0, nfill, q[last + i].contiguous())
        torch.cuda.synchronize()
        _, want, s, _ = cache.debug_intermediates(nfill)
        got = e[:, i // 4, i % 4, :nfill, :].permute(0, 2, 1).reshape(16, nfill).cpu()
        assert torch.equal(got, want), (i, int((got != want).sum()))
        assert torch.equal(sums[:, i // 4, i % 4, :].reshape(16).cpu(), s), i


def test_small_chunk_in_a_decode_workspace():
    """Chunks of 2 to 15 queries are accepted in a workspace sized for decodes (as decode rows), with the
    results of the chunk in a prefill workspace up to the order of the PV sum."""
    pos0, n = 1400, 5
    cache = KvCache(n_layers=1, cap=pos0 + n, k_fmt=BKV_Q8_0, v_fmt=BKV_Q8_0)
    k, v = oracle.synth_kv(pos0 + n, 4, 256, 7, 0, outliers=3)
    cache.append(0, 0, torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    q = queries(n, "normal")
    out, _ = cache.prefill_chunk(0, pos0, q)
    want = torch.empty_like(out)
    rc = lib().bkv_attn_prefill_chunk(ctypes.byref(cache.desc), 0, pos0, n, q.data_ptr(), None, want.data_ptr(), None,
                                      cache.workspace.data_ptr(), cache.workspace.numel(), cache._stream())
    torch.cuda.synchronize()
    assert rc == 0
    # (each output a sum of pos0 + n products with a probability sum of 1)
    assert float((out - want).abs().max()) <= (pos0 + n) * 2.0 ** -24 * float(abs(v).max())
