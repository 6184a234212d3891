"""GPU: the single launch of contexts of at most 512 keys (one workgroup per KV group) against the stream,
resident and chunk kernels, which the other tests hold to the oracle: scores' e, sums and cache bytes bit
for bit, outputs to the fp32 order of the PV sum (each a sum of at most 512 exact products of magnitude
below the row's largest |v|: 512 * 2^-24 of it bounds the difference of two orders)."""
import numpy as np
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache
from tests.gpu_util import pair, qg, say

pytestmark = pytest.mark.gpu
FMTS = [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_F16), (BKV_F16, BKV_Q8_0), (BKV_Q8_0, BKV_F16)]
TOL = 512 * 2.0 ** -24


def caches(n, kf, vf, page):
    kw = {}
    cap = n
    if page:
        pool = -(-n // page) + 3
        kw = {"page_tokens": page, "max_pages": pool, "block_table": torch.randperm(pool, generator=torch.Generator().manual_seed(n))[None]}
        cap = pool * page
    out = []
    k, v = oracle.synth_kv(n, 4, 256, 3, 0, outliers=3)
    k, v = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda()
    for _ in range(2):
        c = KvCache(n_layers=1, cap=cap, k_fmt=kf, v_fmt=vf, max_ctx=n, **kw)
        if n > 1:
            c.append(0, 0, k[:n - 1], v[:n - 1])
        out.append(c)
    return out[0], out[1], k, v


def queries(n, kind):
    q = torch.from_numpy(oracle.normal(n * 16 * 256, 5, 3).reshape(n, 16, 256).copy())
    if kind == "wide":                             # the fp64 path of the q8_0 scores
        q[..., 5] *= 300
        q[..., 70] = 1e-6
    if kind == "third":                            # blocks with three digits
        q[..., ::8] *= 1e-4
    return q.cuda()


def same_caches(a, b):
    return all(x is None or torch.equal(x, y) for x, y in zip(a.host_arrays(), b.host_arrays()))


# edges: 16-key groups, 64-key tiles, 128-key rounds, three and more V tiles, the limit
@pytest.mark.parametrize("kf,vf", FMTS)
@pytest.mark.parametrize("n,page", [(1, 0), (2, 64), (16, 0), (64, 0), (65, 64), (129, 0), (192, 0), (257, 128), (300, 0),
                                    (449, 64), (512, 0)])
def test_short_decode(kf, vf, n, page, monkeypatch):
    say(f"short decode kf={kf} vf={vf} n={n} page={page}")
    monkeypatch.setenv("BKV_KEEP_INTERMEDIATES", "1")
    a, b, k, v = caches(n, kf, vf, page)
    q = queries(1, "wide" if n == 129 else "normal")[0]
    gate = queries(1, "normal")[0].flip(0).contiguous()
    args = (0, n - 1, k[n - 1:], v[n - 1:], q, gate)
    out, og = a.decode_step(*args)
    torch.cuda.synchronize()
    _, e, s, st = a.debug_intermediates(n)
    monkeypatch.setenv("BKV_DECODE", "stream")     # (fp16 V: the resident kernel)
    want, wg = b.decode_step(*args)
    torch.cuda.synchronize()
    _, e2, s2, _ = b.debug_intermediates(n)
    assert torch.equal(e, e2) and torch.equal(s, s2) and int(st.abs().sum()) == 0
    assert same_caches(a, b)
    tol = TOL * float(v.abs().max())
    assert float((out - want).abs().max()) <= tol and float((og - wg).abs().max()) <= tol
    # the same from a window that starts inside a page and a tile, and from interleaved q / gate rows
    if n > 40:
        wb, _ = b.decode_window(0, 37, n, q)
        monkeypatch.delenv("BKV_DECODE")
        wa, _ = a.decode_window(0, 37, n, q)
        qg = torch.stack([q, gate], 1).reshape(16, 512).contiguous()
        oq, ogq = a.decode_qg(0, n, qg)
        torch.cuda.synchronize()
        assert float((wa - wb).abs().max()) <= tol
        assert torch.equal(oq, out) and torch.equal(ogq, og)


@pytest.mark.parametrize("kf,vf", FMTS)
@pytest.mark.parametrize("pos0,n,page,kind", [(0, 2, 0, "normal"), (0, 5, 64, "normal"), (60, 9, 0, "third"), (100, 30, 0, "wide"),
                                              (0, 131, 0, "normal"), (300, 77, 64, "normal"), (495, 17, 0, "third"), (0, 512, 0, "normal")])
def test_short_prefill(kf, vf, pos0, n, page, kind, monkeypatch):
    """Each row of a chunk against the stream or resident decode of the same query."""
    say(f"short prefill kf={kf} vf={vf} pos0={pos0} n={n} page={page} {kind}")
    a, _, k, v = caches(pos0 + n, kf, vf, page)
    a.append(0, pos0 + n - 1, k[-1:], v[-1:])
    q = queries(n, kind)
    gate = queries(n, "normal").flip(1).contiguous()
    out, og = a.prefill_chunk(0, pos0, q, gate)
    monkeypatch.setenv("BKV_DECODE", "stream")
    tol = TOL * float(v.abs().max())
    for i in sorted({0, 1, 2, 3, 4, n // 2, n - 2, n - 1} & set(range(n))):
        want, wg = a.decode(0, pos0 + i + 1, q[i].contiguous(), gate[i].contiguous())
        torch.cuda.synchronize()
        assert float((out[i] - want).abs().max()) <= tol, i
        assert float((og[i] - wg).abs().max()) <= tol, i


# a first token, a token in the middle of a tile, the last of a tile, the first of a tile
@pytest.mark.parametrize("kf,vf", FMTS)
@pytest.mark.parametrize("n", [1, 2, 40, 64, 65, 300])
def test_short_decode_step_into_unwritten_slots(kf, vf, n):
    """What the appended token's slot and those after it held before (here NaN bytes) reaches no output."""
    say(f"short decode into NaN slots kf={kf} vf={vf} n={n}")
    outs = []
    k, v = (torch.from_numpy(x).cuda() for x in oracle.synth_kv(n, 4, 256, 3, 0, outliers=3))
    q = queries(1, "normal")[0]
    for fill in (0, 255):
        c = KvCache(n_layers=1, cap=n + 70, k_fmt=kf, v_fmt=vf, max_ctx=n + 70)
        for t in (c.k_data, c.k_scales, c.v_data, c.v_scales):
            if t is not None:
                t.fill_(fill)
        if n > 1:
            c.append(0, 0, k[:n - 1], v[:n - 1])
        outs.append(c.decode_step(0, n - 1, k[n - 1:], v[n - 1:], q)[0])
    torch.cuda.synchronize()
    assert bool(torch.isfinite(outs[0]).all()) and torch.equal(outs[0], outs[1])


# 16 KV heads: a chunk of a short context in the short kernel, and one of so many workgroups that it leaves it
@pytest.mark.parametrize("kf,vf", [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_F16)])
@pytest.mark.parametrize("pos0,n", [(300, 100), (300, 200), (0, 331)])
def test_short_chunk_of_many_kv_heads(kf, vf, pos0, n):
    say(f"short chunk, 16 KV heads kf={kf} vf={vf} pos0={pos0} n={n}")
    m = pos0 + n
    dev = KvCache(n_layers=1, nh=64, nkv=16, cap=m, k_fmt=kf, v_fmt=vf)
    host = oracle.HostCache(n_layers=1, nh=64, nkv=16, cap=m, k_fmt=kf, v_fmt=vf)
    k, v = oracle.synth_kv(m, 16, 256, 5, 0, outliers=3)
    host.append(0, 0, k, v)
    dev.append(0, 0, torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    q = oracle.normal(n * 64 * 256, 5, 3).reshape(n, 64, 256)
    out, _ = dev.prefill_chunk(0, pos0, torch.from_numpy(q).cuda())
    torch.cuda.synchronize()
    rows = sorted({0, 1, 5, n // 2, n - 1})
    want = [host.decode(0, pos0 + i + 1, q[i], nthreads=8)[0] for i in rows]
    assert max(oracle.rel_err(out[i].cpu().numpy(), w) for i, w in zip(rows, want)) <= 1e-4


@pytest.mark.parametrize("forced", ["split", "resident", "stream"])
@pytest.mark.parametrize("pos0,n", [(100, 3), (700, 5)])
def test_forced_path_in_small_chunks(pos0, n, forced, monkeypatch):
    """BKV_DECODE decides how the rows of a chunk of 2 to 15 queries run: each equals the forced decode."""
    say(f"forced {forced}: chunk of {n} onto {pos0}")
    monkeypatch.setenv("BKV_DECODE", forced)
    c, _, k, v = caches(pos0 + n, BKV_Q8_0, BKV_Q8_0, 0)
    c.append(0, pos0 + n - 1, k[-1:], v[-1:])
    q = queries(n, "normal")
    out, _ = c.prefill_chunk(0, pos0, q)
    for i in range(n):
        want, _ = c.decode(0, pos0 + i + 1, q[i].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(out[i], want), i


SYNC = slice(200 * 1024, 212 * 1024)               # of the workspace: the sync lines of the exchanging kernels


def limit(kf, vf, page):
    """the longest decode the short kernel takes at 4 KV heads"""
    if vf == BKV_Q8_0:
        return 448 if kf == BKV_Q8_0 and not page else 384
    return 448 if page else 512


@pytest.mark.parametrize("kf,vf", FMTS)
@pytest.mark.parametrize("page", [0, 3, 64])
def test_short_decode_against_the_oracle(kf, vf, page, monkeypatch):
    """Unforced decodes on either side of every limit and tile: which kernel ran (the exchanging ones advance their
    generation words in the workspace, the short one leaves them), e, the serial sums and p16 bit for bit the
    oracle's, cache bytes, output; a window; at the limit also appended into slots of NaN bytes."""
    monkeypatch.setenv("BKV_KEEP_INTERMEDIATES", "1")
    say(f"short decode against the oracle kf={kf} vf={vf} page={page}")
    m, kw = 520, {}
    cap = m
    if page:
        pool = -(-m // page) + 2
        kw = dict(page_tokens=page, max_pages=pool, block_table=np.random.default_rng(page).permutation(pool)[None].astype(np.int32))
        cap = pool * page
    dev, host = pair(1, cap, kf, vf, **kw)
    for t in (dev.k_data, dev.k_scales, dev.v_data, dev.v_scales):
        if t is not None:
            t.fill_(255)
    k, v = oracle.synth_kv(m, 4, 256, 17, 0, outliers=3)
    q, g = qg(17, 0)
    qd, gd = torch.from_numpy(q).cuda(), torch.from_numpy(g).cuda()
    done = 0
    for n in (1, 17, 64, 65, 129, 256, 257, 320, 321, 384, 385, 447, 448, 449, 511, 512, 513):
        host.append(0, done, k[done:n], v[done:n])
        if n - 1 > done:
            dev.append(0, done, torch.from_numpy(k[done:n - 1]).cuda(), torch.from_numpy(v[done:n - 1]).cuda())
        done = n
        before = dev.workspace[SYNC].clone()
        out, og = dev.decode_step(0, n - 1, torch.from_numpy(k[n - 1:n]).cuda(), torch.from_numpy(v[n - 1:n]).cuda(), qd, gd)
        torch.cuda.synchronize()
        assert torch.equal(before, dev.workspace[SYNC]) == (n <= limit(kf, vf, page)), n
        want, wg, sc, pr, p16 = host.decode(0, n, q, g, nthreads=8, debug=True)
        _, e, s, st = dev.debug_intermediates(n)
        x = sc * np.float32(0.0625)
        assert oracle.bit_diff(e.numpy(), np.exp((x - x.max(axis=1, keepdims=True)).astype(np.float64)).astype(np.float32)) == 0, n
        p = (e.numpy() / s.numpy()[:, None]).astype(np.float32)
        assert oracle.bit_diff(p, pr) == 0 and np.array_equal(oracle.f32_to_f16(p), p16) and int(st.abs().sum()) == 0, n
        assert oracle.rel_err(out.cpu().numpy(), want) <= 1e-4 and oracle.rel_err(og.cpu().numpy(), wg) <= 1e-4, n
    for a, b in zip(dev.host_arrays(), host.arrays()):
        if b is not None:                          # (the slots after the last token still hold what they did)
            slots = [host.slot(0, i) for i in range(done)]
            assert np.array_equal(a.numpy()[0, slots], b[0, slots])
    _, win = pair(1, 400, kf, vf)
    win.append(0, 0, k[113:513], v[113:513])
    wlen = min(limit(kf, vf, page) - 70, 400)
    out, _ = dev.decode_window(0, 113, 113 + wlen, qd)
    torch.cuda.synchronize()
    assert oracle.rel_err(out.cpu().numpy(), win.decode(0, wlen, q)[0]) <= 1e-4
