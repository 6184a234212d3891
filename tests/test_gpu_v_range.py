"""GPU: V past the range of fp16 products, and non-finite V, in short decodes and chunks against the oracle.

A q8_0 block holds scale * byte up to 8.3 million while fp16 ends at 65504, and a chunk's rows share the
tiles of keys that only some of them see. Bar: 1e-4 of the block's largest output, block by block
(every 32 dimensions have a scale of their own, so a large block must not cover for a small one)."""
import numpy as np
import pytest
import torch

import oracle
from bonsai_vk_amd import BKV_F16, BKV_Q8_0
from tests.gpu_util import pair, qg, say

TOL = 1e-4
pytestmark = pytest.mark.gpu
# decodes (n 1) and chunks: one tile, several, the last token in the middle and at the end of a tile, more tiles
# than V buffers; chunks of the short kernel, of 2 to 15 queries behind it, of several PV workgroups and ranges
SHAPES = [(0, 1), (63, 1), (299, 1), (447, 1), (448, 1), (0, 5), (300, 9), (440, 72), (600, 3), (1400, 6), (1000, 70)]


def filled(pos0, n, kf, vf, v, page=0):
    kw = {}
    cap = pos0 + n
    if page:
        pool = -(-cap // page) + 2
        kw = dict(page_tokens=page, max_pages=pool, block_table=np.random.default_rng(5).permutation(pool)[None].astype(np.int32))
        cap = pool * page
    dev, host = pair(1, cap, kf, vf, **kw)
    k, _ = oracle.synth_kv(pos0 + n, 4, 256, 9, 0, outliers=3)
    for c, f in ((host, lambda x: x), (dev, lambda x: torch.from_numpy(x).cuda())):
        c.append(0, 0, f(k), f(v))
    return dev, host


def both(dev, host, pos0, n):
    q, _ = qg(9, 0, n=n)
    want = host.prefill(0, pos0, q, nthreads=8)[0]
    qd = torch.from_numpy(q).cuda()
    out = dev.decode(0, pos0 + 1, qd[0].contiguous())[0][None] if n == 1 else dev.prefill_chunk(0, pos0, qd)[0]
    torch.cuda.synchronize()
    return out.cpu().numpy(), want


@pytest.mark.parametrize("kf", [BKV_Q8_0, BKV_F16])
@pytest.mark.parametrize("kind", ["blocks", "mixed", "edge"])
@pytest.mark.parametrize("pos0,n", SHAPES)
def test_q8v_past_fp16(pos0, n, kind, kf):
    """blocks: block b of every key near 10^b; mixed: every (key, block) anywhere in 1e-4 .. 8e6, so that large
    and small ones meet in one sum; edge: amax where the scales cross 512 (products at fp16's largest)."""
    say(f"V past fp16: pos0={pos0} n={n} {kind} kf={kf}")
    rng = np.random.default_rng(pos0 + n)
    m = pos0 + n
    v = rng.standard_normal((m, 4, 8, 32)).astype(np.float32)
    if kind == "blocks":
        v *= (10.0 ** np.arange(-1, 7))[None, None, :, None].astype(np.float32) * 0.5
    elif kind == "mixed":
        v *= np.exp(rng.uniform(np.log(1e-4), np.log(2e6), size=(m, 4, 8, 1))).astype(np.float32)
    else:
        amax = 127.0 * rng.choice([511.5, 511.75, 512.0, 512.5, 515.75, 516.0], size=(m, 4, 8, 1))
        v = (v / np.abs(v).max(axis=-1, keepdims=True) * amax).astype(np.float32)
    dev, host = filled(pos0, n, kf, BKV_Q8_0, v.reshape(m, 4, 256).astype(np.float32), page=64 if kind == "mixed" else 0)
    out, want = both(dev, host, pos0, n)
    assert np.isfinite(out).all()
    r = oracle.rel_err(out.reshape(-1, 32), want.reshape(-1, 32))
    say(f"  max err of a block's largest {r:.2e}")
    assert r <= TOL


@pytest.mark.parametrize("kf,vf", [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_F16)])
@pytest.mark.parametrize("what", [np.inf, np.nan, -1e9])
@pytest.mark.parametrize("pos0,n", [s for s in SHAPES if s[1] > 1] + [(100, 40)])
def test_later_tokens_non_finite_v(pos0, n, what, kf, vf):
    """A token whose V is stored as Inf or NaN (also a value past the format's range) in the last token of a
    chunk and in one before it: the queries before each are what they are without it (up to the order of the PV
    sum: at most m steps, each within 2^-23 of a partial sum that the row's largest |v| bounds), and the others
    are finite, Inf and NaN where the oracle is."""
    say(f"non-finite V: pos0={pos0} n={n} {what} kf={kf} vf={vf}")
    m = pos0 + n
    v = oracle.synth_kv(m, 4, 256, 9, 0, outliers=3)[1]
    first = m - 1 - min(n - 1, 2) // 2                 # (the chunk's last token, or the one before it too)
    bad = v.copy()
    bad[m - 1, :, 40:72] = what
    bad[first, 1, 7] = what
    plain, _ = both(*filled(pos0, n, kf, vf, v), pos0, n)
    dev, host = filled(pos0, n, kf, vf, bad)
    out, want = both(dev, host, pos0, n)
    assert np.abs(out[:first - pos0] - plain[:first - pos0]).max(initial=0.0) <= m * 2.0 ** -23 * np.abs(v).max()
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.array_equal(np.isinf(out), np.isinf(want))
    ok = np.isfinite(want)
    assert np.array_equal(np.sign(out[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    assert np.abs(out[ok] - want[ok]).max() <= TOL * np.abs(want[ok]).max()


@pytest.mark.parametrize("kf,vf", [(BKV_Q8_0, BKV_Q8_0), (BKV_F16, BKV_F16)])
@pytest.mark.parametrize("nfill", [1, 40, 64, 300])
def test_short_decode_of_a_non_finite_last_key(nfill, kf, vf):
    """The key a decode's padding repeats holds Inf: the output is Inf where the oracle's is, not NaN."""
    say(f"non-finite last key nfill={nfill} kf={kf} vf={vf}")
    v = oracle.synth_kv(nfill, 4, 256, 9, 0, outliers=3)[1]
    v[nfill - 1, :, 3] = -1e9 if vf == BKV_Q8_0 else np.inf
    out, want = both(*filled(nfill - 1, 1, kf, vf, v), nfill - 1, 1)
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.array_equal(np.isinf(out), np.isinf(want))
