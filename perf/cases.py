"""Timed cases of the KV-cache path: the calls an engine makes per token (decode), per prompt chunk
(prefill), and to fill its cache (norm + rope + append, bulk append), through KvCache.

The model shape is the reference's (16 query heads, 4 KV heads, head_dim 256; 8 attention layers per
token). K ~ N(0, 1) with 3 channels per KV head scaled x8, V ~ N(0, 0.5), Q ~ N(0, 1), the
distributions of bench.py.

A case is a dict:
  kind   "decode"   one token through `layers` layers at context `ctx`: append the token's K/V, attend
                    over ctx + 1 keys (decode_step; front: norm_rope_append, then decode)
         "prefill"  prefill_step of `n` tokens at position `ctx`, one layer
         "front"    norm_rope_append of `n` tokens at position `ctx`, one layer
         "append"   append of `n` tokens at position `ctx`, one layer
  kf, vf cache formats of K and V, "q8_0" or "f16"; page: tokens per page, 0 = contiguous
  gate   the gate is read and the gated output written
"""
import math

import torch

from bonsai_vk_amd import BKV_F16, BKV_Q8_0, KvCache

NH, NKV, HD = 16, 4, 256
NROT, EPS, BASE = 64, 1e-6, 1e7
CHUNK = 8192            # tokens per generated and appended piece of a cache
FMT = {"q8_0": BKV_Q8_0, "f16": BKV_F16}


def _case(name, kind, ctx, n=1, layers=1, kf="q8_0", vf="q8_0", page=0, gate=False, front=False):
    c = {"kind": kind, "ctx": ctx, "n": n, "layers": layers, "kf": kf, "vf": vf, "page": page, "gate": gate,
         "front": front}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the first words of a chat: a token at a few hundred keys, 8 layers, where launches and
        # latencies are all there is
        _case("decode_300", "decode", 300, layers=8, gate=True),
        # a chat turn at 4K keys
        _case("decode_4k", "decode", 4096, layers=8),
        # the engine's own sequence (norm + rope + append, then attention with the gate) in the
        # reference's cache format, mid-size context that is a multiple of nothing
        _case("decode_ref_12k", "decode", 12345, layers=8, kf="f16", gate=True, front=True),
        # the headline workload: a token at 32K keys, 8 layers
        _case("decode_32k", "decode", 32768, layers=8),
        # a long document in fp16, 256-token pages from a shared pool
        _case("decode_64k_paged_f16", "decode", 65536, layers=8, kf="f16", vf="f16", page=256),
        # a very long context: past what one resident workgroup per CU holds
        _case("decode_200k", "decode", 200000, layers=2),
        # a few tokens checked at once (speculative decoding, a short user message)
        _case("prefill_6_at_3k", "prefill", 3000, 6, gate=True),
        # a user's follow-up message in a running conversation
        _case("prefill_48_at_6k", "prefill", 6000, 48, gate=True),
        # an fp16 cache, ragged chunk
        _case("prefill_300_at_2k_f16", "prefill", 2000, 300, kf="f16", vf="f16"),
        # the first prompt of a conversation in the reference's cache format
        _case("prefill_1000_at_0_ref", "prefill", 0, 1000, kf="f16", gate=True),
        # the standard chunk: 512 queries onto 8192 cached keys
        _case("prefill_512_at_8k", "prefill", 8192, 512),
        # a chunk's projected rows: QK norm, rope and quantise-on-write
        _case("front_512", "front", 4096, 512),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Another case of the listed ranges: contexts to 200K keys, chunks of 2 to 2048 tokens, every
    format pair, contiguous and paged. The costs stay below the largest listed case's."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "prefill", "front", "append"])
    kf, vf = rng.choice([("q8_0", "q8_0"), ("q8_0", "q8_0"), ("f16", "q8_0"), ("f16", "f16")])
    page = rng.choice([0, 0, 64, 256])
    gate = rng.random() < 0.5
    if kind == "decode":
        ctx = _log(rng, 1, 190000)
        if ctx > 60000 and kf == "f16":
            ctx //= 3
        return _case(None, kind, ctx, layers=8 if ctx < 40000 else 2, kf=kf, vf=vf, page=page, gate=gate,
                     front=rng.random() < 0.3)
    if kind == "prefill":
        n = _log(rng, 2, 2048)
        # query-key pairs at most half of the largest listed chunk's
        room = int((512 * 8448) * (0.5 if kf == "q8_0" else 0.25) / n - n / 2)
        ctx = rng.choice([0, _log(rng, 1, max(1, min(16000, room)))]) if room > 1 else 0
        return _case(None, kind, ctx, n, kf=kf, vf=vf, page=page, gate=gate)
    return _case(None, kind, _log(rng, 1, 8192), _log(rng, 1, 2048 if kind == "front" else 8192), kf=kf, vf=vf,
                 page=page)


def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 7919 * stream + 1)
    return g


def _pieces(case, seed, layer, n):
    """The cached tokens of a layer, in pieces: (first position, K [m][NKV][HD], V)."""
    g = _gen(seed, 100 + layer)
    ch = torch.stack([torch.randperm(HD, generator=g, device="cuda")[:3] for _ in range(NKV)])
    scale = torch.ones(NKV, HD, device="cuda").scatter_(1, ch, 8.0)
    for s in range(0, n, CHUNK):
        m = min(CHUNK, n - s)
        yield s, torch.randn(m, NKV, HD, generator=g, device="cuda") * scale, \
            torch.randn(m, NKV, HD, generator=g, device="cuda") * 0.5


def _calls(case, seed):
    """The call's own inputs, [layers][n][...]: q, k, v, gate and the norm weights."""
    L, n, g = case["layers"], case["n"], _gen(seed, 1)
    return {"q": torch.randn(L, n, NH, HD, generator=g, device="cuda"),
            "k": torch.randn(L, n, NKV, HD, generator=g, device="cuda"),
            "v": torch.randn(L, n, NKV, HD, generator=g, device="cuda") * 0.5,
            "gate": torch.randn(L, n, NH, HD, generator=g, device="cuda"),
            "qw": 1.0 + 0.1 * torch.randn(HD, generator=g, device="cuda"),
            "kw": 1.0 + 0.1 * torch.randn(HD, generator=g, device="cuda")}


def prepare(case, seed):
    L, ctx, n, page = case["layers"], case["ctx"], case["n"], case["page"]
    total = ctx + n
    kw = {}
    cap = total
    if page:
        need = -(-total // page)
        pool = need + need // 4 + 1
        g = _gen(seed, 2)
        kw = {"page_tokens": page, "max_pages": pool,
              "block_table": torch.stack([torch.randperm(pool, generator=g, device="cuda") for _ in range(L)])}
        cap = pool * page
    cache = KvCache(n_layers=L, nh=NH, nkv=NKV, hd=HD, cap=cap, k_fmt=FMT[case["kf"]], v_fmt=FMT[case["vf"]],
                    max_ctx=total, **kw)
    for layer in range(L):
        for s, k, v in _pieces(case, seed, layer, ctx):
            cache.append(layer, s, k, v)
    if case["kind"] == "prefill":
        cache.prefill_workspace(total)
    state = {"case": dict(case), "cache": cache, "in": _calls(case, seed)}
    if case["kind"] == "decode":
        state["out"] = torch.empty(L, NH, HD, device="cuda")
        state["og"] = torch.empty(L, NH, HD, device="cuda") if case["gate"] else None
    return state


def run(state):
    case, cache, x = state["case"], state["cache"], state["in"]
    pos, kind = case["ctx"], case["kind"]
    res = {}
    if kind == "decode":
        out, og = state["out"], state["og"]
        for layer in range(case["layers"]):
            gate = x["gate"][layer, 0] if case["gate"] else None
            ol, gl = out[layer], og[layer] if case["gate"] else None
            if case["front"]:
                q = cache.norm_rope_append(layer, pos, x["q"][layer], x["k"][layer], x["v"][layer], x["qw"], x["kw"],
                                           NROT, EPS, BASE)
                cache.decode(layer, pos + 1, q[0], gate, ol, gl)
            else:
                cache.decode_step(layer, pos, x["k"][layer], x["v"][layer], x["q"][layer, 0], gate, ol, gl)
        res["out"], res["gated"] = out, og
    elif kind == "prefill":
        res["out"], res["gated"] = cache.prefill_step(0, pos, x["k"][0], x["v"][0], x["q"][0],
                                                      x["gate"][0] if case["gate"] else None)
    elif kind == "front":
        res["q"] = cache.norm_rope_append(0, pos, x["q"][0], x["k"][0], x["v"][0], x["qw"], x["kw"], NROT, EPS, BASE)
    else:
        cache.append(0, pos, x["k"][0], x["v"][0])
    for name in ("k_data", "k_scales", "v_data", "v_scales"):     # the updated state
        res[name] = getattr(cache, name)
    return res


def _row_bytes(fmt):
    return NKV * HD * 2 if fmt == "f16" else NKV * (HD + HD // 16)


def work(case):
    L, ctx, n = case["layers"], case["ctx"], case["n"]
    row = _row_bytes(case["kf"]) + _row_bytes(case["vf"])
    kv_in = n * 2 * NKV * HD * 4
    qo = n * NH * HD * 4
    if case["kind"] in ("append", "front"):
        front = case["kind"] == "front"
        return {"bytes": kv_in + n * row + (2 * qo if front else 0), "flops": 0}
    pairs = n * ctx + n * (n + 1) // 2
    b = ctx * row + n * row + kv_in + 2 * qo + (2 * qo if case["gate"] else 0)
    return {"bytes": L * b, "flops": L * 4 * NH * HD * pairs}


def tolerance(case):
    # The cache bytes are exact. norm + rope is fp32 throughout (measured 1.3e-7 from 64 bits). The
    # attention's probabilities are fp16 values, formed from fp32 scores and a serial fp32 sum: some of
    # them round another way than in 64 bits, and the more keys, the nearer the fp16 subnormals they
    # are (measured 1e-5 to 5e-5 from 64 bits up to 64K keys, 1.9e-4 at 200K). Four times that.
    if case["kind"] == "append":
        return "exact"
    if case["kind"] == "front":
        return {"rel": 5e-7}
    return {"rel": 2e-4 if case["ctx"] + case["n"] <= 70000 else 8e-4}


# ------------------------------------------------------------------ the same in 64 bits
def _stored(x, fmt):
    """What the cache holds of x (fp32 [.., HD]), as fp64."""
    if fmt == "f16":
        return x.half().double()
    b = x.reshape(*x.shape[:-1], HD // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    d = torch.where(amax > 1e-35, amax / 127.0, torch.zeros_like(amax))
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = torch.clamp(torch.round(b * inv), -127, 127)
    return (q.double() * d.half().double()).reshape(x.shape)


def _norm_rope(x, w, pos0):
    """x [n][heads][HD] fp32 -> fp64; the rope's exponent and angle are fp32 values by definition."""
    y = x.double()
    y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + EPS) * w.double()
    half = NROT // 2
    p = torch.arange(half, device=x.device, dtype=torch.float32)
    th = torch.pow(torch.tensor(BASE, dtype=torch.float64, device=x.device), (-2.0 * p / NROT).double()).float()
    pos = torch.arange(pos0, pos0 + x.shape[0], device=x.device, dtype=torch.float32)
    ang = (pos[:, None] * th[None, :]).double()[:, None, :]
    c, s = torch.cos(ang), torch.sin(ang)
    lo, hi = y[..., :half], y[..., half:NROT]
    return torch.cat([lo * c - hi * s, hi * c + lo * s, y[..., NROT:]], -1)


def _attend(q, K, V, pos0):
    """q [n][NH][HD], K, V fp64 [keys][NKV][HD]; query i sees keys 0 .. pos0 + i."""
    n, keys = q.shape[0], K.shape[0]
    q16 = q.float().half().double()
    out = torch.empty(n, NH, HD, dtype=torch.float64, device=q.device)
    j = torch.arange(keys, device=q.device)
    for h in range(NH):
        Kh, Vh = K[:, h // 4].contiguous(), V[:, h // 4].contiguous()
        for a in range(0, n, 512):
            b = min(n, a + 512)
            s = torch.mm(q16[a:b, h], Kh.t().contiguous()) / math.sqrt(HD)
            i = torch.arange(a, b, device=q.device)
            s.masked_fill_(j[None, :] > pos0 + i[:, None], float("-inf"))
            p = torch.softmax(s, -1).half().double()
            out[a:b, h] = torch.mm(p, Vh)
    return out


def exact(case, seed):
    x, pos, L = _calls(case, seed), case["ctx"], case["layers"]
    none = {"k_data": None, "k_scales": None, "v_data": None, "v_scales": None}
    if case["kind"] == "append":
        return None                     # bytes only
    if case["kind"] == "front":
        return {"q": _norm_rope(x["q"][0], x["qw"], pos), **none}
    outs = []
    for layer in range(L):
        q, k, v = x["q"][layer], x["k"][layer], x["v"][layer]
        if case["front"]:
            q, k = _norm_rope(q, x["qw"], pos), _norm_rope(k, x["kw"], pos).float()
        K = [(_stored(a, case["kf"]), _stored(b, case["vf"])) for _, a, b in _pieces(case, seed, layer, pos)]
        K.append((_stored(k, case["kf"]), _stored(v, case["vf"])))
        outs.append(_attend(q, torch.cat([a for a, _ in K]), torch.cat([b for _, b in K]), pos))
    out = torch.stack([o[0] for o in outs]) if case["kind"] == "decode" else outs[0]
    gate = x["gate"][:, 0] if case["kind"] == "decode" else x["gate"][0]
    return {"out": out, "gated": out * torch.sigmoid(gate.double()) if case["gate"] else None, **none}
