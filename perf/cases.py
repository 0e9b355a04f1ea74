"""The attention work a program gives this package: serving (decode over a
KV cache, a decode step over a paged pool, prefill, chunked prefill) and
training (forward + backward), through the public calls of
``stackkernels_amd.torch``.

A case is a dict of plain values.  ``kind`` says which calls a pass makes:

``decode``   one query token per row over a whole contiguous cache.
``step``     one decode step of a server: the new token's key and value go
             into a paged pool (key rotated), then its query (rotated) attends
             to the row's own number of keys.
``prefill``  forward only, of whole sequences; ``layout`` says whether q, k, v
             are (B, H, S, D) tensors or transposed views of a projection's
             (B, S, H, D) output.
``chunk``    chunked prefill: T new tokens are appended to a contiguous cache
             (keys rotated) and their queries (rotated) attend, causally, to
             the filled part of the cache.
``train``    forward, then the gradients of q, k and v for a given dO.
"""

from __future__ import annotations

import math

import torch

from stackkernels_amd._reference.torch.rope import precompute_freqs
from stackkernels_amd.torch import FlashAttention, flash_attention, flash_decode, kv_cache_update

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # One user's decode with a short cache: latency and launches.
        dict(name="decode_one", kind="decode", dtype="bf16", B=1, Hq=32, Hkv=8, Sk=1000, D=128),
        # A full batch over long caches, 8.6 GB of keys and values.
        dict(name="decode_batch", kind="decode", dtype="bf16", B=64, Hq=32, Hkv=8, Sk=32768, D=128),
        # Few KV heads and very long contexts (MQA).
        dict(name="decode_mqa", kind="decode", dtype="fp16", B=8, Hq=64, Hkv=1, Sk=131072, D=128),
        # A server's decode step: ragged lengths in a paged pool, RoPE fused.
        dict(name="step_paged", kind="step", dtype="bf16", B=32, Hq=32, Hkv=8, Sk=4096, D=128,
             page=64),
        # An encoder's batch: short odd sequences, no mask.
        dict(name="encode_short", kind="prefill", dtype="fp16", B=16, Hq=12, Hkv=12, Sq=197,
             Sk=197, D=64, causal=False, layout="bhsd"),
        # An ordinary prompt batch of odd length, straight from the projections.
        dict(name="prefill_ragged", kind="prefill", dtype="bf16", B=2, Hq=32, Hkv=8, Sq=1337,
             Sk=1337, D=128, causal=True, layout="bshd"),
        # The headline forward: long prompts, MHA.
        dict(name="prefill_long", kind="prefill", dtype="bf16", B=4, Hq=32, Hkv=32, Sq=4096,
             Sk=4096, D=128, causal=True, layout="bhsd"),
        # One chunk of a long prompt against what the cache already holds.
        dict(name="chunk_cache", kind="chunk", dtype="bf16", B=1, Hq=32, Hkv=8, Sq=512, Sk=16000,
             D=128, cap=32768),
        # Training steps: a small model's layer, a GQA layer with more keys
        # than queries, a head dim between the powers of two, and 32-bit.
        dict(name="train_small", kind="train", dtype="fp16", B=4, Hq=12, Hkv=12, Sq=1024, Sk=1024,
             D=64, causal=True),
        dict(name="train_gqa", kind="train", dtype="bf16", B=2, Hq=32, Hkv=8, Sq=2048, Sk=8192,
             D=128, causal=True),
        dict(name="train_d96", kind="train", dtype="bf16", B=1, Hq=32, Hkv=8, Sq=2000, Sk=2000,
             D=96, causal=True),
        dict(name="train_f32", kind="train", dtype="fp32", B=2, Hq=8, Hkv=8, Sq=1024, Sk=1024,
             D=64, causal=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(["decode", "step", "prefill", "prefill", "chunk", "train", "train"])
    c = dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"]))
    c["Hq"], c["Hkv"] = rng.choice([(8, 8), (12, 12), (16, 16), (32, 32), (16, 4), (32, 8),
                                    (32, 4), (64, 8), (24, 2), (32, 1), (64, 1)])
    c["D"] = rng.choice([64, 64, 80, 96, 128, 128, 128, 256])
    if kind == "decode":
        c.update(B=_log_int(rng, 1, 64), Sk=_log_int(rng, 17, 131072))
    elif kind == "step":
        c.update(B=_log_int(rng, 1, 64), Sk=_log_int(rng, 64, 16384), page=rng.choice([32, 64, 128]))
    elif kind == "prefill":
        s = _log_int(rng, 17, 16384)
        c.update(B=_log_int(rng, 1, 16), Sq=s, Sk=s, causal=rng.random() < 0.6,
                 layout=rng.choice(["bhsd", "bshd"]))
    elif kind == "chunk":
        sq = _log_int(rng, 16, 2048)
        sk = sq + _log_int(rng, 1, 30000)
        c.update(B=_log_int(rng, 1, 8), Sq=sq, Sk=sk, cap=sk + rng.choice([0, 500, 4096]))
    else:
        s = _log_int(rng, 64, 8192)
        c.update(B=_log_int(rng, 1, 8), Sq=s, Sk=s if rng.random() < 0.7 else s + _log_int(rng, 1, 8192),
                 causal=rng.random() < 0.7)
    return c


def _cost(case):
    """Rough seconds of a pass, only to keep drawn cases below the largest listed one."""
    w = work(case)
    rate = 6e13 if case["dtype"] == "fp32" else 7e14
    return max(w["flops"] / rate, w["bytes"] / 5e12)


def draw(rng):
    most = max(_cost(c) for c in listed()) / 2
    while True:
        c = _draw_once(rng)
        if _cost(c) <= most:
            return c


def _pairs(case):
    """Visible (query, key) pairs of one head."""
    sq, sk = case["Sq"], case["Sk"]
    if not case.get("causal", True):
        return sq * sk
    return sum(min(max(i + 1 + sk - sq, 0), sk) for i in range(sq))


def work(case):
    e = 4 if case["dtype"] == "fp32" else 2
    B, Hq, Hkv, Sk, D = (case[n] for n in ("B", "Hq", "Hkv", "Sk", "D"))
    kind = case["kind"]
    if kind in ("decode", "step"):
        keys = Sk if kind == "decode" else (Sk + 1) / 2  # a step's rows hold 1 .. Sk keys
        data = 2 * B * Hkv * keys * D * e + 2 * B * Hq * D * e
        if kind == "step":
            data += 4 * B * Hkv * D * e
        return {"bytes": data, "flops": 4 * B * Hq * keys * D}
    Sq = case["Sq"]
    q, kv = B * Hq * Sq * D * e, B * Hkv * Sk * D * e
    flops = 4 * D * B * Hq * _pairs(case)
    if kind == "prefill":
        return {"bytes": 2 * q + 2 * kv, "flops": flops}
    if kind == "chunk":
        return {"bytes": 2 * q + 2 * kv + 4 * B * Hkv * Sq * D * e, "flops": flops}
    # q, k, v, dO read, O, dQ, dK, dV written; two products forward, five backward
    return {"bytes": 4 * q + 4 * kv, "flops": flops * 7 / 2}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, Hq, Hkv, Sk, D = (case[n] for n in ("B", "Hq", "Hkv", "Sk", "D"))
    kind = case["kind"]

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=dt)

    s = {"case": case}
    if kind == "decode":
        s.update(q=randn(B, Hq, 1, D), k=randn(B, Hkv, Sk, D), v=randn(B, Hkv, Sk, D))
    elif kind == "step":
        page = case["page"]
        width = (Sk + page - 1) // page
        lens = torch.randint(1, Sk + 1, (B,), generator=g, device=dev, dtype=torch.int32)
        table = torch.randperm(B * width, generator=g, device=dev).to(torch.int32).view(B, width)
        pos = lens - 1
        at = table.gather(1, (pos // page).long().view(B, 1))
        cos, sin = precompute_freqs(D, Sk, device=dev)
        s.update(q=randn(B, Hq, 1, D), k=randn(B, Hkv, 1, D), v=randn(B, Hkv, 1, D),
                 k_pool=randn(B * width, Hkv, page, D), v_pool=randn(B * width, Hkv, page, D),
                 table=table, lens=lens, pos=pos, slots=at.long() * page + (pos % page).view(B, 1),
                 cos=cos, sin=sin)
    elif kind == "prefill":
        Sq = case["Sq"]
        if case["layout"] == "bhsd":
            s.update(q=randn(B, Hq, Sq, D), k=randn(B, Hkv, Sk, D), v=randn(B, Hkv, Sk, D))
        else:
            s.update(q=randn(B, Sq, Hq, D).transpose(1, 2), k=randn(B, Sk, Hkv, D).transpose(1, 2),
                     v=randn(B, Sk, Hkv, D).transpose(1, 2))
    elif kind == "chunk":
        Sq, cap = case["Sq"], case["cap"]
        cos, sin = precompute_freqs(D, cap, device=dev)
        s.update(q=randn(B, Sq, Hq, D).transpose(1, 2), k=randn(B, Sq, Hkv, D).transpose(1, 2),
                 v=randn(B, Sq, Hkv, D).transpose(1, 2), k_cache=randn(B, Hkv, cap, D),
                 v_cache=randn(B, Hkv, cap, D), cos=cos, sin=sin, start=Sk - Sq,
                 slots=torch.arange(Sk - Sq, Sk, device=dev).expand(B, Sq).contiguous())
    else:
        Sq = case["Sq"]
        s.update(layer=FlashAttention(is_causal=case["causal"]),
                 q=randn(B, Hq, Sq, D).requires_grad_(), k=randn(B, Hkv, Sk, D).requires_grad_(),
                 v=randn(B, Hkv, Sk, D).requires_grad_(), do=randn(B, Hq, Sq, D))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        return {"o": flash_decode(s["q"], s["k"], s["v"])}
    if kind == "step":
        kv_cache_update(s["k"], s["v"], s["k_pool"], s["v_pool"], s["slots"], paged=True,
                        rope_cos=s["cos"], rope_sin=s["sin"], start_pos=s["pos"])
        o = flash_decode(s["q"], s["k_pool"], s["v_pool"], cache_seqlens=s["lens"],
                         block_table=s["table"], rope_cos=s["cos"], rope_sin=s["sin"],
                         start_pos=s["pos"])
        return {"o": o, "k_pool": s["k_pool"], "v_pool": s["v_pool"]}
    if kind == "prefill":
        with torch.no_grad():
            return {"o": flash_attention(s["q"], s["k"], s["v"], is_causal=case["causal"])}
    if kind == "chunk":
        n = case["Sk"]
        with torch.no_grad():
            kv_cache_update(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"],
                            rope_cos=s["cos"], rope_sin=s["sin"], start_pos=s["start"])
            o = flash_attention(s["q"], s["k_cache"][:, :, :n], s["v_cache"][:, :, :n],
                                is_causal=True, rope_cos=s["cos"], rope_sin=s["sin"],
                                start_pos=s["start"])
        return {"o": o, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    o = s["layer"](s["q"], s["k"], s["v"])
    dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
    return {"o": o, "dq": dq, "dk": dk, "dv": dv}


def tolerance(case):
    # About four times what the calls show against the 64-bit values over the
    # ranges of draw().  2-norm: 16-bit outputs are off by half a unit in the
    # last place, and so are the 16-bit probabilities that enter a product
    # (bf16 3.0e-3, fp16 3.4e-4); 32-bit sums 1.2e-6.  ``max``, over the root
    # mean square or the value: the first rows under a causal mask, whose
    # gradients are differences of nearly equal terms (bf16 0.12, fp16 0.012,
    # fp32 2.2e-5).
    return {"fp32": {"rel": 5e-6, "max": 9e-5}, "fp16": {"rel": 1.4e-3, "max": 5e-2},
            "bf16": {"rel": 1.2e-2, "max": 0.47}}[case["dtype"]]


def _rotated(x, cos, sin, pos):
    """x (B, H, S, D) rotated in 64 bits, token t of row b at position pos[b, t]."""
    c, s = cos.double()[pos][:, None], sin.double()[pos][:, None]
    half = x.shape[-1] // 2
    return x * c + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * s


def _attend(q, k, v, causal, do=None):
    """One KV head of one batch row: q, do (G, Sq, D), k, v (Sk, D), 64 bits."""
    G, Sq, D = q.shape
    Sk = k.shape[0]
    kt, scale = k.t().contiguous(), 1.0 / math.sqrt(D)
    hide = None
    if causal:
        i = torch.arange(Sq, device=q.device)[:, None]
        hide = torch.arange(Sk, device=q.device)[None] > i + (Sk - Sq)
    o, dq = torch.zeros_like(q), torch.zeros_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    for h in range(G):
        p = torch.mm(q[h], kt) * scale
        if hide is not None:
            p = p.masked_fill(hide, -math.inf)
        p = torch.softmax(p, dim=-1).nan_to_num_(0.0)
        o[h] = torch.mm(p, v)
        if do is not None:
            dv += torch.mm(p.t().contiguous(), do[h])
            ds = torch.mm(do[h], v.t().contiguous())
            ds = p * (ds - (do[h] * o[h]).sum(-1, keepdim=True)) * scale
            dq[h] = torch.mm(ds, k)
            dk += torch.mm(ds.t().contiguous(), q[h])
    return o, dq, dk, dv


def exact(case, seed):
    s = prepare(case, seed)
    B, Hq, Hkv = case["B"], case["Hq"], case["Hkv"]
    G = Hq // Hkv
    kind = case["kind"]
    with torch.no_grad():
        q = s["q"].double()
        o = torch.zeros_like(q, memory_format=torch.contiguous_format)
        if kind == "train":
            do = s["do"].double()
            dq = torch.zeros_like(q)
            dk = torch.zeros_like(s["k"], dtype=torch.float64)
            dv = torch.zeros_like(dk)
            for b in range(B):
                for h in range(Hkv):
                    g = slice(h * G, h * G + G)
                    o[b, g], dq[b, g], dk[b, h], dv[b, h] = _attend(
                        q[b, g], s["k"][b, h].double(), s["v"][b, h].double(), case["causal"],
                        do[b, g])
            return {"o": o, "dq": dq, "dk": dk, "dv": dv}
        out = {"o": o}
        if kind == "step":
            page, pos = case["page"], s["pos"].long().view(B, 1)
            q = _rotated(q, s["cos"], s["sin"], pos)
            kn = _rotated(s["k"].double(), s["cos"], s["sin"], pos)
            kp, vp = s["k_pool"].double(), s["v_pool"].double()
            pg, at = s["slots"][:, 0] // page, s["slots"][:, 0] % page
            kp[pg, :, at] = kn[:, :, 0]
            vp[pg, :, at] = s["v"][:, :, 0].double()
            out.update(k_pool=kp, v_pool=vp)
            lens = s["lens"].tolist()
        elif kind == "chunk":
            pos = torch.arange(case["Sk"] - case["Sq"], case["Sk"], device=q.device).expand(B, -1)
            q = _rotated(q, s["cos"], s["sin"], pos)
            kc, vc = s["k_cache"].double(), s["v_cache"].double()
            kc[:, :, pos[0]] = _rotated(s["k"].double(), s["cos"], s["sin"], pos)
            vc[:, :, pos[0]] = s["v"].double()
            out.update(k_cache=kc, v_cache=vc)
        for b in range(B):
            for h in range(Hkv):
                g = slice(h * G, h * G + G)
                if kind == "step":
                    rows = s["table"][b].long()
                    k = kp[rows, h].reshape(-1, case["D"])[:lens[b]]
                    v = vp[rows, h].reshape(-1, case["D"])[:lens[b]]
                elif kind == "chunk":
                    k, v = kc[b, h, :case["Sk"]], vc[b, h, :case["Sk"]]
                else:
                    k, v = s["k"][b, h].double(), s["v"][b, h].double()
                if kind in ("decode", "step"):  # the heads of the group as one product's rows
                    o[b, g] = _attend(q[b, g].transpose(0, 1), k, v, False)[0].transpose(0, 1)
                else:
                    o[b, g] = _attend(q[b, g], k, v, case.get("causal", True))[0]
    return out
