"""GPU parity of the split dK/dV: the partial sums' chunks and their merge.

``sk_attn_bwd`` splits a key block's query tiles over several workgroups where
its workspace holds the partial sums (``sk_attn_bwd_workspace_best``).  Each
case runs that size and the unsplit one on NaN-filled scratch: dQ must be the
same bits (the dS tiles and the dQ kernel do not depend on the split), dK and
dV within the oracle's rounding bound.  The shapes put chunk seams inside and
between the heads of a group, key blocks of one chunk beside split ones, key
blocks that no query sees, ragged ends, and D = 64 with the dQ kernel forked.
"""

import ctypes

import pytest
import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention.flash_bwd import flash_attn_bwd
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd
from stackkernels_amd._reference.torch.attention import attention_reference

from _bwd_bound import check_backward, rounding_mass
from _gpu_util import make_qkv, np64

pytestmark = pytest.mark.gpu


def _bytes(q, k, causal):
    """(best, unsplit) workspace bytes."""
    b, hq, sq, d = q.shape
    out = []
    for fn in ("sk_attn_bwd_workspace_best", "sk_attn_bwd_workspace"):
        n = ctypes.c_size_t()
        rc = getattr(_lib.load(), fn)(_lib.dtype_code(q.dtype), b, hq, k.shape[1], sq, k.shape[2],
                                      d, int(causal), ctypes.byref(n))
        _lib.check(rc, fn)
        out.append(n.value)
    return out


def _bwd(do, q, k, v, o, lse, causal, ws_bytes):
    b, hq, sq, d = q.shape
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    ws = torch.full((ws_bytes,), 0xFF, dtype=torch.uint8, device=q.device)
    rc = _lib.load().sk_attn_bwd(
        _lib.dtype_code(q.dtype), do.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        o.data_ptr(), lse.data_ptr(), *(t.data_ptr() for t in grads), ws.data_ptr(), ws_bytes, b,
        hq, k.shape[1], sq, k.shape[2], d, int(causal), 1.0 / d ** 0.5,
        torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "sk_attn_bwd")
    return grads


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,causal", [
    (1, 16, 1, 333, 400, 128, True),   # light key blocks of one chunk beside split ones
    (1, 8, 2, 300, 130, 96, True),     # S_q > S_k
    (2, 8, 1, 257, 129, 80, False),    # ragged, one key in the second block
    (1, 16, 1, 200, 1500, 64, True),
    (13, 40, 10, 2000, 200, 64, False),  # 260 key blocks, two rounds
    (1, 8, 1, 190, 260, 256, True),    # head-dim halves
])
def test_split_matches_oracle(device, dtype, b, hq, hkv, sq, sk, d, causal):
    from oracle import attention_oracle as orc

    print(f"split dK/dV case {dtype} {(b, hq, hkv, sq, sk, d, causal)}", flush=True)
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, dtype, seed=sq + sk)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(3)).to(dtype).to(q.device)
    o, lse = flash_attn_fwd(q, k, v, is_causal=causal)
    best, unsplit = _bytes(q, k, causal)
    assert best > unsplit, "the table does not split this shape"
    split = _bwd(do, q, k, v, o, lse, causal, best)
    whole = _bwd(do, q, k, v, o, lse, causal, unsplit)
    again = _bwd(do, q, k, v, o, lse, causal, best)
    torch.cuda.synchronize()
    assert torch.equal(split[0], whole[0]), "dQ differs from the unsplit backward's"
    assert all(torch.equal(x, y) for x, y in zip(split, again)), "two runs differ"
    dt = "bf16" if dtype == torch.bfloat16 else "f16"
    group = hq // hkv
    pairs = {(0, 0), (b - 1, hkv - 1)} if b * hkv > 4 else {(i, j) for i in range(b) for j in range(hkv)}
    for bi, hi in sorted(pairs):  # a pair's gradients do not depend on the others
        def sl(t):
            n = t.shape[1] // hkv
            return t.detach()[bi:bi + 1, hi * n:(hi + 1) * n]

        qs, ks, vs, ds = (np64(sl(t)) for t in (q, k, v, do))
        assert qs.shape[1] == group
        exact = orc.attention_backward(qs, ks, vs, ds, causal)
        mass = rounding_mass(qs, ks, vs, ds, causal, None, dt)
        leaves = [sl(t).cpu().requires_grad_(True) for t in (q, k, v)]
        ref, _ = attention_reference(*leaves, is_causal=causal)
        ref.backward(sl(do).cpu())
        for i, name in enumerate(("dQ", "dK", "dV")):
            check_backward(np64(sl(split[i])), np64(leaves[i].grad), exact[i], mass[i], dt, name)


def test_many_heads_of_few_queries(device):
    """MQA with two query tiles per head: chunk seams fall between heads only."""
    q, k, v = make_qkv(1, 64, 1, 40, 300, 128, torch.bfloat16, seed=1)
    o, lse = flash_attn_fwd(q, k, v, is_causal=True)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(2)).to(q)
    best, unsplit = _bytes(q, k, True)
    a = _bwd(do, q, k, v, o, lse, True, best)
    b = _bwd(do, q, k, v, o, lse, True, unsplit)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.isfinite(x).all() and (x.float() - y.float()).abs().max() <= 2e-2


def test_forked_call_replays_match_eager(device):
    """D = 64, 2,048 x 8,192 (1,024 key blocks, dK/dV of about 400 us): dQ runs on the
    side stream, eagerly and as a captured graph's fork and join."""
    b, hq, hkv, sq, sk, d = 2, 32, 8, 2048, 8192, 64
    gen = torch.Generator(device=device).manual_seed(9)

    def inputs():
        q, do = (torch.randn(b, hq, sq, d, generator=gen, device=device).to(torch.bfloat16)
                 for _ in range(2))
        k, v = (torch.randn(b, hkv, sk, d, generator=gen, device=device).to(torch.bfloat16)
                for _ in range(2))
        return q, k, v, do

    q, k, v, do = inputs()
    o, lse = flash_attn_fwd(q, k, v, is_causal=True)
    cap = torch.cuda.Stream()
    cap.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(cap):
        flash_attn_bwd(do, q, k, v, o, lse, is_causal=True)
    torch.cuda.current_stream().wait_stream(cap)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        grads = flash_attn_bwd(do, q, k, v, o, lse, is_causal=True)
    unsplit = _bytes(q, k, True)[1]
    for step in range(3):
        new = inputs()
        o2, lse2 = flash_attn_fwd(*new[:3], is_causal=True)
        for dst, src in zip((q, k, v, do, o, lse), (*new, o2, lse2)):
            dst.copy_(src)
        want = flash_attn_bwd(new[3], *new[:3], o2, lse2, is_causal=True)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for x, y, name in zip(grads, want, ("dQ", "dK", "dV")):
            assert torch.equal(x, y), f"replay {step}: {name}"
        for x, y in zip(want, _bwd(new[3], *new[:3], o2, lse2, True, unsplit)):
            assert torch.equal(x, y)
