"""The forward reads q, k, v in place when no gradient is asked for: every form
of strides it accepts gives the contiguous copies' bits, and a call that will
run a backward keeps copies of its own (an input changed in place afterwards
neither raises nor reaches the gradients)."""

import pytest
import torch

from stackkernels_amd._reference.torch.rope import precompute_freqs
from stackkernels_amd.torch import flash_attention

from _gpu_util import make_qkv

pytestmark = pytest.mark.gpu


def _forms(t):
    """Views equal to the (B, H, S, D) tensor t with other strides or alignment."""
    b, h, s, d = t.shape
    yield "bshd", t.transpose(1, 2).contiguous().transpose(1, 2)
    yield "sbhd", t.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3)
    big = torch.full((b, h, s + 9, d), float("nan"), dtype=t.dtype, device=t.device)
    big[:, :, :s] = t
    yield "slice", big[:, :, :s]
    odd = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    odd.copy_(t)
    yield "unaligned", odd
    wide = torch.empty(b, h, s, d + 1, dtype=t.dtype, device=t.device)
    wide[..., :d] = t
    yield "odd_rows", wide[..., :d]
    yield "dhbs", t.permute(3, 1, 0, 2).contiguous().permute(2, 1, 3, 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("d,rope", [(128, False), (64, True), (36, False)])
def test_strides_give_the_same_bits(device, dtype, d, rope):
    q, k, v = make_qkv(2, 4, 2, 70, 130, d, dtype, seed=d)
    kw = {}
    if rope:
        cos, sin = precompute_freqs(d, 256, device=device)
        kw = dict(rope_cos=cos, rope_sin=sin, start_pos=3)
    want = flash_attention(q, k, v, is_causal=True, **kw)
    for (name, qs), (_, ks), (_, vs) in zip(_forms(q), _forms(k), _forms(v)):
        print(f"strided forward {dtype} D={d} rope={rope} {name}", flush=True)
        got = flash_attention(qs, ks, vs, is_causal=True, **kw)
        assert got.is_contiguous() and torch.equal(got, want), name
    # one KV head seen by all four through a zero stride
    want = flash_attention(q, k[:, :1].repeat(1, 4, 1, 1), v[:, :1].repeat(1, 4, 1, 1), **kw)
    got = flash_attention(q, k[:, :1].expand(-1, 4, -1, -1), v[:, :1].expand(-1, 4, -1, -1), **kw)
    assert torch.equal(got, want)


def test_backward_keeps_its_own_copies(device):
    q, k, v = make_qkv(1, 4, 2, 40, 60, 64, torch.bfloat16, seed=4)
    base = k.transpose(1, 2).contiguous()
    grads = []
    for change in (False, True):
        kb = base.clone()
        qg = q.clone().requires_grad_(True)
        out = flash_attention(qg, kb.transpose(1, 2), v, is_causal=True)
        if change:
            kb.zero_()
        out.backward(torch.ones_like(out))
        grads.append(qg.grad)
    assert torch.equal(*grads)
