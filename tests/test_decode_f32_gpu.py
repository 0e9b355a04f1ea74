"""fp32 split decode (matrix-core kernel) at the edges of its tiles, splits, head
groups and head dims, against the float64 oracle at the fp32 bound; groups
above 64 heads stay on the fp32 forward's one-row path, unsplit."""

import numpy as np
import pytest
import torch

from stackkernels_amd._core.attention.decode import flash_decode as core_decode
from stackkernels_amd._core.attention.decode import flash_decode_paged
from stackkernels_amd._opt.pick import pick
from stackkernels_amd._reference.torch.rope import precompute_freqs
from stackkernels_amd.torch import flash_decode

from _gpu_util import TOL, assert_close_maxabs, make_qkv, np64, oracle_fwd
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
F32 = torch.float32


@pytest.mark.parametrize("group", [1, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("d", [40, 64, 96, 128, 200])
def test_tile_and_split_edges(device, group, d):
    kernel = pick("flash_decode", (2, 2 * group, 1, d), dtype="float32", kv_len=300,
                  num_kv_heads=2)["kernel_variant"]
    assert kernel == ("decode_split_f32_kernel" if group <= 64 else "fwd_f32_kernel")
    for sk in (1, 31, 33, 300):
        q, k, v = make_qkv(2, 2 * group, 2, 1, sk, d, F32, seed=sk + group + d)
        ref = oracle_fwd(q, k, v, False, -0.3)[0]
        for ns in (None, 1, 3, 9):
            print(f"fp32 decode group={group} D={d} S_k={sk} splits={ns}", flush=True)
            out = core_decode(q, k, v, sm_scale=-0.3, num_splits=ns)
            assert_close_maxabs(out, ref, TOL[F32], f"O (S_k={sk}, splits={ns})")


@pytest.mark.parametrize("d,page", [(64, 32), (128, 64), (256, 32)])
def test_paged_lengths_and_rope(device, d, page):
    """Per-row lengths over a paged pool with a page outside it, q rotated per row."""
    b, hq, hkv, width = 5, 8, 2, 4
    lens = torch.tensor([0, 1, page, 2 * page + 3, width * page], dtype=torch.int32)
    g = torch.Generator().manual_seed(d)
    kp, vp = (torch.randn(b * width, hkv, page, d, generator=g) for _ in range(2))
    q = torch.randn(b, hq, 1, d, generator=g)
    table = torch.randperm(b * width, generator=g).view(b, width).to(torch.int32)
    table[4, 1] = -1
    cos, sin = precompute_freqs(d, 1024)
    pos = torch.tensor([0, 1, 77, 500, 1023], dtype=torch.int32)
    qr = orc.rope_rotate(np64(q), np64(cos), np64(sin), pos.numpy()[:, None])
    ref = orc.decode_paged(qr, np64(kp), np64(vp), table.numpy(), lens.numpy())
    args = [t.to(device) for t in (q, kp, vp)]
    for ns in (None, 1, 5):
        out = flash_decode_paged(*args, table.to(device), lens.to(device), num_splits=ns,
                                 rope_cos=cos.to(device), rope_sin=sin.to(device),
                                 start_pos=pos.to(device))
        assert_close_maxabs(out, ref, TOL[F32], f"O (splits={ns})")
        assert torch.all(out[0] == 0)


def _fp32_in_quarters(q, k, v):
    """Attention of q (H, D) over k, v (H, S, D) in float32: scores as four partial
    sums of D / 4 products each, one running sum over the keys."""
    f = np.float32
    h, s, d = k.shape
    prod = (q[:, None] * k).reshape(h, s, 4, d // 4)
    acc = np.zeros((h, s, 4), f)
    for i in range(d // 4):
        acc += prod[..., i]
    sc = ((acc[..., 0] + acc[..., 1]) + (acc[..., 2] + acc[..., 3])) * f(1 / np.sqrt(d))
    w = np.exp(sc - sc.max(-1, keepdims=True))
    o, den = np.zeros((h, d), f), np.zeros((h, 1), f)
    for j in range(s):
        o += w[:, j:j + 1] * v[:, j]
        den += w[:, j:j + 1]
    return o / den


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("sk", [17, 64, 200])
def test_short_caches_keep_fp32_precision(device, d, sk):
    """No further from 64 bits than fp32 sums in four quarters of the head dim, on
    the same inputs.  (1.15: both are the rounding of as many operations, and its
    2-norm over 8,192 or more outputs varies by a few percent.  One chain over the
    head dim is 1.4 to 1.9 times as far.)"""
    q, k, v = make_qkv(4, 32, 32, 1, sk, d, F32, seed=d + sk)
    exact = oracle_fwd(q, k, v, False)[0].reshape(-1, d)
    want = _fp32_in_quarters(*(t.cpu().numpy().reshape(128, -1, d) if t.shape[2] > 1
                               else t.cpu().numpy().reshape(128, d) for t in (q, k, v)))
    got = np64(core_decode(q, k, v)).reshape(-1, d)
    assert np.linalg.norm(got - exact) <= 1.15 * np.linalg.norm(want - exact)


def test_strided_cache(device):
    """Slices of a larger cache (rows and heads apart) are read in place."""
    q, k, v = make_qkv(3, 4, 2, 1, 700, 128, F32, seed=2)
    kc, vc = (torch.full((3, 2, 900, 160), float("nan"), device=device) for _ in range(2))
    kc[:, :, :700, :128], vc[:, :, :700, :128] = k, v
    out = flash_decode(q, kc[:, :, :700, :128], vc[:, :, :700, :128])
    assert_close_maxabs(out, oracle_fwd(q, k, v, False)[0], TOL[F32], "O")
