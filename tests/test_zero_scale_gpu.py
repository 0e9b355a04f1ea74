"""``sm_scale = 0``: every visible key weighs the same, so O is the mean of the
visible V rows and LSE the logarithm of their number.  Each path that keeps a
running maximum or merges splits is run with masked tails, rows under the
causal mask that see no key of a split, and per-row lengths, against the
float64 oracle."""

import ctypes

import pytest
import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention.decode import flash_decode as core_decode
from stackkernels_amd._core.attention.flash_bwd import flash_attn_bwd
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd
from stackkernels_amd.torch import flash_decode

from _gpu_util import TOL, assert_close_maxabs, assert_lse_close, make_qkv, np64, oracle_fwd
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("group", [1, 20, 64])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_decode(device, dtype, group, d):
    for sk in (1, 33, 300):
        q, k, v = make_qkv(2, 2 * group, 2, 1, sk, d, dtype, seed=sk + group)
        ref = oracle_fwd(q, k, v, False, 0.0)[0]
        for ns in (None, 1, 3):
            out = core_decode(q, k, v, sm_scale=0.0, num_splits=ns)
            assert_close_maxabs(out, ref, TOL[dtype], f"O (S_k={sk}, splits={ns})")


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_decode_per_row_lengths(device, dtype):
    q, k, v = make_qkv(4, 8, 2, 1, 500, 128, dtype, seed=7)
    lens = torch.tensor([0, 1, 33, 500], dtype=torch.int32, device=device)
    ref = orc.decode_varlen(np64(q), np64(k), np64(v), lens.cpu().numpy(), 0.0)
    out = flash_decode(q, k, v, sm_scale=0.0, cache_seqlens=lens)
    assert_close_maxabs(out, ref, TOL[dtype], "O")


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,split", [
    (1, 32, 8, 64, 4096, 128, True),   # 16-bit: heads of a group packed
    (1, 8, 8, 200, 3000, 64, True),    # splits that end inside a tile
    (1, 4, 2, 300, 2100, 256, True),
    (2, 4, 2, 100, 70, 96, False),     # S_q > S_k: rows without a key
])
def test_forward_and_backward(device, dtype, causal, b, hq, hkv, sq, sk, d, split):
    n = ctypes.c_size_t()
    assert _lib.load().sk_attn_fwd_workspace(_lib.dtype_code(dtype), b, hq, hkv, sq, sk, d,
                                             int(causal), ctypes.byref(n)) == 0
    assert (n.value > 0) == (split and not (dtype == torch.float32 and d > 128))
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, dtype, seed=sq)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(3)).to(dtype).to(device)
    o, lse = flash_attn_fwd(q, k, v, is_causal=causal, sm_scale=0.0)
    ref, ref_lse = oracle_fwd(q, k, v, causal, 0.0)
    assert_close_maxabs(o, ref, TOL[dtype], "O")
    assert_lse_close(lse, ref_lse)
    dq, dk, dv = flash_attn_bwd(do, q, k, v, o, lse, is_causal=causal, sm_scale=0.0)
    want = orc.attention_backward(np64(q), np64(k), np64(v), np64(do), causal, 0.0)
    assert torch.all(dq == 0) and torch.all(dk == 0)
    assert_close_maxabs(dv, want[2], TOL[dtype], "dV")
