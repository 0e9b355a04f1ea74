"""fp32 forward and backward whose grids leave CUs idle: key splits of the
forward, chunks of dK/dV and of dQ.  O, LSE and the gradients against the
float64 oracle at the fp32 bound (1e-4), on shapes whose chunks end inside a
head's query tiles, whose blocks differ in their chunk counts (causal), with
rows and keys nobody sees, and the same bits on a second run."""

import ctypes

import pytest
import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention.flash_bwd import flash_attn_bwd
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd

from _gpu_util import TOL, assert_close_maxabs, assert_lse_close, make_qkv, np64, oracle_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,causal,fwd,bwd", [
    (1, 8, 8, 500, 500, 64, True, True, True),
    (1, 8, 1, 150, 1100, 96, True, True, True),
    (2, 4, 4, 300, 260, 128, False, True, True),
    (1, 4, 2, 400, 190, 128, True, True, True),  # S_q > S_k
    (1, 6, 1, 257, 129, 40, False, False, True),
    (1, 2, 2, 40, 1500, 80, True, True, True),    # one query block
])
def test_f32_splits_match_oracle(device, b, hq, hkv, sq, sk, d, causal, fwd, bwd):
    from oracle import attention_oracle as orc

    print(f"fp32 split case {(b, hq, hkv, sq, sk, d, causal)}", flush=True)
    lib, n = _lib.load(), ctypes.c_size_t()
    dims = (0, b, hq, hkv, sq, sk, (d + 7) // 8 * 8, int(causal), ctypes.byref(n))
    assert lib.sk_attn_fwd_workspace(*dims) == 0 and (n.value > 0) == fwd
    assert lib.sk_attn_bwd_workspace(*dims) == 0
    base = n.value
    assert lib.sk_attn_bwd_workspace_best(*dims) == 0 and (n.value > base) == bwd
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, torch.float32, seed=sq)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(3)).to(q.device)
    o, lse = flash_attn_fwd(q, k, v, is_causal=causal)
    grads = flash_attn_bwd(do, q, k, v, o, lse, is_causal=causal)
    again = flash_attn_bwd(do, q, k, v, o, lse, is_causal=causal)
    torch.cuda.synchronize()
    ref, ref_lse = oracle_fwd(q, k, v, causal)
    assert_close_maxabs(o, ref, TOL[torch.float32], "O")
    assert_lse_close(lse, ref_lse)
    exact = orc.attention_backward(np64(q), np64(k), np64(v), np64(do), causal, None)
    for name, x, y, e in zip(("dQ", "dK", "dV"), grads, again, exact):
        assert torch.equal(x, y), f"{name}: two runs differ"
        assert_close_maxabs(x, e, TOL[torch.float32], name)
