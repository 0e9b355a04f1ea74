"""Forward and backward on both sides of the compiled head dims' edges (64, 96,
128): the kernels for D <= 96 run the D = 128 tiles with three quarters of the
matrix instructions, so columns 88-95 and 96-103 fall to different kernels.
O, LSE and the gradients against the float64 oracle, on ragged lengths."""

import pytest
import torch

from stackkernels_amd._core.attention.flash_bwd import flash_attn_bwd
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd

from _gpu_util import TOL, assert_close_maxabs, assert_lse_close, make_qkv, np64, oracle_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("d", [64, 72, 88, 96, 104])
def test_head_dims_match_oracle(device, dtype, d):
    from oracle import attention_oracle as orc

    q, k, v = make_qkv(1, 2, 2, 97, 161, d, dtype, seed=d)
    o, lse = flash_attn_fwd(q, k, v, is_causal=True)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(d)).to(dtype).to(q.device)
    grads = flash_attn_bwd(do, q, k, v, o, lse, is_causal=True)
    torch.cuda.synchronize()
    ref, ref_lse = oracle_fwd(q, k, v, True)
    assert_close_maxabs(o, ref, TOL[dtype], "O")
    assert_lse_close(lse, ref_lse)
    exact = orc.attention_backward(np64(q), np64(k), np64(v), np64(do), True, None)
    for name, x, e in zip(("dQ", "dK", "dV"), grads, exact):
        assert_close_maxabs(x, e, TOL[dtype], name)
