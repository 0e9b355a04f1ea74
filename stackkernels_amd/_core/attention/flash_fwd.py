"""Forward attention launcher over the gfx950 HIP kernel.

Same contract as the reference's ``flash_attn_fwd``
(``src/stackkernels/_core/attention/flash_fwd.py:182-264``): returns
``(out, lse)`` with ``out`` (B, H_q, S_q, D) in the input dtype and ``lse``
(B, H_q, S_q) fp32; GQA/MQA by ``H_q % H_kv == 0``; bottom-right causal mask.
``rope_cos`` / ``rope_sin`` / ``start_pos`` rotate q in the kernel's prologue
(query row i at position ``start_pos + i``): the prefill step with the
reference's ``apply_rope`` on q fused in.  This launcher is forward only; the
torch-level ``flash_attention`` pairs it with a backward that rotates q again
(``sk_rope_rotate``) and carries dQ back through the rotation's adjoint.
"""

from __future__ import annotations

import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention._rope import rope_args
from stackkernels_amd._core.attention._common import (
    check_device,
    default_scale,
    kernel_head_dim,
    operand,
    stream_of,
)
from stackkernels_amd._core.attention.layout import validate_attention_layout
from stackkernels_amd._core.attention.workspace import fwd_workspace


_NO_ROPE = (None, None, 0, 0, 0, None, 0)


def flash_attn_fwd(q, k, v, is_causal: bool = False, sm_scale: float | None = None,
                   rope_cos=None, rope_sin=None, start_pos=0):
    """Launch the HIP forward kernel; see module docstring."""
    b, hq, hkv, sq, sk, d = validate_attention_layout(q, k, v)
    dev = check_device(q, k, v)
    rope = rope_args(rope_cos, rope_sin, start_pos, b, d, dev)
    scale = default_scale(d, sm_scale)
    dk = kernel_head_dim(d)
    qk, qp, qs = operand(q, dk)
    kk, kp, ks = operand(k, dk)
    vk, vp, vs = operand(v, dk)
    out = q.new_empty((b, hq, sq, dk))
    lse = torch.empty((b, hq, sq), dtype=torch.float32, device=dev)
    lib = _lib.load()
    code = _lib.dtype_code(q.dtype)
    ws = fwd_workspace(code, b, hq, hkv, sq, sk, dk, is_causal, dev)
    ptrs = (code, qp, kp, vp, out.data_ptr(), lse.data_ptr())
    shape = (b, hq, hkv, sq, sk, dk, qs, ks, vs, _lib.strides3(out), int(bool(is_causal)))
    with _lib.device_guard(dev):
        if ws is not None:
            rc = lib.sk_attn_fwd_ws(*ptrs, ws.data_ptr(), ws.numel(), 0, *shape,
                                    *(_NO_ROPE if rope is None else rope.args), scale,
                                    stream_of(dev))
        elif rope is None:
            rc = lib.sk_attn_fwd(*ptrs, *shape, scale, stream_of(dev))
        else:
            rc = lib.sk_attn_fwd_rope(*ptrs, *shape, *rope.args, scale, stream_of(dev))
    _lib.check(rc, "flash_attn_fwd")
    if dk != d:
        out = out[..., :d].contiguous()
    return out, lse


__all__ = ["flash_attn_fwd"]
