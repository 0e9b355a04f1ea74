"""Scratch buffers the C ABI takes, sized by the library and allocated by torch.

The reference allocates its scratch in the launchers
(``src/stackkernels/_opt/memory/workspace.py:6-46``: LSE, delta and the
split-KV partials as separate float32 tensors).  Here the library sizes one
byte buffer per call (``sk_attn_fwd_workspace``, ``sk_attn_bwd_workspace``, ``sk_decode_plan`` /
``sk_decode_workspace``) and never allocates; these helpers take that buffer
from torch's caching allocator.  The launchers use them, and callers that bind
the library directly can too.
"""

from __future__ import annotations

import ctypes
import functools

import torch

from stackkernels_amd._core.attention import _lib


@functools.lru_cache(maxsize=512)
def _fwd_workspace_bytes(code: int, B: int, Hq: int, Hkv: int, Sq: int, Sk: int, D: int,
                         is_causal: bool) -> int:
    nb = ctypes.c_size_t(0)
    _lib.check(_lib.load().sk_attn_fwd_workspace(code, B, Hq, Hkv, Sq, Sk, D, int(is_causal),
                                                 ctypes.byref(nb)), "flash_attn_fwd")
    return nb.value


def fwd_workspace(code: int, B: int, Hq: int, Hkv: int, Sq: int, Sk: int, D: int,
                  is_causal: bool, device) -> torch.Tensor | None:
    """uint8 scratch for ``sk_attn_fwd_ws`` (code: the library's dtype code, D:
    the kernel head dim), or None where the forward runs unsplit: the table's
    choice for the shape, or no room for the partials (the same call, slower)."""
    nb = _fwd_workspace_bytes(code, B, Hq, Hkv, Sq, Sk, D, bool(is_causal))
    if nb == 0:
        return None
    try:
        return torch.empty(nb, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        return None


@functools.lru_cache(maxsize=512)
def _bwd_workspace_bytes(code: int, B: int, Hq: int, Hkv: int, Sq: int, Sk: int, D: int,
                         is_causal: bool) -> tuple[int, ...]:
    """The sizes bwd_workspace tries, largest first (each at least 16 bytes)."""
    lib = _lib.load()
    nb = ctypes.c_size_t(0)
    sizes = []
    for fn in (lib.sk_attn_bwd_workspace_best, lib.sk_attn_bwd_workspace,
               lib.sk_attn_bwd_workspace_min):
        _lib.check(fn(code, B, Hq, Hkv, Sq, Sk, D, int(is_causal), ctypes.byref(nb)),
                   "flash_attn_bwd")
        if max(nb.value, 16) not in sizes:
            sizes.append(max(nb.value, 16))
    return tuple(sizes)


def bwd_workspace(dtype: torch.dtype, B: int, Hq: int, Hkv: int, Sq: int, Sk: int, D: int,
                  is_causal: bool, device) -> torch.Tensor:
    """uint8 scratch for ``sk_attn_bwd`` (D: the kernel head dim; at least 16 bytes).

    The most the call makes use of (``sk_attn_bwd_workspace_best``: row
    statistics, one chunk of the five-GEMM backward's dS tiles, at most
    ``SK_BWD_DS_CAP_BYTES`` of them, and the partial sums of gradients split
    over several workgroups, dK/dV and for fp32 dQ, at most
    ``SK_PARTIALS_CAP_BYTES``); if torch cannot allocate that, the size
    without the partial sums, then the minimum (row statistics only), with
    which the call runs the seven-GEMM backward: slower, and those gradients
    summed in one pass, another order than a split one's.
    """
    code = _lib.dtype_code(dtype)
    sizes = _bwd_workspace_bytes(code, B, Hq, Hkv, Sq, Sk, D, bool(is_causal))
    for nb in sizes[:-1]:
        try:
            return torch.empty(nb, dtype=torch.uint8, device=device)
        except torch.OutOfMemoryError:
            pass
    return torch.empty(sizes[-1], dtype=torch.uint8, device=device)


@functools.lru_cache(maxsize=512)
def _decode_plan(code: int, B: int, Hq: int, Hkv: int, Sk: int, D: int,
                 per_row: bool) -> tuple[int, int]:
    """(split count, workspace bytes) of the library's table."""
    lib = _lib.load()
    ns, nb = ctypes.c_int(0), ctypes.c_size_t(0)
    fn = lib.sk_decode_plan_varlen if per_row else lib.sk_decode_plan
    _lib.check(fn(code, B, Hq, Hkv, Sk, D, ctypes.byref(ns), ctypes.byref(nb)),
               "flash_decode plan")
    return ns.value, nb.value


def decode_workspace(dtype: torch.dtype, B: int, Hq: int, Hkv: int, Sk: int, D: int, device,
                     num_splits: int | None = None,
                     per_row: bool = False) -> tuple[torch.Tensor, int]:
    """(uint8 scratch, split count) for ``sk_decode*`` (D: the kernel head dim):
    the gfx950 table's split count when ``num_splits`` is None (``per_row``:
    the plan for per-row cache lengths and paged pools), else the given one."""
    code = _lib.dtype_code(dtype)
    if num_splits is None:
        num_splits, nb = _decode_plan(code, B, Hq, Hkv, Sk, D, bool(per_row))
    else:
        size = ctypes.c_size_t(0)
        num_splits = int(num_splits)
        _lib.check(_lib.load().sk_decode_workspace(code, B, Hq, Hkv, Sk, D, num_splits,
                                                   ctypes.byref(size)), "flash_decode")
        nb = size.value
    return torch.empty(max(nb, 16), dtype=torch.uint8, device=device), num_splits


__all__ = ["fwd_workspace", "bwd_workspace", "decode_workspace"]
