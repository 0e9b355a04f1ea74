"""``pick`` on calls whose work is split: the kernel, grid and scratch that the
launchers use there, the merge passes, and dQ's side stream.  CPU: no launch."""
import ctypes

import pytest

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._opt.pick import pick

CODES = {"float32": 0, "float16": 1, "bfloat16": 2}


def _bytes(fn, dtype, b, hq, hkv, sq, sk, d, causal):
    n = ctypes.c_size_t()
    assert getattr(_lib.load(), fn)(CODES[dtype], b, hq, hkv, sq, sk, d, int(causal),
                                    ctypes.byref(n)) == 0
    return n.value


def _pick(op, dtype, b, hq, hkv, sq, sk, d, causal, **kw):
    return pick(op, (b, hq, sq, d), dtype=dtype, num_kv_heads=hkv, kv_len=sk, is_causal=causal,
                **kw)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,causal,packed", [
    (1, 32, 8, 512, 16000, 128, True, 1),     # key splits of one head's blocks
    (8, 64, 8, 35, 19392, 128, True, 8),      # packed heads, two blocks a unit
    (1, 8, 2, 17, 3000, 128, True, 1),
    (1, 12, 12, 200, 3000, 64, False, 1),
    (4, 32, 4, 40, 12000, 256, True, 8),
])
def test_split_forward(dtype, b, hq, hkv, sq, sk, d, causal, packed):
    dims = (dtype, b, hq, hkv, sq, sk, d, causal)
    f = _pick("flash_attn", *dims)
    ns = f["SPLIT_KV"]
    assert f["packed_heads"] == packed and ns >= 1 and ns * packed > 1
    blocks = -(-packed * sq // 128) * b * (hq // packed)
    assert f["BLOCK_M"] == 128 and f["num_warps"] == 4 and f["grid"] == blocks
    assert not f["paired_causal_blocks"]
    assert f["keys_per_split"] % 64 == 0 and -(-sk // f["keys_per_split"]) == ns
    assert f["workspace_bytes"] == _bytes("sk_attn_fwd_workspace", *dims) == (
        ns * b * hq * sq * (d + 1) * 4)
    assert f["combine"]["kernel_variant"] == "fwd_combine_kernel"
    assert f["combine"]["grid"] == -(-b * hq * sq // f["combine"]["BLOCK_M"])


@pytest.mark.parametrize("b,hq,hkv,sq,sk,split", [
    (1, 12, 12, 2801, 2891, False),  # 264 blocks, just over a round
    (1, 24, 2, 1330, 1330, False),
    (1, 4, 4, 2048, 2048, True),     # 64 blocks
    (1, 12, 12, 2801, 9000, True),   # blocks alike
])
def test_split_forward_d256_causal(b, hq, hkv, sq, sk, split):
    f = _pick("flash_attn", "bfloat16", b, hq, hkv, sq, sk, 256, True)
    assert (f["workspace_bytes"] > 0) == split


def test_split_forward_f32():
    dims = ("float32", 2, 8, 8, 1024, 1024, 64, False)
    f = _pick("flash_attn", *dims)
    ns = f["SPLIT_KV"]
    assert ns > 1 and f["kernel_variant"] == "fwd_f32_mfma_kernel" and f["packed_heads"] == 1
    assert f["grid"] == 4 * 16
    assert f["workspace_bytes"] == _bytes("sk_attn_fwd_workspace", *dims)


@pytest.mark.parametrize("b,hq,hkv,s,d,split", [
    (3, 32, 32, 647, 64, False),   # 288 blocks, three a head
    (2, 32, 1, 1194, 96, False),
    (3, 16, 4, 344, 64, False),    # a thin second block
    (1, 8, 8, 390, 64, True),
    (3, 16, 4, 490, 128, True),
    (2, 16, 4, 2139, 80, True),    # nine blocks a head
])
def test_f32_causal_squares(b, hq, hkv, s, d, split):
    f = _pick("flash_attn", "float32", b, hq, hkv, s, s, d, True)
    assert (f["SPLIT_KV"] > 1) == split


def test_whole_forward_has_no_merge():
    f = _pick("flash_attn", "bfloat16", 4, 32, 32, 4096, 4096, 128, True)
    assert f["SPLIT_KV"] == f["packed_heads"] == 1 and f["workspace_bytes"] == 0
    assert "combine" not in f


@pytest.mark.parametrize("dtype,b,hq,hkv,sq,sk,d,causal,dq_split", [
    ("bfloat16", 1, 32, 8, 2000, 2000, 96, True, False),
    ("float16", 2, 32, 1, 2048, 2048, 128, True, False),
    ("bfloat16", 1, 8, 1, 190, 260, 256, True, False),
    ("float32", 2, 8, 8, 1024, 1024, 64, False, True),
])
def test_split_backward(dtype, b, hq, hkv, sq, sk, d, causal, dq_split):
    dims = (dtype, b, hq, hkv, sq, sk, d, causal)
    w = _pick("flash_bwd", *dims)
    blocks = -(-sk // 128) * b * hkv * (2 if d > 128 else 1)
    assert w["splits"] > 1 and w["grid"] == blocks * w["splits"]
    assert (w["dq"]["splits"] > 1) == dq_split
    assert w["dq"]["grid"] == -(-sq // w["dq"]["BLOCK_M"]) * b * hq * w["dq"]["splits"]
    assert w["workspace_bytes"] == _bytes("sk_attn_bwd_workspace_best", *dims)
    part = 2 * w["splits"] * b * hkv * sk * d * 4 + (
        w["dq"]["splits"] * b * hq * sq * d * 4 if dq_split else 0)
    base = -(-_bytes("sk_attn_bwd_workspace", *dims) // 256) * 256
    assert w["workspace_bytes"] == base + part
    name = "bwd_f32_reduce_kernel" if dtype == "float32" else "bwd_dkv_reduce_kernel"
    assert w["reduce"]["kernel_variant"] == name and w["reduce"]["grid"] > 0


@pytest.mark.parametrize("dims,forks", [
    (("bfloat16", 2, 32, 8, 2048, 8192, 64, True), True),     # long, keys 4 x queries
    (("bfloat16", 4, 32, 8, 1500, 1500, 256, False), True),
    (("bfloat16", 2, 8, 8, 4096, 4096, 64, True), False),     # heavy blocks first
    (("bfloat16", 2, 16, 8, 512, 4096, 64, True), False),     # too short
    (("bfloat16", 2, 32, 8, 2048, 8192, 128, True), False),   # five GEMMs
    (("bfloat16", 2, 12, 12, 320, 7125, 64, False), True),    # few queries: dQ's grid is small
    (("float16", 10, 32, 32, 1744, 1744, 256, True), True),   # 35 rounds: head-major again
    (("bfloat16", 5, 16, 16, 1008, 1008, 64, False), False),  # 130 us: the host would show
    (("float32", 2, 32, 8, 2048, 8192, 64, True), False),
])
def test_side_stream(dims, forks):
    assert _pick("flash_bwd", *dims)["dq"]["side_stream"] == forks


def test_explain_names_the_merges():
    for op in ("flash_attn", "flash_bwd"):
        _, text = _pick(op, "bfloat16", 1, 32, 8, 512, 16000, 128, True, explain=True)
        assert ("fwd_combine_kernel" in text) == (op == "flash_attn")
        assert ("grid 512 workgroups" in text) == (op == "flash_attn")  # 128 in 4 splits
    _, text = _pick("flash_bwd", "bfloat16", 1, 32, 8, 2000, 2000, 96, True, explain=True)
    assert "bwd_dkv_reduce_kernel" in text
