"""GPU parity of the split forward (``sk_attn_fwd_ws``): key splits at tile edges.

Each case runs the forward with explicit split counts on NaN-filled scratch
and outputs, so a partial that is read without having been written, or a row
that is left out, shows as NaN, and compares O and LSE with the float64
oracle: splits that end inside a 64-key tile, splits that rows under the
causal mask cannot see, rows that see no key at all (S_q > S_k), every
compiled head dim, and a shape whose count the table itself picks.
"""

import ctypes
import math

import pytest
import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd
from stackkernels_amd._opt.pick import pick

from _gpu_util import TOL, assert_close_maxabs, assert_lse_close, make_qkv, oracle_fwd

pytestmark = pytest.mark.gpu

NO_ROPE = (None, None, 0, 0, 0, None, 0)


def _fwd(q, k, v, causal, ns):
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1], k.shape[2]
    o = torch.full_like(q, float("nan"))
    lse = torch.full((b, hq, sq), float("nan"), device=q.device)
    ws = torch.full((ns * b * hq * sq * (d + 1),), float("nan"), device=q.device)
    rc = _lib.load().sk_attn_fwd_ws(
        _lib.dtype_code(q.dtype), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
        lse.data_ptr(), ws.data_ptr(), ws.numel() * 4, ns, b, hq, hkv, sq, sk, d,
        *(_lib.strides3(t) for t in (q, k, v, o)), int(causal), *NO_ROPE, 1 / math.sqrt(d),
        torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "sk_attn_fwd_ws")
    return o, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("sq,sk,d", [(1, 65, 128), (33, 129, 64), (130, 400, 80), (300, 191, 96),
                                     (129, 1000, 128), (257, 640, 256)])
def test_splits_match_oracle(device, dtype, causal, sq, sk, d):
    q, k, v = make_qkv(2, 4, 2, sq, sk, d, dtype, seed=sq + sk)
    ref, ref_lse = oracle_fwd(q, k, v, causal)
    for ns in (2, 3, 7):
        print(f"split case {dtype} causal={causal} {sq}x{sk} D={d} splits={ns}", flush=True)
        o, lse = _fwd(q, k, v, causal, ns)
        torch.cuda.synchronize()
        assert_close_maxabs(o, ref, TOL[dtype], f"O (splits={ns})")
        assert_lse_close(lse, ref_lse, f"LSE (splits={ns})")


def test_table_split_matches_oracle_and_replays(device):
    """40 queries against 5,000 keys: the launcher's own scratch, eagerly and as a
    HIP graph replayed on new inputs with eager work in between."""
    shape = (1, 4, 40, 128)
    assert pick("flash_attn", shape, dtype="bfloat16", kv_len=5000, num_kv_heads=1,
                is_causal=True)["SPLIT_KV"] > 1
    q, k, v = make_qkv(1, 4, 1, 40, 5000, 128, torch.bfloat16, seed=1)
    o, lse = flash_attn_fwd(q, k, v, is_causal=True)
    ref, ref_lse = oracle_fwd(q, k, v, True)
    assert_close_maxabs(o, ref, TOL[torch.bfloat16], "O")
    assert_lse_close(lse, ref_lse)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        og, lg = flash_attn_fwd(q, k, v, is_causal=True)
    for step in range(3):
        q2, k2, v2 = make_qkv(1, 4, 1, 40, 5000, 128, torch.bfloat16, seed=10 + step)
        for dst, src in ((q, q2), (k, k2), (v, v2)):
            dst.copy_(src)
        want, want_lse = flash_attn_fwd(q2, k2, v2, is_causal=True)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(og, want) and torch.equal(lg, want_lse), f"replay {step}"


def test_scratch_limits(device):
    """An explicit count without its scratch is refused; the table's count without
    scratch runs unsplit (sk_attn_fwd's result bit for bit)."""
    q, k, v = make_qkv(1, 4, 1, 40, 5000, 128, torch.bfloat16, seed=2)
    lib = _lib.load()
    o, lse = torch.empty_like(q), torch.empty(1, 4, 40, device=q.device)
    ws = torch.empty(1 << 16, dtype=torch.uint8, device=q.device)
    st = [_lib.strides3(t) for t in (q, k, v, o)]
    stream = torch.cuda.current_stream().cuda_stream

    def call(ns, nbytes):
        return lib.sk_attn_fwd_ws(2, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                  lse.data_ptr(), ws.data_ptr(), nbytes, ns, 1, 4, 1, 40, 5000,
                                  128, *st, 1, *NO_ROPE, 0.1, stream)

    need = ctypes.c_size_t()
    assert lib.sk_attn_fwd_workspace(2, 1, 4, 1, 40, 5000, 128, 1, ctypes.byref(need)) == 0
    assert need.value > ws.numel()
    assert call(2, ws.numel()) == _lib.SK_EWORKSPACE
    assert call(0, ws.numel()) == _lib.SK_OK
    o1, l1 = o.clone(), lse.clone()
    assert lib.sk_attn_fwd(2, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                           lse.data_ptr(), 1, 4, 1, 40, 5000, 128, *st, 1, 0.1, stream) == 0
    assert torch.equal(o, o1) and torch.equal(lse, l1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,hq,hkv,sq,sk,d", [
    (1, 8, 2, 17, 3000, 128),   # four heads in one block
    (2, 8, 1, 33, 2500, 64),    # MQA, heads across waves and blocks
    (1, 16, 4, 100, 2000, 80),  # blocks that end inside a head
    (1, 8, 2, 1, 4000, 96),     # one query per head
    (1, 6, 2, 50, 2100, 256),
    (1, 8, 2, 60, 59, 128),     # S_q > S_k: the table leaves it alone
])
def test_packed_heads_match_oracle(device, dtype, causal, b, hq, hkv, sq, sk, d):
    """Few queries per head: the table packs a group's heads into shared 128-row
    blocks (q read from strided heads too) and splits the keys."""
    need = ctypes.c_size_t()
    assert _lib.load().sk_attn_fwd_workspace(_lib.dtype_code(dtype), b, hq, hkv, sq, sk, d,
                                             int(causal), ctypes.byref(need)) == 0
    assert (need.value > 0) == (sk > 100)
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, dtype, seed=sq + sk)
    ref, ref_lse = oracle_fwd(q, k, v, causal)
    for form in (q, q.transpose(1, 2).contiguous().transpose(1, 2)):
        o, lse = flash_attn_fwd(form, k, v, is_causal=causal)
        torch.cuda.synchronize()
        assert_close_maxabs(o, ref, TOL[dtype], "O")
        assert_lse_close(lse, ref_lse)


def test_packed_heads_rotate_by_their_own_query(device):
    """RoPE on packed rows: query i of every head at start + i, as rotated beforehand."""
    from stackkernels_amd._core.attention._rope import rope_args, rope_rotate
    from stackkernels_amd._reference.torch.rope import precompute_freqs

    q, k, v = make_qkv(2, 8, 2, 37, 3000, 128, torch.bfloat16, seed=5)
    cos, sin = precompute_freqs(128, 4096, device=device)
    pos = torch.tensor([2963, 100], dtype=torch.int32, device=device)
    fused, lse = flash_attn_fwd(q, k, v, True, None, cos, sin, pos)
    plain, lse2 = flash_attn_fwd(rope_rotate(q, rope_args(cos, sin, pos, 2, 128, q.device)), k, v,
                                 True)
    assert torch.equal(fused, plain) and torch.equal(lse, lse2)
