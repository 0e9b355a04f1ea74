"""NaN and infinities through the split paths: each gives what the one-pass
kernel of the same call gives.  A NaN in a query, a visible key or a value
reaches the rows it reaches there and no others, an infinite value stays
infinite, keys at -inf weigh nothing (a split, or a row, of only such keys
counts as empty), and the merges pass all of it on."""

import ctypes
import math

import pytest
import torch

from stackkernels_amd._core.attention import _lib
from stackkernels_amd._core.attention.decode import flash_decode as core_decode
from stackkernels_amd._core.attention.flash_fwd import flash_attn_fwd

from _gpu_util import TOL, make_qkv

pytestmark = pytest.mark.gpu
NAN, INF = float("nan"), float("inf")
NO_ROPE = (None, None, 0, 0, 0, None, 0)


def _fwd(q, k, v, causal, ns):
    """sk_attn_fwd_ws with ns splits (0: the table's, which may pack heads)."""
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1], k.shape[2]
    o, lse = torch.empty_like(q), torch.empty(b, hq, sq, device=q.device)
    ws = torch.full((32 * b * hq * sq * (d + 1),), NAN, device=q.device)
    rc = _lib.load().sk_attn_fwd_ws(
        _lib.dtype_code(q.dtype), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
        lse.data_ptr(), ws.data_ptr(), ws.numel() * 4, ns, b, hq, hkv, sq, sk, d,
        *(_lib.strides3(t) for t in (q, k, v, o)), int(causal), *NO_ROPE, 1 / math.sqrt(d),
        torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "sk_attn_fwd_ws")
    return o, lse


def _same(got, want, dtype, what):
    got, want = got.float(), want.float()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want)), f"{what}: {kind.__name__} differs"
    ok = torch.isfinite(want)
    assert (got[ok] - want[ok]).abs().max() <= TOL[dtype], what


def _plant(name, q, k, v, value_at=-1):
    """Writes the named values in place; returns whether rows must come out non-finite.
    (value_at: under the causal mask a key that every row sees.  A NaN in a value
    that a row does not see can still reach it, as 0 * NaN, through the tile it
    shares with rows that do; a split of which the row sees no key drops that.)"""
    hkv = k.shape[1]
    if name == "nan query":
        q[0, 1, -1, 3] = NAN
    elif name == "nan key":
        k[0, hkv - 1, 70, 0] = NAN
    elif name == "nan value":
        v[0, 0, value_at, 5] = NAN
    elif name == "inf value":
        v[0, 0, 2, 5], v[0, 0, 2, 6] = INF, -INF
    elif name == "inf key":
        k[0, 0, 100, 1] = INF
    else:  # scores of -inf: a run of keys, and every key of the last KV head
        q.abs_().clamp_(min=0.1)
        k[:, 0, 40:-30] = -INF
        k[:, hkv - 1] = -INF
        return False
    return True


PLANTS = ["nan query", "nan key", "nan value", "inf value", "inf key", "-inf keys"]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("plant", PLANTS)
@pytest.mark.parametrize("causal", [False, True])
def test_forward_key_splits(device, dtype, plant, causal):
    for sq, sk, d in ((64, 256, 64), (130, 400, 128)):
        q, k, v = make_qkv(1, 4, 2, sq, sk, d, dtype, seed=sk)
        planted = _plant(plant, q, k, v, 70 if causal else -1)
        want, want_lse = _fwd(q, k, v, causal, 1)
        assert bool((~torch.isfinite(want)).any()) == planted
        for ns in (2, 3):
            o, lse = _fwd(q, k, v, causal, ns)
            _same(o, want, dtype, f"O ({plant}, {sq}x{sk}, splits={ns})")
            _same(lse, want_lse, dtype, f"LSE ({plant}, {sq}x{sk}, splits={ns})")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("plant", PLANTS)
def test_forward_packed_heads(device, dtype, plant):
    from stackkernels_amd._opt.pick import pick

    b, hq, hkv, sq, sk, d = 8, 64, 8, 35, 4500, 128
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, dtype, seed=2)
    assert pick("flash_attn", q.shape, dtype=str(dtype), num_kv_heads=hkv,
                kv_len=sk)["packed_heads"] == 8
    planted = _plant(plant, q, k, v)
    want, want_lse = _fwd(q, k, v, False, 1)
    assert bool((~torch.isfinite(want)).any()) == planted
    o, lse = _fwd(q, k, v, False, 0)
    _same(o, want, dtype, f"O ({plant})")
    _same(lse, want_lse, dtype, f"LSE ({plant})")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("plant", PLANTS)
def test_decode(device, dtype, plant):
    for group, sk, d in ((4, 300, 64), (20, 500, 128), (8, 300, 256)):
        q, k, v = make_qkv(2, 2 * group, 2, 1, sk, d, dtype, seed=sk)
        planted = _plant(plant, q, k, v)
        want = flash_attn_fwd(q, k, v, is_causal=False)[0]
        assert bool((~torch.isfinite(want)).any()) == planted
        for ns in (1, 3, 9, None):
            _same(core_decode(q, k, v, num_splits=ns), want, dtype,
                  f"O ({plant}, group {group}, splits={ns})")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("d", [64, 128])
def test_gradient_chunks(device, dtype, d):
    """One dO row of NaN: the same gradients are NaN with partial sums and without."""
    b, hq, hkv, sq, sk = 1, 8, 2, 500, 700
    q, k, v = make_qkv(b, hq, hkv, sq, sk, d, dtype, seed=5)
    do = torch.randn(q.shape, generator=torch.Generator().manual_seed(3)).to(dtype).to(device)
    do[0, 2, 300] = NAN
    o, lse = flash_attn_fwd(q, k, v, is_causal=True)
    lib, n, got = _lib.load(), ctypes.c_size_t(), []
    dims = (b, hq, hkv, sq, sk, d, 1)
    for fn in ("sk_attn_bwd_workspace_best", "sk_attn_bwd_workspace"):
        assert getattr(lib, fn)(_lib.dtype_code(dtype), *dims, ctypes.byref(n)) == 0
        got.append((n.value, [torch.empty_like(t) for t in (q, k, v)]))
        ws = torch.full((n.value,), 0xFF, dtype=torch.uint8, device=device)
        _lib.check(lib.sk_attn_bwd(
            _lib.dtype_code(dtype), do.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
            o.data_ptr(), lse.data_ptr(), *(t.data_ptr() for t in got[-1][1]), ws.data_ptr(),
            n.value, *dims, 1 / math.sqrt(d), torch.cuda.current_stream().cuda_stream), "bwd")
    torch.cuda.synchronize()
    (best, split), (base, whole) = got
    assert best > base, "the table does not split this shape"
    for name, x, y in zip(("dQ", "dK", "dV"), split, whole):
        assert torch.isnan(y).any() and not torch.isnan(y).all(), name
        _same(x, y, dtype, name)
