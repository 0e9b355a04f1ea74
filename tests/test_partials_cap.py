"""The tables never ask for more than SK_PARTIALS_CAP_BYTES of fp32 partials."""
import ctypes
import os
import random
import re

import pytest

from stackkernels_amd._core.attention import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include",
                      "sk_attn.h")
F32, F16, BF16 = 0, 1, 2


def _cap():
    return int(re.search(r"SK_PARTIALS_CAP_BYTES (\d+)", open(HEADER).read()).group(1))


def _bytes(fn, *dims):
    n = ctypes.c_size_t()
    assert getattr(_lib.load(), fn)(*dims, ctypes.byref(n)) == 0
    return n.value


def _partials(*dims):
    """(forward, backward) bytes of partials; the backward's start at a 256-byte boundary."""
    base = (_bytes("sk_attn_bwd_workspace", *dims) + 255) // 256 * 256
    return (_bytes("sk_attn_fwd_workspace", *dims),
            max(0, _bytes("sk_attn_bwd_workspace_best", *dims) - base))


@pytest.mark.parametrize("dims", [
    (F32, 4, 32, 1, 13868, 14160, 128, 1),
    (F16, 3, 64, 1, 10988, 10988, 256, 1),
    (BF16, 1, 64, 1, 26309, 26309, 256, 1),
    (F32, 2, 64, 1, 52404, 52895, 128, 0),
    (F32, 2, 12, 12, 2633, 55973, 128, 0),
])
def test_large_calls(dims):
    assert max(_partials(*dims)) <= _cap()


def test_random_calls():
    rng, seen = random.Random(0), 0
    for _ in range(4000):
        hkv = rng.choice([1, 1, 2, 4, 8, 16])
        sq = int(2 ** rng.uniform(0, 17))
        dims = (rng.choice([F32, F16, BF16]), rng.randint(1, 16), hkv * rng.choice([1, 4, 16, 64]),
                hkv, sq, rng.choice([sq, int(2 ** rng.uniform(0, 19))]),
                rng.choice([64, 96, 128, 256]), rng.randint(0, 1))
        got = _partials(*dims)
        assert max(got) <= _cap(), dims
        seen += max(got) > 0
    assert seen > 500


def test_ordinary_calls_still_split():
    assert _partials(F32, 2, 8, 8, 1024, 1024, 64, 0)[1] > 0
    assert _partials(BF16, 2, 32, 1, 2048, 2048, 128, 1)[1] > 0
    assert _partials(BF16, 1, 32, 8, 512, 16000, 128, 1)[0] > 0
