"""The decode split table's rounds: how many workgroups a planned grid has."""
import ctypes

import pytest

from stackkernels_amd._core.attention import _lib

BF16 = 2


def _plan(fn, b, hq, hkv, sk, d):
    lib = _lib.load()
    ns, nb = ctypes.c_int(0), ctypes.c_size_t(0)
    assert getattr(lib, fn)(BF16, b, hq, hkv, sk, d, ctypes.byref(ns), ctypes.byref(nb)) == 0
    return ns.value


@pytest.mark.parametrize("d,slots", [(64, 2048), (128, 2048), (256, 1024)])
@pytest.mark.parametrize("b,h", [(8, 8), (23, 16), (40, 12), (45, 4), (100, 8)])
def test_uniform_grid_fits_one_round(b, h, d, slots):
    for sk in (192, 500, 976, 4000, 20000):
        n = _plan("sk_decode_plan", b, h, h, sk, d)
        assert 1 <= n and (n == 1 or b * h * n <= slots)


@pytest.mark.parametrize("b,h", [(8, 8), (23, 16), (40, 12), (45, 4), (100, 8), (150, 8), (300, 8)])
def test_per_row_grid_fits_two_rounds(b, h):
    for sk in (192, 500, 976, 4000, 20000):
        n = _plan("sk_decode_plan_varlen", b, h, h, sk, 256)
        assert n == 1 or b * h * n <= 2048


@pytest.mark.parametrize("units", [4096, 4097, 100000])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_more_rows_than_slots_stay_whole(units, d):
    for fn in ("sk_decode_plan", "sk_decode_plan_varlen"):
        assert _plan(fn, units, 1, 1, 4000, d) == 1
