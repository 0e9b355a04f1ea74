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
        assert n == 1 or b * h * n <= 2048 or (n == 2 and 1024 < b * h < 2048)


@pytest.mark.parametrize("heads", [33, 48, 64])
def test_large_groups_split_no_finer_than_pays(heads):
    """Groups above 32: splits of 256 keys, finer only up to 64 splits and 256 workgroups,
    and never into two."""
    for b in (1, 2, 3, 7, 16):
        for sk in (192, 263, 383, 384, 1000, 3356, 8192, 27491, 131072):
            for fn in ("sk_decode_plan", "sk_decode_plan_varlen"):
                n = _plan(fn, b, heads, 1, sk, 128)
                assert n <= max(1, sk // 256, min(64, 256 // b, sk // 128))
                assert sk >= 384 or n == 1


@pytest.mark.parametrize("heads", [17, 32])
def test_groups_of_two_waves_stop_at_64_fine_splits(heads):
    for b in (1, 2, 5):
        for sk in (255, 510, 4422, 12833, 34585, 131072):
            n = _plan("sk_decode_plan", b, heads, 1, sk, 128)
            assert n <= max(1, sk // 256, 64) and (sk >= 256 or n == 1)


@pytest.mark.parametrize("b,h", [(9, 12), (16, 8), (14, 32), (20, 16), (33, 24)])
def test_per_row_small_groups_take_rounds_of_256_keys(b, h):
    """Groups of one head, D <= 128: two rounds, or as many splits of 256 keys as the
    longest row has where that is more than one."""
    for sk in (2000, 4467, 10680, 16384):
        n = _plan("sk_decode_plan_varlen", b, h, h, sk, 128)
        two = -(-4096 // (b * h))
        keys = -(-sk // n)
        assert n <= two and (n >= 0.85 * two or keys <= 352)


@pytest.mark.parametrize("units", [4096, 4097, 100000])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_more_rows_than_slots_stay_whole(units, d):
    for fn in ("sk_decode_plan", "sk_decode_plan_varlen"):
        assert _plan(fn, units, 1, 1, 4000, d) == 1
