"""The key splits of a decode step, which the host plans (infllm_decode_splits): workgroups for the chip's 256 CUs."""
import ctypes as C

import pytest

from infllm_amd import _lib


def splits(B, H, Hkv, dim, blocks, rows, copies, most=64):
    f = _lib.load().infllm_decode_splits
    f.restype, f.argtypes = C.c_int, [C.c_int32] * 4 + [C.c_int64, C.c_int32, C.c_int64, C.c_int64]
    return f(B, H, Hkv, dim, blocks, most, rows, copies)


def workgroups(B, H, Hkv):
    G = H // Hkv
    return B * Hkv * -(-G // (4 if G >= 3 else G))


@pytest.mark.parametrize("H,Hkv,dim", [(32, 8, 128), (8, 8, 128), (16, 8, 128), (40, 40, 128), (28, 4, 128), (16, 1, 128), (36, 36, 64), (32, 8, 64)])
@pytest.mark.parametrize("blocks", [500, 2000])
def test_writers_of_a_row_do_not_cost_places(H, Hkv, dim, blocks):
    for B in range(1, 17):
        wgs, n = workgroups(B, H, Hkv), splits(B, H, Hkv, dim, blocks, B * Hkv, 0)
        assert wgs * n >= 192, (B, wgs, n)                # three of four CUs at least


@pytest.mark.parametrize("H,Hkv", [(16, 1), (64, 8), (28, 4)])
def test_workgroups_that_read_the_same_keys_meet_behind_one_l2(H, Hkv):
    for B in (1, 2, 4, 8):
        assert splits(B, H, Hkv, 128, 2000, B * Hkv, 0) % 8 == 0, B


def test_a_selection_is_two_blocks_of_a_wave():
    """8 splits of 136 blocks behind a selection and 256 others: the selection and 6 blocks a wave beside 7, not 5 beside 8"""
    f = _lib.load().infllm_decode_lead_splits
    f.restype, f.argtypes = C.c_int, [C.c_int32, C.c_int64, C.c_int64]
    assert f(8, 136, 256) == 3
    for n in (2, 3, 8, 32, 64):
        for lead in (1, 136, 100000):
            for rest in (1, 256, 100000):
                assert 1 <= f(n, lead, rest) < n


def test_bounds():
    for H, Hkv in ((32, 8), (40, 40), (16, 1)):
        for blocks in (0, 1, 7, 8, 9, 64, 100000):
            for most in (1, 2, 64):
                for copies in (0, 5, 100000):
                    n = splits(3, H, Hkv, 128, blocks, 24, copies, most)
                    assert 1 <= n <= most and n <= max(1, -(-blocks // 8))
