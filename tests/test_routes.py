"""Which kernels an untuned key switch takes (csrc/routes.hpp) at shapes where
both were timed on an MI355X: the route is the faster one."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["make", "-s", "-C", HERE, "libroutes_emu.so"], check=True)
    lib = C.CDLL(os.path.join(HERE, "libroutes_emu.so"))
    lib.emu_row_mac_pays.argtypes = [C.c_size_t, C.c_size_t]
    lib.emu_row_rotate_pays.argtypes = [C.c_size_t, C.c_size_t, C.c_size_t, C.c_size_t, C.c_uint]
    lib.emu_limb_tiles.argtypes = [C.c_size_t, C.c_size_t, C.c_uint]
    lib.emu_limb_tiles.restype = C.c_size_t
    lib.emu_half_tiles.argtypes = [C.c_int, C.c_size_t, C.c_uint]
    lib.emu_half_tiles.restype = C.c_size_t
    lib.emu_moddown_together.argtypes = [C.c_size_t, C.c_size_t, C.c_int]
    return lib


# digits, key limbs, ciphertexts, log2 N, us of the separate kernels, us fused
@pytest.mark.parametrize("dnum,limbs,cts,logn,separate,fused", [
    (6, 5, 1, 13, 53.7, 53.3), (2, 6, 1, 17, 95.5, 70.0), (10, 10, 1, 13, 69.5, 65.3), (25, 25, 1, 13, 139.2, 129.6),
    (11, 5, 1, 13, 61.7, 70.0), (11, 8, 1, 13, 74.5, 77.9), (11, 5, 1, 14, 69.1, 74.5), (11, 8, 2, 13, 87.8, 81.8),
    (23, 15, 1, 13, 141.2, 148.1), (23, 15, 2, 13, 172.9, 158.5), (34, 8, 1, 13, 117.1, 161.2),
    (34, 8, 2, 13, 144.3, 169.4), (34, 8, 1, 15, 187.9, 199.5), (10, 10, 2, 17, 474.5, 298.4),
])
def test_single_key_switches(emu, dnum, limbs, cts, logn, separate, fused):
    assert emu.emu_row_mac_pays(dnum, emu.emu_limb_tiles(limbs, cts, logn)) == (fused < separate)


# digits, key limbs, ciphertexts, exponents, log2 N, us of the separate kernels, us fused
@pytest.mark.parametrize("dnum,limbs,cts,exps,logn,separate,fused", [
    (2, 6, 1, 1, 13, 25.4, 24.6), (3, 32, 8, 4, 16, 2275.1, 2021.0), (11, 8, 1, 1, 13, 29.4, 33.6),
    (11, 8, 2, 1, 13, 36.6, 34.8), (23, 15, 1, 1, 13, 42.9, 53.0), (23, 15, 4, 1, 13, 65.8, 57.3),
    (10, 10, 1, 1, 13, 30.5, 34.4), (10, 10, 2, 1, 13, 41.4, 36.8), (23, 15, 1, 1, 14, 52.0, 55.0),
    (11, 8, 1, 1, 15, 42.0, 46.7), (11, 8, 2, 1, 15, 55.7, 49.4), (23, 15, 1, 1, 15, 81.4, 93.6),
    (16, 11, 4, 1, 15, 121.4, 140.8), (16, 11, 1, 3, 15, 131.2, 151.2), (16, 11, 4, 2, 15, 214.2, 205.3),
    (25, 25, 4, 1, 15, 353.0, 383.9), (25, 25, 4, 2, 15, 701.2, 595.2), (25, 25, 1, 1, 16, 259.1, 282.6),
    (6, 5, 1, 1, 17, 62.2, 66.2), (10, 10, 1, 1, 17, 122.0, 179.3), (3, 11, 1, 1, 17, 82.9, 91.2),
    (3, 11, 2, 1, 17, 130.6, 116.3), (5, 12, 16, 3, 17, 2596.8, 2755.5), (5, 12, 16, 4, 17, 3680.0, 3623.2),
    (8, 8, 16, 4, 17, 2715.0, 3014.6), (16, 16, 4, 1, 17, 696.9, 798.4), (16, 16, 4, 4, 17, 2861.0, 2495.5), (9, 9, 8, 2, 17, 1065.4, 913.9),
])
def test_hoisted_rotations(emu, dnum, limbs, cts, exps, logn, separate, fused):
    assert emu.emu_row_rotate_pays(dnum, limbs, cts, exps, logn) == (fused < separate)


# rotate, digits, tiles, log2 N, us with whole tiles, us with half ones
@pytest.mark.parametrize("rotate,dnum,tiles,logn,whole,half", [
    (0, 11, 160, 17, 160.5, 176.5), (0, 4, 128, 17, 72.2, 67.0), (1, 23, 120, 13, 68.8, 57.3),
    (1, 4, 256, 13, 47.3, 44.2), (1, 25, 200, 14, 135.7, 151.1), (1, 23, 240, 14, 96.8, 107.8),
    (1, 11, 128, 15, 49.4, 56.9), (1, 6, 40, 15, 36.8, 35.1), (1, 10, 160, 16, 60.2, 86.1),
    (1, 6, 160, 17, 66.2, 98.1),
])
def test_tile_sizes(emu, rotate, dnum, tiles, logn, whole, half):
    assert (tiles <= emu.emu_half_tiles(rotate, dnum, (logn + 1) // 2)) == (half < whole)


# exponents, ciphertexts, log2 N, whether b is added permuted, us in one launch, us in one launch each
@pytest.mark.parametrize("jobs,cts,logn,permuted,together,apart", [
    (4, 4, 16, 1, 1071.4, 1186.0), (4, 16, 16, 1, 3979.4, 3870.6), (3, 16, 16, 1, 1236.4, 1178.4),
    (2, 8, 17, 1, 889.8, 895.6), (4, 4, 17, 1, 2272.1, 2395.3), (3, 16, 17, 1, 2599.8, 2478.8),
    (3, 8, 17, 1, 1375.0, 1317.2), (4, 16, 16, 0, 3616.7, 3707.1), (3, 24, 16, 0, 1124.1, 1133.1),
])
def test_moddown_launches(emu, jobs, cts, logn, permuted, together, apart):
    assert emu.emu_moddown_together(jobs, cts * 2 << (logn - 8), permuted) == (together < apart)
