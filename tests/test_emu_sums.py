"""The sums of the fused passes (csrc/row_sums.hpp) and the tiles of small
launches compiled for the CPU, at the extremes of their operands, against
Python integers and the oracle's transforms."""
from __future__ import annotations

import ctypes as C
import os
import random
import subprocess

import numpy as np
import pytest

from conftest import O, P60, Q0, Q40

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
DIGIT = (1 << 41) - 1  # the largest mixed-radix digit
FP_PRIMES = [O.ntt_primes(41, 65536, 1)[0], O.ntt_primes(36, 65536, 1)[0], O.ntt_primes(20, 1024, 1)[0]]
INT_PRIMES = [O.ntt_primes(42, 65536, 1)[0], O.ntt_primes(55, 65536, 1)[0], Q0[0], O.ntt_primes(61, 65536, 1)[0]]


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["make", "-s", "-C", HERE, "librow_emu.so"], check=True)
    lib = C.CDLL(os.path.join(HERE, "librow_emu.so"))
    lib.emu_block_sum.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_uint64]
    lib.emu_block_sum.restype = C.c_int64
    lib.emu_key_sum.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_uint64, C.POINTER(C.c_uint64)]
    lib.emu_key_sum.restype = C.c_int64
    for name in ("emu_fused_ntt_halved", "emu_small_ntt"):
        getattr(lib, name).argtypes = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint32, C.c_int]
    return lib


def _u64(values):
    return np.array(values, dtype=np.uint64)


@pytest.mark.parametrize("terms", range(1, 14))
@pytest.mark.parametrize("fp", [1, 0])
def test_block_sums_are_the_remainder(emu, fp, terms):
    """sum c W - k q with k right to within the rounding of the quotient: 13
    terms below 2^41 carry an error below 0.04, so the remainder stays within
    0.54 q.  Digits and weights at their largest, remainders at half a q."""
    rng = random.Random(terms * 2 + fp)
    for q in FP_PRIMES if fp else INT_PRIMES:
        draws = []
        for _ in range(300):
            c = [rng.choice([DIGIT, DIGIT, DIGIT - rng.randrange(1000), rng.randrange(DIGIT + 1)]) for _ in range(terms)]
            w = [rng.choice([q - 1, q - 1 - rng.randrange(min(q, 1000)), q // 2, rng.randrange(q)]) for _ in range(terms)]
            if c[-1] % q:  # the last weight puts the remainder next to a tie
                rest = sum(x * y for x, y in zip(c[:-1], w[:-1]))
                w[-1] = (q // 2 + rng.randrange(2) - rest) * pow(c[-1], -1, q) % q
            draws.append((c, w))
        draws += [([DIGIT] * terms, [q - 1] * terms), ([0] * terms, [q - 1] * terms), ([DIGIT] * terms, [0] * terms),
                  ([1] + [0] * (terms - 1), [1] + [0] * (terms - 1))]
        for c, w in draws:
            cc, ww = _u64(c), _u64(w)
            got = emu.emu_block_sum(fp, cc.ctypes.data, ww.ctypes.data, terms, q)
            r = got if fp else (got & ((1 << 64) - 1)) - q
            assert abs(r) <= 0.54 * q and (r - sum(x * y for x, y in zip(c, w))) % q == 0, (q, c, w)


@pytest.mark.parametrize("count", [1, 4, 5, 8, 9, 25, 69])
def test_integer_key_sums(emu, count):
    """Digits below 16 q, canonical key entries: sums below 11 q before a
    reduction, the total below 3 q."""
    rng = random.Random(count)
    for q in INT_PRIMES[:3]:
        top = min(16 * q, 1 << 64) - 1
        for mode in range(40):
            y = [top if mode == 0 else rng.choice([top, top - rng.randrange(1000), rng.randrange(top + 1)]) for _ in range(count)]
            w = [q - 1 if mode == 0 else rng.choice([q - 1, rng.randrange(q)]) for _ in range(count)]
            peak = C.c_uint64()
            yy, ww = _u64(y), _u64(w)
            r = emu.emu_key_sum(0, yy.ctypes.data, ww.ctypes.data, count, q, C.byref(peak)) & ((1 << 64) - 1)
            assert r < 3 * q and peak.value < 11 * q and (r - sum(a * b for a, b in zip(y, w))) % q == 0


@pytest.mark.parametrize("count", [1, 8, 9, 16, 17, 69])
def test_fp64_key_sums(emu, count):
    """Digits below 2^45 in magnitude: exact sums below 2^45, the total within
    half a q."""
    rng = random.Random(count)
    top = (1 << 45) - 1
    for q in FP_PRIMES:
        for mode in range(40):
            sign = rng.choice([1, -1])
            y = [sign * top if mode < 2 else rng.choice([top, -top, rng.randint(-top, top)]) for _ in range(count)]
            w = [q - 1 if mode < 2 else rng.choice([q - 1, q // 2, rng.randrange(q)]) for _ in range(count)]
            peak = C.c_uint64()
            yy, ww = np.array(y, dtype=np.int64), _u64(w)
            r = emu.emu_key_sum(1, yy.ctypes.data, ww.ctypes.data, count, q, C.byref(peak))
            assert abs(r) <= 0.52 * q and peak.value < 1 << 45 and (r - sum(a * b for a, b in zip(y, w))) % q == 0


def _inputs(q, n, seed):
    x = np.random.default_rng(seed).integers(0, q, n, dtype=np.uint64)
    x[:2] = [q - 1, 0]
    return x, np.full(n, q - 1, dtype=np.uint64)


@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_halved_tiles_match_oracle(emu, logn):
    n = 1 << logn
    primes = [Q0[0], Q40[3]] if logn < 17 else [O.ntt_primes(60, n, 1)[0], O.ntt_primes(40, n, 1)[0]]
    for q in primes + O.ntt_primes(55, max(n, 1 << 16), 1):
        plan = O.Plan(q, n)
        for x in _inputs(q, n, logn):
            out = np.zeros(n, dtype=np.uint64)
            assert emu.emu_fused_ntt_halved(x.ctypes.data, out.ctypes.data, q, logn, 1) == 0
            assert (out == plan.forward(x)).all()
            assert emu.emu_fused_ntt_halved(x.ctypes.data, out.ctypes.data, q, logn, 0) == 0
            assert (out == plan.inverse(x)).all()


@pytest.mark.parametrize("logn", [10, 11, 12])
def test_single_pass_tiles_match_oracle(emu, logn):
    n = 1 << logn
    for q in (Q0[0], Q40[3], P60[2], FP_PRIMES[0], INT_PRIMES[0]):
        plan = O.Plan(q, n)
        for x in _inputs(q, n, logn):
            out = np.zeros(n, dtype=np.uint64)
            assert emu.emu_small_ntt(x.ctypes.data, out.ctypes.data, q, logn, 1) == 0
            assert (out == plan.forward(x)).all()
            assert emu.emu_small_ntt(x.ctypes.data, out.ctypes.data, q, logn, 0) == 0
            assert (out == plan.inverse(x)).all()
