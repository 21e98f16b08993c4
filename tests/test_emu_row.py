"""The fused row tile (csrc/row_tile.hpp) compiled for the CPU, every LDS, HBM
and twiddle index bounds-checked, against sums of powers of psi."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import O, P60, Q0, Q40

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["make", "-s", "-C", HERE, "librow_emu.so"], check=True)
    lib = C.CDLL(os.path.join(HERE, "librow_emu.so"))
    lib.emu_row_pass.argtypes = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint32, C.c_int]
    lib.emu_shoup_lazy3.argtypes = [C.c_uint64, C.c_uint64, C.c_uint64]
    lib.emu_shoup_lazy3.restype = C.c_uint64
    return lib


def _bitrev(x, bits):
    return int(format(x, f"0{bits}b")[::-1], 2)


@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_row_tile_evaluates_rows(emu, logn):
    """Forward: row m = bitrev(u) evaluated at psi^(2 (k2 N1 + u) + 1), stored
    at k2 N1 + u; first, last and one other row against Python integers.
    Inverse: gives N2 times the rows back, over the whole limb."""
    n2 = (logn + 1) // 2
    n1, N, N2 = logn - n2, 1 << logn, 1 << n2
    primes = [Q0[0], Q40[3], P60[2]] if logn < 17 else [O.ntt_primes(60, N, 1)[0], O.ntt_primes(40, N, 1)[0]]
    primes += O.ntt_primes(55, max(N, 1 << 16), 1)
    for q in primes:
        plan = O.Plan(q, N)
        psi = plan.psi
        for fill in ("random", "high"):
            rng = np.random.default_rng(logn)
            x = rng.integers(0, q, N, dtype=np.uint64) if fill == "random" else np.full(N, q - 1, dtype=np.uint64)
            x[:2] = [q - 1, 0]
            out, back = np.zeros(N, dtype=np.uint64), np.zeros(N, dtype=np.uint64)
            assert emu.emu_row_pass(x.ctypes.data, out.ctypes.data, q, logn, 1) == 0
            for u in (0, 1, (1 << n1) - 1):
                m = _bitrev(u, n1)
                row = [int(v) for v in x[m * N2:(m + 1) * N2]]
                for k2 in (0, 1, N2 // 2 + 3, N2 - 1):
                    z, acc = pow(psi, 2 * (k2 * (1 << n1) + u) + 1, q), 0
                    for v in reversed(row):
                        acc = (acc * z + v) % q
                    assert int(out[k2 * (1 << n1) + u]) == acc
            assert emu.emu_row_pass(out.ctypes.data, back.ctypes.data, q, logn, 0) == 0
            want = (x.astype(object) * N2) % q
            assert (back == want.astype(np.uint64)).all()


@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_column_and_row_tiles_match_oracle(emu, logn):
    """Column pass and row pass together are the oracle's transform, at the
    largest input bounds the kernels declare."""
    emu.emu_fused_ntt.argtypes = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint32, C.c_int]
    N = 1 << logn
    primes = [Q0[0], Q40[3], P60[2]] if logn < 17 else [O.ntt_primes(60, N, 1)[0], O.ntt_primes(40, N, 1)[0]]
    for q in primes + O.ntt_primes(55, max(N, 1 << 16), 1):
        plan = O.Plan(q, N)
        rng = np.random.default_rng(logn + 1)
        for x in (rng.integers(0, q, N, dtype=np.uint64), np.full(N, q - 1, dtype=np.uint64)):
            out, back = np.zeros(N, dtype=np.uint64), np.zeros(N, dtype=np.uint64)
            assert emu.emu_fused_ntt(x.ctypes.data, out.ctypes.data, q, logn, 1) == 0
            assert (out == plan.forward(x)).all()
            assert emu.emu_fused_ntt(x.ctypes.data, back.ctypes.data, q, logn, 0) == 0
            assert (back == plan.inverse(x)).all()


def test_shoup_lazy3_range(emu):
    """y w - h q stays in [0, 3q) and congruent for any 64-bit y, at the
    largest primes below 2^60 and below 2^41."""
    rng = np.random.default_rng(5)
    top = (1 << 64) - 1
    for q in (Q0[0], O.ntt_primes(41, 65536, 1)[0]):
        ws = [0, 1, 2, q - 1, q // 2, q - 2] + [int(v) for v in rng.integers(0, q, 200, dtype=np.uint64)]
        ys = [0, 1, (1 << 32) - 1, 1 << 32, top, top - 1, 0xffffffff00000000, 16 * q - 1 & top]
        ys += [int(v) for v in rng.integers(0, top, 200, dtype=np.uint64)]
        for w in ws:
            for y in ys:
                r = emu.emu_shoup_lazy3(y, w, q)
                assert r < 3 * q and (r - y * w) % q == 0
