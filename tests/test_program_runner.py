"""ProgramRunner on the CPU, the library's entry points recorded instead of
run: every run makes the calls of the program as it is then."""
from __future__ import annotations

import ctypes as C

import pytest

from conftest import load_pkg

pkg = load_pkg()
S = pkg.serving
N, L = 16, 3


class _Calls:
    """What the library was called with: (entry, [(field, ..) per entry])."""

    def __init__(self):
        self.log = []

    def _entries(self, kind, ptr, count):
        return (kind * count).from_address(C.cast(ptr, C.c_void_p).value)

    def ckks_apply_galois_batch(self, ctx, ptr, count):
        for e in self._entries(pkg.GaloisBatchEntry, ptr, count):
            self.log.append(("rotate", e.key, e.exponent, e.input, e.output, e.n_cts))

    def ckks_ntt_forward_batch(self, ctx, ptr, count):
        for e in self._entries(pkg.NttBatchEntry, ptr, count):
            self.log.append(("ntt", e.input, e.output))

    def ckks_multiply_plain_accumulate_ntt_batch(self, plan, cts, pts, count, outs, n_outs, limbs):
        read = lambda p, n: list((C.c_uint64 * n).from_address(p.value))
        self.log.append(("mac", read(cts, count), read(pts, count * n_outs), read(outs, n_outs)))


class _Plan:
    class ctx:
        handle = 1
    degree, handle = N, 2

    def multiply_plain(self, x, pt, la, out=None):
        pkg.lib().log.append(("mul", pt.data_ptr()))


class _Key(pkg._KeySwitchKey):
    def __init__(self, handle, q_limbs=L):
        self._finish_init(_Plan, handle)
        self.q_limbs = q_limbs

    def close(self):
        pass


@pytest.fixture
def calls(monkeypatch):
    import torch

    c, empty = _Calls(), torch.empty
    for module in (pkg, S):
        monkeypatch.setattr(module, "lib", lambda: c)
        monkeypatch.setattr(module, "_ptr", lambda t, numel=None, **kw: t.data_ptr())
        monkeypatch.setattr(module, "_ptrs", lambda ts, numel, name: [t.data_ptr() for t in ts])
        monkeypatch.setattr(module, "_check", lambda rc: None)
    monkeypatch.setattr(torch, "empty", lambda shape, dtype, device: empty(shape, dtype=dtype))
    return c


def _runner(prog):
    return S.ProgramRunner(_Plan(), L, prog, stream=object())


def _made(runner, calls):
    calls.log.clear()
    runner._run_ops()
    return list(calls.log)


def _pt(value=0):
    import torch

    return torch.full((L * N,), value, dtype=torch.int64)


def _program():
    prog = S.Program(n_regs=4, out_reg=0)
    prog.rotate(1, 0, _Key(11), 5)
    prog.mul_plain(2, 1, _pt())
    prog.ntt(2, 2)
    prog.ntt(3, 0)
    prog.mac_plain(0, 2, [_pt(), _pt()])
    return prog


@pytest.mark.parametrize("field,value", [(5, 25), (4, _Key(12))])
def test_a_rotation_replaced_in_place_runs(calls, field, value):
    prog = _program()
    runner = _runner(prog)
    assert _made(runner, calls)[0][:3] == ("rotate", 11, 5)
    op = list(prog.ops[0])
    op[field] = value
    prog.ops[0] = tuple(op)
    assert _made(runner, calls)[0][:3] == ("rotate", op[4].handle, op[5])


def test_a_product_replaced_in_place_runs(calls):
    prog = _program()
    runner = _runner(prog)
    _made(runner, calls)
    new = _pt(1)
    prog.ops[1] = prog.ops[1][:6] + (new,)
    assert ("mul", new.data_ptr()) in _made(runner, calls)


def test_a_replaced_plaintext_of_a_sum_is_read(calls):
    prog = _program()
    runner = _runner(prog)
    first = [c for c in _made(runner, calls) if c[0] == "mac"]
    assert first[0][2] == [t.data_ptr() for t in prog.ops[4][6]]
    new = _pt(1)
    prog.ops[4][6][1] = new
    again = [c for c in _made(runner, calls) if c[0] == "mac"]
    assert again[0][2] == [prog.ops[4][6][0].data_ptr(), new.data_ptr()]
    # the same tensor with other memory behind it
    other = _pt(2)
    new.set_(other)
    assert [c for c in _made(runner, calls) if c[0] == "mac"][0][2][1] == other.data_ptr()
    prog.ops[4][6].append(_pt())
    with pytest.raises(ValueError):
        runner._run_ops()


def test_another_output_register_is_the_one_that_outlives_the_run(calls):
    prog = S.Program(n_regs=3, out_reg=1)
    prog.rotate(1, 0, _Key(11), 5)
    prog.rotate(2, 0, _Key(11), 25)
    runner = _runner(prog)

    def written(exponent):
        """The row that holds this rotation after a run."""
        return {(c[4] - runner.regs.data_ptr()) // (8 * runner.per)
                for c in _made(runner, calls) if c[0] == "rotate" and c[2] == exponent}

    assert written(5) == {1}
    prog.out_reg = 2
    assert written(25) == {2}
    assert runner.output().data_ptr() == runner.regs[2].data_ptr()


def test_ops_that_can_change_in_place_are_read_on_every_run(calls):
    prog = _program()
    prog.ops[0] = list(prog.ops[0])
    runner = _runner(prog)
    assert _made(runner, calls)[0][2] == 5
    prog.ops[0][5] = 25
    assert _made(runner, calls)[0][2] == 25


def test_appended_and_removed_ops_run(calls):
    prog = _program()
    runner = _runner(prog)
    n = len(_made(runner, calls))
    prog.rotate(0, 0, _Key(13), 125)
    assert _made(runner, calls)[-1][:3] == ("rotate", 13, 125)
    prog.ops.pop()
    assert len(_made(runner, calls)) == n


def test_a_rotation_by_a_key_of_other_limbs_is_refused(calls):
    """As by the key's apply_galois: the register is no batch of its ciphertexts."""
    prog = S.Program(n_regs=2, out_reg=1)
    prog.rotate(1, 0, _Key(11, L - 1), 5)
    with pytest.raises(ValueError):
        _runner(prog)._run_ops()
