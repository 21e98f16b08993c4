"""Grouped execution order of a program (serving.schedule): every register that
outlives a run holds what program order gives it, whatever rows are reused."""
from __future__ import annotations

import random

import pytest

from conftest import load_pkg

S = load_pkg().serving


_names: dict = {}


def _apply(code, ins, op):
    """A result as a number of its own per (op, inputs)."""
    return _names.setdefault((code, tuple(ins), op[5]), len(_names))


def _reads(op):
    code, _, a, b = op[:4]
    if code == S.OP_MAC_PLAIN:
        return list(range(a, a + b))
    return [a, b] if code in (S.OP_ADD, S.OP_SUB, S.OP_MUL_RELIN_RESCALE) else [a]


def _program(rng, n_regs, n_ops):
    prog = S.Program(n_regs=n_regs, out_reg=rng.randrange(n_regs), n_inputs=rng.randint(1, n_regs))
    limbs = [9 if r < prog.n_inputs else 0 for r in range(n_regs)]
    for i in range(n_ops):
        live = [r for r in range(n_regs) if limbs[r] > 1]
        a, dst = rng.choice(live), rng.randrange(n_regs)
        same = [r for r in live if limbs[r] == limbs[a]]
        code = rng.choice([S.OP_ROTATE] * 3 + [S.OP_NTT, S.OP_INTT, S.OP_ADD, S.OP_SUB, S.OP_COPY, S.OP_RESCALE,
                                               S.OP_MUL_PLAIN, S.OP_MAC_PLAIN, S.OP_MUL_RELIN_RESCALE])
        b = 0
        if code in (S.OP_ADD, S.OP_SUB, S.OP_MUL_RELIN_RESCALE):
            b = rng.choice(same)
        if code == S.OP_MAC_PLAIN:
            b = 1
            while a + b < n_regs and limbs[a + b] == limbs[a]:
                b += 1
        if code in (S.OP_RESCALE, S.OP_MUL_RELIN_RESCALE) and limbs[a] < 4:
            code = S.OP_ROTATE
        prog.ops.append((code, dst, a, b, None, i, None))
        limbs[dst] = limbs[a] - (1 if code in (S.OP_RESCALE, S.OP_MUL_RELIN_RESCALE) else 0)
    return prog


@pytest.mark.parametrize("spare", [0, 1, 3, 16])
@pytest.mark.parametrize("n_regs", [1, 2, 5, 12])
def test_groups_give_program_order_results(n_regs, spare):
    for seed in range(60):
        rng = random.Random(seed * 1000 + n_regs * 20 + spare)
        prog = _program(rng, n_regs, rng.randint(0, 60))
        groups, rows = S.schedule(prog, 9, spare)
        assert rows <= n_regs + 2 + spare
        for passes in (1, 2):  # the second on the registers as the first left them
            regs = [("in", r) for r in range(n_regs)]
            phys = [("in", r) for r in range(n_regs)] + [None] * (rows - n_regs)
            for _ in range(passes):
                for op in prog.ops:
                    ins = [regs[r] for r in _reads(op)]
                    regs[op[1]] = ins[0] if op[0] == S.OP_COPY else _apply(op[0], ins, op)
                for code, _, items in groups:
                    assert len(items) <= S._TOGETHER
                    outs = [o for o, _, _ in items]
                    assert len(set(outs)) == len(outs)
                    for out, ins, op in items:
                        others = [r for o, i, _ in items if o != out for r in i]
                        assert out not in others, "a row written and read by two ops of one group"
                        if code not in (S.OP_NTT, S.OP_INTT, S.OP_ADD, S.OP_SUB, S.OP_MUL_PLAIN):
                            assert out not in ins
                    new = [phys[ins[0]] if code == S.OP_COPY else _apply(code, [phys[i] for i in ins], op)
                           for _, ins, op in items]
                    for o, v in zip(outs, new):
                        phys[o] = v
            assert phys[prog.out_reg] == regs[prog.out_reg], (seed, passes)


def test_baby_and_giant_steps_go_out_together():
    import numpy as np

    lin = load_pkg().linear
    b = lin.Builder(4096, lambda limbs, steps: (("k", steps), steps), lambda values, limbs: None, [3] * 8)
    prog = lin.gemv_program(b, np.ones((256, 256)), 8)
    groups, rows = S.schedule(prog, 8, 2 * S._TOGETHER)
    sizes = [(code, len(items)) for code, _, items in groups]
    assert [c for c in sizes if c[0] == S.OP_ROTATE] == [(S.OP_ROTATE, 15)] * 2
    assert [c for c in sizes if c[0] in (S.OP_NTT, S.OP_INTT)] == [(S.OP_NTT, 16), (S.OP_INTT, 16)]
    assert not [c for c in sizes if c[0] == S.OP_COPY]


def test_merged_additions_give_the_same_sums():
    for seed in range(200):
        rng = random.Random(seed)
        rows = 6
        groups = []
        for i in range(rng.randint(1, 80)):
            a, b = rng.randrange(rows), rng.randrange(rows)
            out = a if rng.random() < 0.8 else rng.randrange(rows)
            code = S.OP_ADD if rng.random() < 0.9 else S.OP_SUB
            groups.append((code, 9 - (rng.random() < 0.05), [(out, [a, b], (code, out, a, b, None, 0, None))]))
        merged = S.merge_sums(groups)
        plain, fused = [1 << (8 * i) for i in range(rows)], [1 << (8 * i) for i in range(rows)]
        for regs, gs in ((plain, groups), (fused, merged)):
            for code, _, [(out, ins, _)] in gs:
                assert len(ins) <= 64
                regs[out] = sum(regs[i] for i in ins) if code == S.OP_ADD else regs[ins[0]] - regs[ins[1]]
        assert plain == fused
    chain = [(S.OP_ADD, 8, [(1, [1, r], None)]) for r in range(2, 17)]
    assert S.merge_sums(chain) == [(S.OP_ADD, 8, [(1, [1] + list(range(2, 17)), None)])]


def _outlive(prog, groups, rows):
    """Runs both orders twice; the registers that outlive a run hold the same."""
    n = prog.n_regs
    written, carried = set(), {prog.out_reg}
    for op in prog.ops:
        carried.update(r for r in _reads(op) if r not in written)
        written.add(op[1])
    regs = [("in", r) for r in range(n)]
    phys = regs + [None] * (rows - n)
    for _ in range(2):
        for op in prog.ops:
            ins = [regs[r] for r in _reads(op)]
            regs[op[1]] = ins[0] if op[0] == S.OP_COPY else _apply(op[0], ins, op)
        for code, _, items in groups:
            new = [phys[ins[0]] if code == S.OP_COPY else _apply(code, [phys[i] for i in ins], op)
                   for _, ins, op in items]
            for (o, _, _), v in zip(items, new):
                phys[o] = v
        assert [phys[r] for r in sorted(carried)] == [regs[r] for r in sorted(carried)]


@pytest.mark.parametrize("n_regs,n_inputs,out_reg,ops", [
    # values left in each other's rows and in both rows past the registers
    (3, 2, 2, [(S.OP_COPY, 2, 0, 0, None, 0, None), (S.OP_ROTATE, 1, 1, 0, None, 1, None),
               (S.OP_NTT, 0, 2, 0, None, 2, None)]),
    (4, 4, 1, [(S.OP_MAC_PLAIN, 3, 3, 1, None, 0, None), (S.OP_MUL_PLAIN, 0, 0, 0, None, 1, None),
               (S.OP_NTT, 1, 0, 0, None, 2, None), (S.OP_ROTATE, 0, 1, 0, None, 3, None),
               (S.OP_RESCALE, 0, 2, 0, None, 4, None)]),
])
def test_final_moves_without_a_spare_row(n_regs, n_inputs, out_reg, ops):
    prog = S.Program(n_regs=n_regs, out_reg=out_reg, n_inputs=n_inputs, ops=list(ops))
    groups, rows = S.schedule(prog, 9, 0)
    assert rows <= n_regs + 2
    _outlive(prog, groups, rows)


def test_every_register_that_outlives_a_run_is_in_its_row():
    for seed in range(4000):
        rng = random.Random(seed)
        n_regs, spare = rng.choice([1, 2, 3, 4, 5, 8]), rng.choice([0, 0, 0, 1, 2, 16])
        prog = _program(rng, n_regs, rng.randint(0, 40))
        groups, rows = S.schedule(prog, 9, spare)
        assert rows <= n_regs + 2 + spare
        _outlive(prog, groups, rows)
