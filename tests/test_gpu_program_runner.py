"""ProgramRunner on the GPU: a program changed between runs, against a runner
built for the changed program."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_residues

pytestmark = pytest.mark.gpu


def test_a_program_changed_between_runs(pkg, ctx):
    S = pkg.serving
    n, L = 1 << 12, 3
    q, p = pkg.chain_moduli(L - 1, 1)
    plan, kplan = pkg.PreparedRnsNttPlan(ctx, q, n), pkg.PreparedRnsNttPlan(ctx, q + p, n)
    rng = np.random.default_rng(3)
    keys = [pkg.HybridKeySwitchKey(kplan, L, [1] * L, rand_residues(rng, q + p, n, L), rand_residues(rng, q + p, n, L))
            for _ in range(2)]
    pts = [pkg.to_device(rand_residues(rng, q, n)[0]) for _ in range(4)]
    prog = S.Program(n_regs=4, out_reg=0)
    prog.rotate(1, 0, keys[0], 5)
    prog.ntt(2, 0)
    prog.ntt(3, 1)
    prog.mac_plain(3, 2, pts[:2])
    prog.intt(3, 3)
    prog.mul_plain(2, 1, pts[2])
    prog.add(0, 3, 2)
    x = pkg.to_device(rand_residues(rng, q, n, 2)[None])
    runner = S.ProgramRunner(plan, L, prog)

    def same():
        got = pkg.to_host(runner.run(x).contiguous())
        want = pkg.to_host(S.ProgramRunner(plan, L, prog).run(x).contiguous())
        assert (got == want).all()
        return got

    seen = [same()]
    changes = [lambda: prog.ops.__setitem__(0, prog.ops[0][:5] + (25, None)),
               lambda: prog.ops.__setitem__(0, prog.ops[0][:4] + (keys[1],) + prog.ops[0][5:]),
               lambda: prog.ops.__setitem__(5, prog.ops[5][:6] + (pts[3],)),
               lambda: prog.ops[3][6].__setitem__(1, pts[3]),
               lambda: prog.rescale(0, 0)]
    for change in changes:
        change()
        seen.append(same())
    for i, a in enumerate(seen):
        assert not any(a.shape == b.shape and (a == b).all() for b in seen[:i])
