"""The fused key switch within a chunk (ckks_set_ntt_chunk_bytes): the same
residues by pieces of a batch, and no more inter-pass memory than the chunk."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_residues

pytestmark = pytest.mark.gpu


def _key(pkg, ctx, rng, kind, n, L):
    q, p = pkg.chain_moduli(L - 1, 2)
    if kind == "bounded":
        m = pkg.find_ntt_primes(55, 1 << 16, L + 1)
        plan = pkg.PreparedRnsNttPlan(ctx, m, n)
        d = pkg.bounded_digit_count(plan, L, 30)
        return pkg.BoundedKeySwitchKey(plan, L, 30, rand_residues(rng, m, n, d), rand_residues(rng, m, n, d)), m[:L], d * (L + 1)
    if kind == "gadget":
        plan = pkg.PreparedRnsNttPlan(ctx, q, n)
        return pkg.RnsKeySwitchKey(plan, [1] * L, rand_residues(rng, q, n, L), rand_residues(rng, q, n, L)), q, L * L
    plan = pkg.PreparedRnsNttPlan(ctx, q + p, n)
    return (pkg.HybridKeySwitchKey(plan, L, [L - L // 2, L // 2], rand_residues(rng, q + p, n, 2),
                                   rand_residues(rng, q + p, n, 2)), q, 2 * (L + 2))


@pytest.mark.parametrize("cts", [0.5, 1, 2.5, 4, 100])  # ciphertexts whose digits a chunk holds
def test_chunked_key_switches_give_the_same_residues(pkg, ctx, cts):
    import torch

    n, L = 1 << 13, 4
    rng = np.random.default_rng(2)
    entries = []
    for kind, count in (("hybrid", 5), ("gadget", 3), ("bounded", 6), ("hybrid", 1)):
        key, q, limbs = _key(pkg, ctx, rng, kind, n, L)
        ct = pkg.to_device(rand_residues(rng, q, n, 2 * count).reshape(count, 2, L, n))
        entries.append((key, ct, limbs * n * 8))
    exps = [5, 25, 2 * n - 1, 3]
    want = [k.apply_galois(ct, e) for (k, ct, _), e in zip(entries, exps)]
    switched = [k.switch(ct) for k, ct, _ in entries]
    digits = entries[2][0].digits(entries[2][1])
    try:
        for (key, ct, per), e, w, s in zip(entries, exps, want, switched):
            ctx.set_ntt_chunk_bytes(int(cts * per))
            assert torch.equal(key.apply_galois(ct, e), w)
            again = ct.clone()
            assert torch.equal(key.switch(again, out=again), s)  # in place
        ctx.set_ntt_chunk_bytes(int(cts * entries[2][2]))
        assert torch.equal(entries[2][0].apply_galois_hoisted(entries[2][1], exps[2], digits), want[2])
        ctx.set_ntt_chunk_bytes(int(cts * max(per for _, _, per in entries)))
        outs = [torch.empty_like(ct) for _, ct, _ in entries]
        pkg.apply_galois_batch(ctx, [(k, e, ct, o) for (k, ct, _), e, o in zip(entries, exps, outs)])
        assert all(torch.equal(o, w) for o, w in zip(outs, want))
    finally:
        ctx.set_ntt_chunk_bytes(0)


@pytest.mark.parametrize("batch", [False, True])
def test_a_chunk_bounds_the_inter_pass_buffer(pkg, batch):
    import torch

    n, L, count = 1 << 14, 6, 64
    grown = []
    for chunk in (0, 4):
        c = pkg.Context(0)
        rng = np.random.default_rng(3)
        key, q, limbs = _key(pkg, c, rng, "hybrid", n, L)
        per = limbs * n * 8
        ct = pkg.to_device(rand_residues(rng, q, n, 2 * count).reshape(count, 2, L, n))
        out = torch.empty_like(ct)
        c.set_ntt_chunk_bytes(chunk * per)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        if batch:
            pkg.apply_galois_batch(c, [(key, 5, ct[:40], out[:40]), (key, 25, ct[40:], out[40:])])
        else:
            key.apply_galois(ct, 5, out=out)
        torch.cuda.synchronize()
        grown.append(before - torch.cuda.mem_get_info()[0])
        c.close()
    whole, four = count * per, 4 * per
    assert grown[0] - grown[1] > 0.9 * (whole - four), grown
