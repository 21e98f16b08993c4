"""Key switches and hoisted rotations on both sides of the route rules: the
same residues by the separate kernels, the fused ones in either order and the
ones an untuned key takes."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import O, P60, Q0, rand_residues

pytestmark = pytest.mark.gpu


def _by_mode(ctx, call):
    """{mode: residues}, the context left as it was."""
    out = {}
    try:
        for mode in (ctx.KS_FUSION_OFF, ctx.KS_FUSION_XCD, ctx.KS_FUSION_LINEAR, ctx.KS_FUSION_AUTO):
            ctx.set_key_switch_fusion(mode)
            out[mode] = call()
    finally:
        ctx.set_key_switch_fusion(ctx.KS_FUSION_AUTO)
    return out


@pytest.mark.parametrize("logn,kind,limbs,base_log,cts", [
    (13, "bounded", 2, 10, 1),   # 11 digits, few tiles: separate
    (13, "bounded", 2, 10, 4),   # fused
    (15, "bounded", 2, 8, 2),    # 14 digits
    (14, "gadget", 6, 0, 1),
    (16, "gadget", 5, 0, 1),
    (17, "gadget", 5, 0, 1),     # rotations of a row of 512
    (17, "gadget", 2, 0, 1),     # whole tiles where half ones were taken
])
def test_routes_agree(pkg, ctx, logn, kind, limbs, base_log, cts):
    import torch

    n = 1 << logn
    rng = np.random.default_rng(logn * 100 + limbs)
    if kind == "bounded":
        m = pkg.find_ntt_primes(55, n, limbs + 1)
        q = m[:limbs]
        plan = pkg.PreparedRnsNttPlan(ctx, m, n)
        d = pkg.bounded_digit_count(plan, limbs, base_log)
        make = lambda: pkg.BoundedKeySwitchKey(plan, limbs, base_log, rand_residues(rng, m, n, d),
                                               rand_residues(rng, m, n, d))
    else:
        q = pkg.find_ntt_primes(60, n, 1) + pkg.find_ntt_primes(40, n, limbs - 1)
        plan = pkg.PreparedRnsNttPlan(ctx, q, n)
        make = lambda: pkg.RnsKeySwitchKey(plan, [1] * limbs, rand_residues(rng, q, n, limbs),
                                           rand_residues(rng, q, n, limbs))
    keys = [make() for _ in range(2)]
    exps = [pow(5, i + 1, 2 * n) for i in range(5)]
    batches = [pkg.to_device(rand_residues(rng, q, n, 2 * cts).reshape(cts, 2, limbs, n)) for _ in range(2)]
    digits = [keys[0].hoist(ct) for ct in batches]

    def rotations():
        outs = [torch.empty_like(batches[0]) for _ in range(7)]
        # five exponents of one batch, two of another
        entries = [(digits[i // 5], keys[i % 2], exps[i % 5], batches[i // 5], o) for i, o in enumerate(outs)]
        pkg.rotate_hoisted_batch(ctx, entries)
        single = keys[0].rotate_hoisted(digits[0], batches[0], exps[0])
        return torch.stack(outs + [single])

    def switches():
        return torch.stack([keys[i % 2].apply_galois(batches[i // 5], exps[i % 5]) for i in range(7)]
                           + [keys[0].apply_galois(batches[0], exps[0])])

    want = switches()
    for call in (switches, rotations):
        for mode, got in _by_mode(ctx, call).items():
            assert torch.equal(got, want), (call.__name__, mode)


def test_entries_of_one_batch_on_both_routes(pkg, ctx):
    """Entries counted together where they share launches: one alone of its kind
    on the separate kernels beside fused ones."""
    import torch

    n, m = 1 << 13, pkg.find_ntt_primes(55, 1 << 13, 3)
    rng = np.random.default_rng(4)
    plan = pkg.PreparedRnsNttPlan(ctx, m, n)
    keys = []
    for base_log in (10, 10, 10, 8, 30):
        d = pkg.bounded_digit_count(plan, 2, base_log)
        keys.append(pkg.BoundedKeySwitchKey(plan, 2, base_log, rand_residues(rng, m, n, d), rand_residues(rng, m, n, d)))
    cts = [pkg.to_device(rand_residues(rng, m[:2], n, 2 * c).reshape(c, 2, 2, n)) for c in (1, 1, 2, 1, 1)]
    exps = [5, 25, 125, 625, 3125]
    want = [k.apply_galois(ct, e) for k, ct, e in zip(keys, cts, exps)]

    def batch():
        outs = [torch.empty_like(ct) for ct in cts]
        pkg.apply_galois_batch(ctx, [(k, e, ct, o) for k, e, ct, o in zip(keys, exps, cts, outs)])
        return outs

    for mode, got in _by_mode(ctx, batch).items():
        assert all(torch.equal(g, w) for g, w in zip(got, want)), mode


def test_moddown_of_large_jobs_in_launches_of_their_own(pkg, ctx):
    import torch

    n, L = 1 << 16, 2
    q, p = pkg.chain_moduli(L - 1, 1)
    rng = np.random.default_rng(9)
    plan = pkg.PreparedRnsNttPlan(ctx, q + p, n)
    key = pkg.HybridKeySwitchKey(plan, L, [1, 1], rand_residues(rng, q + p, n, 2), rand_residues(rng, q + p, n, 2))
    ct = pkg.to_device(rand_residues(rng, q, n, 32).reshape(16, 2, L, n))
    exps = [5, 25, 125]
    want = [key.apply_galois(ct, e) for e in exps]
    h = key.hoist(ct)
    for batch in (lambda outs: pkg.rotate_hoisted_batch(ctx, [(h, key, e, ct, o) for e, o in zip(exps, outs)]),
                  lambda outs: pkg.apply_galois_batch(ctx, [(key, e, ct, o) for e, o in zip(exps, outs)])):
        outs = [torch.empty_like(ct) for _ in exps]
        batch(outs)
        assert all(torch.equal(o, w) for o, w in zip(outs, want))


@pytest.mark.parametrize("case", ["blocks_of_12", "basis_over_64"])
def test_large_blocks_and_bases_match_oracle(pkg, ctx, case):
    """Blocks of 10 to 12 limbs (13 terms where the first prime is split) and a
    basis past the limb order's 64, by the fused passes."""
    n = 1 << 13
    blocks = [12, 11, 10] if case == "blocks_of_12" else [12] * 5 + [6]
    L, K = sum(blocks), 8 if case == "blocks_of_12" else 4
    q = Q0 + O.ntt_primes(40, n, L - 1)
    qp = q + P60[:K] if K <= len(P60) else q + P60 + O.ntt_primes(59, 65536, K - len(P60))
    assert len(qp) == L + K == len(set(qp))
    rng = np.random.default_rng(L)
    kb, ka = rand_residues(rng, qp, n, len(blocks)), rand_residues(rng, qp, n, len(blocks))
    key = pkg.HybridKeySwitchKey(pkg.PreparedRnsNttPlan(ctx, qp, n), L, blocks, kb, ka)
    ct = rand_residues(rng, q, n, 2).reshape(1, 2, L, n)
    ct[0, 1, :, :64] = np.array(q, dtype=np.uint64)[:, None] - 1
    ct[0, 1, :, 64:128] = np.array(q, dtype=np.uint64)[:, None] // 2
    want = np.stack(O.hybrid_key_switch(O.RnsPlan(qp, n), L, blocks, ct[0, 0], ct[0, 1], kb, ka))
    x = pkg.to_device(ct)
    for mode, got in _by_mode(ctx, lambda: pkg.to_host(key.switch(x))).items():
        assert (got[0] == want).all(), mode
