"""Paths through the fused row and column passes against the separate
transforms and pointwise kernels: whole residues, so equality."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rand_residues

pytestmark = pytest.mark.gpu

# FP64 limbs (up to 41 bits) beside integer limbs (up to 60), and a limb above
# 2^60 that keeps a plan on the separate passes
MIXES = {"fp": [40, 30, 41], "int": [60, 42], "both": [60, 40, 55, 36, 41], "wide": [61, 40]}


def _moduli(pkg, n, bits):
    out = []
    for b in bits:
        out += pkg.find_ntt_primes(b, n, 1, skip=out)
    return out


def _extremes(rng, moduli, n, polys):
    x = rand_residues(rng, moduli, n, polys)
    x[0, :, : n // 2] = np.array(moduli, dtype=np.uint64)[:, None] - 1
    x[-1, :, n // 2:] = 0
    return x


def _mul(pkg, plan, x, y_ntt):
    """x [p][limbs][N] times y_ntt (the same shape, NTT domain), separate passes."""
    t = pkg.empty(tuple(x.shape))
    plan.forward(x, t)
    plan.pointwise_mul(t, y_ntt, t)
    plan.inverse(t)
    return t


@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_products_match_separate_passes(pkg, ctx, logn, mix):
    import torch

    n, bits = 1 << logn, MIXES[mix]
    moduli = _moduli(pkg, n, bits)
    L, n_cts = len(moduli), 3
    rng = np.random.default_rng(logn * 10 + L)
    plan = pkg.PreparedRnsNttPlan(ctx, moduli, n)
    ct = pkg.to_device(_extremes(rng, moduli, n, 2 * n_cts))
    other = pkg.to_device(_extremes(rng, moduli, n, 2 * n_cts))
    pt = pkg.to_device(_extremes(rng, moduli, n, n_cts))

    # plaintext products: one plaintext for all ciphertexts, one per ciphertext
    c4 = ct.reshape(n_cts, 2, L, n)
    for per_ct in (False, True):
        w = pt if per_ct else pt[:1]
        y = w.reshape(-1, 1, L, n).expand(n_cts, 2, L, n).contiguous().reshape(2 * n_cts, L, n)
        want = _mul(pkg, plan, ct, y)
        got = plan.multiply_plain(c4, w.contiguous(), L)
        assert torch.equal(got.reshape(2 * n_cts, L, n), want), f"plain {per_ct}"
    inplace = c4.clone()
    assert torch.equal(plan.multiply_plain(inplace, pt[:1].contiguous(), L, out=inplace),
                       plan.multiply_plain(c4, pt[:1].contiguous(), L))

    # tensor
    o4 = other.reshape(n_cts, 2, L, n)
    f, g = pkg.empty(tuple(ct.shape)), pkg.empty(tuple(ct.shape))
    plan.forward(ct, f)
    plan.forward(other, g)
    f, g = f.reshape(n_cts, 2, L, n), g.reshape(n_cts, 2, L, n)
    parts = []
    for pairs in (((0, 0),), ((0, 1), (1, 0)), ((1, 1),)):
        acc = None
        for i, j in pairs:
            t = pkg.empty((n_cts, L, n))
            plan.pointwise_mul(f[:, i].contiguous(), g[:, j].contiguous(), t)
            if acc is None:
                acc = t
            else:
                plan.add(acc, t, acc)
        plan.inverse(acc)
        parts.append(acc)
    got = plan.tensor(c4, o4, L)
    for k in range(3):
        assert torch.equal(got[:, k], parts[k]), f"tensor part {k}"

    # encryption and decryption; errors at the ends of int64, secret at int8's
    s = rng.integers(-1, 2, n).astype(np.int8)
    s[:4] = [127, -128, 1, -1]
    e = rng.integers(-(1 << 63), (1 << 63) - 1, (2 * n_cts, n))
    e[0, :4] = [-(1 << 63), (1 << 63) - 1, 0, -1]
    e[-1] = rng.integers(-40, 41, n)
    q = np.array(moduli, dtype=object)[:, None]
    sr = np.array(s.astype(object)[None] % q, dtype=np.uint64)
    er = np.stack([np.array(x.astype(object)[None] % q, dtype=np.uint64) for x in e])
    ds = pkg.to_device(sr)
    plan.forward(ds.reshape(1, L, n), ds.reshape(1, L, n))
    s_ntt = ds.reshape(1, L, n).expand(2 * n_cts, L, n).contiguous()
    as_ = _mul(pkg, plan, other, s_ntt)
    sec = torch.from_numpy(s).cuda()
    b = plan.encrypt_raw(ct, torch.from_numpy(e).cuda(), sec, other)
    want = pkg.empty(tuple(ct.shape))
    plan.add(ct, pkg.to_device(er), want)
    plan.sub(want, as_, want)
    assert torch.equal(b, want), "encrypt"
    got = plan.decrypt_raw(ct, other, sec)
    plan.add(ct, as_, want)
    assert torch.equal(got, want), "decrypt"
    one = plan.decrypt_raw(ct[:1].contiguous(), other[:1].contiguous(), sec, out=ct[:1].clone())
    assert torch.equal(one, want[:1]), "decrypt one"


@pytest.mark.parametrize("with_b", [False, True])
@pytest.mark.parametrize("mix", ["fp", "both"])
@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_hoisted_rotations_match_rotations(pkg, ctx, logn, mix, with_b):
    """sigma_k of the sums inside a tile, for conjugation and exponents of both
    halves, against the rotation that permutes its input instead."""
    import torch

    n, bits = 1 << logn, MIXES[mix]
    q = _moduli(pkg, n, bits)
    qp = q + pkg.find_ntt_primes(59, n, 2, skip=q)
    L = len(q)
    blocks = [L - L // 2, L // 2]
    rng = np.random.default_rng(logn * 10 + L)
    plan = pkg.PreparedRnsNttPlan(ctx, qp, n)
    keys = [pkg.HybridKeySwitchKey(plan, L, blocks, rand_residues(rng, qp, n, 2), rand_residues(rng, qp, n, 2))
            for _ in range(2)]
    ct = rand_residues(rng, q, n, 6).reshape(3, 2, L, n)
    ct[1, 1, :, 1:3] = np.array(q, dtype=np.uint64)[:, None] - 1
    ct = pkg.to_device(ct)
    hoisted = keys[0].hoist(ct, with_b=with_b)
    exps = [(0, 5), (1, 2 * n - 1), (0, n + 1), (1, 2 * n - 5)]
    outs = [pkg.empty(tuple(ct.shape)) for _ in exps]
    pkg.rotate_hoisted_batch(ctx, [(hoisted, keys[i], e, ct, o) for (i, e), o in zip(exps, outs)])
    for (i, e), o in zip(exps, outs):
        want = keys[i].apply_galois(ct, e)
        assert torch.equal(o, want), f"batch exponent {e}"
        assert torch.equal(keys[i].rotate_hoisted(hoisted, ct, e), want), f"exponent {e}"


def test_key_switch_batches_of_one_shape_share_launches(pkg, ctx):
    """Interleaved keys of three shapes (one with single-limb blocks, one at
    another level), uneven ciphertext counts, the most entries a call takes."""
    import torch

    n = 1 << 13
    q = _moduli(pkg, n, [60, 40, 41, 36])
    qp = q + pkg.find_ntt_primes(59, n, 2, skip=q)
    rng = np.random.default_rng(5)
    plan = pkg.PreparedRnsNttPlan(ctx, qp, n)
    low = pkg.PreparedRnsNttPlan(ctx, q[:3] + qp[4:], n)
    shapes = [(plan, 4, [2, 2]), (plan, 4, [1, 1, 1, 1]), (low, 3, [2, 1])]
    entries = []
    for i in range(16):
        p, L, blocks = shapes[i % 3]
        mods = qp if p is plan else q[:3] + qp[4:]
        key = pkg.HybridKeySwitchKey(p, L, blocks, rand_residues(rng, mods, n, len(blocks)),
                                     rand_residues(rng, mods, n, len(blocks)))
        m = 1 + i % 4
        ct = pkg.to_device(rand_residues(rng, mods[:L], n, 2 * m).reshape(m, 2, L, n))
        entries.append((key, 2 * n - 1 if i == 7 else 5 ** i % (2 * n), ct, pkg.empty(tuple(ct.shape))))
    pkg.apply_galois_batch(ctx, entries)
    for i, (key, e, ct, out) in enumerate(entries):
        assert torch.equal(out, key.apply_galois(ct, e)), f"entry {i}"


@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("logn", [10, 11, 12, 13])
def test_key_switches_match_separate_kernels(pkg, ctx, logn, mix):
    """Digits read by the transforms, products formed between them: single-limb
    and larger blocks, hybrid, gadget and bounded keys, conjugation, extremes."""
    import torch

    n, bits = 1 << logn, MIXES[mix]
    q = _moduli(pkg, n, bits)
    qp = q + pkg.find_ntt_primes(60, n, 1, skip=q)
    L = len(q)
    rng = np.random.default_rng(logn * 10 + L)
    plan, q_plan = pkg.PreparedRnsNttPlan(ctx, qp, n), pkg.PreparedRnsNttPlan(ctx, q, n)
    ct = rand_residues(rng, q, n, 6).reshape(3, 2, L, n)
    ct[0, 1, :, : n // 2] = np.array(q, dtype=np.uint64)[:, None] - 1
    ct[1, 1, :, n // 2:] = 0
    ct = pkg.to_device(ct)

    def material(mods, entries):
        return rand_residues(rng, mods, n, entries), rand_residues(rng, mods, n, entries)

    keys = [pkg.HybridKeySwitchKey(plan, L, [1] * L, *material(qp, L)),
            pkg.HybridKeySwitchKey(plan, L, [L - L // 2, L // 2], *material(qp, 2)),
            pkg.RnsKeySwitchKey(q_plan, [1] * L, *material(q, L))]
    for base_log in (7, 31, 61):
        d = pkg.bounded_digit_count(plan, L, base_log)
        keys.append(pkg.BoundedKeySwitchKey(plan, L, base_log, *material(qp, d)))
    for k, key in enumerate(keys):
        for e in (5, 2 * n - 1, n + 1):
            ctx.set_key_switch_fusion(ctx.KS_FUSION_OFF)
            try:
                want = key.apply_galois(ct, e)
            finally:
                ctx.set_key_switch_fusion(ctx.KS_FUSION_AUTO)
            assert torch.equal(key.apply_galois(ct, e), want), f"key {k} exponent {e}"
            one = ct[2:].contiguous()
            assert torch.equal(key.apply_galois(one, e), want[2:]), f"key {k} exponent {e}, one ciphertext"


@pytest.mark.parametrize("bits", [[40, 41], [60, 55]])
@pytest.mark.parametrize("logn", [13, 14, 15, 16, 17])
def test_launches_of_few_tiles(pkg, ctx, logn, bits):
    """One ciphertext over few limbs: halved row tiles, column tiles of 512
    threads, divided ModDown and rescale loops, against larger launches of the
    same ciphertext repeated (whole tiles) and against the separate kernels."""
    import torch

    n = 1 << logn
    q = _moduli(pkg, n, bits)
    qp = q + pkg.find_ntt_primes(59, n, 1, skip=q)
    rng = np.random.default_rng(logn)
    plan = pkg.PreparedRnsNttPlan(ctx, qp, n)
    key = pkg.HybridKeySwitchKey(plan, 2, [2], rand_residues(rng, qp, n, 1), rand_residues(rng, qp, n, 1))
    ct = pkg.to_device(_extremes(rng, q, n, 2).reshape(1, 2, 2, n))
    many = ct.expand(64 if logn < 16 else 8, 2, 2, n).contiguous()
    for e in (5, 2 * n - 1):
        one = key.apply_galois(ct, e)
        assert torch.equal(one[0], key.apply_galois(many, e)[-1]), "rotation"
        assert torch.equal(key.rotate_hoisted(key.hoist(ct), ct, e), one), "hoisted rotation"
        ctx.set_key_switch_fusion(ctx.KS_FUSION_OFF)
        try:
            assert torch.equal(key.apply_galois(ct, e), one), "separate kernels"
        finally:
            ctx.set_key_switch_fusion(ctx.KS_FUSION_AUTO)
    assert torch.equal(plan.tensor(ct, ct, 2)[0], plan.tensor(many, many, 2)[-1]), "tensor"
    assert torch.equal(key.multiply_relinearize_rescale(ct, ct)[0], key.multiply_relinearize_rescale(many, many)[-1])


@pytest.mark.parametrize("mix", ["both", "wide"])
@pytest.mark.parametrize("logn,count,n_outs", [(10, 1, 1), (10, 64, 6), (12, 5, 3), (13, 16, 16), (13, 9, 17), (14, 8, 4)])
def test_shared_inner_sums(pkg, ctx, mix, logn, count, n_outs):
    """Several sums of the same ciphertexts in one call, edges of the groups of
    eight and of a launch's operands, against products and additions."""
    import ctypes as C
    import torch

    n = 1 << logn
    q = _moduli(pkg, n, MIXES[mix])
    L = len(q)
    rng = np.random.default_rng(count * 100 + n_outs)
    plan = pkg.PreparedRnsNttPlan(ctx, q, n)
    cts = [pkg.to_device(_extremes(rng, q, n, 2)) for _ in range(count)]
    pts = [[pkg.to_device(_extremes(rng, q, n, 1)) for _ in range(count)] for _ in range(n_outs)]
    outs = [pkg.empty((2, L, n)) for _ in range(n_outs)]

    def array(ts):
        return (C.c_uint64 * len(ts))(*[t.data_ptr() for t in ts])

    ca, pa, oa = array(cts), array([p for row in pts for p in row]), array(outs)
    rc = pkg.lib().ckks_multiply_plain_accumulate_ntt_batch(plan.handle, C.cast(ca, C.c_void_p), C.cast(pa, C.c_void_p),
                                                            count, C.cast(oa, C.c_void_p), n_outs, L)
    assert rc == 0
    for e in range(n_outs):
        want = torch.zeros((2, L, n), dtype=torch.int64, device="cuda")
        for ct, pt in zip(cts, pts[e]):
            prod = pkg.empty((2, L, n))
            plan.pointwise_mul(ct, pt.expand(2, L, n).contiguous(), prod)
            plan.add(want, prod, want)
        assert torch.equal(outs[e], want), f"sum {e}"


@pytest.mark.parametrize("logn,polys,scale", [(10, 1, 2.0 ** 40), (12, 3, 2.0 ** 55), (13, 2, 1.0), (15, 8, 2.0 ** 40),
                                              (16, 2, 3.7e11)])
def test_embedding_passes_match_torch(pkg, ctx, logn, polys, scale):
    """The scatter, twist and rounding inside the library's kernels give the
    values of the same passes as torch operations, bit for bit."""
    import torch

    n = 1 << logn
    q = _moduli(pkg, n, [60, 40, 41])
    plan, emb = pkg.PreparedRnsNttPlan(ctx, q, n), pkg.encoding.CanonicalEmbedding(n)
    gen = torch.Generator(device="cuda").manual_seed(logn)
    z = torch.randn((polys, n // 2), dtype=torch.complex128, device="cuda", generator=gen)
    for slots in (z, z.conj(), z.real, z[0], torch.zeros_like(z), z.to(torch.complex64).cpu()):
        got = pkg.encoding.encode(plan, emb, slots, scale)
        c = emb.slots_to_coefficients(torch.as_tensor(slots).cuda()).reshape(-1, n)
        want = pkg.empty((c.shape[0], 3, n))
        pkg._check(pkg.lib().ckks_encode_coefficients(plan.handle, pkg._ptr(c, dtype="float64"), scale, pkg._ptr(want),
                                                      c.shape[0], 3))
        assert torch.equal(got.reshape(want.shape), want)
    with pytest.raises(pkg.CkksError):
        pkg.encoding.encode(plan, emb, z, 2.0 ** 70)
    assert torch.equal(pkg.encoding.encode(plan, emb, z, scale).reshape(-1), pkg.encoding.encode(plan, emb, z, scale).reshape(-1))
    x = pkg.to_device(_extremes(np.random.default_rng(logn), q, n, polys))
    want = emb.coefficients_to_slots(pkg.encoding.decode_coefficients(plan, x, scale))
    assert torch.equal(pkg.encoding.decode(plan, emb, x, scale), want)


@pytest.mark.parametrize("logn,count,polys", [(10, 1, 1), (12, 2, 3), (13, 16, 2), (11, 64, 1)])
def test_sums_of_many_match_additions(pkg, ctx, logn, count, polys):
    import ctypes as C
    import torch

    n = 1 << logn
    q = _moduli(pkg, n, MIXES["wide"])
    rng = np.random.default_rng(count)
    plan = pkg.PreparedRnsNttPlan(ctx, q, n)
    xs = [pkg.to_device(_extremes(rng, q, n, polys)) for _ in range(count)]
    want = xs[0].clone()
    for x in xs[1:]:
        plan.add(want, x, want)
    arr = (C.c_uint64 * count)(*[x.data_ptr() for x in xs])
    for out in (pkg.empty(tuple(want.shape)), xs[-1]):
        assert pkg.lib().ckks_poly_sum(plan.handle, C.cast(arr, C.c_void_p), count, C.c_void_p(out.data_ptr()), polys,
                                       len(q), len(q) * n) == 0
        assert torch.equal(out, want)


def test_a_tensor_keeps_only_its_factors(pkg):
    """The products take the place of the factors: four polynomials a pair in
    workspaces, no second buffer."""
    import torch

    n, cts = 1 << 14, 64
    c = pkg.Context(0)
    q, _ = pkg.chain_moduli(7, 0)
    plan = pkg.PreparedRnsNttPlan(c, q, n)
    poly = len(q) * n * 8
    ct = torch.zeros((cts, 2, len(q), n), dtype=torch.int64, device="cuda")
    out = torch.empty((cts, 3, len(q), n), dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    plan.tensor(ct, ct, len(q), out=out)
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    c.close()
    assert grown < 5 * cts * poly, grown
