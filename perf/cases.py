"""The calls whose speed matters to a user of this framework, as cases a
measuring program can prepare, run and check.

Every case goes through the package's public entry points on data that a
program has resident in HBM: one pass is what such a program does per request
or per batch.  Sizes follow the repository's own configurations (the small
pipeline at N = 2^12, the batched primitives at N = 2^16 and 2^15, the CCMM,
GEMV and FFT workloads at N = 2^13 .. 2^16, the bounded-digit rotation shape)
and, between them, generic ones.

Outputs are residues (whole numbers) everywhere except the decoded slots.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _pkg():
    """The package (its folder's name has a hyphen, so it is loaded by path)."""
    name = "ccmm_rs_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(_ROOT, "ccmm-rs_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # One ciphertext's transform in the smallest pipeline (N = 2^12, one
        # 60-bit and three 40-bit primes): a single-pass launch whose latency
        # is what a small program waits for.
        {"name": "ntt_forward_n4096_one_ct", "kind": "ntt", "forward": True, "logn": 12, "limbs": 4, "polys": 2,
         "chain": "mixed"},
        # The smallest rotation: one ciphertext, one special prime, one-limb
        # blocks; a chain of short launches.
        {"name": "rotate_hybrid_n4096_one_ct", "kind": "rotate", "key": "hybrid", "logn": 12, "limbs": 4, "dnum": 4,
         "n_cts": 1, "step": 1},
        # Ciphertext products of the encrypted matrix product (N = 2^13, nine
        # limbs, dnum 2), a few requests batched together.
        {"name": "multiply_relin_rescale_n8192", "kind": "multiply", "logn": 13, "limbs": 9, "dnum": 2, "n_cts": 4},
        # A whole encrypted-vector request: public 256 x 256 matrix times an
        # encrypted vector at N = 2^14, eight limbs (baby-step / giant-step
        # rotations of one ciphertext, NTT-resident inner sums).
        {"name": "gemv_256_n16384", "kind": "gemv", "logn": 14, "limbs": 8, "dim": 256, "dnum": 2},
        # Results leaving the server: raw decryption, exact CRT and the
        # embedding back to slots.
        {"name": "decrypt_decode_n16384", "kind": "decrypt", "logn": 14, "limbs": 8, "n_cts": 4},
        # Inputs entering it: slots encoded and encrypted.
        {"name": "encode_encrypt_n32768", "kind": "encrypt", "logn": 15, "limbs": 13, "n_cts": 8},
        # Plaintext products of a batch (masks, weights), each followed by
        # its rescale.
        {"name": "multiply_plain_rescale_n32768", "kind": "plain", "logn": 15, "limbs": 13, "n_cts": 16},
        # The reference's own rotation: RNS gadget of single limbs (25
        # digits), one ciphertext per call.
        {"name": "rotate_gadget_n65536_one_ct", "kind": "rotate", "key": "gadget", "logn": 16, "limbs": 25,
         "dnum": 25, "n_cts": 1, "step": 4},
        # The reference's bounded-digit rotation (13 + 2 primes of 55 bits,
        # 23 digits of 32 bits) over a small batch.
        {"name": "rotate_bounded_n65536", "kind": "rotate", "key": "bounded", "logn": 16, "limbs": 13, "dnum": 0,
         "n_cts": 8, "step": 8},
        # The inverse transform over a large batch of limbs (accumulators of
        # 32 ciphertexts over 32 key-basis limbs).
        {"name": "ntt_inverse_n65536_2048_limbs", "kind": "ntt", "forward": False, "logn": 16, "limbs": 32,
         "polys": 64, "chain": "mixed"},
        # A batch hoisted once and rotated by four exponents, as every
        # baby-step loop does.
        {"name": "rotate_hoisted_n65536", "kind": "hoisted", "logn": 16, "limbs": 25, "dnum": 3, "n_cts": 16,
         "exponents": 4},
        # The batched rotation the throughput figures are quoted on: 64
        # ciphertexts, 25 limbs, dnum 3.
        {"name": "rotate_hybrid_n65536_batch64", "kind": "rotate", "key": "hybrid", "logn": 16, "limbs": 25, "dnum": 3,
         "n_cts": 64, "step": 1},
    ]


# residues one pass of a drawn key switch may hold as digits: the largest
# listed case's
_MAX_DIGITS = 64 * 3 * 32 << 16


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ntt", "ntt", "rotate", "rotate", "rotate", "hoisted", "multiply", "gemv", "plain", "encrypt",
                       "decrypt"])
    if kind == "ntt":
        logn = rng.randint(10, 17)
        limbs = _log_int(rng, 1, 32)
        polys = _log_int(rng, 1, max(1, min(4096, (2048 << 16) // (limbs << logn))))
        return {"kind": kind, "forward": rng.random() < 0.5, "logn": logn, "limbs": limbs, "polys": polys,
                "chain": rng.choice(["mixed", "mixed", "wide"])}
    if kind == "gemv":
        return {"kind": kind, "logn": rng.randint(12, 15), "limbs": rng.randint(4, 10), "dim": rng.choice([32, 64, 128, 256]),
                "dnum": rng.randint(2, 3)}
    if kind in ("encrypt", "decrypt"):
        logn = rng.randint(12, 16)
        limbs = rng.randint(2, 24)
        return {"kind": kind, "logn": logn, "limbs": limbs,
                "n_cts": _log_int(rng, 1, max(1, min(128, (48 * 24 << 16) // (limbs << logn))))}
    if kind == "plain":
        logn = rng.randint(12, 16)
        limbs = rng.randint(2, 25)
        return {"kind": kind, "logn": logn, "limbs": limbs,
                "n_cts": _log_int(rng, 1, max(1, min(256, (32 * 25 << 16) // (limbs << logn))))}
    if kind == "rotate":
        key = rng.choice(["hybrid", "hybrid", "gadget", "bounded"])
        if key == "bounded":
            logn, limbs = rng.randint(12, 16), rng.randint(3, 13)
            digits, basis = (55 * limbs + 32) // 32, limbs + 2
            dnum = 0
        elif key == "gadget":
            logn, limbs = rng.randint(12, 16), rng.randint(3, 25)
            dnum = digits = limbs
            basis = limbs
        else:
            logn, limbs, dnum, digits, basis = _draw_hybrid(rng)
        most = max(1, min(64, _MAX_DIGITS // 2 // (digits * basis << logn)))
        return {"kind": kind, "key": key, "logn": logn, "limbs": limbs, "dnum": dnum, "n_cts": _log_int(rng, 1, most),
                "step": rng.choice([1, 2, 16, 256, 3, 37])}
    logn, limbs, dnum, digits, basis = _draw_hybrid(rng)
    exps = rng.randint(2, 7) if kind == "hoisted" else 1
    most = max(1, min(64, _MAX_DIGITS // 4 // (digits * basis * exps << logn)))
    case = {"kind": kind, "logn": logn, "limbs": limbs, "dnum": dnum, "n_cts": _log_int(rng, 1, most)}
    if kind == "hoisted":
        case["exponents"] = exps
    return case


def _draw_hybrid(rng):
    logn = rng.randint(12, 16)
    limbs = rng.randint(3, 25)
    low = max(1, -(-limbs // 9))
    dnum = rng.randint(low, max(low, min(limbs, 6)))
    return logn, limbs, dnum, dnum, limbs + _special_primes(limbs, dnum)


# ---------------------------------------------------------------- shapes

def _blocks(limbs, dnum):
    """dnum consecutive blocks, the longer ones first."""
    return [limbs // dnum + (1 if j < limbs % dnum else 0) for j in range(dnum)]


def _special_primes(limbs, dnum):
    """60-bit special primes whose product exceeds the largest block's (the
    first block holds the 60-bit base prime, the others 40-bit ones)."""
    b = _blocks(limbs, dnum)
    bits = max([60 + 40 * (b[0] - 1)] + [40 * n for n in b[1:]])
    return max(1, -(-bits // 60))


def _chain(pkg, limbs, special, degree):
    return pkg.chain_moduli(limbs - 1, special, max(degree, 1 << 16))


# ---------------------------------------------------------------- inputs

class _Inputs:
    """Seeded inputs drawn on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 1000003 + 17)

    def residues(self, lead, moduli, n):
        """Uniform canonical residues [*lead][limbs][n]."""
        out = torch.empty(tuple(lead) + (len(moduli), n), dtype=torch.int64, device="cuda")
        for i, q in enumerate(moduli):
            out[..., i, :] = torch.randint(0, int(q), tuple(lead) + (n,), generator=self.g, dtype=torch.int64,
                                           device="cuda")
        return out

    def normal(self, shape, sigma):
        return torch.randn(shape, generator=self.g, dtype=torch.float64, device="cuda") * sigma

    def uniform(self, shape):
        return torch.rand(shape, generator=self.g, dtype=torch.float64, device="cuda") * 2 - 1

    def ternary(self, n):
        return torch.randint(-1, 2, (n,), generator=self.g, device="cuda", dtype=torch.int64).to(torch.int8)


def _exponent(n, step):
    return pow(5, step % (n // 2), 2 * n)


def _hybrid(pkg, ctx, rnd, case, plan=None):
    """A dnum hybrid key of uniform NTT-domain entries over the case's chain."""
    n, limbs = 1 << case["logn"], case["limbs"]
    if plan is None:
        q, p = _chain(pkg, limbs, _special_primes(limbs, case["dnum"]), n)
        plan = pkg.PreparedRnsNttPlan(ctx, q + p, n)
    kb, ka = (rnd.residues((case["dnum"],), plan.moduli, n) for _ in range(2))
    return pkg.HybridKeySwitchKey(plan, limbs, _blocks(limbs, case["dnum"]), kb, ka)


_BOUNDED_BASE_LOG = 32
_SCALE = float(1 << 40)


def _messages(rnd, case):
    """Integer plaintext coefficients as decryption meets them (scale 2^40,
    slots of magnitude about one) and the encryption errors, on the GPU."""
    n, p = 1 << case["logn"], case["n_cts"]
    m = torch.round(rnd.normal((p, n), 1.0 / math.sqrt(n)) * _SCALE).to(torch.int64)
    e = torch.round(rnd.normal((p, n), 3.2)).to(torch.int64)
    return m, e


def prepare(case, seed):
    pkg = _pkg()
    rnd = _Inputs(seed)
    ctx = pkg.Context(0)
    n = 1 << case["logn"]
    kind = case["kind"]
    s = {"kind": kind, "ctx": ctx, "case": case}
    if kind == "ntt":
        if case["chain"] == "wide":
            moduli = pkg.find_ntt_primes(60, max(n, 1 << 16), case["limbs"])
        else:
            special = min(7, case["limbs"] // 4)  # the special primes' share of a key basis
            q, p = _chain(pkg, case["limbs"] - special, special, n)
            moduli = q + p
        s["plan"] = pkg.PreparedRnsNttPlan(ctx, moduli, n)
        s["x"] = rnd.residues((case["polys"],), moduli, n)
        s["out"] = torch.empty_like(s["x"])
    elif kind == "rotate":
        s["exponent"] = _exponent(n, case["step"])
        if case["key"] == "hybrid":
            s["key"] = _hybrid(pkg, ctx, rnd, case)
            q = s["key"].plan.moduli[:case["limbs"]]
        elif case["key"] == "gadget":
            q, _ = _chain(pkg, case["limbs"], 0, n)
            plan = pkg.PreparedRnsNttPlan(ctx, q, n)
            kb, ka = (rnd.residues((case["limbs"],), q, n) for _ in range(2))
            s["key"] = pkg.RnsKeySwitchKey(plan, [1] * case["limbs"], kb, ka)
        else:
            moduli = pkg.find_ntt_primes(55, 1 << 16, case["limbs"] + 2)
            q = moduli[:case["limbs"]]
            plan = pkg.PreparedRnsNttPlan(ctx, moduli, n)
            count = pkg.bounded_digit_count(plan, case["limbs"], _BOUNDED_BASE_LOG)
            kb, ka = (rnd.residues((count,), moduli, n) for _ in range(2))
            s["key"] = pkg.BoundedKeySwitchKey(plan, case["limbs"], _BOUNDED_BASE_LOG, kb, ka)
        s["ct"] = rnd.residues((case["n_cts"], 2), q, n)
        s["out"] = torch.empty_like(s["ct"])
    elif kind == "hoisted":
        first = _hybrid(pkg, ctx, rnd, case)
        s["keys"] = [first] + [_hybrid(pkg, ctx, rnd, case, first.plan) for _ in range(case["exponents"] - 1)]
        s["exps"] = [_exponent(n, 1 << i) for i in range(case["exponents"])]
        s["ct"] = rnd.residues((case["n_cts"], 2), first.plan.moduli[:case["limbs"]], n)
        s["outs"] = [torch.empty_like(s["ct"]) for _ in s["exps"]]
        # the digit buffers a program keeps; every pass cuts them anew
        s["digits"] = first.hoist(s["ct"], with_b=True)
    elif kind == "multiply":
        s["key"] = _hybrid(pkg, ctx, rnd, case)
        q = s["key"].plan.moduli[:case["limbs"]]
        s["ct0"], s["ct1"] = (rnd.residues((case["n_cts"], 2), q, n) for _ in range(2))
    elif kind == "gemv":
        _prepare_gemv(pkg, ctx, rnd, case, s)
    elif kind == "plain":
        q, _ = _chain(pkg, case["limbs"], 0, n)
        s["plan"] = pkg.PreparedRnsNttPlan(ctx, q, n)
        s["ct"] = rnd.residues((case["n_cts"], 2), q, n)
        s["pt"] = rnd.residues((case["n_cts"],), q, n)
    else:
        q, _ = _chain(pkg, case["limbs"], 0, n)
        s["plan"] = pkg.PreparedRnsNttPlan(ctx, q, n)
        s["emb"] = pkg.encoding.CanonicalEmbedding(n)
        m, e = _messages(rnd, case)
        s["secret"] = rnd.ternary(n)
        s["a"] = rnd.residues((case["n_cts"],), q, n)
        if kind == "encrypt":
            s["error"] = e
            s["slots"] = torch.complex(rnd.uniform((case["n_cts"], n // 2)), rnd.uniform((case["n_cts"], n // 2)))
        else:
            qs = torch.tensor(q, dtype=torch.int64, device="cuda")[None, :, None]
            residues = torch.remainder(m[:, None, :], qs).contiguous()
            s["b"] = s["plan"].encrypt_raw(residues, e, s["secret"], s["a"])
    return s


def _prepare_gemv(pkg, ctx, rnd, case, s):
    n, limbs, dnum = 1 << case["logn"], case["limbs"], min(case["dnum"], case["limbs"])
    special = _special_primes(limbs, dnum)
    q, p = _chain(pkg, limbs, special, n)
    plan = pkg.PreparedRnsNttPlan(ctx, q, n)
    key_plan = pkg.PreparedRnsNttPlan(ctx, q + p, n)
    emb = pkg.encoding.CanonicalEmbedding(n)
    keys = {}

    def key_for(at_limbs, steps):
        if steps not in keys:
            keys[steps] = _hybrid(pkg, ctx, rnd, dict(case, dnum=dnum), key_plan)
        return keys[steps], _exponent(n, steps)

    def encode(values, at_limbs):
        # diagonals at the scale of the level's last prime, NTT domain
        pt = pkg.encoding.encode(plan, emb, torch.from_numpy(np.asarray(values)), float(q[at_limbs - 1]), at_limbs)
        return plan.forward(pt, n_limbs=at_limbs)

    matrix = rnd.uniform((case["dim"], case["dim"])).cpu().numpy()
    builder = pkg.linear.Builder(n // 2, key_for, encode, q)
    s["runner"] = pkg.serving.ProgramRunner(plan, limbs, pkg.linear.gemv_program(builder, matrix, limbs))
    s["keys"], s["plan"] = keys, plan
    s["input"] = rnd.residues((1, 2), q, n)


# ---------------------------------------------------------------- one pass

def run(s):
    kind, pkg = s["kind"], _pkg()
    if kind == "ntt":
        go = s["plan"].forward if s["case"]["forward"] else s["plan"].inverse
        return go(s["x"], out=s["out"])
    if kind == "rotate":
        return s["key"].apply_galois(s["ct"], s["exponent"], out=s["out"])
    if kind == "hoisted":
        s["digits"].rehoist(s["keys"][0], s["ct"])
        pkg.rotate_hoisted_batch(s["ctx"], [(s["digits"], k, e, s["ct"], o)
                                            for k, e, o in zip(s["keys"], s["exps"], s["outs"])])
        return s["outs"]
    if kind == "multiply":
        return s["key"].multiply_relinearize_rescale(s["ct0"], s["ct1"])
    if kind == "gemv":
        return s["runner"].run(s["input"])
    plan, limbs = s["plan"], s["case"]["limbs"]
    if kind == "plain":
        return plan.rescale_to_next(plan.multiply_plain(s["ct"], s["pt"], limbs), limbs)
    if kind == "encrypt":
        m = pkg.encoding.encode(plan, s["emb"], s["slots"], _SCALE)
        return plan.encrypt_raw(m, s["error"], s["secret"], s["a"])
    return pkg.encoding.decode(plan, s["emb"], plan.decrypt_raw(s["b"], s["a"], s["secret"]), _SCALE)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: every input (ciphertexts, keys, plaintexts) read once, every
    output written once, 8 bytes a residue.  flops: residue arithmetic, one
    operation per modular product and per modular sum (a butterfly is
    three)."""
    n, limbs, kind = 1 << case["logn"], case["limbs"], case["kind"]
    fly = 3 * n // 2 * case["logn"]  # one limb transform
    if kind == "ntt":
        t = case["polys"] * limbs
        return {"bytes": 16 * n * t, "flops": fly * t}
    if kind in ("rotate", "hoisted", "multiply"):
        return _switch_work(case, n, limbs, fly)
    c = case.get("n_cts", 1)
    if kind == "gemv":
        dnum = min(case["dnum"], limbs)
        one = _switch_work({"kind": "rotate", "key": "hybrid", "logn": case["logn"], "limbs": limbs, "dnum": dnum,
                            "n_cts": 1}, n, limbs, fly)
        g = int(math.ceil(math.sqrt(case["dim"])))
        giants = -(-case["dim"] // g)
        rotations = g + giants - 2
        basis = limbs + _special_primes(limbs, dnum)
        keys = rotations * 2 * dnum * basis * n
        return {"bytes": 8 * (keys + case["dim"] * limbs * n + 2 * (2 * limbs - 1) * n),
                "flops": rotations * one["flops"] + 2 * limbs * ((g + giants) * fly + 2 * case["dim"] * n)}
    if kind == "plain":
        return {"bytes": 8 * n * c * (3 * limbs + 2 * (limbs - 1)), "flops": c * (4 * limbs * fly + 6 * limbs * n)}
    if kind == "encrypt":
        return {"bytes": 8 * n * (c * (1 + 1 + 2 * limbs)) + n, "flops": c * limbs * (2 * fly + 3 * n)}
    # decrypt: the slots are N/2 complex doubles
    return {"bytes": 8 * n * (c * (2 * limbs + 1)) + n, "flops": c * (limbs * (2 * fly + 2 * n) + limbs * limbs * n)}


def _switch_work(case, n, limbs, fly):
    key = case.get("key", "hybrid")
    if key == "bounded":
        digits, basis, special = (55 * limbs + 1 + _BOUNDED_BASE_LOG - 1) // _BOUNDED_BASE_LOG, limbs + 2, 2
    elif key == "gadget":
        digits, basis, special = limbs, limbs, 0
    else:
        special = _special_primes(limbs, case["dnum"])
        digits, basis = case["dnum"], limbs + special
    c, exps = case["n_cts"], case.get("exponents", 1)
    ct = 2 * limbs * n
    up = digits * basis * (fly + 2 * n * max(1, limbs // max(1, digits)))  # lift and forward transforms
    switch = 2 * basis * (2 * digits * n + fly) + 4 * special * limbs * n  # inner product, inverse, division by P
    out = {"bytes": 8 * (c * ct * (1 + exps) + exps * 2 * digits * basis * n), "flops": c * (up + exps * switch)}
    if case["kind"] == "multiply":
        out["bytes"] += 8 * c * (ct - 2 * n)
        out["flops"] += c * limbs * (7 * fly + 6 * n)
    return out


# ---------------------------------------------------------------- exact values

def exact(case, seed):
    """The decoded slots in double precision from the integers the ciphertexts
    hold (message plus error): evaluation at the roots exp(i pi 5^j / N).
    Every other output is whole numbers."""
    if case["kind"] != "decrypt":
        return None
    m, e = _messages(_Inputs(seed), case)
    n = 1 << case["logn"]
    c = (m + e).cpu().numpy().astype(np.float64) / _SCALE
    values = np.fft.ifft(c * np.exp(1j * np.pi * np.arange(n) / n), axis=-1) * n  # at exp(i pi (2k + 1) / N)
    slot, index = 1, []
    for _ in range(n // 2):
        index.append((slot - 1) // 2)
        slot = slot * 5 % (2 * n)
    return torch.from_numpy(np.ascontiguousarray(values[..., index]))
