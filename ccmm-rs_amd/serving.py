"""Continuous-batching serving loop (libckks_hip.so ckks_server_*) and the
program format its jobs use.

A program is a list of ops over ciphertext registers [2][limbs][N]
(coefficient domain).  Registers 0 .. n_inputs-1 start as the job's inputs;
`out_reg` is copied to the job's output at the end.  The server validates a
program at submission, admits jobs by register footprint against an HBM
budget, and batches the same op of different jobs into one launch.
"""
from __future__ import annotations

import ctypes as C
import operator
from dataclasses import dataclass, field
from typing import Optional

from . import GaloisBatchEntry, NttBatchEntry, PreparedRnsNttPlan, _check, _p, _ptr, _ptrs, _sz, lib

OP_ROTATE, OP_MUL_PLAIN, OP_ADD, OP_RESCALE, OP_MUL_RELIN_RESCALE, OP_COPY, OP_MOD_SWITCH, OP_SUB = 1, 2, 3, 4, 5, 6, 7, 8
OP_NTT, OP_INTT, OP_MAC_PLAIN = 9, 10, 11


class _Op(C.Structure):
    _fields_ = [("code", C.c_uint32), ("dst", C.c_uint32), ("a", C.c_uint32), ("b", C.c_uint32),
                ("key", _p), ("exponent", C.c_uint64), ("plaintext", _p)]


class _Job(C.Structure):
    _fields_ = [("plan", _p), ("n_limbs", C.c_uint32), ("n_regs", C.c_uint32), ("out_reg", C.c_uint32),
                ("n_inputs", C.c_uint32), ("input", _p), ("output", _p), ("ops", _p), ("n_ops", _sz)]


class _Stats(C.Structure):
    _fields_ = [(n, C.c_uint64) for n in ("submitted", "completed", "rejected", "waiting", "active",
                                         "peak_active", "launches", "steps", "peak_bytes")] + \
               [(n, C.c_double) for n in ("p50_ms", "p99_ms", "mean_ms", "max_ms")] + \
               [(n, C.c_uint64) for n in ("cancelled", "failed", "resident_bytes")]


def _fn(name):
    return getattr(lib(), name)


@dataclass
class Program:
    """Straight-line op list; `keep` holds device plaintexts alive."""
    n_regs: int
    out_reg: int
    n_inputs: int = 1
    ops: list = field(default_factory=list)
    keep: list = field(default_factory=list)

    meta: list = field(default_factory=list)  # per op: slot rotation or plaintext slot values
    _scratch_base: int = -1
    _scratch_n: int = 0

    def scratch(self, k: int) -> list:
        """k scratch registers after the program's own (one shared area,
        grown as needed; consecutive indices)."""
        if self._scratch_base < 0:
            self._scratch_base = self.n_regs
        if k > self._scratch_n:
            self._scratch_n = k
            self.n_regs = self._scratch_base + k
        return list(range(self._scratch_base, self._scratch_base + k))

    def rotate(self, dst, a, key, exponent, steps=None):
        self.ops.append((OP_ROTATE, dst, a, 0, key, int(exponent), None))
        self.meta.append(steps)

    def mul_plain(self, dst, a, pt, values=None):
        if pt is not None:
            self.keep.append(pt)
        self.ops.append((OP_MUL_PLAIN, dst, a, 0, None, 0, pt))
        self.meta.append(values)

    def add(self, dst, a, b):
        self.ops.append((OP_ADD, dst, a, b, None, 0, None))
        self.meta.append(None)

    def ntt(self, dst, a):
        """dst = NTT(a): the register moves to the NTT domain."""
        self.ops.append((OP_NTT, dst, a, 0, None, 0, None))
        self.meta.append(None)

    def intt(self, dst, a):
        self.ops.append((OP_INTT, dst, a, 0, None, 0, None))
        self.meta.append(None)

    def mac_plain(self, dst, first, pts, values=None):
        """dst = sum_t reg[first + t] * pts[t] over NTT-domain registers and
        NTT-domain plaintexts (ckks_multiply_plain_accumulate_ntt): one
        launch for a whole baby-step inner sum."""
        pts = list(pts)
        self.keep.extend(p for p in pts if p is not None)
        self.ops.append((OP_MAC_PLAIN, dst, first, len(pts), None, 0, pts))
        self.meta.append(values)

    def sub(self, dst, a, b):
        self.ops.append((OP_SUB, dst, a, b, None, 0, None))
        self.meta.append(None)

    def rescale(self, dst, a):
        self.ops.append((OP_RESCALE, dst, a, 0, None, 0, None))
        self.meta.append(None)

    def mul_relin_rescale(self, dst, a, b, key):
        self.ops.append((OP_MUL_RELIN_RESCALE, dst, a, b, key, 0, None))
        self.meta.append(None)

    def copy(self, dst, a):
        self.ops.append((OP_COPY, dst, a, 0, None, 0, None))
        self.meta.append(None)

    def mod_switch(self, dst, a):
        self.ops.append((OP_MOD_SWITCH, dst, a, 0, None, 0, None))
        self.meta.append(None)

    def simulate(self, inputs):
        """Runs the program on cleartext slot vectors (FP64): rotations are
        cyclic shifts, plaintext products elementwise, rescale and
        mod-switch identities.  The FP64 reference of a program's result."""
        import numpy as np

        regs = [None] * self.n_regs
        for i, v in enumerate(inputs):
            regs[i] = np.asarray(v, dtype=np.complex128)
        for (code, dst, a, b, _k, _e, _pt), meta in zip(self.ops, self.meta):
            if code == OP_ROTATE:
                regs[dst] = np.roll(regs[a], -int(meta))
            elif code == OP_MUL_PLAIN:
                regs[dst] = regs[a] * meta
            elif code == OP_ADD:
                regs[dst] = regs[a] + regs[b]
            elif code == OP_SUB:
                regs[dst] = regs[a] - regs[b]
            elif code == OP_MAC_PLAIN:
                regs[dst] = sum(regs[a + t] * meta[t] for t in range(b))
            elif code == OP_MUL_RELIN_RESCALE:
                regs[dst] = regs[a] * regs[b]
            else:
                regs[dst] = regs[a].copy()
        return regs[self.out_reg]

    def register_limbs(self, n_limbs: int):
        """Per op, (limbs of its source register a, limbs of the output
        register after the program) as levels move: rescale, mod switch and
        multiply+relinearize+rescale drop one limb; everything else keeps a's.
        The last entry's second field is the output's limb count (the server
        itself rejects programs that read empty registers)."""
        regs = [int(n_limbs) if i < self.n_inputs else 0 for i in range(self.n_regs)]
        out = []
        for code, dst, a, _b, _k, _e, _pt in self.ops:
            la = regs[a] if 0 <= a < self.n_regs else 0
            if 0 <= dst < self.n_regs:
                regs[dst] = la - 1 if code in (OP_RESCALE, OP_MOD_SWITCH, OP_MUL_RELIN_RESCALE) else la
            out.append((la, 0))
        final = regs[self.out_reg] if 0 <= self.out_reg < self.n_regs else 0
        return [(la, final) for la, _ in out] or [(0, final)]

    def footprint(self, n_limbs: int, degree: int) -> int:
        """Bytes the server charges to admit this program alone: its registers
        (n_regs x 2 x n_limbs x N x 8) plus each distinct key and plaintext it
        reads (ckks_server_submit's admission model)."""
        regs = self.n_regs * 2 * int(n_limbs) * int(degree) * 8
        seen, res = set(), 0
        for (code, _d, _a, _b, key, _e, pt), (la, _) in zip(self.ops, self.register_limbs(n_limbs)):
            if key is not None and code in (OP_ROTATE, OP_MUL_RELIN_RESCALE) and id(key) not in seen:
                seen.add(id(key))
                res += key.nbytes
            for p in (pt if code == OP_MAC_PLAIN else [pt] if code == OP_MUL_PLAIN else []):
                if p is not None and id(p) not in seen:
                    seen.add(id(p))
                    res += la * int(degree) * 8
        return regs + res

    def counts(self) -> dict:
        names = {OP_ROTATE: "rotate", OP_MUL_PLAIN: "mul_plain", OP_ADD: "add", OP_SUB: "sub", OP_RESCALE: "rescale",
                 OP_NTT: "ntt", OP_INTT: "intt", OP_MAC_PLAIN: "mac_plain",
                 OP_MUL_RELIN_RESCALE: "mul_relin_rescale", OP_COPY: "copy", OP_MOD_SWITCH: "mod_switch"}
        out: dict = {}
        for op in self.ops:
            out[names[op[0]]] = out.get(names[op[0]], 0) + 1
        return out


class Server:
    WAITING, ADMITTED, DONE, CANCELLED, FAILED = 0, 1, 2, 3, 4

    def __init__(self, ctx, hbm_budget_bytes: int, max_active: int = 0):
        self.ctx = ctx
        h = _p()
        _check(_fn("ckks_server_create")(ctx.handle, int(hbm_budget_bytes), int(max_active), C.byref(h)))
        self._h = h
        self._jobs = {}  # ticket -> (job struct, op array, program, tensors) kept alive until done

    def submit(self, plan: PreparedRnsNttPlan, n_limbs: int, inputs, output, program: Program) -> int:
        ops = (_Op * max(len(program.ops), 1))()
        n = plan.degree
        limbs = program.register_limbs(int(n_limbs))
        tables = []
        for i, (code, dst, a, b, key, exp, pt) in enumerate(program.ops):
            if code == OP_MAC_PLAIN:
                # a host array of the terms' device pointers (copied at submission)
                tab = (C.c_uint64 * len(pt))(*[_ptr(p, limbs[i][0] * n, name="plaintext") for p in pt])
                tables.append(tab)
                ptr = C.cast(tab, _p)
            else:
                ptr = _ptr(pt, limbs[i][0] * n, name="plaintext") if pt is not None else None
            ops[i] = _Op(code, dst, a, b, key.handle if key is not None else None, exp, ptr)
        job = _Job(plan.handle, int(n_limbs), program.n_regs, program.out_reg, program.n_inputs,
                   _ptr(inputs, program.n_inputs * 2 * int(n_limbs) * n, name="inputs"),
                   _ptr(output, 2 * limbs[-1][1] * n, name="output"), C.cast(ops, _p), len(program.ops))
        t = C.c_uint64()
        _check(_fn("ckks_server_submit")(self._h, C.addressof(job), C.byref(t)))
        self._jobs[t.value] = (job, ops, program, inputs, output, tables)
        return t.value

    def step(self) -> int:
        n = _sz()
        _check(_fn("ckks_server_step")(self._h, C.byref(n)))
        return n.value

    def poll(self, ticket: int):
        st, lat = C.c_int(), C.c_double()
        _check(_fn("ckks_server_poll")(self._h, int(ticket), C.byref(st), C.byref(lat)))
        if st.value in (self.DONE, self.CANCELLED, self.FAILED):
            self._jobs.pop(ticket, None)
        return st.value, (lat.value if st.value == self.DONE else None)

    def cancel(self, ticket: int):
        """Drop a waiting or admitted request (ckks_server_cancel)."""
        _check(_fn("ckks_server_cancel")(self._h, int(ticket)))
        self._jobs.pop(ticket, None) if self.poll(ticket)[0] == self.CANCELLED else None

    def drain(self):
        _check(_fn("ckks_server_drain")(self._h))

    def stats(self) -> dict:
        s = _Stats()
        _check(_fn("ckks_server_stats")(self._h, C.addressof(s)))
        return {n: getattr(s, n) for n, _ in _Stats._fields_}

    def close(self):
        # the context destroys its servers itself when it is closed first
        if getattr(self, "_h", None) and self.ctx.handle:
            _fn("ckks_server_destroy")(self._h)
        self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


_LEVEL_DROP = (OP_RESCALE, OP_MOD_SWITCH, OP_MUL_RELIN_RESCALE)
_TOGETHER = 16  # rotations or transforms of one library call


@dataclass
class _Value:
    """One result of a program: the registers' contents over time."""
    limbs: int
    reads: int = 0    # ops that still read it
    home: int = -1    # the register whose row it has to end in (-1: any)
    row: int = -1


def schedule(prog: Program, n_limbs: int, spare: int):
    """Groups of independent ops of one kind, in an order that gives every op
    the values it reads in program order.  Every op writes a row of its own
    (a register reused for unrelated results orders nothing), out of n_regs +
    2 + spare rows; copies only rename.  Ops behind the oldest unfinished one
    hold at most `spare` rows, so the oldest always finds one: the values that
    program order keeps alive take n_regs rows at most.

    Returns (groups, rows used): a group is (code, limbs, [(out row, [input
    rows], op)]), code OP_COPY for the final moves of registers whose contents
    outlive the run (the output, and what the program reads before writing)."""
    n = prog.n_regs
    cur = [_Value(n_limbs if i < prog.n_inputs else 0, row=i) for i in range(n)]
    first = list(cur)
    written, carried = set(), {prog.out_reg}
    todo = []  # [op index, code, inputs, output, waits, dependants]
    source = {}
    for i, op in enumerate(prog.ops):
        code, dst, a, b = op[:4]
        regs = list(range(a, a + b)) if code == OP_MAC_PLAIN else \
            [a, b] if code in (OP_ADD, OP_SUB, OP_MUL_RELIN_RESCALE) else [a]
        carried.update(r for r in regs if r not in written)
        written.add(dst)
        if code == OP_COPY:
            cur[dst] = cur[a]
            continue
        ins = [cur[r] for r in regs]
        out = _Value(ins[0].limbs - (1 if code in _LEVEL_DROP else 0))
        node = [i, code, ins, out, 0, []]
        for v in {id(v): v for v in ins}.values():
            if id(v) in source:
                source[id(v)][5].append(node)
                node[4] += 1
        for v in ins:
            v.reads += 1
        source[id(out)] = node
        cur[dst] = out
        todo.append(node)
    final = [(r, cur[r]) for r in sorted(carried)]
    for r, v in final:
        v.reads += 1  # by the end of the run
        if v.home < 0:
            v.home = r

    free = set(range(n + 2 + spare)) - {v.row for v in first if v.reads}
    used = n
    groups = []
    ready = [t for t in todo if t[4] == 0]
    done, oldest = set(), 0
    early = {}  # rows of results behind the oldest unfinished op -> their op

    def place(t):
        """Row of t's output, or None."""
        code, ins, out = t[1], t[2], t[3]
        if code in (OP_NTT, OP_INTT, OP_ADD, OP_SUB, OP_MUL_PLAIN) and ins[0].reads == 1 and ins[0].limbs:
            return ins[0].row  # in place: nothing else reads it
        if not free:
            return None
        if out.home in free:
            return out.home
        return min(free, key=lambda r: (r < n, r))

    while oldest < len(todo):
        kinds = {}
        for t in ready:
            kinds.setdefault((t[1], t[2][0].limbs), []).append(t)
        # the fullest group first: what waits on it is then ready together
        members = max(kinds.values(), key=lambda g: (len(g), -g[0][0]))
        group = []
        for attempt in (members, [todo[oldest]]):
            for t in sorted(attempt, key=lambda t: t[0])[:_TOGETHER]:
                row = place(t)
                if row is None or (t is not todo[oldest] and row not in early and len(early) >= spare):
                    break
                t[3].row = row
                free.discard(row)
                used = max(used, row + 1)
                early[row] = t[0]
                group.append(t)
            if group:
                break
        groups.append((group[0][1], group[0][2][0].limbs,
                       [(t[3].row, [v.row for v in t[2]], prog.ops[t[0]]) for t in group]))
        for t in group:
            done.add(t[0])
            ready.remove(t)
            for v in t[2]:
                v.reads -= 1
                if v.reads == 0 and all(u[3].row != v.row for u in group):
                    free.add(v.row)
                    early.pop(v.row, None)
            if t[3].reads == 0:  # written for nobody: the row is free again
                free.add(t[3].row)
                early.pop(t[3].row, None)
            for d in t[5]:
                d[4] -= 1
                if d[4] == 0:
                    ready.append(d)
        while oldest < len(todo) and todo[oldest][0] in done:
            oldest += 1
        if oldest < len(todo):
            early = {r: i for r, i in early.items() if i >= todo[oldest][0]}
    # the registers that outlive the run move to their own rows: first those
    # whose row holds nothing another move still reads.  Where none is left, the
    # moves' rows are the registers' own (as many of them as values to move), so
    # row n is free: one value steps aside there and its row takes what it awaits
    moves = []
    pending = {r: v.row for r, v in final if v.row != r}
    while pending:
        read = set(pending.values())
        r = next((r for r in pending if r not in read), None)
        if r is None:
            q, row = next(iter(pending.items()))
            moves.append((n, [row], (OP_COPY, q, row, 0, None, 0, None)))
            used = max(used, n + 1)
            pending = {z: n if x == row else x for z, x in pending.items()}
        else:
            row = pending.pop(r)
            moves.append((r, [row], (OP_COPY, r, row, 0, None, 0, None)))
    for m in moves:
        groups.append((OP_COPY, n_limbs, [m]))
    return groups, used


def merge_sums(groups):
    """Chains of in-place additions that follow each other directly (an
    accumulator and what is added to it) as one addition of up to 64 operands:
    nothing runs between them, and sums of canonical residues do not depend on
    their order."""
    out = []
    for g in groups:
        code, la, items = g
        if code == OP_ADD and len(items) == 1 and out and out[-1][0] == OP_ADD and out[-1][1] == la \
                and len(out[-1][2]) == 1:
            row, ins, op = items[0]
            acc, terms, first = out[-1][2][0]
            if row == acc and ins[0] == acc and ins[1] != acc and len(terms) < 64:
                out[-1] = (code, la, [(acc, terms + [ins[1]], first)])
                continue
        out.append(g)
    return out


class ProgramRunner:
    """Runs one Program directly on registers it owns, outside the serving
    loop, so that a whole rotation schedule can be captured once as a hipGraph
    (capture()) and replayed (replay()) without per-op host work.  Independent
    rotations and transforms go out together, one library call for up to 16
    of them (schedule): a baby-step / giant-step request at N = 2^14 is 30
    rotations of one ciphertext, whose kernels each fill a third of the chip
    one at a time (256 x 256, 8 limbs: 3.06 ms one by one, 0.53 ms).  Registers hold compact [2][limbs][N]
    ciphertexts at their current level (as the server's); after a run the
    output register and those the program reads before it writes them hold
    their program-order values, the others whatever was last put there.  The program's
    keys must belong to the plan's context; each run switches that context
    to the runner's own (non-null, default-priority) stream and back, which
    waits for the run.  The first run() sizes every library workspace and
    builds the calls (1.7 ms where later runs take 0.53), so
    run() must precede capture(); nothing is allocated while capturing.  A
    program changed after a run is planned anew by the next one."""

    # rows of results that wait for others of their kind, and the library's
    # workspaces per group grow with them: bounded at large degrees, where a
    # single rotation fills the chip
    _SPARE_BYTES = 512 << 20

    def __init__(self, plan: PreparedRnsNttPlan, n_limbs: int, program: Program, stream=None):
        import torch

        self.ctx, self.plan, self.prog = plan.ctx, plan, program
        self.stream = stream if stream is not None else torch.cuda.Stream()
        self.L = int(n_limbs)
        n = plan.degree
        self.per = 2 * self.L * n
        self.spare = max(0, min(2 * _TOGETHER, self._SPARE_BYTES // (8 * self.per) - 1))
        self._plan_ops()
        self.regs = torch.empty((max(self.rows, program.n_regs + 2), self.per), dtype=torch.int64, device="cuda")
        self.graph = None

    def _plan_ops(self):
        prog = self.prog
        self.planned = list(prog.ops), (prog.n_regs, prog.n_inputs, prog.out_reg)
        self.mutable = any(type(op) is not tuple for op in prog.ops)
        self.limbs = prog.register_limbs(self.L)
        groups, self.rows = schedule(prog, self.L, self.spare)
        self.groups = merge_sums(groups)
        self.calls = None

    def _stale(self):
        """Whether the program differs from the planned one.  An op is a tuple,
        the same as long as it is the same object; one that could change in
        place is not taken for the same.  What an op refers to (a key's handle,
        a plaintext's address, the list of a mac_plain) is read on every run."""
        prog, (ops, shape) = self.prog, self.planned
        return (self.mutable or len(ops) != len(prog.ops) or shape != (prog.n_regs, prog.n_inputs, prog.out_reg)
                or not all(map(operator.is_, prog.ops, ops)))

    def _reg(self, i, limbs):
        return self.regs[i, : 2 * limbs * self.plan.degree]

    def _ct(self, i, limbs):
        return self._reg(i, limbs).view(1, 2, limbs, self.plan.degree)

    def _call(self, code, la, items):
        """The library call of one group as a function without arguments."""
        plan, ctx, n = self.plan, self.ctx, self.plan.degree
        if code == OP_ROTATE:
            keys = [op[4] for _, _, op in items]
            arr = (GaloisBatchEntry * len(items))()
            for e, (out, (a,), op) in zip(arr, items):
                key, ct = op[4], self._ct(a, la)
                e.exponent, e.n_cts = op[5], key._n_cts(ct, 2)
                e.input, e.output = key._ct_ptrs(e.n_cts, [("ct", ct, 2)], self._ct(out, la))
            ptr = C.cast(arr, _p)

            def rotate():
                for e, key in zip(arr, keys):
                    e.key = key.handle
                _check(lib().ckks_apply_galois_batch(ctx.handle, ptr, len(arr)))
            return rotate
        if code in (OP_NTT, OP_INTT):
            arr = (NttBatchEntry * len(items))()
            for e, (out, (a,), _) in zip(arr, items):
                p_in, p_out = (_ptr(self._reg(i, la)) for i in (a, out))
                e.input, e.output, e.n_polys, e.n_limbs, e.poly_stride = p_in, p_out, 2, la, la * n
            ptr = C.cast(arr, _p)

            def transform():
                for e in arr:
                    e.plan = plan.handle
                fn = lib().ckks_ntt_forward_batch if code == OP_NTT else lib().ckks_ntt_inverse_batch
                _check(fn(ctx.handle, ptr, len(arr)))
            return transform
        if code == OP_MAC_PLAIN:
            # sums of the same ciphertexts share a call
            shared = {}
            for out, ins, op in items:
                shared.setdefault(tuple(ins), []).append((_ptr(self._reg(out, la)), op[6]))
            sums = [([_ptr(self._reg(i, la)) for i in ins], [pts for _, pts in group],
                     (C.c_uint64 * len(group))(*[out for out, _ in group])) for ins, group in shared.items()]

            def accumulate():
                for ins, lists, outs in sums:
                    if not ins or any(len(pts) != len(ins) for pts in lists):
                        raise ValueError("one plaintext per ciphertext, at least one term")
                    cts = (C.c_uint64 * len(ins))(*ins)
                    pts = (C.c_uint64 * (len(ins) * len(lists)))(*[p for pts in lists for p in _ptrs(pts, la * n, "pt")])
                    _check(lib().ckks_multiply_plain_accumulate_ntt_batch(
                        plan.handle, C.cast(cts, _p), C.cast(pts, _p), len(ins), C.cast(outs, _p), len(outs), la))
            return accumulate
        steps = []
        for out, ins, op in items:
            _, _, _, _, key, _, pt = op
            if code == OP_MUL_PLAIN:
                def step(x=self._ct(ins[0], la), pt=pt, out=self._ct(out, la)):
                    plan.multiply_plain(x, pt, la, out=out)
            elif code == OP_ADD and len(ins) > 2:
                xs = (C.c_uint64 * len(ins))(*[_ptr(self._reg(i, la)) for i in ins])

                def step(xs=xs, out=_ptr(self._reg(out, la))):
                    _check(lib().ckks_poly_sum(plan.handle, C.cast(xs, _p), len(xs), out, 2, la, la * n))
            elif code in (OP_ADD, OP_SUB):
                def step(fn=plan.add if code == OP_ADD else plan.sub, x=self._reg(ins[0], la),
                         y=self._reg(ins[1], la), out=self._reg(out, la)):
                    fn(x, y, out=out, n_limbs=la)
            elif code in (OP_RESCALE, OP_MOD_SWITCH):
                def step(fn=plan.rescale_to_next if code == OP_RESCALE else plan.mod_switch_to_next,
                         x=self._ct(ins[0], la), out=self._ct(out, la - 1)):
                    fn(x, la, out=out)
            elif code == OP_MUL_RELIN_RESCALE:
                def step(key=key, x=self._ct(ins[0], la), y=self._ct(ins[1], la), out=self._ct(out, la - 1)):
                    key.multiply_relinearize_rescale(x, y, out=out)
            elif code == OP_COPY:
                def step(x=self.regs[ins[0]], out=self.regs[out]):
                    out.copy_(x)
            else:
                raise ValueError(f"unknown op code {code}")
            steps.append(step)

        def each():
            for s in steps:
                s()
        return each

    def _run_ops(self):
        if self._stale():
            # the rows there are stay: a captured graph and the caller's views hold them
            self.spare = max(0, self.regs.shape[0] - self.prog.n_regs - 2)
            self._plan_ops()
            if max(self.rows, self.prog.n_regs) > self.regs.shape[0]:
                self.planned = [], ()
                raise ValueError("the program outgrew the runner's registers")
        if self.calls is None:
            self.calls = [self._call(*g) for g in self.groups]
        for call in self.calls:
            call()

    def _on_stream(self):
        import contextlib

        import torch

        @contextlib.contextmanager
        def cm():
            prev = self.ctx.stream
            torch.cuda.current_stream().synchronize()
            self.ctx.set_stream(self.stream)
            try:
                with torch.cuda.stream(self.stream):
                    yield
            finally:
                self.ctx.set_stream(prev)  # waits for the runner's stream
        return cm()

    def _load(self, inputs):
        self.regs[: self.prog.n_inputs].copy_(inputs.reshape(self.prog.n_inputs, self.per))

    def output(self):
        lo = self.limbs[-1][1]
        return self._ct(self.prog.out_reg, lo)[0]

    def run(self, inputs=None):
        """Run the program on `inputs` ([n_inputs][2][n_limbs][N]; None: the
        registers as they are); returns the output register (complete)."""
        with self._on_stream():
            if inputs is not None:
                self._load(inputs)
            self._run_ops()
        return self.output()

    def capture(self):
        """Record one run of the ops (not the input load) as a graph."""
        with self._on_stream():
            self.ctx.graph_begin()
            try:
                self._run_ops()
            finally:
                self.graph = self.ctx.graph_end()
        return self.graph

    def replay(self, inputs=None):
        with self._on_stream():
            if inputs is not None:
                self._load(inputs)
            self.graph.launch()
        return self.output()
