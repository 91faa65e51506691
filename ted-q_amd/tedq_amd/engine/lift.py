"""Lifted plans: rounds of in-place register ops for the interpreted pass kernels (csrc/sv_lift.hip).

What bounds an interpreted pass is VALU issue, and most of it is not arithmetic when every op is dispatched
by itself: each arm of the dispatch leaves its results in registers of its own and the join copies them
back.  A lifted pass is a list of *rounds* over the register bits of a stage instead.  A round does, in
order and without any dispatch: a diagonal D0, an RX or RY per register bit, a diagonal D1 (each optional),
then a list of general ops (dense 4x4s, controlled rotations, user matrices: dispatched, rare), then a signed
permutation of the thread's 2^r amplitudes (every CZ, CNOT, Toffoli, SWAP).

* A rotation is applied as [[1, -q], [q, 1]] or [[q, -1], [1, q]], whichever has |q| <= 1 (q = tan or cot of
  half its angle): one multiply-add per output, and its common factor (cos or sin) goes into D1.  (A form with
  two in-place multiply-adds and different scales for the two outputs needs no moves but rounds the scales
  apart: expectation values of 20-qubit circuits then have 1.1 times the error of plain 2x2 matrices.)
* D1 holds, per amplitude, the product of those factors and of the phases of every diagonal gate that
  follows the rotations on any register bit: one complex multiply for all of them.
* The permutation is free: it is the order in which the round writes its amplitudes to LDS.

Every form drops its global phase, as the specialised plan's diagonal gates do, so lifted plans serve
forward sweeps of expectation values and probabilities, and every adjoint sweep (psi and lambda receive the
same phase).

Table row of a round (csrc/sv_tables.hip, complex64 entries): D1 (2^r), then per register bit (q, 0), then one
entry whose real part's bits are the mask of bits in the second form, then D0 (2^r) if it has one.
"""

from dataclasses import dataclass, field

import numpy as np

from .planner import (Component, Slot, OP_CD1, OP_CU1, OP_D1, OP_DAGGER, OP_PGRAD, OP_R1, OP_U1, OP_U2, SLOT_1Q, SLOT_2Q,
                      Unit, _const_comp)

OP_PHL = 15                    # controlled phase of a lifted program (general op)

# how a slot is used (csrc/sv_tables.hip, SlotRec.form); 0: by its matrix.  FORM_PHASE: a controlled phase,
# stored as that complex number; FORM_DENSE: a 4x4 followed by its adjoint; FORM_PART: it was multiplied into
# another slot; the others are parts of a round.
FORM_X, FORM_Y, FORM_DIAG, FORM_EULER, FORM_PHASE, FORM_DENSE, FORM_PART = 1, 2, 3, 4, 5, 6, 7

GROUP_UNITS = 12               # units of one two-qubit user matrix (planner.two_qubit_units)

# stage words of a lifted program (csrc/sv_lift.hip)
STAGE_WORDS = 80
(W_FLAGS, W_REGMASK, W_ROT, W_COEF, W_SIGN, W_NGEN, W_GEN, W_GRADS, W_KINDP, W_GROUP, W_GROUP_PRE) = range(11)
W_IN, W_OUT = 12, 44
SKIP_READ, SKIP_WRITE, BARRIER, HAS_D0, HAS_D1, HAS_SCALE = 1, 2, 4, 8, 16, 32
ROUND_WORDS = 18               # round records of the table kernel: table offset, flags, 5 slots each (or -1) of
                               # D0, rotations and D1, 0
HDR_STAGES = 100


def lift_units(units, const_pool):
    """Units of a lifted plan: a whole two-qubit user matrix is one dense "u2" unit (its decomposition serves
    the other plans), consecutive ones on the same pair are multiplied into one, and Rot(phi, theta, omega)
    is RZ(phi), RY(theta), RZ(omega), whose gradients are single values."""
    out, last = [], {}

    def put(u):
        out.append(u)
        for b in u.bits:
            last[b] = len(out) - 1

    i = 0
    while i < len(units):
        u = units[i]
        run = units[i:i + GROUP_UNITS]
        if u.group is not None and [x.group for x in run] == [(u.group[0], j) for j in range(GROUP_UNITS)]:
            i += GROUP_UNITS
            lo, hi = u.bits                           # the first multiplexor: target low, control high
            m = np.asarray(const_pool[u.group[0]:u.group[0] + 16]).reshape(4, 4)
            if hi < lo:                               # stored with the higher bit first
                hi, lo = lo, hi
                swap = [0, 2, 1, 3]
                m = m[np.ix_(swap, swap)]
            prev = last.get(hi)
            if prev is not None and prev == last.get(lo) and out[prev].kind == "u2":
                c = out[prev].comp.const_mat
                m = m @ np.asarray(const_pool[c:c + 16]).reshape(4, 4)
                out[prev] = Unit("u2", (hi, lo), _const_comp(m, const_pool))
            else:
                put(Unit("u2", (hi, lo), _const_comp(m, const_pool)))
            continue
        i += 1
        if u.kind == "u1" and u.comp.code == 17 and u.comp.const_mat < 0:
            phi, theta, omega = u.comp.srcs
            parts = [(16, phi), (15, theta), (16, omega)]
            for code, src in (reversed(parts) if u.comp.dagger else parts):
                put(Unit("u1", u.bits, Component(code, u.comp.dagger, (src,)), u.index))
            continue
        put(u)
    return out


def slot_form(slot, trained=True):
    """Form of a slot: RX / RY as a rotation, diagonal slots in D0 or D1, other products of known (hence
    unitary) gates as diagonal - RY - diagonal.  Controlled slots keep their matrix (their block's phase is not
    global) unless the block is diag(1, p); user matrices, which need not be unitary, keep theirs.  ``trained``:
    the plan serves the adjoint, whose gradients need trained gates unfused."""
    if slot.kind == SLOT_2Q:
        return FORM_DENSE
    if any(c.const_mat >= 0 for c in slot.comps):
        return 0
    codes = [c.code for c in slot.comps]
    if slot.controlled:
        return FORM_PHASE if codes == [18] else 0
    if slot.diagonal:
        return FORM_DIAG
    if codes in ([14], [15]):
        return FORM_X if codes == [14] else FORM_Y
    if trained and slot.trainable:
        raise ValueError("a lifted plan has no form for this trainable slot")
    return FORM_EULER


@dataclass
class Round:
    """One round of a stage (see module note); slots by register bit."""
    reg_bits: list
    pre: dict = field(default_factory=dict)
    rot: dict = field(default_factory=dict)
    post: dict = field(default_factory=dict)
    gen: list = field(default_factory=list)      # plan ops (kind, b0, b1, cmask, slot)
    perm: list = None                            # amplitude m moves to position perm[m] ...
    sign: int = 0                                # ... and is negated where bit m is set
    coef: int = 0
    group: int = -1                              # gradient slot of rotations (comp b) and last phases (4 + b)
    group_pre: int = -1                          # gradient slot of first phases (comp 4 + b)
    last: bool = False                           # last round of its stage

    def has_d0(self, slots):
        return bool(self.pre) or any(slots[si].form == FORM_EULER for si in self.rot.values())

    def has_d1(self, slots):
        """Phases in D1 (otherwise it is the rotations' factor, or 1)."""
        return bool(self.post) or any(slots[si].form == FORM_EULER for si in self.rot.values())

    @property
    def moves(self):
        return any(p != m for m, p in enumerate(self.perm))


def _stage_rounds(stage, slots, r, fuse):
    """The stage's ops in order, each in the newest round if the round's order allows it, else in a new one.
    ``fuse`` (forward plans): a gate whose register bit has its rotation and diagonals already is multiplied
    with them into one general rotation instead (fewer rounds and roundings)."""
    R = 1 << r
    rounds = []

    def new():
        rounds.append(Round(stage.reg_bits, perm=list(range(R))))
        return {"level": [0] * r, "gen": 0, "move": 0}
    st = new()
    for op in stage.ops:
        kind, b0, b1, cmask, si = op
        cur = rounds[-1]
        if kind in ("cx", "cz"):
            for m in range(R):
                p = cur.perm[m]
                if (p & cmask) != cmask:
                    continue
                if kind == "cx":
                    cur.perm[m] = p ^ (1 << b0)
                else:
                    cur.sign ^= 1 << m
            st["move"] |= cmask | ((1 << b0) if kind == "cx" else 0)
            continue
        form = slot_form(slots[si], not fuse)
        slots[si].form = form
        if kind == "u1" and form:
            bit = 1 << b0
            mine = [part[b0] for part in (cur.pre, cur.rot, cur.post) if b0 in part]
            if fuse and mine and not (st["gen"] | st["move"]) & bit and (
                    form == FORM_EULER or st["level"][b0] > (1 if form != FORM_DIAG else 2)):
                slots.append(Slot(SLOT_1Q, [c for s in mine for c in slots[s].comps] + slots[si].comps))
                for s in mine + [si]:
                    slots[s].form = FORM_PART
                si = len(slots) - 1
                form = slots[si].form = slot_form(slots[si], False) or FORM_EULER
                for part in (cur.pre, cur.rot, cur.post):
                    part.pop(b0, None)
                st["level"][b0] = 0
            need = {FORM_EULER: 0, FORM_X: 1, FORM_Y: 1, FORM_DIAG: 2}[form]
            if (st["gen"] | st["move"]) & bit or st["level"][b0] > need:
                st = new()
                cur = rounds[-1]
            if form == FORM_EULER:
                cur.rot[b0], st["level"][b0] = si, 3
            elif form != FORM_DIAG:
                cur.rot[b0], st["level"][b0] = si, 2
            elif st["level"][b0] == 0:
                cur.pre[b0], st["level"][b0] = si, 1
            else:
                cur.post[b0], st["level"][b0] = si, 3
            continue
        bits = cmask | (1 << b0) | ((1 << b1) if kind == "u2" else 0)
        if st["move"] & bits:
            st = new()
        rounds[-1].gen.append(op)
        st["gen"] |= bits
    for rd in rounds:
        # a first diagonal with nothing after it is part of D1 (its gradient then shares the rotations' group)
        for b in [b for b in rd.pre if b not in rd.rot and b not in rd.post]:
            rd.post[b] = rd.pre.pop(b)
    rounds[-1].last = True
    return rounds


def assign_rounds(passes, slots, r, fuse=False):
    """Rounds of every pass, and the table offsets and gradient slots of their slots: (rounds per pass, complex64
    entries per table row, gradient slots)."""
    off = gslot = 0
    out = []
    for p in passes:
        mine = [rd for st in p.stages for rd in _stage_rounds(st, slots, r, fuse)]
        for rd in mine:
            rd.coef = off
            if rd.pre or rd.rot or rd.post:
                off += (1 << r) + r + 1 + ((1 << r) if rd.has_d0(slots) else 0)
            if fuse:
                for op in rd.gen:
                    slots[op[4]].mat_off = off
                    off += 32 if slots[op[4]].kind == SLOT_2Q else 4
                continue
            trained = [(b, si, c) for part, c in ((rd.rot, 0), (rd.post, 4)) for b, si in part.items()
                       if slots[si].trainable]
            if trained:
                rd.group = gslot
                gslot += 1
                for b, si, c in trained:
                    slots[si].gslot, slots[si].scomp = rd.group, b + c
            pre = [(b, si) for b, si in rd.pre.items() if slots[si].trainable]
            if pre:
                rd.group_pre = gslot
                gslot += 1
                for b, si in pre:
                    slots[si].gslot, slots[si].scomp = rd.group_pre, 4 + b
            for op in rd.gen:
                sl = slots[op[4]]
                sl.mat_off = off
                off += 32 if sl.kind == SLOT_2Q else 4
                if sl.trainable:
                    sl.gslot, sl.scomp = gslot, 0
                    gslot += 1
        out.append(mine)
    return out, off, gslot


def _gen_words(op, slots, adjoint):
    """Words of one general op; in the adjoint its gradient first, then its inverse."""
    kind, b0, b1, cmask, si = op
    sl = slots[si]
    dag = OP_DAGGER if adjoint else 0
    words = []
    if adjoint and sl.gslot >= 0:
        pk, neg = sl.pauli
        words.append([OP_PGRAD, b0, 0, cmask, 0, sl.gslot, pk | (int(neg) << 4), 0])
    if kind == "u2":
        words.append([OP_U2, b0, b1, 0, sl.mat_off + (16 if adjoint else 0), -1, 0, 0])
    elif sl.form == FORM_PHASE:
        words.append([OP_PHL | dag, b0, 0, cmask, sl.mat_off, -1, 0, 0])
    else:
        t = OP_R1 if sl.real else (OP_D1 if kind == "u1" else OP_CD1) if sl.diagonal else (
            OP_U1 if kind == "u1" else OP_CU1)
        words.append([t | dag, b0, 0, cmask, sl.mat_off, -1, 0, 0])
    return words


def _round_words(rd, r, slots, adjoint, skip_read, skip_write, barrier, pdep, swizzle):
    """(stage words, general op words) of one round."""
    w = np.zeros(STAGE_WORDS, dtype=np.int64)
    d1 = rd.has_d1(slots)
    w[W_FLAGS] = ((SKIP_READ if skip_read else 0) | (SKIP_WRITE if skip_write else 0) | (BARRIER if barrier else 0)
                  | (HAS_D0 if rd.has_d0(slots) else 0) | (HAS_D1 if d1 else 0)
                  | (HAS_SCALE if rd.rot and not d1 else 0))
    w[W_REGMASK] = sum(1 << b for b in rd.reg_bits)
    grads, kindp = [0, 0, 0], [0, 0]             # bits of trained rotations, D1 gates, D0 gates; PhaseShifts
    for b, si in rd.rot.items():
        w[W_ROT] |= 1 << b << (0 if slots[si].form == FORM_X else 8)
        if slots[si].gslot >= 0:
            grads[0] |= 1 << b
    for i, part in enumerate((rd.post, rd.pre)):
        for b, si in part.items():
            if slots[si].gslot >= 0:
                grads[1 + i] |= 1 << b
                kindp[i] |= int(slots[si].pauli[0] == 3) << b
    # a round of general ops only has no table row: the kernel, which reads ahead, finds row 0
    w[W_COEF], w[W_SIGN] = (rd.coef if rd.pre or rd.rot or rd.post else 0), rd.sign
    w[W_GRADS] = grads[0] | grads[1] << 8 | grads[2] << 16
    w[W_KINDP] = kindp[0] | kindp[1] << 8
    w[W_GROUP], w[W_GROUP_PRE] = rd.group, rd.group_pre
    plain = [swizzle(pdep(m, rd.reg_bits)) for m in range(1 << r)]
    moved = [plain[rd.perm[m]] for m in range(1 << r)]
    w[W_IN:W_IN + (1 << r)] = moved if adjoint else plain
    w[W_OUT:W_OUT + (1 << r)] = plain if adjoint else moved
    gen = []
    for op in (reversed(rd.gen) if adjoint else rd.gen):
        gen += _gen_words(op, slots, adjoint)
    w[W_NGEN] = len(gen)
    return w, gen


def encode_rounds(rounds, plan, adjoint, pdep, swizzle):
    """Stage words and general op words of one pass: (list of stage words with W_GEN relative to the first
    general op, list of general op words)."""
    seq = rounds[::-1] if adjoint else rounds
    stages, gens = [], []
    for i, rd in enumerate(seq):
        # between two rounds of a stage the amplitudes stay in registers unless the earlier one permutes them
        # (then each thread writes and reads its own LDS positions, without a barrier)
        prev, nxt = (seq[i - 1] if i else None), (seq[i + 1] if i + 1 < len(seq) else None)
        if adjoint:
            first, last = rd.last, nxt is None or nxt.last
            keep_in = not first and not rd.moves
            keep_out = not last and not nxt.moves
        else:
            first, last = prev is None or prev.last, rd.last
            keep_in = not first and not prev.moves
            keep_out = not last and not rd.moves
        w, gen = _round_words(rd, plan.r, plan.slots, adjoint, keep_in, keep_out, last, pdep, swizzle)
        w[W_GEN] = len(gens)
        stages.append(w)
        gens += gen
    return stages, gens



def round_records(plan):
    """Round records of the table kernel (ROUND_WORDS int32 each) of every round that has a table row part."""
    out = []
    for rd in (x for rounds in plan.rounds for x in rounds):
        if not (rd.pre or rd.rot or rd.post):
            continue
        rec = [rd.coef, int(rd.has_d0(plan.slots))]
        for part in (rd.pre, rd.rot, rd.post):
            rec += [part.get(b, -1) for b in range(5)]
        out.append(rec + [0])
    return np.asarray(out if out else np.zeros((0, ROUND_WORDS)), dtype=np.int32).reshape(-1, ROUND_WORDS)
