"""Runs of gates on one large tensor, executed as passes over LDS tiles.

A contraction path applies gate-sized tensors one after another to the same
state-like intermediate; done step by step, each of them reads and writes the
whole intermediate.  Here such a chain of steps becomes *ops* (dense 4 x 4 or
8 x 8 matrices on two or three address bits, in place), and the ops become
*passes*: a tile of address bits is chosen, every op that fits it and is not
behind one that does not is applied while the tile is in LDS, and the large
tensor crosses HBM once per pass (tedq_tn_run_pass, tedq_tn_run_backward).

Terms: a *wire* is an address bit of the chain's input tensor; an op consumes
the index symbols on its wires and leaves others there.  Steps that change
the rank, or that share a kept (hyper-)index with the large tensor, join an op
together with their neighbours when the group as a whole is square: the
kernel forms the group's matrix from its factors (sums over the symbols that
live only inside the group, equality where an index goes straight through).
"""

from dataclasses import dataclass, field

import numpy as np

MIN_WIRES = 9      # smallest large operand: a wave of 64 rows of an 8 x 8 op
TILE_WIRES = 12    # largest tile: 2^12 amplitudes, 32 KB of LDS
LOW_WIRES = 3      # lowest address bits of every tile: 64-byte segments (four cost 51 forward passes against 44 on
                   # a 5x5 lattice, 50 against 43 with gradients, and 37.6 against 37.0 ms: the longer segments do
                   # not repay the passes)
MAX_ARITY = 3
MAX_FACTORS = 4
MAX_INTERNAL = 3
MAX_FACTOR_RANK = 6
MAX_PASS_OPS = 32
COEF_BUDGET = 512          # matrix entries of one pass (4 KB of LDS, twice that in the backward)
OP_WORDS = 12 + 10 * MAX_FACTORS
PASS_WORDS = 128


@dataclass
class Op:
    """One square group of steps: symbols on its wires before and after, its factors (tensor ids)."""
    ins: list
    outs: list
    factors: list
    internal: list
    wires: list = field(default_factory=list)


@dataclass
class RunPass:
    local: list        # wires of the tile, ascending
    ops: list          # Ops in order
    words: np.ndarray = None
    head: int = 0      # first op row in the network's op table


@dataclass
class Run:
    a: int             # input tensor id
    c: int             # result tensor id
    steps: list        # step numbers covered
    wires: int
    out_bit: list      # address bit of every wire in the result
    passes: list

    def parts(self):
        """The run pass by pass."""
        return [Run(self.a, self.c, self.steps, self.wires, self.out_bit, [ps]) for ps in self.passes]


def _symbols(lay, st, big, small):
    sb, ss, sc = set(lay[big]), set(lay[small]), set(lay[st.c])
    used = [s for s in lay[big] if s in ss]
    return used, [s for s in used if s not in sc], [s for s in lay[small] if s not in sb]


def _group(chain, i, lay, single):
    """Shortest square group of chain steps starting at i: (Op, next) or None."""
    ins, live, internal, factors = [], [], [], []
    made = set()
    for j in range(i, min(len(chain), i + (1 if single else MAX_FACTORS))):
        _, small, used, gone, new = chain[j]
        if len(lay[small]) > MAX_FACTOR_RANK:
            return None
        if single and len(used) != len(gone):
            return None
        factors.append(small)
        for s in used:
            if s not in live:
                ins.append(s)
                live.append(s)
        for s in gone:
            live.remove(s)
            if s in made:
                internal.append(s)
        live += new
        made.update(new)
        if len(ins) > MAX_ARITY or len(internal) > MAX_INTERNAL:
            return None
        if len(live) == len(ins) and ins:
            return Op(ins, list(live), factors, internal), j + 1
    return None


def _absorb(ops, op):
    """Merge ``op`` with the earlier ops on its symbols where one matrix of at most 4 x 4 (or the larger
    of the two) holds both: products of small matrices instead of passes over the tile."""
    def limit(*o):
        return max([2] + [len(x.ins) for x in o])
    while True:
        last = {}
        for k, o in enumerate(ops):
            for s in o.outs:
                if s in op.ins:
                    last[s] = k
        merged = False
        for k in sorted(set(last.values()), reverse=True):
            o = ops[k]
            shared = [s for s in o.outs if s in op.ins]
            rest = [s for s in op.ins if s not in shared]
            # o moves to op's place: no op in between may use its results
            if any(s in x.ins for x in ops[k + 1:] for s in o.outs):
                continue
            gone = [s for s in shared if s not in op.outs]
            ins = o.ins + rest
            outs = [s for s in o.outs if s not in gone] + [s for s in op.outs if s not in o.outs]
            internal = o.internal + op.internal + [s for s in gone if s not in o.ins]
            if (len(ins) > limit(o, op) or len(o.factors) + len(op.factors) > MAX_FACTORS
                    or len(internal) > MAX_INTERNAL):
                continue
            op = Op(ins, outs, o.factors + op.factors, internal)
            del ops[k]
            merged = True
            break
        if not merged:
            return op


def _split_passes(ops, n):
    """Greedy passes: each takes, in order, every op that fits its tile and is not behind one left out."""
    passes = []
    pending = list(ops)
    while pending:
        local = set(range(min(LOW_WIRES, n)))
        cap = min(TILE_WIRES, n)
        taken, left, blocked, coef = [], [], set(), 0
        for op in pending:
            w = set(op.wires)
            size = 4 ** _arity(op)
            if (blocked & w or len(local | w) > cap or len(taken) == MAX_PASS_OPS or coef + size > COEF_BUDGET):
                blocked |= w
                left.append(op)
                continue
            local |= w
            coef += size
            taken.append(op)
        # a tile of at least 2^10 amplitudes, of 2^12 where many tiles remain
        want = min(n, cap if n >= 20 else 10)
        for w in range(n):
            if len(local) >= want:
                break
            local.add(w)
        passes.append(RunPass(sorted(local), taken))
        pending = left
    return passes


def _arity(op):
    return max(2, len(op.wires))


def find_runs(net, small_offs, grad, unitary=None):
    """The runs of a network: maximal chains of steps with a large and a gate-sized operand (a leaf or a
    small step's result), cut into square ops.  With ``grad`` only single-step ops that ``unitary`` (tensor
    id, symbols of one side) accepts, whose input the backward recovers from their result."""
    lay, steps = net.lay, net.steps

    def ready(t):
        return t < net.n_inputs or t in small_offs

    def link(st):
        if st.c in small_offs:
            return None
        big, small = (st.a, st.b) if net.ranks[st.a] >= net.ranks[st.b] else (st.b, st.a)
        if not ready(small) or net.ranks[big] < MIN_WIRES or net.ranks[small] > MAX_FACTOR_RANK:
            return None
        return big, small

    runs, seen = [], set()
    for s0, st0 in enumerate(steps):
        if s0 in seen or link(st0) is None:
            continue
        chain, s = [], s0
        while True:
            lk = link(steps[s])
            if lk is None or (chain and lk[0] != steps[chain[-1][0]].c):
                break
            chain.append((s, lk[1]) + _symbols(lay, steps[s], *lk))
            seen.add(s)
            s = net.consumer.get(steps[s].c, -1)
            if s < 0:
                break
        i = 0
        while i < len(chain):
            ops, j = [], i
            big0 = link(steps[chain[i][0]])[0]
            while j < len(chain):
                got = _group(chain, j, lay, grad)
                if got is None or (grad and not unitary(chain[j][1], chain[j][3])):
                    break
                op, j = got
                ops.append(op if grad else _absorb(ops, op))
            if j - i >= 2:
                run = _place(net, big0, steps[chain[j - 1][0]].c, [c[0] for c in chain[i:j]], ops)
                if run is not None:
                    runs.append(run)
            i = max(j, i + 1)
    return runs


def _place(net, a, c, covered, ops):
    n = net.ranks[a]
    if net.ranks[c] != n:
        return None
    wire = {s: n - 1 - i for i, s in enumerate(net.lay[a])}
    for op in ops:
        pairs = [(s, wire[s]) for s in op.ins]
        stay = {s for s in op.ins if s in op.outs}
        free = sorted(w for s, w in pairs if s not in stay)
        op.wires = sorted(w for _, w in pairs)
        # several results on one op: the order among the freed wires only fixes names
        named = {s: wire[s] for s in stay}
        for s, w in zip([s for s in op.outs if s not in stay], reversed(free)):
            named[s] = w
        op.in_wire = dict(pairs)
        op.out_wire = named
        for s in op.ins:
            del wire[s]
        wire.update(named)
    out_pos = {s: n - 1 - i for i, s in enumerate(net.lay[c])}
    out_bit = [0] * n
    for s, w in wire.items():
        out_bit[w] = out_pos[s]
    return Run(a, c, covered, n, out_bit, _split_passes(ops, n))


def encode_op(op, local, source, lay):
    """Words of one op: arity, slots, delta mask, internal count, factors (base, offset, per address bit the
    variable it follows: 0..2 in, 3..5 out, 6..8 internal).  An op on one wire carries a spectator slot."""
    slot = {w: i for i, w in enumerate(local)}
    slots = sorted(slot[w] for w in op.wires)
    delta = 0
    if len(slots) == 1:
        slots = sorted(slots + [0 if slots[0] != 0 else 1])
    num = {s: j for j, s in enumerate(slots)}
    words = np.zeros(OP_WORDS, dtype=np.int32)
    var = {}
    used = set()
    for s in op.ins:
        used.add(num[slot[op.in_wire[s]]])
        if s in op.out_wire:
            delta |= 1 << num[slot[op.in_wire[s]]]
        var[s] = num[slot[op.in_wire[s]]]
    for s in op.outs:
        if s not in op.in_wire:
            var[s] = 3 + num[slot[op.out_wire[s]]]
    for j in range(len(slots)):
        if j not in used:
            delta |= 1 << j
    for j, s in enumerate(op.internal):
        var[s] = 6 + j
    words[0] = len(slots)
    words[1:1 + len(slots)] = slots
    words[4] = delta
    words[5] = len(op.internal)
    words[6] = len(op.factors)
    for f, tid in enumerate(op.factors):
        base, off = source(tid)
        w = words[12 + 10 * f:]
        w[0], w[1], w[2] = base, off, len(lay[tid])
        for i, s in enumerate(reversed(lay[tid])):
            w[3 + i] = var[s]
    return words


def encode_run(run, source, lay):
    """Fill every pass's words (head, slots and address bits) and return its op rows."""
    rows = []
    n = run.wires
    for p, ps in enumerate(run.passes):
        last = p == len(run.passes) - 1
        out = run.out_bit if last else list(range(n))
        outer = [w for w in range(n) if w not in set(ps.local)]
        by_out = sorted(ps.local, key=lambda w: out[w])
        words = np.zeros(PASS_WORDS, dtype=np.int32)
        words[0], words[1], words[2] = len(ps.local), len(outer), len(ps.ops)
        L = len(ps.local)
        words[4:4 + L] = ps.local                                     # address bit of slot i in the input
        words[16:16 + L] = [ps.local.index(w) for w in by_out]        # slot of the i-th lowest result bit
        words[28:28 + L] = [out[w] for w in by_out]                   # its address bit in the result
        words[40:40 + len(outer)] = outer
        words[72:72 + len(outer)] = [out[w] for w in outer]
        ps.words = words
        coef = 0
        for op in ps.ops:
            row = encode_op(op, ps.local, source, lay)
            row[7] = coef
            coef += 4 ** int(row[0])
            rows.append(row)
        words[3] = coef
    return rows


class Unitarity:
    """Which gate-sized tensors are unitary maps between two halves of their indices: whole gate leaves by their
    operator (``leaf_unitary(source, rank)``: False for reduced ones), small products when one factor's whole
    contact lies in one half of each operand."""

    def __init__(self, net, leaf_unitary):
        self.net = net
        self.leaf = leaf_unitary
        self.maker = {st.c: st for st in net.steps}
        self.memo = {}

    def halves(self, tid):
        if tid not in self.memo:
            self.memo[tid] = self._halves(tid)
        return self.memo[tid]

    def _halves(self, tid):
        lay = self.net.lay
        if tid < self.net.n_inputs:
            r = len(lay[tid])
            if r % 2 or not self.leaf(self.net.sources[tid], r):
                return None
            return frozenset(lay[tid][:r // 2]), frozenset(lay[tid][r // 2:])
        st = self.maker[tid]
        a, b = self.halves(st.a), self.halves(st.b)
        if a is None or b is None:
            return None
        common = set(lay[st.a]) & set(lay[st.b])
        if common & set(lay[tid]):
            return None
        for x, x2 in (a, a[::-1]):
            for y, y2 in (b, b[::-1]):
                if common <= x and common <= y:
                    return frozenset(x2 | (y - common)), frozenset(y2 | (x - common))
        return None

    def __call__(self, tid, summed):
        h = self.halves(tid)
        return h is not None and frozenset(summed) in h and len(h[0]) == len(h[1])
