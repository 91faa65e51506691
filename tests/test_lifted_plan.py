"""Lifted plans (rounds of in-place ops, tedq_amd/engine/lift.py) emulated on the CPU against the oracle.

The emulator decodes the encoded rounds -- LDS offsets, masks, round tables, signed permutations, general
ops, gradient groups -- and runs them in float64 with the table entries that the table kernel stores, so the
planner, the encoder and the algebra of the rounds are checked without a GPU: states up to the global
phase that lifted plans drop, and gradients.  All gates of the state-vector engine occur, on tiles and
register counts small enough to force several passes, stages and rounds.
"""

import math

import numpy as np
import pytest
import torch

import tedq_amd as qai
from oracle import sv_oracle as O
from sv_emulator import _comp_matrix, _pdep
from tedq_amd.engine import lift as LF
from tedq_amd.engine import program as P
from tedq_amd.engine.lowering import lower_circuit
from tedq_amd.engine.planner import build_plan
from test_plan_emulated import oracle_gates, random_spec, trace

DAG = 1 << 8


def _unit(z):
    return z / abs(z) if abs(z) > 0 else 1.0


def _euler(S):
    """(e^ig, c, s, e^ia) with S = e^id diag(1, e^ia) [[c, -s], [s, c]] diag(1, e^ig)."""
    c, s = abs(S[0, 0]), abs(S[1, 0])
    ea = _unit(S[1, 0] * np.conj(S[0, 0]))
    eg = _unit(S[1, 1] * np.conj(S[0, 0]) * np.conj(ea)) if c >= s else _unit(-S[0, 1] * np.conj(S[1, 0]) * ea)
    return eg, c, s, ea


def tables(enc, plan, row):
    """Table row (complex), and where and with which sign each parameter's gradient value is found."""
    pool = enc.const_pool
    mats = np.full(plan.mat_stride, np.nan + 0j)
    grads, S = {}, []
    for si, s in enumerate(plan.slots):
        rec = [int(x) for x in enc.slot_recs[si]]
        comps = enc.comp_recs[rec[2]:rec[2] + rec[1]]
        off, form = rec[3], rec[7]
        m = np.eye(2, dtype=np.complex128)
        if rec[0] == 1:
            o = int(comps[0][5])
            d = (pool[o:o + 16, 0] + 1j * pool[o:o + 16, 1]).reshape(4, 4)
            mats[off:off + 32] = np.concatenate([d.reshape(-1), d.conj().T.reshape(-1)])
            S.append(m)
            continue
        for c in comps:
            m = _comp_matrix(c, row, pool) @ m
        S.append(m)
        for c in comps:
            for src in (int(x) for x in c[2:5]):
                if src != P.NO_SRC and src >= 0:
                    grads[src] = (rec[4], abs(rec[5]) - 1, math.copysign(1.0, rec[5]))
        if form == 0:
            mats[off:off + 4] = m.reshape(-1)
        elif form == LF.FORM_PHASE:
            mats[off] = m[1, 1]
    r = plan.r
    R = 1 << r
    for rec in enc.round_recs:
        coef, has_d0 = int(rec[0]), int(rec[1])
        pre, rot, post = (rec[2 + 5 * i:2 + 5 * i + 5] for i in range(3))
        d0, d1, cots = np.ones(R, dtype=np.complex128), np.ones(R, dtype=np.complex128), 0
        for b in range(r):
            one = np.array([(m >> b) & 1 for m in range(R)], dtype=bool)
            for si, d in ((int(pre[b]), d0), (int(post[b]), d1)):
                if si >= 0:
                    d[one] *= S[si][1, 1] * np.conj(S[si][0, 0])
            si = int(rot[b])
            if si < 0:
                continue
            form = int(enc.slot_recs[si][7])
            if form == LF.FORM_EULER:
                eg, c, s, ea = _euler(S[si])
                d0[one] *= eg
                d1[one] *= ea
            else:
                c, s = S[si][0, 0].real, (-S[si][1, 0].imag if form == LF.FORM_X else S[si][1, 0].real)
            cot = abs(s) > abs(c)
            d1 *= s if cot else c
            cots |= int(cot) << b
            mats[coef + R + b] = c / s if cot else s / c
            assert abs(mats[coef + R + b].real) <= 1
        mats[coef:coef + R] = d1
        mats[coef + R + r] = cots
        if has_d0:
            mats[coef + R + r + 1:coef + 2 * R + r + 1] = d0
        else:
            assert np.allclose(d0, 1)
    return mats, grads


def _pairs(R, b, cm=0):
    i = np.array([m for m in range(R) if not m & (1 << b) and (m & cm) == cm])
    return i, i | (1 << b)


def _grad(p, l, b, cm, kind):
    i, j = _pairs(p.shape[1], b, cm)

    def c(x, y):
        return np.sum(np.conj(l[:, x]) * p[:, y])
    return [(c(i, j) + c(j, i)).imag, (c(j, i) - c(i, j)).real, (c(i, i) - c(j, j)).imag, -2 * c(j, j).imag][kind]


def run_lifted(words, n, states, mats, acc):
    """One lifted pass over psi, or psi and lambda (adjoint), in place."""
    k, r, nst = (int(x) for x in words[:3])
    R, adj = 1 << r, len(states) == 2
    tile_bits = [int(b) for b in words[P.HDR_TILE_BITS:P.HDR_TILE_BITS + k]]
    rest = [b for b in range(n) if b not in tile_bits]
    phys = np.array([_pdep(j, tile_bits) for j in range(1 << k)])
    for t in range(1 << (n - k)):
        base = _pdep(t, rest)
        tiles = [s[base + phys].copy() for s in states]
        regs = None
        for i in range(nst):
            st = [int(x) for x in words[LF.HDR_STAGES + LF.STAGE_WORDS * i:LF.HDR_STAGES + LF.STAGE_WORDS * (i + 1)]]
            free = [b for b in range(k) if not (st[LF.W_REGMASK] >> b) & 1]
            tb = np.array([_pdep(x, free) for x in range(1 << (k - r))])[:, None]

            def at(word, st=st, tb=tb):
                return tb + np.array([P.lds_swizzle(x) for x in st[word:word + R]])[None, :]
            if not st[LF.W_FLAGS] & LF.SKIP_READ:
                regs = [x[at(LF.W_IN)] for x in tiles]
            flags, rots = st[LF.W_FLAGS], (st[LF.W_ROT] & 31, (st[LF.W_ROT] >> 8) & 31)
            at1 = st[LF.W_COEF]
            rt, at0 = at1 + R, at1 + R + r + 1
            sign = np.array([1 - 2 * ((st[LF.W_SIGN] >> m) & 1) for m in range(R)])

            def diagonal(flag, at, flags=flags):
                for v in regs if flags & flag else []:
                    d = mats[at:at + R]
                    v *= np.conj(d) if adj else d

            def factor(flags=flags, at1=at1):
                for v in regs if flags & LF.HAS_SCALE else []:
                    assert np.all(mats[at1:at1 + R] == mats[at1].real)
                    v *= mats[at1].real

            def rotations(kind, rots=rots, rt=rt):
                for b in range(r):
                    if not (rots[kind] >> b) & 1:
                        continue
                    q = mats[rt + b].real
                    m = np.array([[q, -1], [1, q]] if (int(mats[rt + r].real) >> b) & 1 else [[1, -q], [q, 1]])
                    m = m.T if adj else m
                    x, y = _pairs(R, b)
                    for v in regs:
                        u, w = v[:, x].copy(), v[:, y].copy()
                        if kind:
                            v[:, x], v[:, y] = m[0, 0] * u + m[0, 1] * w, m[1, 0] * u + m[1, 1] * w
                        else:
                            yi, xr = m[0, 0] * w.imag + m[0, 1] * u.real, m[1, 0] * w.imag + m[1, 1] * u.real
                            xi, yr = m[0, 0] * u.imag + m[0, 1] * w.real, m[1, 0] * u.imag + m[1, 1] * w.real
                            v[:, x], v[:, y] = xr + 1j * xi, yr + 1j * yi

            def general(st=st):
                for o in range(st[LF.W_NGEN]):
                    w = [int(x) for x in words[st[LF.W_GEN] + 8 * o:st[LF.W_GEN] + 8 * o + 8]]
                    typ, dag = w[0] & 255, bool(w[0] & DAG)
                    if typ == LF.OP_PGRAD:
                        val = _grad(regs[0], regs[1], w[1], w[3], w[6] & 15) * (-1 if w[6] >> 4 else 1)
                        acc[w[5]] = acc.get(w[5], np.zeros(8)) + np.array([val] + [0.0] * 7)
                        continue
                    for v in regs:
                        if typ == LF.OP_PHL:
                            idx = [x for x in range(R) if (x & (w[3] | 1 << w[1])) == w[3] | 1 << w[1]]
                            v[:, idx] *= np.conj(mats[w[4]]) if dag else mats[w[4]]
                        elif typ == LF.OP_U2:
                            m = mats[w[4]:w[4] + 16].reshape(4, 4)
                            assert w[1] > w[2]
                            for x in range(R):
                                if not x & (1 << w[1] | 1 << w[2]):
                                    idx = [x, x | 1 << w[2], x | 1 << w[1], x | 1 << w[1] | 1 << w[2]]
                                    v[:, idx] = v[:, idx] @ m.T
                        else:
                            m = mats[w[4]:w[4] + 4].reshape(2, 2)
                            m = m.conj().T if dag else m
                            x, y = _pairs(R, w[1], w[3])
                            v[:, x], v[:, y] = m[0, 0] * v[:, x] + m[0, 1] * v[:, y], m[1, 0] * v[:, x] + m[1, 1] * v[:, y]

            def phase_grads(group, shift, st=st):
                if st[group] < 0:
                    return
                val = acc.setdefault(st[group], np.zeros(8))
                kp = st[LF.W_KINDP] >> (8 if shift == 16 else 0)
                for b in range(r):
                    if (st[LF.W_GRADS] >> shift >> b) & 1:
                        val[4 + b] += _grad(regs[0], regs[1], b, 0, 3 if (kp >> b) & 1 else 2)
            if not adj:
                diagonal(LF.HAS_D0, at0)
                rotations(0)
                rotations(1)
                diagonal(LF.HAS_D1, at1)
                factor()
                general()
                regs = [v * sign for v in regs]
            else:
                regs = [v * sign for v in regs]
                general()
                phase_grads(LF.W_GROUP, 8)
                diagonal(LF.HAS_D1, at1)
                factor()
                rotations(0)
                rotations(1)
                for b in range(r):
                    if (st[LF.W_GRADS] >> b) & 1:
                        acc[st[LF.W_GROUP]][b] += _grad(regs[0], regs[1], b, 0, (rots[1] >> b) & 1)
                phase_grads(LF.W_GROUP_PRE, 16)
                diagonal(LF.HAS_D0, at0)
            if not st[LF.W_FLAGS] & LF.SKIP_WRITE:
                for tile, v in zip(tiles, regs):
                    tile[at(LF.W_OUT)] = v
        for s, tile in zip(states, tiles):
            s[base + phys] = tile


def lifted_value_and_grad(circ, values, zfun, k, r):
    n, units, npar, pool = lower_circuit(circ.compilecircuit(backend="pytorch"))
    runs = []
    for lift in ("fwd", True):                  # the forward-only plan, whose trained gates may be fused, too
        plan = build_plan(n, units, npar, list(pool), k_max=k, r=r, lift=lift)
        enc = P.encode_plan(plan)
        mats, where = tables(enc, plan, np.asarray(values))
        psi = np.zeros(2 ** n, dtype=np.complex128)
        psi[0] = 1
        for off in enc.fwd_offsets:
            run_lifted(enc.prog[off:], n, [psi], mats, {})
        runs.append(psi)
    ph = np.vdot(runs[0], runs[1])
    assert abs(abs(ph) - 1) < 1e-10 and np.allclose(runs[0] * ph, runs[1], atol=1e-10)
    out, lam, acc = psi.copy(), zfun * psi, {}
    for off in enc.adj_offsets:
        run_lifted(enc.prog[off:], n, [psi, lam], mats, acc)
    e0 = np.zeros(2 ** n)
    e0[0] = 1
    assert abs(abs(psi[0]) - 1) < 1e-10 and np.allclose(psi * np.conj(psi[0]), e0, atol=1e-10)   # walked back
    grad = np.array([where[p][2] * acc[where[p][0]][where[p][1]] for p in range(npar)])
    assert all(int(enc.pgslot[p]) == where[p][0] for p in range(npar))
    return out, grad, plan


def check(n, spec, values, k, r, rng):
    circ = trace(n, spec, values, lambda: qai.expval(qai.PauliZ(qubits=[0])))
    z = rng.normal(size=2 ** n)
    psi, grad, plan = lifted_value_and_grad(circ, values, z, k, r)
    ref = O.propagate(n, oracle_gates(spec, values)).numpy().reshape(-1)
    ph = np.vdot(psi, ref)
    assert abs(abs(ph) - 1) < 1e-10 and np.allclose(psi * ph, ref, atol=1e-10)
    t = torch.tensor(values, dtype=torch.float64, requires_grad=True)
    out = O.propagate(n, oracle_gates(spec, list(t))).reshape(-1)
    (out.abs() ** 2 * torch.tensor(z)).sum().backward()
    assert np.allclose(grad, t.grad.numpy(), atol=1e-9)
    return plan


@pytest.mark.parametrize("seed,n,k,r", [(0, 5, 3, 2), (1, 6, 4, 3), (2, 7, 5, 4), (3, 6, 6, 4), (4, 8, 5, 2), (5, 3, 3, 1),
                                        (6, 9, 7, 4), (7, 8, 8, 3), (8, 4, 4, 4)])
def test_lifted_plan_of_random_circuits(seed, n, k, r):
    rng = np.random.default_rng(seed)
    spec = random_spec(n, 60, rng) + [("Rot", [0], 3)]
    values = [float(x) for x in rng.uniform(-2 * math.pi, 2 * math.pi, sum(s[2] for s in spec))]
    check(n, spec, values, k, r, rng)


@pytest.mark.parametrize("angle", [0.0, math.pi, -math.pi, 2 * math.pi, math.pi / 2, 3 * math.pi / 2, 3 * math.pi, 1e-9])
def test_lifted_rotations_at_the_ends_of_the_tangent_range(angle):
    """Angles where cos vanishes or changes sign, where a rotation is the identity, and where it is -1."""
    spec = [("Hadamard", [0], 0), ("RX", [0], 1), ("RZ", [0], 1), ("CNOT", [0, 1], 0), ("RY", [1], 1), ("PhaseShift", [1], 1),
            ("Rot", [0], 3), ("ControlledPhaseShift", [0, 1], 1), ("SX", [1], 0), ("CRX", [1, 0], 1), ("PauliY", [0], 0)]
    values = [angle] * sum(s[2] for s in spec)
    check(2, spec, values, 2, 2, np.random.default_rng(3))


def test_lifted_plan_makes_user_matrices_dense_and_keeps_registers_between_rounds():
    """Consecutive two-qubit user matrices on a pair are one dense op, also with the qubits reversed, and a
    one-qubit user matrix keeps its 2x2; rounds of one stage without a permutation skip the LDS exchange."""
    rng = np.random.default_rng(5)

    def unitary(d):
        return np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))[0]
    a, b, c, v = unitary(4), unitary(4), unitary(4), unitary(2)
    vals = [0.3, -0.7, 1.1, 2.9]

    def circuit_def():
        qai.RX(vals[0], qubits=[0])
        qai.Unitary(a, qubits=[0, 1])
        qai.Unitary(b, qubits=[0, 1])
        qai.RY(vals[1], qubits=[1])
        qai.Unitary(c, qubits=[2, 1])
        qai.Unitary(v, qubits=[2])
        qai.RZ(vals[2], qubits=[2])
        qai.RX(vals[3], qubits=[2])
        return qai.expval(qai.PauliZ(qubits=[0]))
    z = rng.normal(size=8)
    psi, grad, plan = lifted_value_and_grad(qai.Circuit(circuit_def, 3), vals, z, 3, 3)

    def gates(t):
        return [("RX", [0], [t[0]]), (a, [0, 1], []), (b, [0, 1], []), ("RY", [1], [t[1]]), (c, [2, 1], []), (v, [2], []),
                ("RZ", [2], [t[2]]), ("RX", [2], [t[3]])]

    def apply(t):
        state = torch.zeros(8, dtype=torch.complex128)
        state[0] = 1
        for g, qs, ps in gates(t):
            m = O.gate_matrix(g, ps) if isinstance(g, str) else torch.as_tensor(g)
            m = m.reshape([2] * (2 * len(qs))).to(torch.complex128)
            s = torch.tensordot(m, state.reshape(2, 2, 2), (list(range(len(qs), 2 * len(qs))), qs))
            order = qs + [q for q in range(3) if q not in qs]
            state = s.permute([order.index(q) for q in range(3)]).reshape(-1)
        return state
    t = torch.tensor(vals, dtype=torch.float64, requires_grad=True)
    ref = apply(t)
    (ref.abs() ** 2 * torch.tensor(z)).sum().backward()
    ph = np.vdot(psi, ref.detach().numpy())
    assert abs(abs(ph) - 1) < 1e-10 and np.allclose(psi * ph, ref.detach().numpy(), atol=1e-10)
    assert np.allclose(grad, t.grad.numpy(), atol=1e-9)
    rounds = [rd for p in plan.rounds for rd in p]
    assert sum(1 for rd in rounds for op in rd.gen if op[0] == "u2") == 2       # a and b in one
    assert len(rounds) > 1 and not any(rd.moves for rd in rounds)
    words = P.encode_plan(plan).prog
    flags = [int(words[LF.HDR_STAGES + LF.STAGE_WORDS * i]) for i in range(len(rounds))]
    assert all(f & LF.SKIP_WRITE for f in flags[:-1])
    assert flags[-1] & (LF.SKIP_READ | LF.SKIP_WRITE | LF.BARRIER) == LF.SKIP_READ | LF.BARRIER


@pytest.mark.parametrize("last", ["matrix", "controlled", "rotation"])
def test_every_round_leaves_a_whole_row_to_read_ahead(last):
    """The kernels read 2^r + r + 1 table entries of the next round before they know whether it uses them: also
    for rounds of general ops only (no row of their own), the last of them at the end of the table."""
    rng = np.random.default_rng(2)
    u = np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))[0]

    def circuit_def():
        qai.Unitary(u, qubits=[0, 1])
        qai.RY(0.4, qubits=[2])
        if last == "matrix":
            qai.Unitary(u, qubits=[2, 3])
            qai.Unitary(u, qubits=[1, 2])
        elif last == "controlled":
            qai.CRX(0.3, qubits=[0, 3])
        return qai.expval(qai.PauliZ(qubits=[0]))
    n, units, npar, pool = lower_circuit(qai.Circuit(circuit_def, 4).compilecircuit(backend="pytorch"))
    for lift in ("fwd", True):
        for k, r in ((4, 4), (3, 2), (2, 1)):
            plan = build_plan(n, units, npar, list(pool), k_max=k, r=r, lift=lift)
            enc = P.encode_plan(plan)
            for off in list(enc.fwd_offsets) + list(enc.adj_offsets):
                for s in range(int(enc.prog[off + 2])):
                    st = enc.prog[off + P.HDR_STAGES + LF.STAGE_WORDS * s:]
                    assert 0 <= st[LF.W_COEF] <= plan.mat_stride - ((1 << r) + r + 1)
