"""Runs of gates on one large tensor (tedq_amd.tn.runs, tedq_tn_run_*).

On the CPU the encoded passes are executed by a numpy model of the kernels
(same words, slots, address bits and matrices) and compared with the
step-by-step contraction of the same network; on the GPU the kernels are
compared with the step-by-step kernels and the oracle's gradients at the
sizes where a tile, an op or a layout changes form.

Tolerances: a value is a sum of unit-norm amplitudes with fp32 rounding of
at most ~2e-7 per gate and random sign, so a few hundred gates stay below
1e-5 of the scale; both sides of a comparison carry that.
"""

import ctypes

import numpy as np
import pytest
import torch

import tedq_amd as qai
from tedq_amd.engine import hip
from tedq_amd.tn import runs as R
from tedq_amd.tn.executor import TNExecutor, make_desc

from tn_emulator import contract_np, install

TOL = 1e-5


def lattice(rows, cols, layers, obs, simplify):
    n = rows * cols
    bonds = [(r * cols + c, r * cols + c + 1) for r in range(rows) for c in range(cols - 1)]
    bonds += [(r * cols + c, (r + 1) * cols + c) for r in range(rows - 1) for c in range(cols)]

    def cd(*p):
        it = iter(p)
        for _ in range(layers):
            for q in range(n):
                qai.RX(next(it), qubits=[q])
                qai.RZ(next(it), qubits=[q])
            for a, b in bonds:
                qai.CZ(qubits=[a, b])
        return [qai.expval(qai.PauliZ(qubits=[obs]))]
    return qai.Circuit(cd, n, *([0.1] * (2 * n * layers))).compilecircuit(backend="pytorch", tn_mode=True,
                                                                          tn_simplify=simplify), 2 * n * layers


def chain(n, layers, simplify):
    zz = np.diag(np.exp(-0.1j * np.array([1, -1, -1, 1])))
    xy = np.eye(4, dtype=complex)
    xy[1:3, 1:3] = [[np.cos(0.2), -1j * np.sin(0.2)], [-1j * np.sin(0.2), np.cos(0.2)]]

    def cd(*p):
        it = iter(p)
        for _ in range(layers):
            for q in range(n):
                qai.RZ(next(it), qubits=[q])
                qai.RY(next(it), qubits=[q])
            for q in range(n - 1):
                qai.Unitary(zz, qubits=[q, q + 1])
                qai.Unitary(xy, qubits=[q, q + 1])
        return [qai.expval(qai.PauliZ(qubits=[n // 2]))]
    return qai.Circuit(cd, n, *([0.1] * (2 * n * layers))).compilecircuit(backend="pytorch", tn_mode=True,
                                                                      tn_simplify=simplify), 2 * n * layers


def rows_for(n_params, batch, seed):
    rng = np.random.default_rng(seed)
    return torch.tensor(rng.uniform(0, 2 * np.pi, size=(batch, n_params)), dtype=torch.float32)


# --- numpy model of the kernels ------------------------------------------------
def _offsets(count, bits):
    i = np.arange(1 << count)
    return sum(((i >> k) & 1) << int(bits[k]) for k in range(count)) if count else np.zeros(1, dtype=int)


def _matrix(w, bases):
    a = int(w[0])
    m = np.zeros((1 << a, 1 << a), dtype=np.complex128)
    for out in range(1 << a):
        for inn in range(1 << a):
            if (inn ^ out) & int(w[4]):
                continue
            for z in range(1 << int(w[5])):
                v = inn | out << 3 | z << 6
                p = 1.0
                for f in range(int(w[6])):
                    d = w[12 + 10 * f:]
                    off = sum(((v >> int(d[3 + i])) & 1) << i for i in range(int(d[2])))
                    p = p * bases[int(d[0])][int(d[1]) + off]
                m[out, inn] += p
    return m


def _op_index(w, n_local):
    slots = [int(x) for x in w[1:1 + int(w[0])]]
    rest = [s for s in range(n_local) if s not in slots]
    return _offsets(len(rest), rest)[:, None] | _offsets(len(slots), slots)[None, :]


def emulate(ex):
    install(ex)
    ex._use_runs = lambda dev: ex.run_passes and ex.small_batch  # pylint: disable=protected-access

    def coefs(plan, small, arena, leaves, buf, B, dev):  # pylint: disable=unused-argument
        consts = buf["consts"].numpy().astype(np.complex128)
        return [[_matrix(w, (leaves[b].numpy().astype(np.complex128), consts,
                             arena[b].numpy().astype(np.complex128))) for w in plan["ops"]] for b in range(B)]

    def forward(run, plan, coef, x, B, dev, keep):  # pylint: disable=unused-argument
        outs = []
        cur = x[0].reshape(B, -1)[:, x[2]:x[2] + (1 << run.wires)].numpy().astype(np.complex128)
        for ps in run.passes:
            L, no, ops = (int(v) for v in ps.words[:3])
            res = np.full_like(cur, np.nan)
            oin, oout = _offsets(no, ps.words[40:]), _offsets(no, ps.words[72:])
            lin, lout, lslot = (_offsets(L, ps.words[k:]) for k in (4, 28, 16))
            for b in range(B):
                tile = cur[b][oin[:, None] | lin[None, :]]
                for k in range(ops):
                    idx = _op_index(plan["ops"][ps.head + k], L)
                    tile[:, idx] = np.einsum("qk,trk->trq", coef[b][ps.head + k], tile[:, idx])
                res[b][oout[:, None] | lout[None, :]] = tile[:, lslot]
            cur = res
            outs.append(torch.from_numpy(res.astype(np.complex64)))
        return outs if keep else outs[-1:]

    def backward(run, plan, coef, outs, env, env_arena, env_small, B, dev):  # pylint: disable=unused-argument
        e = env[0].reshape(B, -1)[:, env[2]:env[2] + (1 << run.wires)].numpy().astype(np.complex128)
        arenas = (env_arena.numpy(), env_small.numpy())
        for ps, c in zip(reversed(run.passes), reversed(outs)):
            L, no, ops = (int(v) for v in ps.words[:3])
            oin, oout = _offsets(no, ps.words[40:]), _offsets(no, ps.words[72:])
            lin, lout, lslot = (_offsets(L, ps.words[k:]) for k in (4, 28, 16))
            res = np.full_like(e, np.nan)
            for b in range(B):
                xt = np.zeros((1 << no, 1 << L), dtype=np.complex128)
                et = xt.copy()
                at = oout[:, None] | lout[None, :]
                xt[:, lslot] = c.numpy()[b].astype(np.complex128)[at]
                et[:, lslot] = e[b][at]
                for k in reversed(range(ops)):
                    w, m = plan["ops"][ps.head + k], coef[b][ps.head + k]
                    idx = _op_index(w, L)
                    xt[:, idx] = np.einsum("qk,trq->trk", m.conj(), xt[:, idx])
                    g = np.einsum("trq,trk->qk", et[:, idx], xt[:, idx])
                    et[:, idx] = np.einsum("qk,trq->trk", m, et[:, idx])
                    if int(w[8]) < 0:
                        continue
                    d = w[12:]
                    for o in range(1 << int(d[2])):
                        v = sum(((o >> i) & 1) << int(d[3 + i]) for i in range(int(d[2])))
                        arenas[int(w[8])][b, int(w[9]) + o] = sum(
                            g[((v >> 3) & 7) | z, (v & 7) | z] for z in range(1 << int(w[0])) if not z & ~int(w[4]))
                res[b][oin[:, None] | lin[None, :]] = et
            e = res
        return torch.from_numpy(e.astype(np.complex64))

    def small_backward(net, arena, env_small, env_arena, leaves, buf, B, dev):  # pylint: disable=unused-argument
        env = ex._small_env_plan(net)  # pylint: disable=protected-access
        bases = [leaves.numpy(), np.broadcast_to(buf["consts"].numpy(), (B, buf["consts"].numel())), arena.numpy(),
                 env_small.numpy(), env_arena.numpy()]
        for s, e in env["bounds"]:
            for row, ia, oa, ib, ob, oc, size, ic in env["recs"][s:e]:
                desc = ex._descs[row]  # pylint: disable=protected-access
                nh, nm, nn, nk = (int(v) for v in desc[:4])
                out = np.zeros((B, size), dtype=np.complex128)
                contract_np(desc, bases[ia][:, oa:oa + (1 << (nh + nm + nk))].astype(np.complex128),
                            bases[ib][:, ob:ob + (1 << (nh + nk + nn))].astype(np.complex128), out)
                bases[ic][:, oc:oc + size] = out

    # pylint: disable=protected-access
    ex._run_coefs, ex._run_forward_passes, ex._run_backward_passes = coefs, forward, backward
    ex._batch_small_backward, ex._small_backward = (lambda dev: ex.small_batch), small_backward
    return ex


def _run_ops(ex, grad):
    return [op for net in ex.networks for run in ex._run_plan(net, grad)["first"].values()  # pylint: disable=protected-access
            for ps in run.passes for op in ps.ops]


# gates merged to one, two and three bits; hyper-indices (simplify) with several factors per op;
# a last pass whose result layout differs
@pytest.mark.parametrize("build,args,grad", [
    (lattice, (3, 4, 4, 5, False), True), (lattice, (4, 4, 3, 5, False), True), (lattice, (4, 4, 2, 5, True), False),
    (chain, (14, 4, True), False), (chain, (13, 4, False), True)])
def test_passes_equal_the_steps(build, args, grad):
    cc, npar = build(*args)
    rows = rows_for(npar, 2, 7)
    # the circuit-order sweep: a state-like intermediate at every size
    ex = emulate(TNExecutor(cc, trials=(), diagonal_reduction=args[-1]))
    plain = install(TNExecutor(cc, trials=(), diagonal_reduction=args[-1]))
    ex.SMALL_RANK = 6          # keep the batched small steps to gate merges, so that the rest is a run
    assert _run_ops(ex, grad), "the network has no run"
    got = ex.measure(ex.run_forward(rows))[0].numpy()
    want = plain.measure(plain.run_forward(rows))[0].numpy()
    assert np.max(np.abs(got - want)) < TOL
    if grad:
        up = [torch.ones(2)]
        (v, g), (_, gw) = ex.value_and_grad(rows, up), plain.value_and_grad(rows, up)
        assert np.max(np.abs(v[0].numpy() - want)) < TOL
        assert np.max(np.abs(g.numpy() - gw.numpy())) < TOL * max(1.0, float(gw.abs().max()))


def test_a_matrix_that_is_not_unitary_is_not_undone():
    """The backward recovers an op's input from its result only for unitary matrices."""
    n = 10
    skew = np.array([[1.0, 0.5], [0.0, 1.0]], dtype=complex)

    def cd(*p):
        it = iter(p)
        for _ in range(3):
            for q in range(n):
                qai.RX(next(it), qubits=[q])
            for q in range(n - 1):
                qai.CNOT(qubits=[q, q + 1])
            for q in range(n):
                qai.Unitary(skew, qubits=[q])
        return [qai.expval(qai.PauliZ(qubits=[n // 2]))]
    cc = qai.Circuit(cd, n, *([0.1] * (3 * n))).compilecircuit(backend="pytorch", tn_mode=True, tn_simplify=False)
    rows = rows_for(3 * n, 1, 3)
    ex, plain = emulate(TNExecutor(cc, trials=())), install(TNExecutor(cc, trials=()))
    (v, g), (vw, gw) = ex.value_and_grad(rows, [torch.ones(1)]), plain.value_and_grad(rows, [torch.ones(1)])
    scale = max(1.0, float(vw[0].abs().max()), float(gw.abs().max()))
    assert abs(float(v[0][0] - vw[0][0])) < TOL * scale
    assert np.max(np.abs(g.numpy() - gw.numpy())) < TOL * scale


# --- kernels --------------------------------------------------------------------
def _random_run(n, arities, seed, permute):
    """A run of random unitary ops on n wires: plan, factors (arena values) and pass words."""
    rng = np.random.default_rng(seed)
    ops, arena = [], []
    for a in arities:
        w = sorted(int(x) for x in rng.choice(n, size=a, replace=False))
        ins, outs = [f"i{len(ops)}.{k}" for k in range(a)], [f"o{len(ops)}.{k}" for k in range(a)]
        q, _ = np.linalg.qr(rng.normal(size=(1 << a, 1 << a)) + 1j * rng.normal(size=(1 << a, 1 << a)))
        op = R.Op(ins, outs, [len(ops)], [], w)
        op.in_wire, op.out_wire = dict(zip(ins, w)), dict(zip(outs, w))
        ops.append(op)
        arena.append(q.reshape(-1))
    lay = [list(reversed(op.outs)) + list(reversed(op.ins)) for op in ops]   # [out][in], most significant first
    offs = np.concatenate([[0], np.cumsum([v.size for v in arena])]).astype(int)
    out_bit = [int(x) for x in rng.permutation(n)] if permute else list(range(n))
    run = R.Run(0, 1, [], n, out_bit, R._split_passes(list(ops), n))  # pylint: disable=protected-access
    rows = R.encode_run(run, lambda t: (0, int(offs[t])), lay)
    order = [op for ps in run.passes for op in ps.ops]
    coef = head = 0
    for ps in run.passes:
        ps.head = head
        head += len(ps.ops)
        for row in rows[ps.head:head]:
            row[7] += coef
            row[8], row[9] = row[13] % 2, row[13]          # either environment arena, at the leaf's offset
        coef += int(ps.words[3])
    plan = {"ops": np.array(rows, dtype=np.int32), "coef": coef, "dev": {}}
    return run, plan, np.concatenate(arena), order, offs


@pytest.mark.gpu
@pytest.mark.parametrize("n,arities,batch,permute", [
    (9, [2, 3, 1, 2], 1, False), (9, [1, 1], 3, True), (10, [3, 3, 2], 2, True), (11, [2] * 6, 1, False),
    (12, [1, 2, 3] * 4, 2, True), (13, [2] * 40, 1, True), (15, [2, 3] * 8, 3, False), (20, [2] * 20, 1, True)])
def test_run_kernels_vs_reference(n, arities, batch, permute):
    """Passes forward and backward against float64: results, recovered input's environment and gate
    environments.  Up to 40 unitary ops of fp32 matrices: 40 * 2e-7 of the largest entry's scale."""
    dev = torch.device("cuda", 0)
    run, plan, arena, order, offs = _random_run(n, arities, n, permute)
    rng = np.random.default_rng(1)
    x = rng.normal(size=(batch, 1 << n)) + 1j * rng.normal(size=(batch, 1 << n))
    e = rng.normal(size=(batch, 1 << n)) + 1j * rng.normal(size=(batch, 1 << n))
    leaves = torch.tensor(np.tile(arena, (batch, 1)), dtype=torch.complex64, device=dev)
    ex = TNExecutor.__new__(TNExecutor)
    ex.leaf_stride = arena.size
    small = {"len": arena.size}
    buf = {"consts": torch.zeros(2, dtype=torch.complex64, device=dev)}
    # pylint: disable=protected-access
    coef = ex._run_coefs(plan, small, leaves, leaves, buf, batch, dev)
    tx = torch.tensor(x, dtype=torch.complex64, device=dev)
    outs = ex._run_forward_passes(run, plan, coef, (tx, tx.shape[1], 0), batch, dev, True)
    last = ex._run_forward_passes(run, plan, coef, (tx, tx.shape[1], 0), batch, dev, False)[-1]
    assert torch.equal(outs[-1], last)
    te = torch.tensor(e, dtype=torch.complex64, device=dev)
    envs = [torch.zeros((batch, arena.size), dtype=torch.complex64, device=dev) for _ in range(2)]
    ein = ex._run_backward_passes(run, plan, coef, outs, (te, te.shape[1], 0), envs[0], envs[1], batch, dev)
    # float64 reference: wires as axes, one op after the other in the order of the passes
    src = np.zeros(1 << n, dtype=int)
    for w in range(n):
        src |= ((np.arange(1 << n) >> w) & 1) << run.out_bit[w]
    states = [tx.cpu().numpy().astype(np.complex128)]
    for op in order:
        m = arena[offs[op.factors[0]]:offs[op.factors[0] + 1]].reshape(1 << len(op.wires), -1)
        states.append(_apply(states[-1], m, op.wires, n))
    scale = np.abs(states[-1]).max()
    assert np.max(np.abs(last.cpu().numpy()[:, src] - states[-1])) < TOL * scale
    env = te.cpu().numpy().astype(np.complex128)[:, src]
    got = [v.cpu().numpy() for v in envs]
    for k in range(len(order) - 1, -1, -1):
        op, t = order[k], order[k].factors[0]
        m = arena[offs[t]:offs[t + 1]].reshape(1 << len(op.wires), -1)
        D = m.shape[0]
        want = np.einsum("brq,brk->bqk", _rows(env, op.wires, n), _rows(states[k], op.wires, n)).reshape(batch, D * D)
        base = int(offs[t]) % 2
        g = got[base][:, offs[t]:offs[t + 1]]
        # a sum of 2^n products of unit normals: its rounding scales with sqrt(2^n)
        assert np.max(np.abs(g - want)) < TOL * 4 * 2 ** (n / 2) * np.sqrt(n), (k, op.wires)
        env = _apply(env, m.T, op.wires, n)
    assert np.max(np.abs(ein.cpu().numpy() - env)) < TOL * np.abs(env).max()


def _index(wires, n):
    rest = [w for w in range(n) if w not in wires]
    return _offsets(len(rest), rest)[:, None] | _offsets(len(wires), wires)[None, :]


def _rows(x, wires, n):
    return x[:, _index(wires, n)]


def _apply(x, m, wires, n):
    out = np.empty_like(x)
    idx = _index(wires, n)
    out[:, idx] = x[:, idx] @ m.T
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("na,nb,nk,batch", [(0, 0, 0, 1), (0, 0, 12, 2), (2, 2, 10, 3), (1, 0, 11, 1), (4, 4, 8, 2),
                                            (6, 6, 6, 1), (11, 1, 1, 2), (3, 9, 0, 1)])
def test_small_environments_vs_reference(na, nb, nk, batch):
    """One step per shape: few outputs over long sums (lanes per output, k past the table), many outputs;
    sums of 2^nk products of unit normals, fp32: 2^(nk/2) * 1e-6 of their scale."""
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(nk)
    la = [f"m{i}" for i in range(na)] + [f"k{i}" for i in range(nk)]
    lb = [f"k{i}" for i in range(nk)] + [f"n{i}" for i in range(nb)]
    lc = [f"m{i}" for i in range(na)] + [f"n{i}" for i in range(nb)]
    la, lb, lc = (list(rng.permutation(v)) for v in (la, lb, lc))
    desc = make_desc(la, lb, lc)
    a = rng.normal(size=(batch, 1 << (na + nk))) + 1j * rng.normal(size=(batch, 1 << (na + nk)))
    b = rng.normal(size=(batch, 1 << (nb + nk))) + 1j * rng.normal(size=(batch, 1 << (nb + nk)))
    ta, tb = (torch.tensor(v, dtype=torch.complex64, device=dev) for v in (a, b))
    outs = [torch.zeros((batch, (1 << (na + nb)) + 3), dtype=torch.complex64, device=dev) for _ in range(2)]
    ten = [ta, tb, outs[0], outs[1], outs[1]]
    bases = (ctypes.c_void_p * 5)(*[t.data_ptr() for t in ten])
    sizes = (ctypes.c_int64 * 5)(*[t.shape[1] for t in ten])
    recs = np.array([[0, 0, 0, 1, 0, 3, 1 << (na + nb), 2], [0, 0, 0, 1, 0, 1, 1 << (na + nb), 4]], dtype=np.int64)
    drecs, ddesc = torch.from_numpy(recs).to(dev), torch.from_numpy(desc).to(dev)
    hip.call("tedq_tn_small_environments", bases, sizes, sizes, recs.ctypes.data_as(hip.c_vp), hip.ptr(drecs), 2, batch,
             desc.ctypes.data_as(hip.c_vp), hip.ptr(ddesc), 1, hip.stream_handle(dev))
    want = np.zeros((batch, 1 << (na + nb)), dtype=np.complex128)
    contract_np(desc, ta.cpu().numpy().astype(np.complex128), tb.cpu().numpy().astype(np.complex128), want)
    tol = 2 ** (nk / 2) * 1e-6 * 8
    assert np.max(np.abs(outs[0][:, 3:].cpu().numpy() - want)) < tol
    assert np.max(np.abs(outs[1][:, 1:-2].cpu().numpy() - want)) < tol


@pytest.mark.gpu
@pytest.mark.parametrize("build,args,grad,batch", [
    (lattice, (3, 4, 4, 5, False), True, 3), (lattice, (4, 4, 4, 5, False), True, 2),
    (lattice, (4, 5, 4, 9, False), True, 1), (chain, (20, 5, True), False, 4), (chain, (14, 4, False), True, 2)])
def test_networks_with_and_without_runs(build, args, grad, batch):
    """Whole networks on the device, runs on and off: values, and gradients where the runs have them."""
    dev = torch.device("cuda", 0)
    cc, npar = build(*args)
    rows = rows_for(npar, batch, 11).to(dev)
    ex = TNExecutor(cc)
    res = []
    for on in (True, False):
        ex.run_passes = on
        v = ex.measure(ex.run_forward(rows))[0]
        res.append((v,) + ((ex.value_and_grad(rows, [torch.ones(batch, device=dev)])[1],) if grad else ()))
    for a, b in zip(*res):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("args", [(3, 3, 2, 4, False), (4, 4, 4, 5, False), (3, 4, 3, 5, True)])
def test_backward_from_a_kept_forward(args):
    """A forward that keeps its intermediates serves one backward; a second backward through the same graph
    and a forward that kept nothing contract again: the same launches on the same values, so equal bits."""
    dev = torch.device("cuda", 0)
    cc, npar = lattice(*args)
    rows = rows_for(npar, 2, 5).to(dev)
    ex = TNExecutor(cc)
    up = [torch.ones(2, device=dev)]
    grads = []
    for need in (True, False):
        run = ex.run_forward(rows, need_grad=need)
        assert (run["kept"][0] is not None) == need
        for _ in range(2):
            grads.append(ex.run_backward(rows, run, ex.seed_adjoint(run, up)))
            assert run["kept"][0] is None
    assert all(torch.equal(grads[0], g) for g in grads[1:])
    assert float(grads[0].abs().max()) > 1e-3
