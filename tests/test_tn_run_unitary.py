"""Which gates the backward of runs may undo (tedq_amd.tn.runs.Unitarity).

The backward of a run recovers an op's input as M^H of its result, so every
matrix of a backward run has to be unitary.  Diagonal reduction stores a
diagonal gate as its diagonal and a controlled gate per control value: such a
leaf is no map between the halves of its indices, whatever its rank.

Tolerance of M^H M = 1: the matrices are products of complex64 entries, whose
rounding of 6e-8 per entry gives at most 4 * 8 * 6e-8 = 2e-6 for an 8 x 8
matrix.  Gradients: as in test_tn_runs.
"""

import numpy as np
import pytest
import torch

import tedq_amd as qai
from tedq_amd.tn import runs as R
from tedq_amd.tn.executor import TNExecutor

from test_tn_runs import TOL, _apply, _rows, chain, emulate, lattice, rows_for
from tn_emulator import install

UNITARY_TOL = 2e-6
_DIAG = np.diag(np.exp(1j * np.array([0.1, 0.7, -0.4, 0.9])))


def grid(n, width):
    return [(q, q + 1) for q in range(n - 1) if (q + 1) % width] + [(q, q + width) for q in range(n - width)]


def circuit(gate, n, width, layers, obs):
    """Layers of RX on every qubit, then ``gate`` on every bond of a grid (Toffoli: also on the next qubit)."""
    bonds = grid(n, width)
    trained = gate in ("CRZ", "ControlledPhaseShift")
    n_params = layers * (n + (len(bonds) if trained else 0))

    def cd(*p):
        it = iter(p)
        for _ in range(layers):
            for q in range(n):
                qai.RX(next(it), qubits=[q])
            for a, b in bonds:
                if gate == "Unitary":
                    qai.Unitary(_DIAG, qubits=[a, b])
                elif gate == "Toffoli":
                    qai.Toffoli(qubits=[a, b, next(q % n for q in (b + 1, b + 2) if q % n not in (a, b))])
                else:
                    getattr(qai, gate)(*([next(it)] if trained else []), qubits=[a, b])
        return [qai.expval(qai.PauliZ(qubits=[obs]))]
    return qai.Circuit(cd, n, *([0.1] * n_params)).compilecircuit(backend="pytorch", tn_mode=True), n_params


class _Offered(R.Unitarity):
    """Counts the ops with a reduced leaf that the selection was asked about; no such leaf has halves."""
    reduced = 0

    def __init__(self, net, leaf_unitary):
        super().__init__(net, leaf_unitary)
        for t, src in enumerate(net.sources):
            if self._reduced(t):
                assert self.halves(t) is None, (src, net.lay[t])

    def _reduced(self, t):
        src = self.net.sources[t]
        return src[0] in ("gate", "adj") and len(self.net.lay[t]) < 2 * self.qubits[src[1]]

    def _leaves(self, tid):
        if tid < self.net.n_inputs:
            return [tid]
        st = self.maker[tid]
        return self._leaves(st.a) + self._leaves(st.b)

    def __call__(self, tid, summed):
        _Offered.reduced += any(self._reduced(t) for t in self._leaves(tid))
        return super().__call__(tid, summed)


def _backward_matrices(ex, rows):
    """The matrices of every backward run, and the number of forward run ops (``ex`` emulated)."""
    leaves, _ = ex._leaves(rows)  # pylint: disable=protected-access
    buf, mats, forward = ex._buffers(None), [], 0  # pylint: disable=protected-access
    for net in ex.networks:
        small = ex._small_plan(net)  # pylint: disable=protected-access
        arena = torch.zeros((1, small["len"]), dtype=torch.complex64)
        ex._small_levels(small, arena, leaves, buf, 1, None)  # pylint: disable=protected-access
        plan = ex._run_plan(net, True)  # pylint: disable=protected-access
        mats += ex._run_coefs(plan, small, arena, leaves, buf, 1, None)[0]  # pylint: disable=protected-access
        forward += len(ex._run_plan(net, False)["ops"])  # pylint: disable=protected-access
    return mats, forward


# default options (the reduction is chosen by the path model), then reduction forced; the last two have merged
# controls of one wire (rank 3: the small steps kept to gate merges) and of two (rank 4)
@pytest.mark.parametrize("gate,n,width,layers,obs,forced", [
    ("CRZ", 19, 4, 3, 9, False), ("CRZ", 17, 4, 4, 8, False), ("CRZ", 21, 5, 3, 11, False),
    ("ControlledPhaseShift", 19, 4, 3, 9, False), ("CZ", 19, 4, 3, 9, False), ("Unitary", 17, 4, 4, 8, False),
    ("CRZ", 16, 4, 4, 8, True), ("ControlledPhaseShift", 15, 5, 4, 7, True), ("CNOT", 17, 4, 3, 8, True),
    ("Toffoli", 12, 4, 4, 6, True)])
def test_backward_runs_hold_unitary_matrices(gate, n, width, layers, obs, forced, monkeypatch):
    cc, n_params = circuit(gate, n, width, layers, obs)
    rows = rows_for(n_params, 1, 3)
    opts = {"diagonal_reduction": True} if forced else {}
    ex, plain = emulate(TNExecutor(cc, **opts)), install(TNExecutor(cc, **opts))
    assert ex.simplify
    if forced:
        ex.SMALL_RANK = 6
    _Offered.qubits = {idx: len(op.qubits) for idx, op in cc._operators.items()}  # pylint: disable=protected-access
    _Offered.reduced = 0
    monkeypatch.setattr(R, "Unitarity", _Offered)
    mats, forward = _backward_matrices(ex, rows)
    assert forward, "the network has no run"
    assert _Offered.reduced, "no op with a reduced leaf was offered to the backward"
    for m in mats:
        assert np.max(np.abs(m.conj().T @ m - np.eye(len(m)))) < UNITARY_TOL
    up = [torch.ones(1)]
    monkeypatch.undo()
    (v, g), (vw, gw) = ex.value_and_grad(rows, up), plain.value_and_grad(rows, up)
    assert abs(float(v[0][0] - vw[0][0])) < TOL
    assert float((g - gw).abs().max()) < TOL * max(1.0, float(gw.abs().max()))


def test_a_matrix_near_a_unitary_one_is_not_undone():
    """Four copies per layer of a matrix that is unitary but for a factor of 1 + 4.5e-7: undone, each adds 9e-7
    of the gradients of the gates before it.  The two paths round about 800 results to complex64 with random
    sign: 800^(1/2) * 6e-8 = 1.7e-6 of the gradients' scale, within 4e-6."""
    n, layers, copies = 10, 8, 4
    near = (1 + 4.5e-7) * np.array([[np.cos(0.3), -np.sin(0.3)], [np.sin(0.3), np.cos(0.3)]])

    def cd(*p):
        it = iter(p)
        for _ in range(layers):
            for q in range(n):
                qai.RX(next(it), qubits=[q])
            for q in range(n - 1):
                qai.CNOT(qubits=[q, q + 1])
            for q in list(range(n)) * copies:
                qai.Unitary(near, qubits=[q])
        return [qai.expval(qai.PauliZ(qubits=[n // 2]))]
    cc = qai.Circuit(cd, n, *([0.1] * (layers * n))).compilecircuit(backend="pytorch", tn_mode=True,
                                                                     tn_simplify=False)
    rows, up = rows_for(layers * n, 1, 3), [torch.ones(1)]
    ex, plain = emulate(TNExecutor(cc, trials=())), install(TNExecutor(cc, trials=()))
    ex.SMALL_RANK = 4
    assert ex._run_plan(ex.networks[0], False)["first"], "the network has no run"  # pylint: disable=protected-access
    (v, g), (vw, gw) = ex.value_and_grad(rows, up), plain.value_and_grad(rows, up)
    assert abs(float(v[0][0] - vw[0][0])) < 4e-6
    assert float((g - gw).abs().max()) < 4e-6 * float(gw.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("gate,n,width,layers,obs,batch", [
    ("CRZ", 19, 4, 3, 9, 2), ("CRZ", 17, 4, 4, 8, 1), ("ControlledPhaseShift", 17, 4, 4, 8, 2), ("CZ", 19, 4, 3, 9, 1),
    ("Unitary", 17, 4, 4, 8, 2), ("Toffoli", 17, 4, 4, 8, 2)])
def test_gradients_with_and_without_runs(gate, n, width, layers, obs, batch):
    """Default options on the device: values and gradients of the runs against the steps, where the backward
    has runs beside steps that it must not undo (Toffoli: unreduced, all of its large steps in runs)."""
    cc, n_params = circuit(gate, n, width, layers, obs)
    dev = torch.device("cuda", 0)
    rows = rows_for(n_params, batch, 5).to(dev)
    ex = TNExecutor(cc)
    assert all(len(ex._run_plan(ex.networks[0], grad)["ops"]) for grad in (False, True))  # pylint: disable=protected-access
    up, res = [torch.ones(batch, device=dev)], []
    for on in (True, False):
        ex.run_passes = on
        v, g = ex.value_and_grad(rows, up)
        run = ex.run_forward(rows, need_grad=True)
        res.append((v[0], g, ex.measure(run)[0], ex.run_backward(rows, run, ex.seed_adjoint(run, up))))
    for a, b in zip(*res):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))
    assert float(res[0][1].abs().max()) > 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("build,args,backward,batch", [
    (chain, (40, 8, True), True, 1), (lattice, (3, 5, 5, 7, False), True, 2), (lattice, (4, 5, 6, 9, True), True, 1),
    (lattice, (5, 5, 3, 12, True), False, 2)])
def test_networks_that_have_runs(build, args, backward, batch):
    """Networks whose runs are known to exist (forward only in the last, where reduction leaves the backward
    none): values, gradients, and the gradient from a kept forward against the steps."""
    cc, n_params = build(*args)
    dev = torch.device("cuda", 0)
    rows = rows_for(n_params, batch, 11).to(dev)
    ex = TNExecutor(cc)
    net = ex.networks[0]
    covered = [len(ex._run_plan(net, grad)["covered"]) for grad in (False, True)]  # pylint: disable=protected-access
    assert covered[0] > 20 and (covered[1] > 20) == backward
    up, res = [torch.ones(batch, device=dev)], []
    for on in (True, False):
        ex.run_passes = on
        v, g = ex.value_and_grad(rows, up)
        run = ex.run_forward(rows, need_grad=True)
        if on and covered[1] >= 0.9 * covered[0]:
            assert run["kept"][0] is not None
        res.append((v[0], g, ex.measure(run)[0], ex.run_backward(rows, run, ex.seed_adjoint(run, up)),
                    ex.measure(ex.run_forward(rows))[0]))
    for a, b in zip(*res):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))
    assert float(res[0][1].abs().max()) > 1e-3


def _rounded_rotation(sign):
    """The RY in fp32, of many angles, whose c^2 + s^2 is furthest from 1 on one side."""
    a = np.linspace(0.1, 1.4, 4001)
    c, s = np.cos(a).astype(np.float32).astype(np.float64), np.sin(a).astype(np.float32).astype(np.float64)
    i = int(np.argmax(sign * (c * c + s * s - 1)))
    assert sign * (c[i] ** 2 + s[i] ** 2 - 1) > 5e-8
    return np.array([[c[i], -s[i]], [s[i], c[i]]], dtype=np.complex128)


@pytest.mark.gpu
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("n,ops,batch", [(9, 32, 2), (12, 32, 1), (14, 20, 2)])
def test_rounding_of_the_undone_matrices_does_not_add_up(sign, n, ops, batch):
    """One pass of rotations that are all rounded to the same side of unitary: undone, each scales the recovered
    input by up to 1 + 1e-7.  Against float64 with the stored inputs, environments whose sums do not cancel:
    3e-7 of their size (rounding of the results 6e-8, of sums of at most 16 terms per lane with random sign, and
    of random signs elsewhere); left in, the factors give up to 32 * 1e-7."""
    dev, rng = torch.device("cuda", 0), np.random.default_rng(n)
    m = _rounded_rotation(sign)
    chain_ops = []
    for k in range(ops):
        w = k % min(n, 9)
        op = R.Op([f"i{k}"], [f"o{k}"], [k], [], [w])
        op.in_wire, op.out_wire = {f"i{k}": w}, {f"o{k}": w}
        chain_ops.append(op)
    run = R.Run(0, 1, [], n, list(range(n)), R._split_passes(chain_ops, n))  # pylint: disable=protected-access
    assert len(run.passes) == 1
    rows = R.encode_run(run, lambda t: (0, 4 * t), [list(reversed(op.outs)) + list(reversed(op.ins)) for op in chain_ops])
    for row in rows:
        row[8], row[9] = 0, row[13]
    plan = {"ops": np.array(rows, dtype=np.int32), "coef": int(run.passes[0].words[3]), "dev": {}}
    ex = TNExecutor.__new__(TNExecutor)
    ex.leaf_stride = 4 * ops
    leaves = torch.tensor(np.tile(m.reshape(-1), (batch, ops)), dtype=torch.complex64, device=dev)
    buf = {"consts": torch.zeros(2, dtype=torch.complex64, device=dev)}
    # pylint: disable=protected-access
    coef = ex._run_coefs(plan, {"len": 4 * ops}, leaves, leaves, buf, batch, dev)
    x = rng.normal(size=(batch, 1 << n)) + 1j * rng.normal(size=(batch, 1 << n))
    tx = torch.tensor(x, dtype=torch.complex64, device=dev)
    outs = ex._run_forward_passes(run, plan, coef, (tx, tx.shape[1], 0), batch, dev, True)
    te = outs[-1].conj().resolve_conj().contiguous()
    envs = [torch.zeros((batch, 4 * ops), dtype=torch.complex64, device=dev) for _ in range(2)]
    ex._run_backward_passes(run, plan, coef, outs, (te, te.shape[1], 0), envs[0], envs[1], batch, dev)
    states = [tx.cpu().numpy().astype(np.complex128)]
    for op in run.passes[0].ops:
        states.append(_apply(states[-1], m, op.wires, n))
    env, got = te.cpu().numpy().astype(np.complex128), envs[0].cpu().numpy()
    for k in range(ops - 1, -1, -1):
        op = run.passes[0].ops[k]
        want = np.einsum("brq,brk->bqk", _rows(env, op.wires, n), _rows(states[k], op.wires, n)).reshape(batch, 4)
        t = op.factors[0]
        assert np.max(np.abs(got[:, 4 * t:4 * t + 4] - want)) < 3e-7 * np.max(np.abs(want)), k
        env = _apply(env, m.T, op.wires, n)


@pytest.mark.gpu
@pytest.mark.parametrize("products,singles,batch", [(1, 0, 1), (40, 3, 2), (300, 0, 2)])
def test_rounding_of_products_does_not_add_up(products, singles, batch):
    """Matrices of ops that are the product of two rotations, all the same and so all rounded alike, then ops of one
    factor: the scale of the roundings, |M| against the product in float64, is balanced in one op, whose own
    rounding remains (6e-8 at most); the matrices themselves are right to 4 roundings and the balance."""
    dev, arena = torch.device("cuda", 0), []
    rng = np.random.default_rng(3)

    def rotation(a):
        return np.array([[np.cos(a), -np.sin(a)], [np.sin(a), np.cos(a)]]).astype(np.complex64).astype(np.complex128)
    cands = [(rotation(a), rotation(b)) for a, b in rng.uniform(0.2, 1.3, size=(2000, 2))]

    def scale(m, p):
        return 0.5 * (np.sum(np.abs(m) ** 2) / np.sum(np.abs(p) ** 2) - 1)
    a, b = max(cands, key=lambda f: scale((f[1] @ f[0]).astype(np.complex64).astype(np.complex128), f[1] @ f[0]))
    assert scale((b @ a).astype(np.complex64).astype(np.complex128), b @ a) > 3e-8
    ops, lay = [], []
    for k in range(products + singles):
        names, w = [len(lay)] + ([len(lay) + 1] if k < products else []), k % 9
        lay += [["x", f"i{k}"], [f"o{k}", "x"]] if k < products else [[f"o{k}", f"i{k}"]]
        arena += [a, b] if k < products else [a]
        op = R.Op([f"i{k}"], [f"o{k}"], names, ["x"] if k < products else [], [w])
        op.in_wire, op.out_wire = {f"i{k}": w}, {f"o{k}": w}
        ops.append(op)
    rows = [R.encode_op(op, list(range(9)), lambda t: (0, 4 * t), lay) for op in ops]
    for k, row in enumerate(rows):
        row[7] = 16 * k
    plan = {"ops": np.array(rows, dtype=np.int32), "coef": 16 * len(ops), "dev": {}}
    ex = TNExecutor.__new__(TNExecutor)
    ex.leaf_stride = 4 * len(arena)
    leaves = torch.tensor(np.tile(np.concatenate([m.reshape(-1) for m in arena]), (batch, 1)), dtype=torch.complex64,
                          device=dev)
    buf = {"consts": torch.zeros(2, dtype=torch.complex64, device=dev)}
    coef = ex._run_coefs(plan, {"len": 4 * len(arena)}, leaves, leaves, buf, batch, dev)  # pylint: disable=protected-access
    got = coef.cpu().numpy().astype(np.complex128)
    for e in range(batch):
        total = 0.0
        for k in range(len(ops)):
            m = got[e, 16 * k:16 * k + 16].reshape(4, 4)
            p = b @ a if k < products else a
            want = np.kron(np.eye(2), p) if ops[k].wires[0] == 0 else np.kron(p, np.eye(2))
            # (the spectator slot is the lowest other one)
            assert np.max(np.abs(m - want)) < 4 * 6e-8 + products * 6e-8 * (k == products - 1)
            total += scale(m, want)
        assert abs(total) <= 6e-8
