"""Gradients through a returned state for complex upstream gradients, as a tensor holds them or as torch marks them
(conjugated or negated lazily, which the kernels, reading memory, do not see)."""

import numpy as np
import pytest
import torch

import tedq_amd as qai
from oracle import sv_oracle as O
from tedq_amd.tn.executor import TNExecutor
from test_tn_runs import emulate
from tn_emulator import install

TOL = 1e-5


def circuit(n, tn_mode):
    spec = [("RX", [q], 1) for q in range(n)] + [("CNOT", [q, q + 1], 0) for q in range(n - 1)]
    spec += [("RZ", [q], 1) for q in range(n)] + [("RY", [q], 1) for q in range(0, n, 2)]
    n_params = sum(s[2] for s in spec)

    def cd(*p):
        it = iter(p)
        for name, qubits, k in spec:
            getattr(qai, name)(*[next(it) for _ in range(k)], qubits=qubits)
        return [qai.state()]
    return qai.Circuit(cd, n, *([0.1] * n_params)).compilecircuit(backend="pytorch", tn_mode=tn_mode), spec, n_params


def upstream(n, form, dev):
    rng = np.random.default_rng(n)
    g = torch.tensor(rng.normal(size=(1,) + (2,) * n) + 1j * rng.normal(size=(1,) + (2,) * n), dtype=torch.complex64,
                     device=dev)
    if form == "conjugated":
        return g.conj()
    if form == "negated":
        return torch._neg_view(g)  # pylint: disable=protected-access
    return g


def reference(n, spec, row, g):
    t = torch.tensor(row.astype(np.float64), requires_grad=True)
    it = iter(t)
    psi = O.propagate(n, [(name, q, [next(it) for _ in range(k)]) for name, q, k in spec])
    w = g.cpu().resolve_conj().resolve_neg().to(torch.complex128).reshape(psi.shape)
    (psi * w.conj()).sum().real.backward()
    return t.grad.numpy()


def row_of(n_params):
    return np.random.default_rng(3).uniform(0, 2 * np.pi, n_params).astype(np.float32)


@pytest.mark.parametrize("form", ["plain", "conjugated", "negated"])
@pytest.mark.parametrize("small", [True, False])
def test_root_environment_is_conjugated_in_memory(form, small):
    """On the CPU, with the root a small step's result or its own tensor."""
    n = 6
    cc, spec, n_params = circuit(n, True)
    ex = (emulate if small else install)(TNExecutor(cc))
    row, g = row_of(n_params), upstream(n, form, "cpu")
    _, grad = ex.value_and_grad(torch.tensor(row[None]), [g])
    want = reference(n, spec, row, g)
    assert np.max(np.abs(grad[0].numpy() - want)) < TOL * np.max(np.abs(want))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "conjugated", "negated"])
@pytest.mark.parametrize("n,tn_mode", [(6, True), (13, True), (14, True), (6, False), (13, False)])
def test_state_gradients_for_complex_upstream_gradients(n, tn_mode, form):
    dev = torch.device("cuda", 0)
    cc, spec, n_params = circuit(n, tn_mode)
    row, g = row_of(n_params), upstream(n, form, dev)
    _, grad = cc.executor().value_and_grad(torch.tensor(row[None], device=dev), [g])
    want = reference(n, spec, row, g)
    assert np.max(np.abs(grad[0].cpu().numpy() - want)) < TOL * np.max(np.abs(want))


@pytest.mark.gpu
@pytest.mark.parametrize("tn_mode", [False, True])
def test_fidelity_loss_of_a_state(tn_mode):
    """Through autograd: 1 - |<target|psi>|^2 of 13 qubits."""
    n, dev = 13, torch.device("cuda", 0)
    cc, spec, n_params = circuit(n, tn_mode)
    row = row_of(n_params)
    target = upstream(n, "plain", "cpu").reshape(-1).to(torch.complex128)
    target = target / target.abs().pow(2).sum().sqrt()
    p = torch.tensor(row, device=dev, requires_grad=True)
    (1 - torch.vdot(target.to(dev, torch.complex64), cc(p).reshape(-1)).abs() ** 2).backward()
    t = torch.tensor(row.astype(np.float64), requires_grad=True)
    it = iter(t)
    psi = O.propagate(n, [(name, q, [next(it) for _ in range(k)]) for name, q, k in spec])
    (1 - torch.vdot(target, psi.reshape(-1)).abs() ** 2).backward()
    want = t.grad.numpy()
    # both sides' amplitudes are about 2^(-n/2), the loss's gradient about 2^-n of unit scale: fp32 rounding of
    # 2^13 products relative to the largest derivative
    assert np.max(np.abs(p.grad.cpu().numpy() - want)) < TOL * np.max(np.abs(want))
