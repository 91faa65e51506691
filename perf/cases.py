"""Performance cases: the work that programs built on this framework have it do.

A case names a circuit family, its size, what is measured and how it is called:

* ``sv``: state-vector mode through the compiled callable (``entry="call"``, one parameter row, as the
  reference's scripts train) or ``execute_batch`` (``entry="batch"``), forward only or with the gradient;
* ``tn``: contraction mode (``tn_mode=True``) through ``execute_batch``;
* ``serve``: a closed-loop stream of mixed requests through ``ServingEngine``.

Circuit families (workloads.py): ``hea`` (RY RZ on every qubit, then the CNOT chain), ``lattice`` (RX RZ,
then CZ on the grid's bonds), ``chain`` (Trotterised disordered chain of two-qubit unitaries).  Compiled
circuits are kept per structure, as a program keeps them; parameters, disorder fields and upstream weights
come from the seed.
"""

import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "ted-q_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "ted-q_amd"))

import tedq_amd as qai  # noqa: E402  pylint: disable=wrong-import-position
from tedq_amd import workloads  # noqa: E402  pylint: disable=wrong-import-position
from tedq_amd.serving.engine import Request, ServingEngine  # noqa: E402  pylint: disable=wrong-import-position

_J, _DT = 1.0, 0.1


def _sv(name, ansatz, n, layers, batch, measure, grad, entry="batch", jit=False, tile=12):
    return {"name": name, "kind": "sv", "ansatz": ansatz, "n": n, "layers": layers, "batch": batch,
            "measure": measure, "grad": grad, "entry": entry, "jit": jit, "tile": tile}


def _tn(name, ansatz, n, layers, batch, grad):
    return {"name": name, "kind": "tn", "ansatz": ansatz, "n": n, "layers": layers, "batch": batch,
            "measure": "site", "grad": grad}


def listed():
    return [
        # the reference's CPU-runnable training step: one small circuit, one parameter row, one value
        _sv("call_8q_d4_z0", "hea", 8, 4, 1, "z0", True, entry="call"),
        # a mini-batch of small circuits (quantum layers in a classical model): whole circuits in a tile
        _sv("train_12q_d6_b64", "hea", 12, 6, 64, "z", True),
        # a variational energy: transverse-field Ising terms (ZZ bonds and X sites) of a 15-qubit chain
        _sv("ising_15q_d4_b16", "hea", 15, 4, 16, "ising", True),
        # medium circuits in a mini-batch, default kernels
        _sv("train_17q_d8_b32", "hea", 17, 8, 32, "z", True),
        # inference on a batch of 20-qubit circuits: forward only
        _sv("infer_20q_d10_b48", "hea", 20, 10, 48, "z", False),
        # one row of a 20-qubit circuit through the compiled callable, default kernels
        _sv("call_20q_d10", "hea", 20, 10, 1, "z", True, entry="call"),
        # the disordered chain in state-vector mode with a marginal probability, as the reference's
        # many-body-localisation script measures it
        _sv("mbl_18q_s8_probs", "chain", 18, 8, 8, "probs", True),
        # the largest single state of the serving range
        _sv("call_24q_d4", "hea", 24, 4, 1, "z", True, entry="call"),
        # the headline workload: 20 qubits, 10 layers, 256 rows, all <Z_i>, generated pass kernels
        _sv("train_20q_d10_b256", "hea", 20, 10, 256, "z", True, jit=True, tile=13),
        # contraction mode: the 40-qubit disordered chain, 32 disorder seeds, forward
        _tn("tn_chain40_s8_b32", "chain", 40, 8, 32, False),
        # contraction mode with gradients: the 5x5 lattice, the network of its central site
        _tn("tn_lattice5x5_l6", "lattice", 25, 6, 1, True),
        # a backlog of mixed requests (6-24 qubits, 2-20 layers, value and gradient) served to the end
        {"name": "serve_96", "kind": "serve", "structures": 24, "requests": 96, "pool": 7},
    ]


def draw(rng):
    kind = rng.choice(["sv", "sv", "sv", "sv", "sv", "sv", "tn", "serve"])
    if kind == "serve":
        return {"kind": "serve", "structures": rng.randint(8, 32), "requests": rng.randint(24, 128),
                "pool": rng.randint(0, 10 ** 6)}
    if kind == "tn":
        if rng.random() < 0.5:
            c = _tn("", "chain", rng.randint(20, 40), rng.randint(4, 8), _log_int(rng, 1, 32), False)
        else:
            c = _tn("", "lattice", rng.choice([9, 12, 15, 16, 20]), rng.randint(3, 6), rng.randint(1, 2), True)
        del c["name"]
        return c
    while True:
        n, batch = rng.randint(6, 24), _log_int(rng, 1, 256)
        ansatz = rng.choice(["hea", "hea", "hea", "lattice", "chain"])
        layers = rng.randint(1, 12)
        if ansatz == "lattice":
            n = rng.choice([6, 8, 9, 12, 15, 16, 20])
        measure = "probs" if ansatz == "chain" else rng.choice(["z", "z", "z0", "ising", "probs"])
        grad = rng.random() < 0.75
        jit = n >= 15 and rng.random() < 0.3
        c = _sv("", ansatz, n, layers, batch, measure, grad, "call" if batch == 1 else "batch", jit,
                rng.choice([12, 13]) if jit else 12)
        del c["name"]
        if work(c)["flops"] <= 0.5 * work(_sv("", "hea", 20, 10, 256, "z", True))["flops"] and batch << n <= 1 << 27:
            return c


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ---------------------------------------------------------------------------
# circuits
# ---------------------------------------------------------------------------
def _grid(n):
    rows = int(math.isqrt(n))
    while n % rows:
        rows -= 1
    return rows, n // rows


def _bonds(n):
    """Bonds of the lattice family on a rows x cols grid: all horizontal ones, then all vertical ones."""
    rows, cols = _grid(n)
    out = [(r * cols + c, r * cols + c + 1) for r in range(rows) for c in range(cols - 1)]
    return out + [(r * cols + c, (r + 1) * cols + c) for r in range(rows - 1) for c in range(cols)]


def _n_params(case):
    return case["n"] * case["layers"] * (1 if case["ansatz"] == "chain" else 2)


def _measurements(case):
    n, m = case["n"], case["measure"]
    if m == "probs":
        return qai.probs(qubits=[n - 1])
    if m == "z0":
        return qai.expval(qai.PauliZ(qubits=[0]))
    if m == "site":
        return qai.expval(qai.PauliZ(qubits=[n // 2]))
    if m == "z":
        return [qai.expval(qai.PauliZ(qubits=[q])) for q in range(n)]
    out = [qai.expval([qai.PauliZ(qubits=[q]), qai.PauliZ(qubits=[q + 1])]) for q in range(n - 1)]
    return out + [qai.expval(qai.PauliX(qubits=[q])) for q in range(n)]


@functools.lru_cache(maxsize=None)
def _compiled(kind, ansatz, n, layers, measure, jit, tile):
    case = {"n": n, "layers": layers, "ansatz": ansatz, "measure": measure}
    zz, xy = workloads.exchange_unitaries(_J, _DT)

    def circuit_def(*p):
        it = iter(p)
        if ansatz == "chain":
            for q in range(1, n, 2):
                qai.PauliX(qubits=[q])
        for _ in range(layers):
            for q in range(n):
                if ansatz == "hea":
                    qai.RY(next(it), qubits=[q])
                elif ansatz == "lattice":
                    qai.RX(next(it), qubits=[q])
                qai.RZ(next(it), qubits=[q])
            if ansatz == "hea":
                for q in range(n - 1):
                    qai.CNOT(qubits=[q, q + 1])
            elif ansatz == "lattice":
                for a, b in _bonds(n):
                    qai.CZ(qubits=[a, b])
            else:
                for q in range(n - 1):
                    qai.Unitary(zz, qubits=[q, q + 1])
                    qai.Unitary(xy, qubits=[q, q + 1])
        return _measurements(case)

    kwargs = {"tn_mode": True} if kind == "tn" else ({"jit": True, "tile_bits": tile} if jit else {})
    circuit = qai.Circuit(circuit_def, n, *([0.1] * _n_params(case)))
    return circuit.compilecircuit(backend="pytorch", **kwargs)


@functools.lru_cache(maxsize=None)
def _engine(keys):
    engine = ServingEngine(lambda key: _compiled("sv", "hea", key[0], key[1], "z0", False, 12),
                           hbm_budget=64 << 30, max_batch=64, n_streams=4, max_inflight=8, ragged=True)
    engine.prepare(keys, buckets=(1, 2, 4))
    return engine


def _n_out(case):
    n, m = case["n"], case["measure"]
    return {"probs": 2, "z0": 1, "site": 1, "z": n, "ising": 2 * n - 1}[m]


def _rows(case, seed):
    """Parameter rows [B, P] and upstream weights [B, outputs], float32 numpy, from the seed."""
    rng = np.random.default_rng(seed)
    B, n = case["batch"], case["n"]
    if case["ansatz"] == "chain":
        rows = workloads.chain_rows(rng.uniform(-5, 5, size=(B, n)), case["layers"], _DT)
    else:
        rows = rng.uniform(0, 2 * np.pi, size=(B, _n_params(case))).astype(np.float32)
    return rows, rng.uniform(0.5, 1.5, size=(B, _n_out(case))).astype(np.float32)


def _stream(case, seed):
    """(structure keys, [(key, parameter row)]) of a serving case."""
    pool = np.random.default_rng(case["pool"])
    keys = [(int(n), int(d)) for n, d in zip(pool.integers(6, 25, size=case["structures"]),
                                             pool.integers(2, 21, size=case["structures"]))]
    rng = np.random.default_rng(seed)
    order = np.arange(case["requests"]) % len(keys)
    return tuple(sorted(set(keys))), [(keys[i], rng.uniform(0, 2 * np.pi, 2 * keys[i][0] * keys[i][1])
                                       .astype(np.float32)) for i in order]


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "serve":
        keys, reqs = _stream(case, seed)
        return {"case": case, "engine": _engine(keys), "reqs": reqs}
    rows, w = _rows(case, seed)
    compiled = _compiled(case["kind"], case["ansatz"], case["n"], case["layers"], case["measure"],
                         case.get("jit", False), case.get("tile", 12))
    compiled.executor()
    dev = torch.device("cuda", torch.cuda.current_device())
    return {"case": case, "compiled": compiled, "rows": torch.from_numpy(rows).to(dev),
            "w": torch.from_numpy(w).to(dev)}


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        engine = state["engine"]
        engine.completed.clear()
        engine.batch_sizes.clear()
        reqs = [Request(i, key, params, 0.0) for i, (key, params) in enumerate(state["reqs"])]
        engine.run(reqs)
        return {"values": np.concatenate([r.value.reshape(-1) for r in reqs]),
                "grads": np.concatenate([r.grad.reshape(-1) for r in reqs])}
    compiled, rows, w = state["compiled"], state["rows"], state["w"]
    call = case.get("entry") == "call"
    if not case["grad"]:
        with torch.no_grad():
            return {"values": compiled(rows[0]) if call else compiled.execute_batch(rows)}
    p = (rows[0] if call else rows).detach().clone().requires_grad_(True)
    out = compiled(p) if call else compiled.execute_batch(p)
    (out.reshape(w.shape) * w).sum().backward()
    return {"values": out.detach(), "grad": p.grad}


# ---------------------------------------------------------------------------
# what a pass cannot do without: its parameters in, its values and gradients out, and the arithmetic of
# the gates on the state (a real rotation 6 flops per amplitude, a phase 3, a dense two-qubit gate 30),
# twice that plus 4 flops per amplitude and parameter for the reverse sweep
# ---------------------------------------------------------------------------
def _flops(n, layers, ansatz, grad):
    if ansatz == "chain":
        gates, params = layers * (3.0 * n + 30.0 * (n - 1)), layers * n
    else:
        gates, params = layers * 9.0 * n, 2 * layers * n
    return 2.0 ** n * (gates + (2.0 * gates + 4.0 * params if grad else 0.0))


def work(case):
    if case["kind"] == "serve":
        _, reqs = _stream(case, 0)
        flops = sum(_flops(min(n, d), d, "hea", True) for (n, d), _ in reqs)   # the light cone of <Z_0>
        return {"bytes": float(sum(8 * p.size + 4 for _, p in reqs)), "flops": flops}
    B, n = case["batch"], case["n"]
    nbytes = 4.0 * B * (_n_params(case) * (2 if case["grad"] else 1) + _n_out(case))
    if case["kind"] == "tn":
        macs = sum(r["macs"] for r in _compiled("tn", case["ansatz"], n, case["layers"], case["measure"], False, 12)
                   .executor().path_report())
        return {"bytes": nbytes, "flops": 8.0 * B * macs * (3 if case["grad"] else 1)}
    m = min(n, case["layers"]) if case["measure"] == "z0" and case["ansatz"] == "hea" else n
    return {"bytes": nbytes, "flops": B * _flops(m, case["layers"], case["ansatz"], case["grad"])}


# ---------------------------------------------------------------------------
# the same in complex128 with torch alone: states [B, 2^n], qubit q = bit n-1-q
# ---------------------------------------------------------------------------
class _Exact:
    def __init__(self, case, rows, dev):
        self.n, self.case, self.dev = case["n"], case, dev
        self.rows = torch.as_tensor(rows, dtype=torch.float64, device=dev)
        n, x = self.n, torch.arange(1 << case["n"], device=dev)
        self.x = x
        self.src = self.sign = self.u4 = None
        if case["ansatz"] == "hea":
            src = x.clone()
            for q in reversed(range(n - 1)):                 # CNOT(q, q+1) in order: gather through all of them
                src = src ^ (((src >> (n - 1 - q)) & 1) << (n - 2 - q))
            self.src = src
            self.inv = torch.empty_like(src)
            self.inv[src] = x
        elif case["ansatz"] == "lattice":
            odd = torch.zeros_like(x)
            for a, b in _bonds(n):
                odd ^= (x >> (n - 1 - a)) & (x >> (n - 1 - b)) & 1
            self.sign = (1 - 2 * odd).to(torch.float64)
        else:
            zz, xy = workloads.exchange_unitaries(_J, _DT)
            self.u4 = torch.as_tensor(xy @ zz, dtype=torch.complex128, device=dev)

    def layer_matrices(self, layer):
        """Per qubit [B, 2, 2]: the product of the layer's rotations, and dU U^dagger per parameter."""
        n, per = self.n, (1 if self.case["ansatz"] == "chain" else 2)
        th = self.rows[:, layer * per * n:(layer + 1) * per * n].reshape(-1, n, per)
        zero = torch.zeros(2, 2, dtype=torch.complex128, device=self.dev)
        X, Y, Z = zero.clone(), zero.clone(), zero.clone()
        X[0, 1] = X[1, 0] = 1
        Y[0, 1], Y[1, 0] = -1j, 1j
        Z[0, 0], Z[1, 1] = 1, -1
        eye = torch.eye(2, dtype=torch.complex128, device=self.dev)

        def rot(P, t):
            c, s = torch.cos(t / 2)[..., None, None], torch.sin(t / 2)[..., None, None]
            return c * eye - 1j * s * P
        rz = rot(Z, th[..., per - 1])
        if per == 1:
            return rz, [(-0.5j * Z).expand(rz.shape)]
        first = X if self.case["ansatz"] == "lattice" else Y
        a = rz @ (-0.5j * first) @ rz.conj().transpose(-1, -2)
        return rz @ rot(first, th[..., 0]), [a, (-0.5j * Z).expand(rz.shape)]

    def blocks(self):
        return [list(range(q, min(q + 4, self.n))) for q in range(0, self.n, 4)]

    def kron(self, U, qs):
        out = U[:, qs[0]]
        for q in qs[1:]:
            out = (out[:, :, None, :, None] * U[:, q][:, None, :, None, :]).reshape(out.shape[0], out.shape[1] * 2, -1)
        return out.contiguous()

    def apply_layer(self, U, psi):
        """The 1-qubit layer: the top block of qubits is multiplied, then moved to the bottom."""
        B = psi.shape[0]
        for qs in self.blocks():
            M = self.kron(U, qs)
            psi = torch.bmm(M, psi.reshape(B, 1 << len(qs), -1)).transpose(1, 2).contiguous()
        return psi.reshape(B, -1)

    def densities(self, psi, lam):
        """Per qubit [B, 2, 2]: rho_ab = sum over the rest of psi_a conj(lam_b)."""
        B, n = psi.shape[0], self.n
        out = []
        for q in range(n):
            p = psi.view(B, 1 << q, 2, -1)
            l = lam.view(B, 1 << q, 2, -1).conj()
            out.append(torch.stack([torch.stack([(p[:, :, a] * l[:, :, b]).sum((1, 2)) for b in (0, 1)], -1)
                                    for a in (0, 1)], -2))
        return torch.stack(out, 1)

    def bond(self, psi, q, u):
        B = psi.shape[0]
        v = psi.view(B, 1 << q, 4, -1)
        return torch.stack([sum(u[i, j] * v[:, :, j] for j in range(4)) for i in range(4)], 2).reshape(B, -1)

    def entangle(self, psi, back=False):
        if self.src is not None:
            return psi[:, self.inv if back else self.src]
        if self.sign is not None:
            return psi * self.sign
        u = self.u4.conj().T if back else self.u4
        for q in (reversed(range(self.n - 1)) if back else range(self.n - 1)):
            psi = self.bond(psi, q, u)
        return psi

    def z(self, *qs):
        s = torch.ones(1 << self.n, dtype=torch.float64, device=self.dev)
        for q in qs:
            s = s * (1 - 2 * ((self.x >> (self.n - 1 - q)) & 1))
        return s

    def observables(self):
        n, m = self.n, self.case["measure"]
        if m == "probs":
            return [("d", (1 + self.z(n - 1)) / 2), ("d", (1 - self.z(n - 1)) / 2)]
        if m == "ising":
            return [("d", self.z(q, q + 1)) for q in range(n - 1)] + [("x", q) for q in range(n)]
        return [("d", self.z(q)) for q in ({"z0": [0], "site": [n // 2]}.get(m) or range(n))]

    def run(self, w):
        B, n = self.rows.shape[0], self.n
        psi = torch.zeros(B, 1 << n, dtype=torch.complex128, device=self.dev)
        start = sum(1 << (n - 1 - q) for q in range(1, n, 2)) if self.u4 is not None else 0
        psi[:, start] = 1
        for layer in range(self.case["layers"]):
            psi = self.entangle(self.apply_layer(self.layer_matrices(layer)[0], psi))
        vals, lam = [], torch.zeros_like(psi)
        w = torch.as_tensor(w, dtype=torch.float64, device=self.dev)
        for m, (kind, o) in enumerate(self.observables()):
            opsi = psi * o if kind == "d" else psi[:, self.x ^ (1 << (n - 1 - o))]
            vals.append((psi.conj() * opsi).sum(1).real)
            lam += w[:, m:m + 1] * opsi
        vals = torch.stack(vals, 1)
        if not self.case["grad"]:
            return vals, None
        grads = []
        for layer in reversed(range(self.case["layers"])):
            psi, lam = self.entangle(psi, True), self.entangle(lam, True)
            U, gens = self.layer_matrices(layer)
            rho = self.densities(psi, lam)
            g = torch.stack([2 * (a * rho.transpose(-1, -2)).sum((-1, -2)).real for a in gens], -1)
            grads.append(g.reshape(B, -1))
            Ud = U.conj().transpose(-1, -2).contiguous()
            psi, lam = self.apply_layer(Ud, psi), self.apply_layer(Ud, lam)
        return vals, torch.cat(list(reversed(grads)), 1)


def _exact_rows(case, rows, w, dev):
    step = max(1, (1 << 24) >> case["n"])
    parts = [_Exact(case, rows[i:i + step], dev).run(w[i:i + step]) for i in range(0, rows.shape[0], step)]
    vals = torch.cat([v for v, _ in parts])
    return vals, (torch.cat([g for _, g in parts]) if case["grad"] else None)


def exact(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")
    if case["kind"] == "serve":
        vals, grads = [], []
        for (n, d), params in _stream(case, seed)[1]:
            m = min(n, d)   # qubits past the layer count are outside the light cone of <Z_0>
            c = {"n": m, "layers": d, "ansatz": "hea", "measure": "z0", "grad": True}
            rows = params.reshape(d, n, 2)[:, :m].reshape(1, -1)
            v, g = _exact_rows(c, rows, np.ones((1, 1)), dev)
            full = torch.zeros(d, n, 2, dtype=torch.float64, device=dev)
            full[:, :m] = g.reshape(d, m, 2)
            vals.append(v.reshape(-1))
            grads.append(full.reshape(-1))
        return {"values": torch.cat(vals).cpu().numpy(), "grads": torch.cat(grads).cpu().numpy()}
    if case["n"] > 25 or (case["ansatz"] == "chain" and case["batch"] * case["layers"] * 2.0 ** case["n"] > 2.0 ** 29):
        return None          # the 40-qubit chain has no state vector here
    rows, w = _rows(case, seed)
    vals, grads = _exact_rows(case, rows, w, dev)
    if case.get("entry") == "call":
        vals = vals.reshape(2) if case["measure"] == "probs" else vals.reshape(-1)
        if case["measure"] == "z0":
            vals = vals.reshape(1)
        grads = grads[0] if grads is not None else None
    elif case["measure"] == "probs":
        vals = vals.reshape(-1, 1, 2)
    return {"values": vals, "grad": grads} if grads is not None else {"values": vals}
