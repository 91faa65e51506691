"""Pass kernels that the default plans do not choose: op lists on the library's kernels (executors set up for
generated kernels run them in ragged batches), lifted forward plans with 32 amplitudes per thread (a shape of the
autotuner), and the generated form of op lists.

Tolerances: 1e-5 relative to the complex128 oracle, as in test_gpu_sv; gradients against at least 0.1.
"""

import math
import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

import tedq_amd as qai
from oracle import sv_oracle as O
from tedq_amd.engine import jit
from tedq_amd.engine.lowering import lower_circuit
from tedq_amd.engine.ragged import ragged_value_and_grad
from tedq_amd.engine.sv import SVExecutor
from test_plan_emulated import oracle_gates, random_spec

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL, GFLOOR = 1e-5, 0.1
OBS = (0, 2, 3)


def executor(n, spec, k, r, k_bwd=None, r_bwd=None):
    """Executor of the whole circuit (nothing folded away) measuring <Z> of three qubits."""
    n_params = sum(s[2] for s in spec)

    def cd(*p):
        it = iter(p)
        for name, qubits, count in spec:
            getattr(qai, name)(*[next(it) for _ in range(count)], qubits=qubits)
        return [qai.expval(qai.PauliZ(qubits=[q])) for q in OBS]
    cc = qai.Circuit(cd, n, *([0.1] * n_params)).compilecircuit(backend="pytorch")
    nq, units, P, pool = lower_circuit(cc)
    return SVExecutor(nq, units, P, pool, cc._measurements, k_max=k, r=r, k_bwd=k_bwd, r_bwd=r_bwd), n_params  # pylint: disable=protected-access


def op_lists(ex, specialize):
    """The executor on op lists, as before a generated kernel takes their place."""
    # pylint: disable=protected-access
    ex.fwd = ex._program(ex.fwd.plan.k, ex.fwd.plan.r, specialize=specialize)
    ex.bwd = ex._program(ex.bwd.plan.k, ex.bwd.plan.r, specialize=specialize)
    assert not ex.fwd.plan.lift and not ex.bwd.plan.lift
    return ex


def compare(n, spec, row, values, grad):
    t = torch.tensor(row.astype(np.float64), requires_grad=True)
    ref = O.execute(n, oracle_gates(spec, list(t)), [("expval", ("PauliZ", [q])) for q in OBS])
    ref.sum().backward()
    want, g = ref.detach().numpy(), t.grad.numpy()
    assert np.max(np.abs(values - want)) < TOL * max(np.max(np.abs(want)), GFLOOR)
    assert np.max(np.abs(grad - g)) < TOL * max(np.max(np.abs(g)), GFLOOR)


def rows_of(n_params, batch, rng):
    return rng.uniform(-math.pi, math.pi, size=(batch, n_params)).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("specialize", [False, True])
@pytest.mark.parametrize("n,k,r,batch", [(4, 4, 2, 3), (7, 7, 4, 5), (9, 6, 3, 2), (12, 12, 4, 2), (13, 11, 4, 2)])
def test_op_lists_on_the_library_kernels(specialize, n, k, r, batch):
    """Whole circuits in a tile (several per workgroup, and one that fills it) and tiled states."""
    dev, rng = torch.device("cuda", 0), np.random.default_rng(n)
    spec = random_spec(n, 50, rng) + [("Rot", [0], 3)]
    ex, n_params = executor(n, spec, k, r)
    op_lists(ex, specialize)
    p = rows_of(n_params, batch, rng)
    outs, grad = ex.value_and_grad(torch.tensor(p, device=dev), [torch.ones(batch, device=dev)] * 3)
    for b in range(batch):
        compare(n, spec, p[b], np.array([float(o[b]) for o in outs]), grad[b].cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["op lists", "specialised", "lifted", "mixed"])
def test_ragged_batches_of_both_plan_forms(kind):
    """Structures of both forms in one ragged batch: each result equals the oracle's."""
    dev, rng = torch.device("cuda", 0), np.random.default_rng(8)
    items, cases = [], []
    for i, n in enumerate((9, 12, 10, 13)):
        spec = random_spec(n, 40, rng) + [("Rot", [1], 3)]
        ex, n_params = executor(n, spec, 9, 3)
        if kind != "lifted" and (kind != "mixed" or i % 2):
            op_lists(ex, kind == "specialised" or i == 3)
        p = rows_of(n_params, 1 + i % 2, rng)
        items.append((ex, torch.tensor(p, device=dev), [torch.ones(len(p), device=dev)] * 3))
        cases.append((n, spec, p))
    results, keep = ragged_value_and_grad(items, dev)
    torch.cuda.synchronize()
    del keep
    for (n, spec, p), (outs, grad) in zip(cases, results):
        for b, row in enumerate(p):
            compare(n, spec, row, np.array([float(o[b]) for o in outs]), grad[b].cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n,k,batch", [(5, 5, 7), (8, 8, 3), (12, 12, 2), (13, 13, 1), (14, 12, 2)])
def test_lifted_forward_with_five_register_bits(general, n, k, batch):
    """k_lift with 32 amplitudes per thread, with and without general ops: several circuits per workgroup, one
    that fills it, and tiles of a larger state.  The adjoint of the same executor has four register bits."""
    dev, rng = torch.device("cuda", 0), np.random.default_rng(n)
    spec = random_spec(n, 50, rng)
    if not general:
        spec = [s for s in spec if not (s[0].startswith("CR") or s[0] in ("CY", "ControlledPhaseShift"))]
    spec += [(name, [q], 1) for q in range(n) for name in ("RX", "RZ")] + [("Rot", [0], 3)]
    ex, n_params = executor(n, spec, k, 5, min(k, 12), 4)
    assert ex.fwd.plan.r == 5 and ex.fwd.plan.lift and ex.bwd.plan.r == 4
    assert any(ex.fwd.general) == general
    p = rows_of(n_params, batch, rng)
    outs, grad = ex.value_and_grad(torch.tensor(p, device=dev), [torch.ones(batch, device=dev)] * 3)
    for b in range(batch):
        compare(n, spec, p[b], np.array([float(o[b]) for o in outs]), grad[b].cpu().numpy())


def test_generated_op_lists_compile_for_gfx950(tmp_path):
    """The kernels that enable_jit generates, one tile per workgroup and looping over tiles with the fused seed."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    rng = np.random.default_rng(4)
    ex, _ = executor(9, random_spec(9, 40, rng) + [("Rot", [0], 3)], 6, 3)
    csrc = os.path.join(ROOT, "ted-q_amd", "csrc")
    for specialize in (False, True):
        enc = op_lists(ex, specialize).fwd.enc
        for tag, kw in (("plain", {}), ("persistent", {"seed_masks": tuple(ex.zmasks), "persistent": True})):
            src = jit.program_source(enc, len(enc.fwd_offsets), len(enc.adj_offsets), **kw)
            assert ("TILE += gridDim.x" in src) == (tag == "persistent")
            path = tmp_path / f"gen_{tag}.hip"
            path.write_text(src)
            out = subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                                  "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-c", "-I", csrc, str(path),
                                  "-o", str(tmp_path / f"gen_{tag}.o")], capture_output=True, text=True, timeout=300)
            assert out.returncode == 0, out.stderr[-2000:]
