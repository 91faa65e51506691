"""Device memory that contraction mode holds (tedq_amd.tn.executor)."""

import weakref

import pytest
import torch

import tedq_amd as qai
from tedq_amd.engine import hip
from tedq_amd.tn import executor as X
from tedq_amd.tn.executor import TNExecutor

from test_tn_runs import lattice, rows_for


class _Live:
    """Stands in for the library: counts the tensors of at least ``size`` elements alive at each launch."""

    def __init__(self, monkeypatch, size):
        self.seen, self.size, self.most = [], size, 0
        self.launches = 0
        empty = torch.empty

        def traced(*args, **kwargs):
            t = empty(*args, **kwargs)
            if t.numel() >= size:
                self.seen.append(weakref.ref(t))
            return t
        monkeypatch.setattr(torch, "empty", traced)
        monkeypatch.setattr(hip, "stream_handle", lambda dev: None)
        monkeypatch.setattr(hip, "call", self.call)

    def call(self, name, *args):  # pylint: disable=unused-argument
        if name == "tedq_tn_gate_tensors":
            return
        self.launches += name == "tedq_tn_run_pass"
        self.most = max(self.most, sum(r() is not None for r in self.seen))


def test_a_forward_run_holds_two_large_tensors(monkeypatch):
    """A pass needs its input and its result, as a step does: a run's input goes once its first pass is issued."""
    cc, n_params = lattice(4, 4, 4, 5, False)
    ex = TNExecutor(cc, trials=())
    net = ex.networks[0]
    plan = ex._run_plan(net, False)  # pylint: disable=protected-access
    assert max(len(run.passes) for run in plan["first"].values()) >= 4
    monkeypatch.setattr(ex, "_use_runs", lambda dev: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    live = _Live(monkeypatch, 1 << max(net.ranks))
    rows = rows_for(n_params, 1, 3)
    leaves, _ = ex._leaves(rows)  # pylint: disable=protected-access
    ex._forward_network(net, leaves, 1, rows.device)  # pylint: disable=protected-access
    assert live.launches >= 4
    assert live.most == 2


def many_values(rows, cols, layers):
    """A lattice circuit with <Z> of every qubit: one network each."""
    n = rows * cols
    bonds = [(r * cols + c, r * cols + c + 1) for r in range(rows) for c in range(cols - 1)]
    bonds += [(r * cols + c, (r + 1) * cols + c) for r in range(rows - 1) for c in range(cols)]

    def cd(*p):
        it = iter(p)
        for _ in range(layers):
            for q in range(n):
                qai.RX(next(it), qubits=[q])
            for a, b in bonds:
                qai.CZ(qubits=[a, b])
        return [qai.expval(qai.PauliZ(qubits=[q])) for q in range(n)]
    return qai.Circuit(cd, n, *([0.1] * (n * layers))).compilecircuit(backend="pytorch", tn_mode=True,
                                                                      tn_simplify=False), n * layers


def test_waiting_forwards_share_one_budget(monkeypatch):
    """Over all networks, graphs and executors on a device: no more than is kept freely without a look at the free
    memory, no more than the share of it, no more than an executor's cap; a dropped forward gives its bytes back."""
    cc, _ = many_values(3, 3, 3)
    dev, batch, freely = torch.device("cuda", 0), 1, 4 << 20
    free, asked = [0], []
    monkeypatch.setattr(X, "_KEPT_FREELY", freely)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: asked.append(d) or (free[0], 1 << 38))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda d: 0)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda d: 0)
    executors = [TNExecutor(cc, trials=(), max_bytes=1 << 40) for _ in range(2)]

    def graph(ex):
        return [ex._keep_forward(net, batch, dev) for net in ex.networks]  # pylint: disable=protected-access

    def total(graphs):
        return sum(k.nbytes for g in graphs for k in g if k is not None)
    graphs = [graph(ex) for ex in executors * 3]
    assert 0 < total(graphs) <= freely and asked
    assert any(k is None for k in graphs[-1])
    held = total(graphs)
    free[0] = 32 * freely                                   # what is free beside the forwards that wait
    graphs += [graph(ex) for ex in executors * 3]
    assert held < total(graphs) <= (free[0] + total(graphs)) // 16
    first = graphs[0][0].nbytes
    del graphs[:]
    free[0] = 0
    assert executors[0]._keep_forward(executors[0].networks[0], batch, dev).nbytes == first  # pylint: disable=protected-access
    # an executor's cap: its waiting forwards and what a backward may keep beside them
    free[0] = 1 << 38
    capped = TNExecutor(cc, trials=(), max_bytes=3 * first)
    graphs = [graph(capped) for _ in range(3)]
    assert 0 < total(graphs) <= capped.max_bytes
    assert capped._keep_budget(dev) == capped.max_bytes - total(graphs)  # pylint: disable=protected-access


def test_a_captured_forward_asks_for_no_memory_info(monkeypatch):
    cc, _ = many_values(3, 3, 3)
    ex = TNExecutor(cc, trials=(), max_bytes=1 << 40)
    dev = torch.device("cuda", 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: pytest.fail("asked while a stream is captured"))
    kept = ex._keep_forward(ex.networks[0], 1, dev)  # pylint: disable=protected-access
    assert kept is not None and kept.nbytes <= X._KEPT_FREELY  # pylint: disable=protected-access
    monkeypatch.setattr(X, "_KEPT_FREELY", 2 * kept.nbytes - 1)
    assert ex._keep_forward(ex.networks[0], 1, dev) is None  # pylint: disable=protected-access


def test_both_run_plans_are_on_the_device_together(monkeypatch):
    """Whether a forward waits for its backward decides which of the two run plans it uses, and may differ between
    an eager call and the same call under capture, when no table may be copied to the device any more."""
    cc, n_params = lattice(4, 4, 4, 5, False)
    ex = TNExecutor(cc, trials=())
    net = ex.networks[0]
    monkeypatch.setattr(ex, "_use_runs", lambda dev: True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(hip, "stream_handle", lambda dev: None)
    monkeypatch.setattr(hip, "call", lambda name, *args: None)
    rows = rows_for(n_params, 1, 3)
    leaves, _ = ex._leaves(rows)  # pylint: disable=protected-access
    ex._forward_stored(net, leaves, 1, rows.device)  # pylint: disable=protected-access
    copied = []
    monkeypatch.setattr(torch, "from_numpy", copied.append)
    ex._forward_network(net, leaves, 1, rows.device)  # pylint: disable=protected-access
    ex._forward_stored(net, leaves, 1, rows.device)  # pylint: disable=protected-access
    assert not copied


@pytest.mark.gpu
@pytest.mark.parametrize("need_free", [False, True])
def test_memory_between_forward_and_backward(need_free, monkeypatch):
    """Three live graphs of 16 networks: what they hold between forward and backward beyond leaves and values
    stays within the budget, and their gradients equal those of graphs that hold nothing, in any order."""
    cc, n_params = many_values(4, 4, 4)
    dev, batch, freely = torch.device("cuda", 0), 2, 128 << 20
    ex = TNExecutor(cc)
    up = [torch.full((batch,), 1.0 + i, device=dev) for i in range(16)]
    rows = [rows_for(n_params, batch, s).to(dev) for s in range(3)]
    monkeypatch.setattr(X, "_KEPT_FREELY", freely)
    if not need_free:
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (0, 0))
        monkeypatch.setattr(torch.cuda, "memory_reserved", torch.cuda.memory_allocated)
    want = []
    for r in rows:
        run = ex.run_forward(r)
        want.append(ex.run_backward(r, run, ex.seed_adjoint(run, up)))
    del run
    before = torch.cuda.memory_allocated(dev)
    runs = [ex.run_forward(r, need_grad=True) for r in rows]
    grown = torch.cuda.memory_allocated(dev) - before
    kept = sum(k.nbytes for run in runs for k in run["kept"] if k is not None)
    assert kept > 0
    if not need_free:
        assert kept <= freely
    # leaves, derivative blocks, roots and the small results' arenas, in blocks of at least 512 bytes
    small = sum(ex._small_plan(net)["len"] for net in ex.networks)  # pylint: disable=protected-access
    other = 3 * (8 * batch * (ex.leaf_stride + 4 * n_params + small) + 16 * 2 * (1 << 20))
    assert grown <= kept + other
    for i in (1, 2, 0):
        g = ex.run_backward(rows[i], runs[i], ex.seed_adjoint(runs[i], up))
        assert float((g - want[i]).abs().max()) < 1e-5 * max(1.0, float(want[i].abs().max()))
    assert all(k is None for run in runs for k in run["kept"])


@pytest.mark.gpu
def test_capture_of_a_forward_that_may_not_wait(monkeypatch):
    """Value and gradient captured after an eager call that kept its forward, with the budget used up: every replay
    equals the eager result of its parameters."""
    cc, n_params = lattice(4, 4, 4, 5, False)
    dev = torch.device("cuda", 0)
    ex = TNExecutor(cc)
    rows = rows_for(n_params, 2, 5).to(dev)
    up = [torch.ones(2, device=dev)]

    def step():
        run = ex.run_forward(rows, need_grad=True)
        return ex.measure(run)[0], ex.run_backward(rows, run, ex.seed_adjoint(run, up)), run["kept"]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        held = ex._keep_forward(ex.networks[0], 2, dev)  # pylint: disable=protected-access
        assert held is not None
        del held
        step()
        torch.cuda.synchronize()
        monkeypatch.setattr(X, "_KEPT_FREELY", 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            value, grad, _ = step()
    monkeypatch.undo()
    torch.cuda.synchronize()
    for seed in (7, 8, 9):
        rows.copy_(rows_for(n_params, 2, seed))
        want_v, want_g, _ = step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert float((value - want_v).abs().max()) < 1e-5
        assert float((grad - want_g).abs().max()) < 1e-5 * max(1.0, float(want_g.abs().max()))


@pytest.mark.gpu
def test_a_backward_on_another_stream_contracts_again(monkeypatch):
    """The intermediates belong to the forward's stream; a backward elsewhere, after waiting for the forward, leaves
    them alone and gives the same gradient."""
    cc, n_params = lattice(4, 4, 4, 5, False)
    dev = torch.device("cuda", 0)
    ex = TNExecutor(cc)
    rows, up = rows_for(n_params, 2, 5).to(dev), [torch.ones(2, device=dev)]
    run = ex.run_forward(rows, need_grad=True)
    want = ex.run_backward(rows, run, ex.seed_adjoint(run, up))
    run = ex.run_forward(rows, need_grad=True)
    used, backward = [], ex._backward_network  # pylint: disable=protected-access

    def traced(*args):
        used.append(args[-1])
        return backward(*args)
    monkeypatch.setattr(ex, "_backward_network", traced)
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(other):
        got = ex.run_backward(rows, run, ex.seed_adjoint(run, up))
    torch.cuda.synchronize()
    assert used == [None]
    assert torch.equal(got, want)
