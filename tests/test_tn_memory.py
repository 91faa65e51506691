"""Device memory that contraction mode holds (tedq_amd.tn.executor)."""

import weakref

import torch

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
