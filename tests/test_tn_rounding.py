"""Rounding of the batched environments of small steps (tedq_tn_small_environments)."""

import ctypes

import numpy as np
import pytest
import torch

from tedq_amd.engine import hip
from tedq_amd.tn.executor import make_desc

from tn_emulator import contract_np


@pytest.mark.gpu
@pytest.mark.parametrize("na,nb,nk,lanes", [(4, 4, 8, 1), (6, 6, 6, 1), (4, 2, 8, 4), (3, 3, 9, 4), (2, 2, 10, 16)])
def test_rounding_of_small_environments(na, nb, nk, lanes):
    """Outputs that share a workgroup's threads, so that a lane has many terms: it keeps eight sums of c terms, two
    roundings each, and everything after that is pairwise.  A sum of random signs rounds by (j / c)^(1/2) of its size
    after j terms, so the result's root mean square error is 2^-24 (c + 3 + log2 lanes + 1)^(1/2) of its size at
    most; one sum per lane would have about sqrt(8) times the first part."""
    dev, rng = torch.device("cuda", 0), np.random.default_rng(na + nk)
    la = [f"m{i}" for i in range(na)] + [f"k{i}" for i in range(nk)]
    lb = [f"k{i}" for i in range(nk)] + [f"n{i}" for i in range(nb)]
    lc = [f"m{i}" for i in range(na)] + [f"n{i}" for i in range(nb)]
    desc = make_desc(la, lb, lc)
    size = 1 << (na + nb)
    a, b = (torch.tensor(rng.normal(size=(1, n)) + 1j * rng.normal(size=(1, n)), dtype=torch.complex64, device=dev)
            for n in (1 << (na + nk), 1 << (nb + nk)))
    out = torch.zeros((1, size), dtype=torch.complex64, device=dev)
    ten = [a, b, out, out, out]
    bases = (ctypes.c_void_p * 5)(*[t.data_ptr() for t in ten])
    sizes = (ctypes.c_int64 * 5)(*[t.shape[1] for t in ten])
    recs = np.array([[0, 0, 0, 1, 0, 0, size, 2]], dtype=np.int64)
    drecs, ddesc = torch.from_numpy(recs).to(dev), torch.from_numpy(desc).to(dev)
    hip.call("tedq_tn_small_environments", bases, sizes, sizes, recs.ctypes.data_as(hip.c_vp), hip.ptr(drecs), 1, 1,
             desc.ctypes.data_as(hip.c_vp), hip.ptr(ddesc), 1, hip.stream_handle(dev))
    want = np.zeros((1, size), dtype=np.complex128)
    contract_np(desc, a.cpu().numpy().astype(np.complex128), b.cpu().numpy().astype(np.complex128), want)
    err = np.sqrt(np.mean(np.abs(out.cpu().numpy() - want) ** 2) / np.mean(np.abs(want) ** 2))
    terms = (1 << nk) // (8 * lanes)
    assert err < 2.0 ** -24 * np.sqrt(terms + 3 + np.log2(lanes) + 1)
