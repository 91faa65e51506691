"""Measurement kernels at the sizes where they change form: chunk sums around the switch between their
two kernels, factored observables batched per factor count, marginals around one thread block.

References are float64.  Sums are accumulated in fp64, so they agree to 1e-12 of the sum of magnitudes;
quantities that pass through fp32 products (factors of magnitude about 1 on unit-norm states: four fp32
roundings per factor) to 2e-6; lambda, an fp32 sum of `count` such terms of size max |psi|, to
count * 1e-6 of that.
"""

import ctypes

import numpy as np
import pytest
import torch

from tedq_amd.engine import hip

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _hp(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _state(batch, n, seed):
    rng = np.random.default_rng(seed)
    psi = rng.normal(size=(batch, 1 << n)) + 1j * rng.normal(size=(batch, 1 << n))
    psi /= np.linalg.norm(psi, axis=1, keepdims=True)
    t = torch.tensor(psi, dtype=torch.complex64, device=DEV)
    return t, t.cpu().numpy().astype(np.complex128)


@pytest.mark.parametrize("batch,chunks,m", [(3, 15, 5), (3, 16, 5), (2, 17, 1), (5, 1000, 25), (1, 256, 32), (2, 64, 33),
                                            (1, 31, 100)])
def test_sum_partials(batch, chunks, m):
    rng = np.random.default_rng(chunks)
    p = rng.normal(size=(batch, chunks, m)) * 10.0 ** rng.integers(-6, 6, size=(batch, chunks, m))
    t = torch.tensor(p, device=DEV)
    out = torch.empty((batch, m), dtype=torch.float64, device=DEV)
    hip.call("tedq_sum_partials", hip.ptr(t), batch, chunks, m, hip.ptr(out), hip.stream_handle(DEV))
    assert np.max(np.abs(out.cpu().numpy() - p.sum(1)) / np.abs(p).sum(1)) < 1e-12


def _operator_row(psi, bits, fac, zmask, n):
    x = np.arange(1 << n)
    out = psi
    for b, f in zip(bits, fac):
        flip = out[:, x ^ (1 << b)]
        one = (x >> b) & 1
        out = np.where(one, f[1, 0] * flip + f[1, 1] * out, f[0, 0] * out + f[0, 1] * flip)
    # the sign is that of the group: the factors' own bits are clear in it
    clear = x & ~np.int64(sum(1 << b for b in bits))
    sign = np.array([1 - 2 * (bin(int(c) & zmask).count("1") & 1) for c in clear])
    return sign * out


@pytest.mark.parametrize("n,q,count,batch", [(1, 1, 1, 3), (4, 4, 2, 2), (5, 2, 3, 1), (9, 0, 2, 2), (12, 1, 5, 2),
                                             (13, 1, 13, 1), (14, 3, 2, 1), (16, 2, 3, 2), (18, 1, 4, 1)])
def test_factored_batch(n, q, count, batch):
    rng = np.random.default_rng(10 * n + q)
    psi, ref = _state(batch, n, n)
    size = hip.load().tedq_sv_factored_record_bytes()
    recs = np.zeros((count, size), dtype=np.uint8)
    want, lam = np.zeros((batch, count)), np.zeros_like(ref)
    coef = rng.normal(size=(batch, count))
    for o in range(count):
        bits = rng.permutation(n)[:q].astype(np.int32)
        fac = (rng.normal(size=(q, 2, 2)) + 1j * rng.normal(size=(q, 2, 2))) / 2
        zmask = int(rng.integers(0, 1 << n)) & ~int(sum(1 << int(b) for b in bits))
        f32 = np.ascontiguousarray(fac.astype(np.complex64)).view(np.float32).reshape(-1)
        hip.call("tedq_sv_factored_record", _hp(recs[o]), n, q, _hp(bits), _hp(f32), zmask)
        fac = fac.astype(np.complex64).astype(np.complex128)
        row = _operator_row(ref, bits, fac, zmask, n)
        want[:, o] = (ref.conj() * row).sum(1).real
        dag = _operator_row(ref, bits, [f.conj().T for f in fac], zmask, n)
        lam += coef[:, o:o + 1] * 0.5 * (row + dag)
    drecs = torch.from_numpy(recs.copy()).to(DEV)
    part = torch.empty((batch, count, hip.load().tedq_sv_factored_chunks(n, q)), dtype=torch.float64, device=DEV)
    out = torch.empty((batch, count), dtype=torch.float64, device=DEV)
    st = hip.stream_handle(DEV)
    hip.call("tedq_sv_expval_factored_batch", hip.ptr(psi), batch, n, q, _hp(recs), hip.ptr(drecs), count, hip.ptr(part),
             hip.ptr(out), st)
    assert np.max(np.abs(out.cpu().numpy() - want)) < 2e-6
    if q == 1:
        got = torch.zeros_like(psi)
        tc = torch.tensor(coef, device=DEV)
        hip.call("tedq_sv_lambda_factored_batch", hip.ptr(psi), hip.ptr(got), batch, n, _hp(recs), hip.ptr(drecs), count,
                 hip.ptr(tc), st)
        assert np.max(np.abs(got.cpu().numpy() - lam)) < count * 1e-6 * np.abs(ref).max() * max(1, np.abs(coef).max())


@pytest.mark.parametrize("n,bits", [(3, [1]), (8, [0]), (9, [8]), (10, [3, 7]), (11, [10, 0]), (13, [5]), (15, [2]),
                                    (17, [16, 1, 9])])
def test_marginals(n, bits):
    psi, ref = _state(2, n, n)
    k = len(bits)
    b32 = np.asarray(bits, dtype=np.int32)
    part = torch.empty((2, hip.load().tedq_sv_probs_chunks(n, k), 1 << k), dtype=torch.float64, device=DEV)
    out = torch.empty((2, 1 << k), dtype=torch.float32, device=DEV)
    hip.call("tedq_sv_probs", hip.ptr(psi), 2, n, k, _hp(b32), hip.ptr(part), hip.ptr(out), hip.stream_handle(DEV))
    x = np.arange(1 << n)
    y = np.zeros_like(x)
    for b in bits:
        y = (y << 1) | ((x >> b) & 1)
    want = np.stack([np.bincount(y, weights=np.abs(r) ** 2, minlength=1 << k) for r in ref])
    assert np.max(np.abs(out.cpu().numpy() - want)) < 2e-7
