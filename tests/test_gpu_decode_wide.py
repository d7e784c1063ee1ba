"""The 8-coordinates-per-thread decode kernels against the oracle, bit for bit, at row counts off
the wave and block sizes, and against the general kernels where a view is off their alignment."""

import numpy as np
import pytest

from conftest import rand_codebooks, randn16, rng
from oracle import numerics as nx

pytestmark = pytest.mark.gpu


def _dev(a, device):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


@pytest.mark.parametrize("D,M,Mr,k", [(64, 16, 16, 4), (64, 16, 0, 4), (64, 8, 8, 0), (128, 8, 8, 4), (128, 4, 0, 0),
                                      (256, 16, 16, 4), (96, 12, 12, 4), (64, 8, 16, 4)])
@pytest.mark.parametrize("n", [1, 63, 777])
def test_decode_ext(device, D, M, Mr, k, n):
    from apple_amd import kernels as K

    g = rng(n + D + Mr)
    C = 200
    pq_cb, rvq_cb = rand_codebooks(g, M, C, D // M), rand_codebooks(g, Mr, C, D // Mr) if Mr else None
    pq = g.integers(0, C, (n, M), dtype=np.uint8)
    rvq = g.integers(0, C, (n, Mr), dtype=np.uint8) if Mr else None
    idx = np.stack([g.permutation(D)[:k] for _ in range(n)]).astype(np.uint8).reshape(n, k) if k else None
    val = randn16(g, n, k) if k else None
    want = nx.ext_decode(pq, pq_cb, rvq, rvq_cb, idx, val)
    t = [None if a is None else _dev(a, device) for a in (pq, pq_cb, rvq, rvq_cb, idx, val)]
    fmt = K.WarmFormat(D, M, C, Mr, C if Mr else 0, k)
    got = K.decode(fmt, *t).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
    if n > 1:  # rows from a view one code row in (8 or 16 B) and one byte off where the rows allow it
        sub = [t[0][1:], t[1], None if t[2] is None else t[2][1:], t[3], None if t[4] is None else t[4][1:],
               None if t[5] is None else t[5][1:]]
        odd = _dev(np.concatenate([np.zeros(1, np.uint8), pq.reshape(-1)]), device)[1:].view(n, M)
        assert np.array_equal(K.decode(fmt, *sub).cpu().numpy().view(np.uint16), want[1:].view(np.uint16))
        assert np.array_equal(K.decode(fmt, odd, *t[1:]).cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("D,M,L", [(64, 8, 2), (128, 8, 4), (128, 4, 5), (256, 32, 4), (128, 32, 3)])
@pytest.mark.parametrize("active", ["all", "most", "one", "none", "shuffled"])
def test_decode_ref(device, D, M, L, active):
    import torch
    from apple_amd import kernels as K

    g = rng(D + L)
    n, C, Cr = 333, 256, 1000
    pq_cb, rvq_cb = rand_codebooks(g, M, C, D // M), rand_codebooks(g, L, Cr, D)
    pq = g.integers(0, C, (n, M), dtype=np.uint8)
    offs = {"all": np.arange(n), "most": np.flatnonzero(g.random(n) < 0.9), "one": np.array([n - 1]),
            "none": np.zeros(0, int), "shuffled": g.permutation(n)[:200]}[active].astype(np.int32)
    codes = g.integers(0, Cr, (offs.size, L), dtype=np.uint16)
    mask = np.zeros(n, bool)
    mask[offs] = True
    want = nx.hybrid_decode(pq, codes, mask, offs, pq_cb, rvq_cb)
    got = K.decode_ref(_dev(pq, device), _dev(pq_cb, device), _dev(codes, device), _dev(offs, device),
                       _dev(rvq_cb, device))
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    if offs.size:  # offsets outside the rows are ignored; codebooks off 16-byte alignment take the general kernel
        far = np.concatenate([offs, [n, -1]]).astype(np.int32)
        more = np.concatenate([codes, codes[:1], codes[:1]])
        flat = torch.empty(rvq_cb.size + 1, dtype=torch.float16, device=device)
        flat[1:] = _dev(rvq_cb, device).view(-1)
        got = K.decode_ref(_dev(pq, device), _dev(pq_cb, device), _dev(more, device), _dev(far, device),
                           flat[1:].view(rvq_cb.shape))
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
        got = K.decode_ref(_dev(pq, device), _dev(pq_cb, device), _dev(more, device), _dev(far, device),
                           _dev(rvq_cb, device))
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
