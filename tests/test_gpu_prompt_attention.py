"""Many-query exact attention on the matrix cores against float64.

The kernel takes 64, 128 or 256 query rows per block, 64-token tiles and one or
more token splits; the shapes sit at those edges.  Tolerance: the fp16 result's
rounding (2^-11 of the value) plus fp32 sums of weights kept to 22 bits, so
2^-11 |out| + 2^-15 max|v| (2^-22 per weight and 2^-24 per product would be
far below the second term; it covers the exponent of a score of up to 64)."""

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ref(q, k, v, scale, pos):
    B, Hq, D = q.shape
    T, Hkv, _ = k.shape
    G = Hq // Hkv
    kk, vv = k.astype(np.float64), v.astype(np.float64)
    out = np.zeros((B, Hq, D))
    for h in range(Hq):
        s = q[:, h].astype(np.float64) @ kk[:, h // G].T * scale
        if pos is not None:
            s = np.where(np.arange(T)[None] <= pos[:, h, None], s, -np.inf)
        m = s.max(1, keepdims=True)
        w = np.where(np.isfinite(s), np.exp(s - np.where(np.isfinite(m), m, 0)), 0)
        n = w.sum(1, keepdims=True)
        out[:, h] = (w @ vv[:, h // G]) / np.where(n > 0, n, 1)
    return out


CASES = [  # B, Hq, Hkv, T, D
    (4, 2, 2, 1, 64), (5, 8, 4, 63, 64), (33, 4, 2, 64, 128), (16, 8, 2, 65, 64), (64, 2, 2, 129, 128),
    (65, 2, 2, 1537, 128), (150, 4, 2, 1600, 64), (257, 4, 4, 2000, 64), (600, 4, 2, 6200, 64), (7, 8, 1, 5000, 64),
]


@pytest.mark.parametrize("B,Hq,Hkv,T,D", CASES)
@pytest.mark.parametrize("mode", ["full", "causal", "mixed"])
def test_prompt_attention(device, B, Hq, Hkv, T, D, mode):
    import torch
    from apple_amd import kernels as K

    g = np.random.default_rng(B * 1000 + T)
    q, k, v = (g.standard_normal(s, dtype=np.float32).astype(np.float16)
               for s in ((B, Hq, D), (T, Hkv, D), (T, Hkv, D)))
    q[B // 2] *= np.float16(8)  # one sharp query
    if mode == "full":
        pos = None
    elif mode == "causal":
        pos = np.repeat((np.arange(B) + T - B)[:, None], Hq, 1).astype(np.int32)  # negative: nothing allowed
    else:
        pos = g.integers(-2, T + 2, (B, Hq)).astype(np.int32)
    dev = lambda a: torch.from_numpy(a).to(device)
    got = K.blockwise_attention(dev(q), dev(k), dev(v), D ** -0.5, pos is not None,
                                None if pos is None else dev(pos)).double().cpu().numpy()
    want = _ref(q, k, v, D ** -0.5, pos)
    assert np.all(np.abs(got - want) <= np.abs(want) * 2.0 ** -11 + np.abs(v).max().astype(np.float64) * 2.0 ** -15)
    if pos is not None:
        assert not got[pos < 0].any()


def test_prompt_attention_strides_and_views(device):
    """Strided K/V rows (a head-major ring), and a query view off 16-byte alignment (the scalar kernel's)."""
    import torch
    from apple_amd import kernels as K

    g = torch.Generator().manual_seed(5)
    ring = torch.randn(2, 3, 200, 64, generator=g).half().to(device)  # [K/V][head][token][D]
    k, v = (ring[i].permute(1, 0, 2)[7:190] for i in range(2))
    q = torch.randn(9 * 3 * 64 + 1, generator=g).half().to(device)
    want = _ref(q[1:].view(9, 3, 64).cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), 0.125, None)
    for qq in (q[1:].view(9, 3, 64), q[1:].view(9, 3, 64).clone()):
        got = K.blockwise_attention(qq, k, v, 0.125, False, None).double().cpu().numpy()
        assert np.all(np.abs(got - want) <= np.abs(want) * 2.0 ** -11 + 5 * 2.0 ** -15)


@pytest.mark.parametrize("fmt", ["gated", "subspace"])
def test_hybrid_attention_decodes_once_for_many_queries(device, monkeypatch, fmt):
    """A chunk past ``decode_first``'s line decodes both stores once and agrees with the decode-in-register
    kernel (which a chunk below the line keeps) and with float64 over the decoded rows."""
    import torch
    from apple_amd import attention as A
    from apple_amd import kernels as K
    from apple_amd.quantization import HybridQuantizerMLX, _compress_tensor_sequence, _decode_compressed_tensor
    from apple_amd.storage import RFSNConfig

    B, Hq, Hkv, T, D = 150, 8, 4, 301, 128
    ext = dict(rvq_subspaces=8, sparse_topk=4, rvq_codebook_size=256) if fmt == "subspace" else dict(rvq_codebook_size=64)
    cfg = RFSNConfig(hidden_dim=Hq * D, num_heads=Hq, head_dim=D, num_kv_heads=Hkv, num_rvq_layers=3,
                     rvq_sparsity_threshold=9.0, **ext)
    g = torch.Generator().manual_seed(11)
    qz = HybridQuantizerMLX(cfg, device=device, generator=g)
    r = lambda *s: torch.randn(*s, generator=g).half().to(device)
    ks, vs = (_compress_tensor_sequence(r(T, Hkv, D), qz) for _ in range(2))
    q, pos = r(B, Hq, D), torch.arange(T - B, T, dtype=torch.int32, device=device)
    assert K.decode_first(B, Hq, Hkv, D, T, False)
    att = A.RFSNHybridAttentionMLX(cfg)
    got = att(q, ks, vs, qz, causal=True, query_positions=pos)
    # without room for the decoded window, or where the caller declines it, the chunk keeps the kernel in registers
    decoded = []

    def no_room(store, quantizer):
        decoded.append(store)
        raise torch.OutOfMemoryError("no room")

    with monkeypatch.context() as m:
        m.setattr(A, "_decode_compressed_tensor", no_room)
        reg = att(q, ks, vs, qz, causal=True, query_positions=pos)
        assert len(decoded) == 1
        qz.config = dataclasses.replace(cfg, hybrid_window_bytes=0)
        declined = att(q, ks, vs, qz, causal=True, query_positions=pos)
        assert len(decoded) == 1 and torch.equal(declined, reg)
        qz.config = cfg
    monkeypatch.setattr(K, "decode_first", lambda *a: False)
    assert torch.equal(att(q, ks, vs, qz, causal=True, query_positions=pos), reg)
    k, v = (_decode_compressed_tensor(s, qz).cpu().numpy() for s in (ks, vs))
    want = _ref(q.cpu().numpy(), k, v, D ** -0.5, np.repeat(pos.cpu().numpy()[:, None], Hq, 1))
    for out in (got, reg):
        err = np.abs(out.double().cpu().numpy() - want)
        assert np.all(err <= np.abs(want) * 2.0 ** -11 + np.abs(v).max().astype(np.float64) * 2.0 ** -15)


@pytest.mark.parametrize("T", [0, 5])
@pytest.mark.parametrize("B,Hkv", [(0, 2), (3, 0)])
def test_empty_sizes_are_refused(device, T, B, Hkv):
    """No queries, or no KV heads: the launch's ValueError, whatever the window."""
    import torch
    from apple_amd import kernels as K

    z = lambda *s: torch.zeros(s, dtype=torch.float16, device=device)
    with pytest.raises(ValueError):
        K.blockwise_attention(z(B, 2, 64), z(T, Hkv, 64), z(T, Hkv, 64), 0.125, False, None)


@pytest.mark.parametrize("B,Hq,Hkv,T,D", [(4, 2, 2, 1, 64), (5, 8, 4, 63, 64), (33, 4, 2, 65, 128), (65, 2, 2, 1537, 128),
                                          (150, 4, 2, 1600, 64), (600, 4, 2, 6200, 64), (7, 8, 1, 5000, 64)])
def test_infinite_values(device, B, Hq, Hkv, T, D):
    """Infinite values meet every weight as p * V does: infinities where one sign is seen, NaN where both are, and the
    other coordinates as without them; from many query rows as from one (the scalar kernel)."""
    import torch
    from apple_amd import kernels as K

    g = np.random.default_rng(T)
    q, k, v = (g.standard_normal(s, dtype=np.float32).astype(np.float16)
               for s in ((B, Hq, D), (T, Hkv, D), (T, Hkv, D)))
    want = _ref(q, k, v, D ** -0.5, None)
    v[T - 1, :, 1] = np.inf                              # the last token, which the tiles' ends repeat
    v[T // 2, :, 7] = v[T // 3, :, 7] = -np.inf
    v[0, :, D - 1], v[T - 1, :, D - 1] = np.inf, -np.inf
    v[T // 2, 0, 9] = np.nan
    want[:, :, 1], want[:, :, 7] = np.inf, -np.inf
    want[:, :, D - 1] = np.nan if T > 1 else -np.inf
    want[:, :Hq // Hkv, 9] = np.nan
    dev = lambda a: torch.from_numpy(a).to(device)
    tol = np.where(np.isfinite(want), np.abs(want), 0) * 2.0 ** -11 + 6 * 2.0 ** -15
    runs = [K.blockwise_attention(dev(q), dev(k), dev(v), D ** -0.5, False, None, dense=d) for d in (False, True)]
    if Hq == Hkv:  # one query row per KV head: the scalar kernel
        runs.append(torch.cat([K.blockwise_attention(dev(q[i:i + 1]), dev(k), dev(v), D ** -0.5, False, None)
                               for i in range(B)]))
    for got in runs:
        got = got.double().cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        same = np.isfinite(want)
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        assert np.all(np.abs(got[same] - want[same]) <= tol[same])
    # a causal chunk: every row as the values it may read make it, and no others
    if B * Hq // Hkv >= 4:
        pos = g.integers(-1, T, (B, Hq)).astype(np.int32)
        got = K.blockwise_attention(dev(q), dev(k), dev(v), D ** -0.5, True, dev(pos)).double().cpu().numpy()
        fin = np.where(np.isfinite(v), v, np.float16(0))
        want = _ref(q, k, fin, D ** -0.5, pos)
        seen = (np.arange(T)[None, None] <= pos[..., None])[..., None]           # [B, Hq, T, 1]
        vh = np.repeat(v, Hq // Hkv, 1).transpose(1, 0, 2)[None]                   # [1, Hq, T, D]
        up, down, nan = ((seen & f(vh)).any(2) for f in (np.isposinf, np.isneginf, np.isnan))
        want[up], want[down], want[nan | (up & down)] = np.inf, -np.inf, np.nan
        same = np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        assert np.all(np.abs(got[same] - want[same]) <= np.abs(want[same]) * 2.0 ** -11 + 6 * 2.0 ** -15)


@pytest.mark.parametrize("B,Hq,Hkv,T,D", [(1, 2, 2, 70, 64), (6, 2, 2, 70, 64), (40, 4, 2, 1500, 128)])
def test_scores_that_are_no_numbers(device, B, Hq, Hkv, T, D):
    """A NaN in a query, or in a key it may see: zeros from blockwise attention, whatever the number of query rows
    (one is the scalar kernel's), and NaN from dense attention; keys past a query's position change nothing."""
    import torch
    from apple_amd import kernels as K

    g = np.random.default_rng(T)
    q, k, v = (g.standard_normal(s, dtype=np.float32).astype(np.float16)
               for s in ((B, Hq, D), (T, Hkv, D), (T, Hkv, D)))
    pos = np.repeat((np.arange(B) + T - B)[:, None], Hq, 1).astype(np.int32)
    want = _ref(q, k, v, D ** -0.5, pos)
    k[T - 1, 0, 3] = np.nan                              # the last query's own key
    q[B // 2, -1, 5] = np.nan
    bad = np.zeros((B, Hq), bool)
    bad[B - 1, :Hq // Hkv] = bad[B // 2, -1] = True
    dev = lambda a: torch.from_numpy(a).to(device)
    for dense in (False, True) if B * Hq // Hkv >= 4 else (False,):
        got = K.blockwise_attention(dev(q), dev(k), dev(v), D ** -0.5, True, dev(pos), dense=dense)
        got = got.double().cpu().numpy()
        assert (np.isnan(got[bad]).all() if dense else not got[bad].any())
        assert np.all(np.abs(got - want)[~bad] <= np.abs(want[~bad]) * 2.0 ** -11 + 5 * 2.0 ** -15)
    if B == 1:
        with pytest.raises(Exception, match="dense_attention"):
            K.blockwise_attention(dev(q), dev(k), dev(v), D ** -0.5, True, dev(pos), dense=True)
