"""Decoder layers over the MI355X cache (rfsn_v10_mlx_ane_complete.py:55-172,
llama32_adapter.py:375-662): the reference suite's layer test, and each
layer's cache-backed decode step against a float64 restatement of the layer
around the oracle's blockwise attention over the window the cache holds."""

import numpy as np
import pytest
import torch

from oracle import numerics as nx
from tests.conftest import randn16, rng

pytestmark = pytest.mark.gpu


def H(t):
    return t.detach().float().cpu().numpy()


def f16(a):
    return np.asarray(a, dtype=np.float64).astype(np.float16)


def _rms(x, w, eps):
    x = x.astype(np.float64)
    return f16(x / np.sqrt((x * x).mean(-1, keepdims=True) + eps) * w)


def _gelu(x):
    return 0.5 * x * (1.0 + np.tanh(0.7978845608 * (x + 0.044715 * x ** 3)))


def test_decoder_layer_api(device, tmp_path):
    """rfsn_v10_mlx_ane_complete.py:556-574 (the reference suite's config)."""
    from apple_amd.layer import RFSNDecoderLayerMLX
    from apple_amd.storage import RFSNConfig

    cfg = RFSNConfig(hidden_dim=512, num_heads=4, head_dim=128, num_layers=2, num_subspaces=8, subspace_dim=16,
                     num_rvq_layers=3, rvq_codebook_size=256, rvq_sparsity_threshold=0.25, hot_capacity=16,
                     warm_capacity=24, cold_capacity=128, block_size_seq=16, disk_cache_dir=str(tmp_path),
                     prefetch_throttle_s=0.0)
    layer = RFSNDecoderLayerMLX(cfg, layer_idx=0, device=device)
    g = rng(31)
    out = layer(torch.from_numpy(randn16(g, 2, 6, 512)).to(device), use_cache=False)
    assert out.shape == (2, 6, 512) and out.dtype == torch.float16
    layer.prefill_cache(torch.from_numpy(randn16(g, 1, 4, 512)).to(device))
    assert layer.cache_tokens == 4
    dec = layer(torch.from_numpy(randn16(g, 1, 1, 512)).to(device), use_cache=True, context_window=8)
    assert dec.shape == (1, 1, 512) and layer.cache_tokens == 5
    layer.reset_cache(remove_disk=True)
    assert layer.cache_tokens == 0
    with pytest.raises(ValueError):
        layer(torch.zeros((1, 2, 512), dtype=torch.float16, device=device), use_cache=True)


def _ext_config(tmp_path, **kw):
    from apple_amd.storage import RFSNConfig

    base = dict(hidden_dim=512, num_heads=8, head_dim=64, num_subspaces=16, subspace_dim=4, num_rvq_layers=1,
                rvq_codebook_size=256, rvq_sparsity_threshold=0.0, hot_capacity=64, warm_capacity=256,
                block_size_seq=64, num_kv_heads=4, rvq_subspaces=16, sparse_topk=4, tier_policy="recency",
                cold_medium="pinned", cold_chunk_tokens=64, disk_cache_dir=str(tmp_path))
    base.update(kw)
    return RFSNConfig(**base)


def _ext_quantizer(cfg, device, seed):
    from apple_amd.quantization import HybridQuantizerMLX
    from tests.conftest import rand_codebooks

    g = rng(seed)
    return HybridQuantizerMLX(cfg, device=device, pq_codebooks=torch.from_numpy(rand_codebooks(g, 16, 256, 4)),
                              rvq_codebooks=torch.from_numpy(rand_codebooks(g, 16, 256, 4) * np.float16(0.35)))


def test_rfsn_layer_decode_matches_restatement(device, tmp_path):
    """Prompt prefill, then three cache-backed decode steps of the reference
    layer on the long-context format (grouped KV heads, pinned cold chunks):
    each step equals RMSNorm -> o_proj(attention over the cache's window) ->
    residual -> GELU FFN restated in float64, the attention by the oracle
    over the window the cache materializes, within 2e-2."""
    from apple_amd.layer import RFSNDecoderLayerMLX

    cfg = _ext_config(tmp_path)
    layer = RFSNDecoderLayerMLX(cfg, device=device, quantizer=_ext_quantizer(cfg, device, 7))
    g = rng(32)
    layer.prefill_cache(torch.from_numpy(randn16(g, 1, 500, 512)).to(device))
    assert layer.cache.num_cold > 0 and layer.cache._fused_ok()
    W = {n: H(getattr(layer, n)).astype(np.float64) for n in ("q_proj", "o_proj", "ffn_up", "ffn_down")}
    for step in range(3):
        x = randn16(g, 1, 1, 512)
        out = H(layer(torch.from_numpy(x).to(device), use_cache=True))
        pos = layer.cache.total_tokens - 1
        window = max(cfg.block_size_seq, min(layer.cache.total_tokens, cfg.warm_capacity))
        mk, mv, adj = layer.cache.materialize_window(query_positions=torch.tensor([pos], device=device),
                                                     context_window=window)
        a = _rms(x[0], 1.0, 1e-5)
        q = f16(a.astype(np.float64) @ W["q_proj"].T).reshape(1, 8, 64)
        att = nx.blockwise_attention(q, H(mk).astype(np.float16), H(mv).astype(np.float16), 64 ** -0.5,
                                     cfg.block_size_seq, True, H(adj).astype(np.int32))
        hidden = f16(x[0].astype(np.float64) + f16(att.reshape(1, 512).astype(np.float64) @ W["o_proj"].T))
        ffn = f16(_gelu(_rms(hidden, 1.0, 1e-5).astype(np.float64) @ W["ffn_up"].T) @ W["ffn_down"].T)
        ref = f16(hidden.astype(np.float64) + ffn)
        assert np.abs(out[0] - ref.astype(np.float32)).max() <= 2e-2, step
    assert layer.cache_tokens == 503


def test_llama_layer_decode_matches_restatement(device, tmp_path):
    """The Llama layer: rotary embeddings on q and k (positions continue
    after the prompt), grouped KV heads stored as they are, SwiGLU MLP; a
    decode step against a float64 restatement around the oracle attention,
    and the prompt path (dense attention over repeated KV heads) against the
    same restatement."""
    from apple_amd.layer import LLAMA3_ROPE_SCALING, Llama32DecoderLayerMLX, rope_cos_sin

    cfg = _ext_config(tmp_path)
    layer = Llama32DecoderLayerMLX(cfg, intermediate_size=1024, device=device, quantizer=_ext_quantizer(cfg, device, 8))
    W = {n: H(getattr(layer, n)).astype(np.float64) for n in Llama32DecoderLayerMLX.WEIGHTS}
    g = rng(33)
    S = 400
    prompt = randn16(g, 1, S, 512)
    layer.prefill_cache(torch.from_numpy(prompt).to(device))

    def rope(x, pos):                      # x [S, h, 64] fp16 -> fp16
        cos, sin = (t.double().cpu().numpy() for t in rope_cos_sin(torch.tensor(pos), 64, 500000.0,
                                                                      LLAMA3_ROPE_SCALING))
        xf = x.astype(np.float64)
        rot = np.concatenate([-xf[..., 32:], xf[..., :32]], -1)
        return f16(xf * cos[:, None, :] + rot * sin[:, None, :])

    def mlp(h):
        m = _rms(h, W["post_attention_layernorm"], 1e-5).astype(np.float64)
        gate = f16(m @ W["gate_proj"].T).astype(np.float64)
        up = f16(m @ W["up_proj"].T).astype(np.float64)
        act = f16(gate / (1.0 + np.exp(-gate))).astype(np.float64)
        return f16(f16(act * up).astype(np.float64) @ W["down_proj"].T)

    x = randn16(g, 1, 1, 512)
    out = H(layer(torch.from_numpy(x).to(device), use_cache=True))
    n = _rms(x[0], W["input_layernorm"], 1e-5).astype(np.float64)
    q = rope(f16(n @ W["q_proj"].T).reshape(1, 8, 64), [S])
    mk, mv, _ = layer.cache.materialize_window()
    att = nx.blockwise_attention(q, H(mk).astype(np.float16), H(mv).astype(np.float16), 0.125, 64, False, None)
    hidden = f16(x[0].astype(np.float64) + f16(att.reshape(1, 512).astype(np.float64) @ W["o_proj"].T))
    ref = f16(hidden.astype(np.float64) + mlp(hidden))
    assert np.abs(out[0] - ref.astype(np.float32)).max() <= 2e-2
    # the newest key in the cache is the rotated projection of the decode token
    k_new = rope(f16(n @ W["k_proj"].T).reshape(1, 4, 64), [S])
    assert np.abs(H(layer.cache.hot_keys[-1]) - k_new[0].astype(np.float32)).max() <= 4e-3  # one fp16 ulp
    # prompt path: dense causal attention over the KV heads repeated to the query heads
    xs = randn16(g, 1, 24, 512)
    layer.reset_cache()
    dense = H(layer(torch.from_numpy(xs).to(device), use_cache=False))
    n = _rms(xs[0], W["input_layernorm"], 1e-5).astype(np.float64)
    pos = list(range(24))
    qs = rope(f16(n @ W["q_proj"].T).reshape(24, 8, 64), pos)
    ks = np.repeat(rope(f16(n @ W["k_proj"].T).reshape(24, 4, 64), pos), 2, axis=1)
    vs = np.repeat(f16(n @ W["v_proj"].T).reshape(24, 4, 64), 2, axis=1)
    ctx = np.zeros((24, 8, 64))
    for t in range(24):
        s = np.einsum("hd,thd->ht", qs[t].astype(np.float64), ks[:t + 1].astype(np.float64)) * 0.125
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        ctx[t] = np.einsum("ht,thd->hd", p, vs[:t + 1].astype(np.float64))
    hidden = f16(xs[0].astype(np.float64) + f16(f16(ctx).reshape(24, 512).astype(np.float64) @ W["o_proj"].T))
    ref = f16(hidden.astype(np.float64) + mlp(hidden))
    assert np.abs(dense[0] - ref.astype(np.float32)).max() <= 2e-2


def test_llama_layer_cpu_rotary_module(device, tmp_path):
    """A rotary module whose buffers live on the CPU is called on the CPU
    (llama32_adapter.py:535-553 resolves the device from the module) and its
    tables give the same decode step as the layer's own rope_cos_sin."""
    from apple_amd.layer import LLAMA3_ROPE_SCALING, Llama32DecoderLayerMLX, rope_cos_sin

    class CpuRotary(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.register_buffer("anchor", torch.zeros(1))
            self.calls = 0

        def forward(self, hidden, position_ids):
            assert hidden.device.type == "cpu" and position_ids.device.type == "cpu"
            self.calls += 1
            cos, sin = rope_cos_sin(position_ids.reshape(-1), 64, 500000.0, LLAMA3_ROPE_SCALING)
            return cos[None], sin[None]

    cfg = _ext_config(tmp_path)
    base = Llama32DecoderLayerMLX(cfg, intermediate_size=256, device=device, quantizer=_ext_quantizer(cfg, device, 8),
                                  generator=torch.Generator().manual_seed(4))
    weights = {n: getattr(base, n).detach().clone() for n in Llama32DecoderLayerMLX.WEIGHTS}
    rot = CpuRotary()
    other = Llama32DecoderLayerMLX(_ext_config(tmp_path / "b"), intermediate_size=256, device=device,
                                   quantizer=_ext_quantizer(cfg, device, 8), weights=weights, rotary_module=rot)
    g = rng(34)
    prompt = torch.from_numpy(randn16(g, 1, 40, 512)).to(device)
    x = torch.from_numpy(randn16(g, 1, 1, 512)).to(device)
    outs = []
    for layer in (base, other):
        layer.prefill_cache(prompt)
        outs.append(H(layer(x, use_cache=True)))
    assert rot.calls >= 2
    np.testing.assert_array_equal(outs[0], outs[1])


def test_llama_layer_session_follows_its_cache(device, tmp_path):
    """The layer's cached steps through its decode session against the general update + attention_forward: the
    same cache rows and access counters and attention within a rounding of fp16, over demotions, writes and
    recalibration from outside between steps, another stream, a smaller window, the first cold spill and a reset."""
    from apple_amd.layer import Llama32DecoderLayerMLX

    layers = []
    for sub in ("a", "b"):
        cfg = _ext_config(tmp_path / sub, warm_capacity=192)
        layers.append(Llama32DecoderLayerMLX(cfg, intermediate_size=256, device=device,
                                             quantizer=_ext_quantizer(cfg, device, 8),
                                             generator=torch.Generator().manual_seed(4)))
    ours, general = layers
    general._session = lambda: None
    g = rng(35)
    t = lambda *s: torch.from_numpy(randn16(g, *s)).to(device)
    prompt = t(1, 90, 512)
    for layer in layers:
        layer.prefill_cache(prompt)
    used = 0
    for step in range(150):
        if step in (7, 40):                      # tokens written past the layer
            k, v = t(step, 4, 64), t(step, 4, 64)
            for layer in layers:
                layer.cache.update(k, v, layer.quantizer)
        if step == 20:                           # codebooks recalibrated in place
            for layer in layers:
                layer.quantizer.pq.codebooks.mul_(1.01)
        kw = dict(context_window=70) if step in (11, 12) else {}
        x = t(1, 1, 512)
        with torch.cuda.stream(torch.cuda.Stream(device) if step in (30, 31) else torch.cuda.current_stream(device)):
            torch.cuda.synchronize()
            outs = [layer(x, use_cache=True, **kw) for layer in layers]
            torch.cuda.synchronize()
        used += ours._session() is not None
        a, b = (H(o) for o in outs)
        assert np.abs(a - b).max() <= 4e-3, step   # one fp16 step of the hidden state's values below 4
        assert ours.cache.get_last_access_stats() == general.cache.get_last_access_stats(), step
        assert torch.equal(ours.cache.hot_keys, general.cache.hot_keys)
        assert torch.equal(ours.cache.warm_keys.pq_codes, general.cache.warm_keys.pq_codes)
    assert 60 < used < 140 and ours.cache.num_cold > 0 and ours._decode.regrows + ours._decode.rebuilds > 1
    for layer in layers:
        layer.prefill_cache(prompt)
    a, b = (H(layer(x, use_cache=True)) for layer in layers)
    assert np.abs(a - b).max() <= 4e-3


def _llama(device, tmp_path, **kw):
    from apple_amd.layer import Llama32DecoderLayerMLX

    cfg = _ext_config(tmp_path)
    return Llama32DecoderLayerMLX(cfg, intermediate_size=256, device=device, quantizer=_ext_quantizer(cfg, device, 8),
                                  generator=torch.Generator().manual_seed(4), **kw)


def test_llama_layer_watched_tables(device, tmp_path):
    """Gradients of rotary tables (given, or made by a trainable rotary module) and tables mapped by vmap go through
    torch's operators; the same tables unwatched agree with them."""
    from apple_amd.layer import rope_cos_sin

    layer = _llama(device, tmp_path / "a")
    g = rng(36)
    x = torch.from_numpy(randn16(g, 1, 6, 512)).to(device)
    cos, sin = rope_cos_sin(torch.arange(3, 9, device=device), 64)
    plain = layer(x, position_embeddings=(cos, sin))
    assert layer._native(x, (cos, sin)) and not plain.requires_grad
    for i in (0, 1):
        t = [cos.clone(), sin.clone()]
        t[i].requires_grad_()
        out = layer(x, position_embeddings=tuple(t))
        assert out.requires_grad and (out - plain).abs().max() <= 4e-3
        out.float().sum().backward()
        assert t[i].grad is not None and bool(t[i].grad.any())
        with torch.no_grad():
            assert torch.equal(layer(x, position_embeddings=tuple(t)), plain)
    many = torch.func.vmap(lambda c, s: layer(x, position_embeddings=(c, s)))(torch.stack([cos, sin]), torch.stack([sin, cos]))
    assert (many[0] - plain).abs().max() <= 4e-3

    class Trained(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.shift = torch.nn.Parameter(torch.zeros((), device=device))

        def forward(self, hidden, position_ids):
            return tuple(t + self.shift for t in rope_cos_sin(position_ids.reshape(-1), 64))

    rot = Trained()
    layer = _llama(device, tmp_path / "b", rotary_module=rot)
    out = layer(x)
    assert out.requires_grad
    out.float().sum().backward()
    assert rot.shift.grad is not None and float(rot.shift.grad) != 0.0


def test_llama_layer_functional_weights(device, tmp_path):
    """torch.func.grad and vmap over the layer's weights with a plain input."""
    layer = _llama(device, tmp_path)
    x = torch.from_numpy(randn16(rng(37), 1, 5, 512)).to(device)
    w = layer.down_proj.detach()
    call = lambda t: torch.func.functional_call(layer, {"down_proj": t}, (x,))
    grad = torch.func.grad(lambda t: call(t).float().sum())(w)
    assert grad.shape == w.shape and bool(grad.any())
    many = torch.func.vmap(call)(torch.stack([w, 2 * w]))
    plain = layer(x)
    assert (many[0] - plain).abs().max() <= 4e-3 and not torch.equal(many[0], many[1])


def test_llama_layer_frequencies_on_every_stream(device, tmp_path):
    """The rotary frequencies that calls on any stream read are complete before the first of them; a graph capture
    that finds none leaves none behind, and its replays agree with the eager call."""
    layer = _llama(device, tmp_path)
    x = torch.from_numpy(randn16(rng(38), 1, 70, 512)).to(device)
    kept = layer.__dict__["_inv_freq_kept"]
    with torch.cuda.stream(torch.cuda.Stream(device)):
        plain = layer(x)
        assert layer.__dict__["_inv_freq_kept"] is kept  # nothing made on the call's stream
        torch.cuda.synchronize()
    del layer._inv_freq_kept
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(x)
    assert "_inv_freq_kept" not in layer.__dict__
    eager = layer(x)  # before any replay: reads frequencies of its own
    torch.cuda.synchronize()
    assert torch.equal(eager, plain) and "_inv_freq_kept" in layer.__dict__
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, plain) and torch.equal(layer(x), plain)
    layer.rope_theta = 10000.0
    assert not torch.equal(layer(x), plain) and layer._inv_freq_kept[0][1] == 10000.0


def test_llama_layer_saved_without_shapes(device, tmp_path):
    """A layer pickled before it kept its weights' shapes runs, and as the one it was saved from."""
    import copy

    layer = _llama(device, tmp_path)
    x = torch.from_numpy(randn16(rng(39), 1, 9, 512)).to(device)
    for names in (["_shapes", "_linear_ok"], ["_linear_ok"]):
        state = copy.deepcopy(layer.__getstate__())
        for n in names:
            del state[n]
        old = type(layer).__new__(type(layer))
        old.__setstate__(state)
        assert old._shapes == layer._shapes and old._native(x) and torch.equal(old(x), layer(x))


def test_llama_layer_carries_infinite_and_nan_tokens(device, tmp_path):
    """A prompt token that is no number reaches itself and the tokens after it, and none before."""
    layer = _llama(device, tmp_path)
    x = torch.from_numpy(randn16(rng(40), 1, 90, 512)).to(device)
    plain = layer(x)
    for value in (float("nan"), float("inf")):
        y = x.clone()
        y[0, 50, 3] = value
        out = layer(y)
        assert (out[0, :50] - plain[0, :50]).abs().max() <= 4e-3  # blocks that repeat their sums round anew
        assert bool(out[0, 50:].isnan().all())  # the norm of an infinite row holds inf * 0


def test_llama_layer_calls_the_methods_of_its_cache(device, tmp_path):
    """A cache class of the caller's sees every cached step through its own methods."""
    from apple_amd.cache import RFSNv10KVCacheMLX

    calls = []

    class Counted(RFSNv10KVCacheMLX):
        def update(self, *a, **kw):
            calls.append("update")
            return super().update(*a, **kw)

        def attention_forward(self, *a, **kw):
            calls.append("attend")
            return super().attention_forward(*a, **kw)

    layer = _llama(device, tmp_path)
    layer.cache = Counted(layer.config, layer_idx=0, device=device)
    g = rng(41)
    layer.prefill_cache(torch.from_numpy(randn16(g, 1, 70, 512)).to(device), reset=False)
    for _ in range(3):
        layer(torch.from_numpy(randn16(g, 1, 1, 512)).to(device), use_cache=True)
    assert calls == ["update"] + ["update", "attend"] * 3
