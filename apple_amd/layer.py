"""Decoder layers over the MI355X cache: the caller one step up from the
decode path.

* ``RFSNDecoderLayerMLX`` -- the reference's layer
  (rfsn_v10_mlx_ane_complete.py:55-172): RMSNorm, q/k/v projections into the
  tiered cache, cache-backed single-token decode, o_proj and a GELU FFN.
* ``Llama32DecoderLayerMLX`` -- the Llama layer of llama32_adapter.py
  (375-662): RMSNorm with weights, rotary position embeddings on q and k,
  grouped KV heads and a SwiGLU MLP.  The cache stores the KV heads as they
  are (``num_kv_heads``); the reference repeats them to the query heads
  first (llama32_adapter.py:380-386, 578-579).

Norms, projections and activations are computed in fp32 from fp16
activations with fp16 results at the reference's cast points: by torch ops
in the reference's layer, and in the Llama layer by ``rfsn_layer_linear``
(RMSNorm, projection, rotary embedding / SwiGLU / residual in one pass over
the weights) with the prompt's attention on the matrix cores; where autograd,
a tracer, autocast or a tensor subclass watches the call, or weights are not
plain fp32 matrices, the Llama layer runs the same steps as torch ops.
Cache-backed decode goes through the cache's fused dequant-attention kernel.
Weights are module parameters: the reference's initialisation or a local
state dict; nothing is downloaded.
"""

from __future__ import annotations

import itertools
import math
import shutil
import threading
from pathlib import Path
from typing import Dict, Optional, Tuple

import torch

from . import kernels as K
from .cache import RFSNv10KVCacheMLX
from .quantization import HybridQuantizerMLX
from .storage import AsyncHierarchicalRouterMLX, RFSNConfig

MASK_FILL_VALUE = -1e30

_PLAIN_TYPES = (torch.Tensor, torch.nn.Parameter)
_wrapped = torch._C._functorch.is_functorch_wrapped_tensor  # a tensor that torch.func maps or differentiates

_INV_FREQ_LOCK = threading.Lock()  # two calls that miss a layer's kept frequencies make them once


def _gelu(x: torch.Tensor) -> torch.Tensor:
    """attention.py:137-138 (tanh form)."""
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608 * (x + 0.044715 * (x ** 3))))


def _dense_exact_attention(q: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, scale: float,
                           causal: bool = True) -> torch.Tensor:
    """attention.py:108-134: q [B, S, H, D], keys/values [B, T, H, D] ->
    [B, S, H, D] in q's dtype; fp32 scores, mask k_pos <= q_pos."""
    qf = q.float().permute(0, 2, 1, 3).contiguous()          # [B, H, S, D]
    kf = keys.float().permute(0, 2, 3, 1).contiguous()       # [B, H, D, T]
    vf = values.float().permute(0, 2, 1, 3).contiguous()     # [B, H, T, D]
    scores = torch.matmul(qf, kf) * scale
    if causal:
        qp = torch.arange(q.shape[1], device=q.device)
        kp = torch.arange(keys.shape[1], device=q.device)
        allowed = kp[None, :] <= qp[:, None]
        scores = torch.where(allowed[None, None], scores, torch.full_like(scores, MASK_FILL_VALUE))
    probs = torch.softmax(scores, dim=-1)
    return torch.matmul(probs, vf).permute(0, 2, 1, 3).to(q.dtype)


def _repeat_kv(x: torch.Tensor, repeats: int) -> torch.Tensor:
    """llama32_adapter.py:380-386: [B, T, Hkv, D] -> [B, T, Hkv * repeats, D]."""
    if repeats == 1:
        return x
    B, T, H, D = x.shape
    return x[:, :, :, None, :].expand(B, T, H, repeats, D).reshape(B, T, H * repeats, D)


def _linear_weight(out_features: int, in_features: int, generator, device) -> torch.nn.Parameter:
    """fp32 weights drawn U(-1/sqrt(in), 1/sqrt(in)), the initialisation of the reference's nn.Linear."""
    bound = 1.0 / math.sqrt(in_features)
    w = (torch.rand((out_features, in_features), generator=generator, dtype=torch.float32) * 2 - 1) * bound
    return torch.nn.Parameter(w.to(device), requires_grad=False)


def _project(x16: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """fp16 activations times fp32 weights in fp32, result fp16."""
    return (x16.float() @ weight.t()).to(torch.float16)


def _rms_norm(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    xf = x.float()
    y = xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + eps)
    if weight is not None:
        y = y * weight.float()
    return y.to(torch.float16)


def _unwatched(x: torch.Tensor) -> bool:
    """Whether a call on ``x`` may pass torch's operators by: nothing records
    gradients of it (reverse or forward mode), maps, traces or compiles it,
    intercepts its operators or casts them, and it is a plain tensor (or
    parameter).  A tensor that torch.func maps or differentiates has a plain
    type and no address: it is told by its wrapper, before anything reads it."""
    return (type(x) in _PLAIN_TYPES and not (x.requires_grad and torch.is_grad_enabled())
            and not torch.is_autocast_enabled() and not torch.compiler.is_compiling()
            and torch._C._get_tracing_state() is None and torch._C._len_torch_dispatch_stack() == 0
            and torch._C._len_torch_function_stack() == 0 and torch.autograd.forward_ad._current_level < 0
            and not _wrapped(x))


def _plain_weight(w: torch.Tensor, device: torch.device) -> bool:
    """A weight the projection kernel reads as it is: fp32, contiguous, aligned, on the device, and nothing
    watches it (``_unwatched``, whose checks of the call itself the caller has made for its input)."""
    return (type(w) in _PLAIN_TYPES and not _wrapped(w) and not (w.requires_grad and torch.is_grad_enabled())
            and w.dtype is torch.float32 and w.device == device and w.is_contiguous() and w.data_ptr() % 16 == 0)


class RFSNDecoderLayerMLX(torch.nn.Module):
    """Decoder layer that owns its projections, quantizer and cache-backed
    decode path (rfsn_v10_mlx_ane_complete.py:55-172).  With
    ``config.num_kv_heads`` below ``num_heads`` the K/V projections produce
    only the KV heads and the cache serves the query heads grouped."""

    def __init__(self, config: RFSNConfig, layer_idx: int = 0, ffn_multiplier: int = 2, device=None,
                 generator: Optional[torch.Generator] = None, quantizer=None):
        super().__init__()
        if device is None:
            if not torch.cuda.is_available():
                raise RuntimeError("the RFSN MI355X decoder layer needs a ROCm GPU; none is visible")
            device = torch.device("cuda", torch.cuda.current_device())
        self.device = torch.device(device)
        self.config = config
        self.layer_idx = layer_idx
        self.num_heads = config.num_heads
        self.num_kv_heads = config.kv_heads
        self.head_dim = config.head_dim
        self.model_dim = config.hidden_dim
        self.ffn_hidden_dim = max(config.hidden_dim * ffn_multiplier, config.hidden_dim)
        self.scale = config.head_dim ** -0.5
        self.eps = 1e-5
        g = generator if generator is not None else torch.Generator().manual_seed(1234 + layer_idx)
        D, H, Hkv = config.hidden_dim, config.num_heads, self.num_kv_heads
        self.attn_norm_weight = torch.nn.Parameter(torch.ones(D, device=self.device), requires_grad=False)
        self.ffn_norm_weight = torch.nn.Parameter(torch.ones(D, device=self.device), requires_grad=False)
        self.q_proj = _linear_weight(H * self.head_dim, D, g, self.device)
        self.k_proj = _linear_weight(Hkv * self.head_dim, D, g, self.device)
        self.v_proj = _linear_weight(Hkv * self.head_dim, D, g, self.device)
        self.o_proj = _linear_weight(D, H * self.head_dim, g, self.device)
        self.ffn_up = _linear_weight(self.ffn_hidden_dim, D, g, self.device)
        self.ffn_down = _linear_weight(D, self.ffn_hidden_dim, g, self.device)
        self.quantizer = quantizer if quantizer is not None else HybridQuantizerMLX(config, device=self.device)
        self.disk_cache_dir = Path(config.disk_cache_dir) / f"decoder_layer_{layer_idx}"
        self.cache = RFSNv10KVCacheMLX(config, layer_idx=layer_idx, device=self.device)

    @property
    def cache_tokens(self) -> int:
        return self.cache.total_tokens

    def reset_cache(self, remove_disk: bool = True) -> None:
        if remove_disk and self.disk_cache_dir.exists():
            shutil.rmtree(self.disk_cache_dir)
        self.cache = RFSNv10KVCacheMLX(self.config, layer_idx=self.layer_idx, device=self.device)

    def _heads(self, projected: torch.Tensor, heads: int) -> torch.Tensor:
        B, S, _ = projected.shape
        return projected.reshape(B, S, heads, self.head_dim).to(torch.float16)

    def _qkv(self, x16: torch.Tensor):
        a = _rms_norm(x16, self.attn_norm_weight, self.eps)
        return (self._heads(_project(a, self.q_proj), self.num_heads),
                self._heads(_project(a, self.k_proj), self.num_kv_heads),
                self._heads(_project(a, self.v_proj), self.num_kv_heads))

    def prefill_cache(self, x: torch.Tensor, reset: bool = True) -> None:
        """rfsn_v10_mlx_ane_complete.py:90-104: the prompt's K/V into the cache."""
        if x.dim() != 3 or int(x.shape[0]) != 1:
            raise ValueError("prefill_cache expects input shape [1, seq_len, hidden_dim]")
        if reset:
            self.reset_cache(remove_disk=True)
        _, keys, values = self._qkv(x.to(self.device, torch.float16))
        self.cache.update(keys[0], values[0], self.quantizer, disk_dir=self.disk_cache_dir)

    def forward(self, x: torch.Tensor, use_cache: bool = False,
                router: Optional[AsyncHierarchicalRouterMLX] = None,
                context_window: Optional[int] = None) -> torch.Tensor:
        """rfsn_v10_mlx_ane_complete.py:114-172."""
        if x.dim() != 3:
            raise ValueError("Decoder layer expects input shape [batch, seq_len, hidden_dim]")
        if int(x.shape[-1]) != self.model_dim:
            raise ValueError(f"Expected hidden_dim {self.model_dim}, got {int(x.shape[-1])}")
        residual = x.to(self.device, torch.float16)
        q, k, v = self._qkv(residual)
        if use_cache:
            if tuple(int(d) for d in x.shape[:2]) != (1, 1):
                raise ValueError("cache-backed decoding currently supports input shape [1, 1, hidden_dim]; "
                                 "use prefill_cache() for longer prompts")
            self.cache.update(k[0], v[0], self.quantizer, disk_dir=self.disk_cache_dir)
            pos = self.cache.total_tokens - 1
            window = context_window
            if window is None:
                window = max(self.config.block_size_seq, min(self.cache.total_tokens, self.config.warm_capacity))
            # the query is the newest token: attention_forward's default position
            # (a device tensor here would be read back to the host for the window)
            attended = self.cache.attention_forward(
                q[:, 0], causal=True, router=router, current_position=pos, context_window=window,
            ).reshape(1, 1, self.num_heads, self.head_dim)
        else:
            rep = self.num_heads // self.num_kv_heads
            attended = _dense_exact_attention(q, _repeat_kv(k, rep), _repeat_kv(v, rep), self.scale, causal=True)
        B, S = attended.shape[:2]
        attn_out = _project(attended.reshape(B, S, self.num_heads * self.head_dim), self.o_proj)
        hidden = residual + attn_out
        f = _rms_norm(hidden, self.ffn_norm_weight, self.eps)
        ffn_out = (_gelu(f.float() @ self.ffn_up.t()) @ self.ffn_down.t()).to(torch.float16)  # fp32 until the end
        return hidden + ffn_out


# Rotary frequency scaling of the Llama 3.1 / 3.2 checkpoints (their
# config.json "rope_scaling"; Llama-3.2-1B: factor 32, low / high frequency
# factors 1 / 4, original context 8192).
LLAMA3_ROPE_SCALING = {"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                       "original_max_position_embeddings": 8192}


def rope_inv_freq(head_dim: int, theta: float = 500000.0, rope_scaling: Optional[Dict] = None,
                  device=None) -> torch.Tensor:
    """Rotary inverse frequencies [head_dim / 2] (float64): theta^(-2i/D),
    then, for ``rope_scaling`` of type "llama3", Meta's published Llama 3.1
    frequency scaling: components whose wavelength 2*pi/f is shorter than
    original / high_freq_factor keep f, longer than original /
    low_freq_factor become f / factor, and those between interpolate
    linearly in original / wavelength between the two."""
    inv = theta ** (-torch.arange(0, head_dim, 2, dtype=torch.float64, device=device) / head_dim)
    if not rope_scaling:
        return inv
    kind = rope_scaling.get("rope_type", rope_scaling.get("type"))
    if kind != "llama3":
        raise ValueError(f"unsupported rope_scaling type {kind!r} (only 'llama3')")
    factor = float(rope_scaling["factor"])
    lo, hi = float(rope_scaling["low_freq_factor"]), float(rope_scaling["high_freq_factor"])
    orig = float(rope_scaling["original_max_position_embeddings"])
    ratio = orig * inv / (2 * math.pi)           # periods of each component within the original context
    smooth = ((ratio - lo) / (hi - lo)).clamp(0.0, 1.0)
    return inv / factor * (1.0 - smooth) + inv * smooth


def rope_cos_sin(positions: torch.Tensor, head_dim: int, theta: float = 500000.0,
                 rope_scaling: Optional[Dict] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Rotary tables [S, head_dim] (fp32): angle p * f_i (``rope_inv_freq``),
    the two halves repeated, as the rotary module the adapter calls returns
    them (llama32_adapter.py:528-553)."""
    inv = rope_inv_freq(head_dim, theta, rope_scaling, positions.device)
    ang = positions.to(torch.float64)[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)
    return ang.cos().float(), ang.sin().float()


def _rotate_half(x: torch.Tensor) -> torch.Tensor:
    """llama32_adapter.py:375-377."""
    half = x.shape[-1] // 2
    return torch.cat([-x[..., half:], x[..., :half]], dim=-1)


class Llama32DecoderLayerMLX(torch.nn.Module):
    """The Llama decoder layer of llama32_adapter.py on the MI355X cache.

    ``weights`` (optional) maps ``input_layernorm``, ``post_attention_layernorm``,
    ``q_proj``, ``k_proj``, ``v_proj``, ``o_proj``, ``gate_proj``, ``up_proj``,
    ``down_proj`` to tensors of the Hugging Face layer's shapes (a local state
    dict); otherwise weights are drawn as an untrained layer's would be.

    Rotary tables come, in this order, from the call's ``position_embeddings``
    (cos, sin), from ``rotary_module`` (the reference's argument: called as
    ``module(hidden, position_ids)``, else ``module(position_ids)``), or from
    ``rope_cos_sin`` with ``rope_theta`` and ``rope_scaling`` (default: the
    Llama-3.2 checkpoints' llama3 scaling).  Without ``position_ids`` a call's
    positions continue after the cached tokens (the reference's adapter
    defaults to 0 .. seq_len-1 and leaves positions to its caller)."""

    WEIGHTS = ("input_layernorm", "post_attention_layernorm", "q_proj", "k_proj", "v_proj", "o_proj",
               "gate_proj", "up_proj", "down_proj")

    def __init__(self, config: RFSNConfig, intermediate_size: int, layer_idx: int = 0, rms_norm_eps: float = 1e-5,
                 rope_theta: float = 500000.0, weights: Optional[Dict[str, torch.Tensor]] = None, device=None,
                 generator: Optional[torch.Generator] = None, quantizer=None,
                 rope_scaling: Optional[Dict] = LLAMA3_ROPE_SCALING, rotary_module=None):
        super().__init__()
        if device is None:
            if not torch.cuda.is_available():
                raise RuntimeError("the RFSN MI355X decoder layer needs a ROCm GPU; none is visible")
            device = torch.device("cuda", torch.cuda.current_device())
        self.device = torch.device(device)
        self.config = config
        self.layer_idx = layer_idx
        self.num_heads = config.num_heads
        self.num_kv_heads = config.kv_heads
        self.num_key_value_groups = self.num_heads // self.num_kv_heads
        self.head_dim = config.head_dim
        self.hidden_dim = config.hidden_dim
        self.scale = config.head_dim ** -0.5
        self.rms_norm_eps = rms_norm_eps
        self.rope_theta = rope_theta
        self.rope_scaling = dict(rope_scaling) if rope_scaling else None
        if self.device.type == "cuda":
            self._inv_freq()  # rejects unsupported scaling types now
        elif self.rope_scaling:
            rope_inv_freq(config.head_dim, rope_theta, self.rope_scaling)
        self.rotary_module = rotary_module
        shapes = self._set_shapes(intermediate_size)
        g = generator if generator is not None else torch.Generator().manual_seed(4321 + layer_idx)
        for name in self.WEIGHTS:
            if weights is not None:
                w = torch.as_tensor(weights[name]).float()
                if w.shape != shapes[name]:
                    raise ValueError(f"{name}: expected shape {tuple(shapes[name])}, got {tuple(w.shape)}")
                p = torch.nn.Parameter(w.to(self.device), requires_grad=False)
            elif len(shapes[name]) == 1:
                p = torch.nn.Parameter(torch.ones(shapes[name], device=self.device), requires_grad=False)
            else:
                p = _linear_weight(shapes[name][0], shapes[name][1], g, self.device)
            setattr(self, name, p)
        self.quantizer = quantizer if quantizer is not None else HybridQuantizerMLX(config, device=self.device)
        self.disk_cache_dir = Path(config.disk_cache_dir) / f"llama_layer_{layer_idx}"
        self.cache = RFSNv10KVCacheMLX(config, layer_idx=layer_idx, device=self.device)

    def _set_shapes(self, inter: int) -> Dict[str, torch.Size]:
        """The weights' shapes, and whether ``rfsn_layer_linear`` takes projections of them."""
        D, qd, kvd = self.hidden_dim, self.num_heads * self.head_dim, self.num_kv_heads * self.head_dim
        shapes = {"input_layernorm": (D,), "post_attention_layernorm": (D,), "q_proj": (qd, D), "k_proj": (kvd, D),
                  "v_proj": (kvd, D), "o_proj": (D, qd), "gate_proj": (inter, D), "up_proj": (inter, D),
                  "down_proj": (D, inter)}
        self._shapes = {n: torch.Size(s) for n, s in shapes.items()}
        self._linear_ok = (K.layer_linear_ok(D, (qd + 2 * kvd,), self.head_dim) and K.layer_linear_ok(D, (inter, inter))
                           and K.layer_linear_ok(qd, (D,)) and K.layer_linear_ok(inter, (D,)))
        return self._shapes

    @property
    def cache_tokens(self) -> int:
        return self.cache.total_tokens

    def reset_cache(self, remove_disk: bool = True) -> None:
        if remove_disk and self.disk_cache_dir.exists():
            shutil.rmtree(self.disk_cache_dir)
        self.cache = RFSNv10KVCacheMLX(self.config, layer_idx=self.layer_idx, device=self.device)

    def _positions(self, seq_len: int, position_embeddings, position_ids) -> Tuple[torch.Tensor, torch.Tensor]:
        if position_embeddings is not None:
            cos, sin = (torch.as_tensor(t, device=self.device).float().reshape(-1, self.head_dim)[-seq_len:]
                        for t in position_embeddings)
            return cos, sin
        if position_ids is None:
            start = self.cache.total_tokens
            position_ids = torch.arange(start, start + seq_len, device=self.device)
        pid = torch.as_tensor(position_ids, device=self.device).reshape(-1)
        if self.rotary_module is not None:
            # llama32_adapter.py:535-553: HF rotary modules take (hidden, position_ids)
            # on the device of their own buffers or parameters
            first = next(itertools.chain(self.rotary_module.buffers(), self.rotary_module.parameters()), None)
            rdev = self.device if first is None else first.device
            ids = pid.reshape(1, -1).to(rdev)
            hidden = torch.zeros((1, seq_len, self.hidden_dim), dtype=torch.float32, device=rdev)
            try:
                cos, sin = self.rotary_module(hidden, ids)
            except TypeError:
                cos, sin = self.rotary_module(ids)
            return tuple(torch.as_tensor(t, device=self.device).float().reshape(-1, self.head_dim)[-seq_len:]
                         for t in (cos, sin))
        return rope_cos_sin(pid, self.head_dim, self.rope_theta, self.rope_scaling)

    def _given_tables(self, seq_len: int, position_embeddings, position_ids) -> Optional[Tuple]:
        """The call's rotary tables where the caller or ``rotary_module`` determines them (``_positions``), or None
        where they follow from the layer's own settings and the cached tokens."""
        if position_embeddings is None and position_ids is None and self.rotary_module is None:
            return None
        return self._positions(seq_len, position_embeddings, position_ids)

    def _native(self, h16: torch.Tensor, tables: Optional[Tuple] = None) -> bool:
        """Whether ``rfsn_layer_linear`` runs this call's projections: a plain
        [1, S, hidden] fp16 input and rotary tables nothing watches, weights
        as it reads them."""
        if (not self._linear_ok or not _unwatched(h16) or h16.dim() != 3 or h16.shape[1] == 0
                or int(h16.shape[2]) != self.hidden_dim or not h16.is_cuda
                or h16.device.index != torch.cuda.current_device()
                or tables is not None and not all(_unwatched(t) and t.device == h16.device for t in tables)):
            return False
        device, weights = h16.device, self._parameters
        for name, shape in self._shapes.items():
            w = weights.get(name)
            if w is None or w.shape != shape or not _plain_weight(w, device):
                return False
        return True

    def _rows(self, h16: torch.Tensor) -> torch.Tensor:
        """[1, S, hidden] as the contiguous, aligned rows [S, hidden] the projection kernel reads."""
        x = h16.reshape(-1, self.hidden_dim).contiguous()
        return x.clone() if x.data_ptr() % 16 else x

    def _inv_freq(self) -> torch.Tensor:
        """``rope_inv_freq`` on the device, kept for the layer's present rotary settings.  Calls on any stream read
        it: it is copied from host memory, which is done when the copy returns, at construction for the first
        settings; before one of other settings is dropped the device is waited for.  Inside a graph capture, which
        allows neither, a missing one is made on the device for the call alone."""
        key = (self.head_dim, self.rope_theta, None if not self.rope_scaling else dict(self.rope_scaling))
        kept = self.__dict__.get("_inv_freq_kept")
        if kept is None or kept[0] != key:
            if torch.cuda.is_current_stream_capturing():
                return rope_inv_freq(*key, self.device).contiguous()
            with _INV_FREQ_LOCK:
                kept = self.__dict__.get("_inv_freq_kept")
                if kept is None or kept[0] != key:
                    made = (key, rope_inv_freq(*key, torch.device("cpu")).to(self.device))
                    if kept is not None:
                        torch.cuda.synchronize(self.device)
                    self._inv_freq_kept = kept = made
        return kept[1]

    def _session(self):
        """The decode session of a cached step over the whole hot + warm window
        (``DecodeSession``: most steps re-issue one prepared launch, which
        appends the token itself), or None where the general ``update`` +
        ``attention_forward`` has to run: a cold tier, or a step that may spill
        into one, another tier policy, a format the fused kernel does not
        serve, or a cache class of the caller's (whose methods a session would
        pass by).  A cache that was written, reconfigured or recalibrated since
        the session's last step has its launch built anew."""
        c = self.cache
        if (type(c) is not RFSNv10KVCacheMLX or not c._recency or not c._subspace or c.num_cold or c._kq is None or c.hot_capacity < 2 * c.HOT_BLOCK
                or c.num_warm + c.HOT_BLOCK > c.warm_capacity or not c._fused_ok(self.num_heads)):
            return None
        s = getattr(self, "_decode", None)
        if s is None or s.cache is not c or s.quantizer is not self.quantizer:
            q = torch.empty((1, self.num_heads, self.head_dim), dtype=torch.float16, device=c._hot_k.device)
            s = self._decode = c.decode_session(q, self.quantizer)
        elif s.left != s.state() or s.splits_stale():
            s.forget()
        return s

    def __getstate__(self):
        # the session's prepared launch and the kept frequencies belong to this layer's device: a copy makes its own
        return {n: v for n, v in self.__dict__.items() if n not in ("_decode", "_inv_freq_kept")}

    def __setstate__(self, state):
        super().__setstate__(state)
        if "_linear_ok" not in self.__dict__:  # a layer saved before it kept what its weights' shapes allow
            self._set_shapes(int(self.down_proj.shape[1]))

    def _session_step(self, session, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        session.left = None  # a step that raises leaves a launch to rebuild
        out = session.step(k, v)
        self.cache.last_access_stats = self.cache.whole_window_stats()
        session.left = session.state()
        return out

    def _qkv(self, h16: torch.Tensor, native: bool, tables: Optional[Tuple], q_out=None):
        """Rotated q and k, and v, [1, S, heads, head_dim] (llama32_adapter.py:570-580); ``tables`` as
        ``_given_tables`` returns them."""
        S = int(h16.shape[1])
        if not native:
            return self._project_qkv(h16, *(self._positions(S, None, None) if tables is None else tables))
        w = self._parameters
        if tables is None:
            rope = dict(inv_freq=self._inv_freq(), pos0=self.cache.total_tokens)
        else:
            cos, sin = tables
            shape = (S, self.head_dim)
            rope = dict(tables=(cos.expand(shape).contiguous(), sin.expand(shape).contiguous()))
        outs = K.layer_linear(self._rows(h16), [w["q_proj"], w["k_proj"], w["v_proj"]], head_dim=self.head_dim,
                              norm=(w["input_layernorm"], self.rms_norm_eps),
                              out0=None if q_out is None else q_out.view(1, -1), **rope)
        return tuple(o.view(1, S, -1, self.head_dim) for o in outs)

    def _project_qkv(self, h16: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor):
        """llama32_adapter.py:570-580 without the KV repeat (the cache groups heads)."""
        n = _rms_norm(h16, self.input_layernorm, self.rms_norm_eps)
        B, S, _ = h16.shape
        q = _project(n, self.q_proj).reshape(B, S, self.num_heads, self.head_dim)
        k = _project(n, self.k_proj).reshape(B, S, self.num_kv_heads, self.head_dim)
        v = _project(n, self.v_proj).reshape(B, S, self.num_kv_heads, self.head_dim)
        c, s = cos[None, :, None, :], sin[None, :, None, :]
        qf, kf = q.float(), k.float()
        q = (qf * c + _rotate_half(qf) * s).to(torch.float16)       # llama32_adapter.py:555-568
        k = (kf * c + _rotate_half(kf) * s).to(torch.float16)
        return q, k, v

    def _mlp(self, h16: torch.Tensor) -> torch.Tensor:
        """llama32_adapter.py:582-587."""
        m = _rms_norm(h16, self.post_attention_layernorm, self.rms_norm_eps)
        gate = _project(m, self.gate_proj).float()
        up = _project(m, self.up_proj)
        act = (gate * torch.sigmoid(gate)).to(torch.float16)
        return _project((act.float() * up.float()).to(torch.float16), self.down_proj)

    def prefill_cache(self, hidden_states: torch.Tensor, position_embeddings=None, position_ids=None,
                      reset: bool = True) -> None:
        """llama32_adapter.py:589-614."""
        if int(hidden_states.shape[0]) != 1:
            raise ValueError("prefill_cache currently supports batch size 1 only")
        if reset:
            self.reset_cache(remove_disk=True)
        S = int(hidden_states.shape[1])
        if S == 0:
            return
        h16 = hidden_states.to(self.device, torch.float16)
        tables = self._given_tables(S, position_embeddings, position_ids)
        _, k, v = self._qkv(h16, self._native(h16, tables), tables)
        self.cache.update(k[0], v[0], self.quantizer, disk_dir=self.disk_cache_dir)

    def forward(self, hidden_states: torch.Tensor, position_embeddings=None, position_ids=None,
                use_cache: bool = False, router: Optional[AsyncHierarchicalRouterMLX] = None,
                context_window: Optional[int] = None) -> torch.Tensor:
        """llama32_adapter.py:616-662."""
        if int(hidden_states.shape[0]) != 1:
            raise ValueError("The Llama adapter currently supports batch size 1 only")
        S = int(hidden_states.shape[1])
        residual = hidden_states.to(self.device, torch.float16)
        tables = self._given_tables(S, position_embeddings, position_ids)
        native = self._native(residual, tables)
        session = None
        if use_cache and native and S == 1 and router is None and context_window is None:
            session = self._session()
        q, k, v = self._qkv(residual, native, tables, None if session is None else session.q)
        if session is not None:
            attended = self._session_step(session, k[0], v[0])
        elif use_cache:
            if S != 1:
                raise ValueError("cache-backed decode expects input shape [1, 1, hidden_dim]")
            self.cache.update(k[0], v[0], self.quantizer, disk_dir=self.disk_cache_dir)
            pos = self.cache.total_tokens - 1
            attended = self.cache.attention_forward(
                q[:, 0], causal=True, router=router, current_position=pos, context_window=context_window,
            ).reshape(1, 1, self.num_heads, self.head_dim)
        elif native and K.dense_attention_ok(S, self.num_heads, self.num_kv_heads, self.head_dim, self.scale):
            own = torch.arange(S, dtype=torch.int32, device=self.device)[:, None].expand(S, self.num_heads)
            attended = K.blockwise_attention(q[0], k[0], v[0], self.scale, True, own, dense=True)
        else:
            g = self.num_key_value_groups
            attended = _dense_exact_attention(q, _repeat_kv(k, g), _repeat_kv(v, g), self.scale, causal=True)
        attended = attended.reshape(1, S, self.num_heads * self.head_dim)
        if native:
            w = self._parameters
            hidden, = K.layer_linear(attended.reshape(S, -1), [w["o_proj"]], K.LINEAR_RESIDUAL,
                                     residual=self._rows(residual))
            act, = K.layer_linear(hidden, [w["gate_proj"], w["up_proj"]], K.LINEAR_SWIGLU,
                                  norm=(w["post_attention_layernorm"], self.rms_norm_eps))
            out, = K.layer_linear(act, [w["down_proj"]], K.LINEAR_RESIDUAL, residual=hidden)
            return out.reshape(1, S, self.hidden_dim)
        attn = _project(attended, self.o_proj)
        hidden = residual + attn
        return hidden + self._mlp(hidden)
