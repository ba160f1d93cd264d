"""Caller-side pieces around the attention operator: the attention module of the reference's vision
model and a manager for the depth stream it feeds.

``MoDAAttention`` has the constructor, parameter names (``q``, ``kv``, ``proj``) and return value of the
reference's module (vision_tasks/deit/models.py:215-267), so its ``state_dict`` loads unchanged; it
hands the strided ``k``/``v`` views of the fused projection to the kernels as they are (the reference's
operator copies them first) and can take a partially filled depth cache (``depth_valid``).

``DepthStream`` replaces the model-side loop of vision_tasks/deit/models.py:383-387, which re-stacks the
K/V of all previous layers for every layer (and lets autograd scatter the gradient of every such stack
back): one token-major cache is preallocated per forward pass and each layer's K/V is written into its
slot once.
  * With gradients flowing, a second buffer of the same shape collects the depth gradients: the backward
    of the attention that saw ``n`` slots adds its share to slots ``< n`` (the kernels' accumulate mode),
    and the gradient of a layer's K/V is its own attention's plus the slice of that buffer for its slot,
    joined when autograd reaches the layer.  Neither direction touches a slot more than once per consumer.
    The autograd nodes and the bookkeeping are native (csrc/host.cpp: TrainStream).
  * Without gradients only the cache is kept.
  * ``inplace=False`` keeps the reference's behaviour (rebuild per layer, differentiable ``stack_depth``).
"""
from __future__ import annotations

from typing import List, Optional, Tuple

import torch
from torch import nn

from . import _lib
from .depth_cache import DepthCache, stack_depth
from .ops import _chunk_tokens, _tracing, parallel_moda, parallel_moda_chunk_visible


class DepthStream:
    """Depth K/V of the layers seen so far, in the layout the kernels read.

    Per layer: ``o = stream.attend(q, k, v, scale=..., moda_group_num=..., is_causal=...)`` (attention over
    the sequence and over everything pushed so far), then ``stream.push(k, v)`` with the layer's
    ``[B, T, H, D]`` tensors (any number of pushes per layer, e.g. K/V projected from the FFN output as
    well).  ``max_layers`` sizes the cache.  ``inplace=None`` keeps one cache in place (with gradient
    accumulators when gradients flow), ``inplace=False`` rebuilds the cache per layer as the reference does; so does a
    stream whose first push ``torch.jit.trace`` records (what writes a cache in place leaves nothing to replay).

    ``context()`` -> ``(cached_k, cached_v, depth_valid)`` is the lower-level access for callers that
    invoke ``parallel_moda`` themselves; with gradients flowing it uses the rebuilding path (the in-place
    gradient path needs ``attend``).  Each backward pass over the stream's graph fills the accumulators anew."""

    def __init__(self, max_layers: int, inplace: Optional[bool] = None):
        self.max_layers = int(max_layers)
        self._layers: List[Tuple[torch.Tensor, torch.Tensor]] = []
        self._cache: Optional[DepthCache] = None
        self._train = None  # native TrainStream, from the first call with gradients flowing
        self._n = 0
        self._inplace: Optional[bool] = inplace
        self._mode: Optional[str] = None  # 'train' | 'infer' | 'rebuild', fixed by the first push
        self._used_context = False

    def __len__(self):
        return self._n

    def _decide(self, k, v):
        if self._mode is not None:
            return
        grads = torch.is_grad_enabled() and (k.requires_grad or v.requires_grad)
        if self._inplace is False or (grads and self._used_context) or _tracing():
            self._mode = "rebuild"
        else:
            self._mode = "train" if grads else "infer"

    def push(self, k: torch.Tensor, v: torch.Tensor):
        assert self._n < self.max_layers, "depth stream is full"
        self._decide(k, v)
        if self._mode == "train":
            self._native().push(k, v)
        elif self._mode == "infer":
            if self._cache is None:
                B, T, H, D = k.shape
                self._cache = DepthCache(B, T, self.max_layers, H, D, k.dtype, k.device)
            self._cache.append(k.detach(), v.detach())
        else:
            self._layers.append((k, v))
        self._n += 1

    def _native(self):
        if _tracing():
            raise RuntimeError("a depth stream that began in place cannot be traced: create it inside the traced function")
        if self._train is None:
            self._train = _lib.host().TrainStream(self.max_layers)
        return self._train

    def context(self):
        self._used_context = True
        if self._n == 0:
            return None, None, None
        if self._mode == "infer":
            return self._cache.filled()
        assert self._mode == "rebuild", \
            "with gradients flowing through an in-place depth stream use attend(): the depth gradients are " \
            "collected by the stream, not by autograd"
        return stack_depth([kv[0] for kv in self._layers]), stack_depth([kv[1] for kv in self._layers]), None

    def attend(self, q, k, v, scale=None, moda_group_num=1, is_causal=True, chunk_rows=None):
        """``parallel_moda(q, k, v, cached_k, cached_v, ...)`` over what has been pushed so far; with ``chunk_rows``
        (query rows per chunk, the reference's 64) ``parallel_moda_chunk_visible`` instead: a token also sees the
        depth slots of the earlier tokens of its chunk (causal by definition)."""
        chunk_visible = chunk_rows is not None
        assert not chunk_visible or is_causal, "chunk-visible attention is causal"
        if self._mode == "train" or (self._mode is None and self._inplace is not False and not self._used_context
                                     and not _tracing() and torch.is_grad_enabled()
                                     and (q.requires_grad or k.requires_grad)):
            # the same argument contract as parallel_moda, which is bypassed here
            assert q.shape[2] == k.shape[2] and q.shape[1] == k.shape[1] * moda_group_num, \
                "q must be [B, T*moda_group_num, H, D] for k [B, T, H, D]"
            assert 128 % moda_group_num == 0, \
                "To keep depth alignment consistent with backward, BT % moda_group_num must be 0"
            if scale is None:
                scale = q.shape[-1] ** -0.5
            mode = _lib.CHUNK_VISIBLE if chunk_visible else _lib.CAUSAL if is_causal else _lib.NONCAUSAL
            cb = _chunk_tokens(moda_group_num, chunk_rows) if chunk_visible else 0
            return self._native().attend(q, k, v, scale, moda_group_num, mode, cb)
        if self._n == 0:
            dk = dv = n = None
        elif self._mode == "infer":
            dk, dv, n = self._cache.filled()
        else:
            dk, dv = stack_depth([kv[0] for kv in self._layers]), stack_depth([kv[1] for kv in self._layers])
            n = None
        if chunk_visible:
            return parallel_moda_chunk_visible(q=q, k=k, v=v, g=None, scale=scale, cu_seqlens=None, cached_k=dk,
                                               cached_v=dv, moda_group_num=moda_group_num, head_first=False,
                                               warn_shape=False, chunk_rows=chunk_rows, depth_valid=n)
        return parallel_moda(q=q, k=k, v=v, g=None, scale=scale, cu_seqlens=None, cached_k=dk, cached_v=dv,
                             moda_group_num=moda_group_num, is_causal=is_causal, head_first=False, warn_shape=False,
                             depth_valid=n)


class MoDAAttention(nn.Module):
    """Attention over the sequence and over the depth stream; GQA groups are folded into the query
    rows (``q [B, N*G, num_kv_heads, head_dim]``, ``moda_group_num = G``) exactly as in
    vision_tasks/deit/models.py:244-267.  ``is_causal`` defaults to the vision model's ``False``.

    ``forward(x, depth_k, depth_v)`` is the reference's call; ``forward(x, stream=DepthStream)`` attends
    over the stream instead.  Either way the layer's own ``k, v`` are returned for the caller to push.

    ``ffn_kv=True`` adds a second projection ``kv_ffn`` and the method ``project_depth_kv`` that maps
    another hidden state (e.g. the block's FFN output) to depth K/V, for callers that also feed the
    depth stream from their feed-forward layers."""

    def __init__(self, dim, num_heads=8, num_kv_heads=1, qkv_bias=False, attn_drop=0., proj_drop=0.,
                 is_causal=False, ffn_kv=False, chunk_rows=None):
        super().__init__()
        self.chunk_rows = chunk_rows  # not None: chunk-visible attention with chunks of that many query rows
        if dim % num_heads != 0:
            raise ValueError(f"dim ({dim}) must be divisible by num_heads ({num_heads})")
        if num_heads % num_kv_heads != 0:
            raise ValueError(f"num_heads ({num_heads}) must be divisible by num_kv_heads ({num_kv_heads})")
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.moda_group_num = num_heads // num_kv_heads
        self.head_dim = dim // num_heads
        self.scale = self.head_dim ** -0.5
        self.is_causal = is_causal
        self.q = nn.Linear(dim, dim, bias=qkv_bias)
        self.kv = nn.Linear(dim, 2 * num_kv_heads * self.head_dim, bias=qkv_bias)
        self.proj = nn.Linear(dim, dim)
        self.proj_drop = nn.Dropout(proj_drop)
        self.kv_ffn = nn.Linear(dim, 2 * num_kv_heads * self.head_dim, bias=qkv_bias) if ffn_kv else None

    def _split_kv(self, kv: torch.Tensor):
        B, N, _ = kv.shape
        kv = kv.reshape(B, N, 2, self.num_kv_heads, self.head_dim)
        return kv[:, :, 0], kv[:, :, 1]

    def project_depth_kv(self, h: torch.Tensor):
        """Depth K/V ``[B, N, num_kv_heads, head_dim]`` of a hidden state other than the attention input."""
        assert self.kv_ffn is not None, "constructed without ffn_kv=True"
        return self._split_kv(self.kv_ffn(h))

    def forward(self, x, depth_k=None, depth_v=None, depth_valid=None, stream: Optional[DepthStream] = None):
        B, N, C = x.shape
        G = self.moda_group_num
        q = self.q(x).reshape(B, N * G, self.num_kv_heads, self.head_dim)
        k, v = self._split_kv(self.kv(x))
        if stream is not None:
            assert depth_k is None and depth_v is None, "pass either a stream or explicit depth tensors"
            o = stream.attend(q, k, v, scale=self.scale, moda_group_num=G, is_causal=self.is_causal,
                              chunk_rows=self.chunk_rows)
        elif self.chunk_rows is not None:
            o = parallel_moda_chunk_visible(q=q, k=k, v=v, g=None, scale=self.scale, cu_seqlens=None, cached_k=depth_k,
                                            cached_v=depth_v, moda_group_num=G, head_first=False, warn_shape=False,
                                            chunk_rows=self.chunk_rows, depth_valid=depth_valid)
        else:
            o = parallel_moda(q=q, k=k, v=v, g=None, scale=self.scale, cu_seqlens=None, cached_k=depth_k,
                              cached_v=depth_v, moda_group_num=G, is_causal=self.is_causal, head_first=False,
                              warn_shape=False, depth_valid=depth_valid)
        x = self.proj_drop(self.proj(o.reshape(B, N, C)))
        return x, k, v


_MISSING = object()


class MoDAStack(nn.Module):
    """``depth`` blocks (attention + MLP) chained through one ``DepthStream``: the body of
    ``MoDAVisionTransformer.forward_features`` (vision_tasks/deit/models.py:376-390) without the patch
    embedding and the classifier, for timing and testing whole-model steps.  Pre-norm blocks as in the
    reference (``x + f(norm(x))``, deit/models.py:288-292) or, with ``post_norm=True``, ``norm(x + f(x))``;
    ``ffn_kv=True`` also pushes K/V projected from every block's output into the stream (two slots per
    block)."""

    def __init__(self, dim, depth, num_heads, num_kv_heads, mlp_ratio=4., qkv_bias=True, is_causal=False,
                 post_norm=False, ffn_kv=False, chunk_rows=None):
        super().__init__()
        self.post_norm, self.ffn_kv = post_norm, ffn_kv
        self.blocks = nn.ModuleList()
        for _ in range(depth):
            blk = nn.Module()
            blk.norm1 = nn.LayerNorm(dim, eps=1e-6)
            blk.attn = MoDAAttention(dim, num_heads, num_kv_heads, qkv_bias=qkv_bias, is_causal=is_causal,
                                     ffn_kv=ffn_kv, chunk_rows=chunk_rows)
            blk.norm2 = nn.LayerNorm(dim, eps=1e-6)
            hidden = int(dim * mlp_ratio)
            blk.mlp = nn.Sequential(nn.Linear(dim, hidden), nn.GELU(), nn.Linear(hidden, dim))
            self.blocks.append(blk)

    def _plain_parameters(self):
        """Parameters and norm epsilons of every block for the native forward pass, or None when a block is not what
        the constructor made: a replaced, subclassed, patched or hooked module, blocks that differ, active dropout."""
        params, eps, first = [], [], None
        for blk in self.blocks:
            attn, mlp, norm1, norm2 = (blk._modules.get(n) for n in ("attn", "mlp", "norm1", "norm2"))  # none: wrapped
            if type(attn) is not MoDAAttention or type(mlp) is not nn.Sequential or len(mlp) != 3:
                return None
            q, kv, proj, drop, kv_ffn = (attn._modules.get(n) for n in ("q", "kv", "proj", "proj_drop", "kv_ffn"))
            fc1, act, fc2 = mlp._modules.values()
            linears = (q, kv, proj, fc1, fc2) if kv_ffn is None else (q, kv, proj, fc1, fc2, kv_ffn)
            if not (all(type(m) is nn.Linear for m in linears) and type(norm1) is nn.LayerNorm and type(norm2) is nn.LayerNorm
                    and type(act) is nn.GELU and act.approximate == "none" and type(drop) is nn.Dropout):
                return None
            if (drop.training and drop.p > 0) or (self.ffn_kv and kv_ffn is None):
                return None
            for m in (attn, mlp, norm1, norm2, act, drop, *linears):
                if m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__:
                    return None
            what = (attn.num_heads, attn.num_kv_heads, attn.is_causal, attn.chunk_rows, attn.scale)
            if first is None:
                first = what
            if what != first or attn.scale != attn.head_dim ** -0.5:
                return None
            # a replica, and a module whose parameters are slices of one flat tensor, hold them as plain attributes
            tensors = [m._parameters.get(n, _MISSING) for m in (norm1, q, kv, proj, norm2, fc1, fc2) for n in ("weight", "bias")]
            tensors += [None if kv_ffn is None or not self.ffn_kv else kv_ffn._parameters.get(n, _MISSING) for n in ("weight", "bias")]
            if not all(t is None or type(t) is nn.Parameter for t in tensors):
                return None
            params.append(tensors)
            eps.append((norm1.eps, norm2.eps))
        return (params, eps) if params else None

    def _forward_native(self, x):
        """The whole stack as kernel launches from native code (csrc/host.cpp: stack_forward), for calls through which
        no gradient flows, backward or forward (an open level of forward-mode differentiation: no_grad does not close
        it), and while nothing watches the framework's operations (a dispatch mode); None where the modules have to
        run one by one.  Twelve blocks of width 256 on 64 x 197 tokens issue some 200 framework operations of about
        10 us host time each when run as modules."""
        attn = self.blocks[0].attn if len(self.blocks) else None
        if (torch.is_grad_enabled() or torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling() or _tracing()
                or torch.autograd.forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() or type(attn) is not MoDAAttention
                or nn.modules.module._global_forward_hooks or nn.modules.module._global_forward_pre_hooks
                or type(x) is not torch.Tensor or x.dim() != 3 or x.shape[-1] != attn.num_heads * attn.head_dim):
            return None
        if 128 % attn.moda_group_num or (attn.chunk_rows is not None and not attn.is_causal):
            return None  # attend() refuses these
        plain = self._plain_parameters()
        if plain is None:
            return None
        cb = 0 if attn.chunk_rows is None else _chunk_tokens(attn.moda_group_num, attn.chunk_rows)
        return _lib.host().stack_forward(x, plain[0], plain[1], attn.num_heads, attn.num_kv_heads, bool(attn.is_causal), cb, self.post_norm)

    def forward(self, x, inplace_cache: Optional[bool] = None):
        if inplace_cache is not False:
            y = self._forward_native(x)
            if y is not None:
                return y
        stream = DepthStream(len(self.blocks) * (2 if self.ffn_kv else 1), inplace=inplace_cache)
        for blk in self.blocks:
            if self.post_norm:
                a, k, v = blk.attn(x, stream=stream)
                x = blk.norm1(x + a)
                x = blk.norm2(x + blk.mlp(x))
            else:
                a, k, v = blk.attn(blk.norm1(x), stream=stream)
                x = x + a
                x = x + blk.mlp(blk.norm2(x))
            stream.push(k, v)
            if self.ffn_kv:
                stream.push(*blk.attn.project_depth_kv(x))
        return x
