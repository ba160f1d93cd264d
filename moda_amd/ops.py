"""Host side of the fused sequence+depth attention operators.

Mirrors the reference's Python operator interface -- same function names,
argument meaning, assertions and return conventions -- on top of the C ABI of
``libmoda_hip.so``:

  * ``parallel_moda`` / ``parallel_moda_fwd`` / ``parallel_moda_bwd``
    (libs/moda_triton/fla/ops/moda/moda_v14.py:2792-2893, 381-522, 1470-1842)
  * ``parallel_moda_chunk_visible`` / ``_fwd`` / ``_bwd``
    (moda_v16.py:3614-3651, 498-633, 2099-2343)
  * ``parallel_fda`` / ``_fwd`` / ``_bwd`` (fda_v12.py:1346-1449, 261-400, 881-1135)
  * ``parallel_attn`` (fla/ops/attn/parallel.py:678-730), the plain causal comparator.

Tensors stay torch tensors; torch is used for allocation, streams and autograd
only.  Every compute step is a HIP kernel of the shared library; the host work of
a call (contract checks, descriptor, allocation, launch, autograd node) is native
(``csrc/host.cpp``), this file is the interface.
"""
from __future__ import annotations

import ctypes
import warnings
from typing import NamedTuple, Optional, Tuple

import torch

from . import _lib
from ._lib import Desc, Strides

_tracing = torch._C._get_tracing_state  # true while torch.jit.trace records (torch.jit.is_tracing takes twice as long)

_DTYPES = {torch.bfloat16: _lib.BF16, torch.float16: _lib.FP16, torch.float32: _lib.FP32}

# How fp32 tensors are computed.  "fp32": fp32 products and sums throughout, on the fp32 matrix instruction (head dims up
# to 128, rows on the 16-byte grid; 2 x 4096 tokens, 16 query heads, head dim 128: 9.5 ms forward and backward, through
# fp16 1.1 ms) or on the vector ALU.  "fp16" / "bf16": the inputs are rounded to that type, the 16-bit matrix
# kernels run, the results are widened again.  "fp16" is what the reference's own fp32 path amounts to: its
# tl.dot calls (moda_v14.py:188, 209, 699-712) take the default input precision, which rounds fp32 operands to a
# 10-bit mantissa (TF32) and accumulates in fp32 -- fp16 has the same mantissa; its range (6e-8 .. 65504) is the
# caller's responsibility, "bf16" trades three mantissa bits for the fp32 range.
_FP32_COMPUTE = "fp32"


def set_fp32_compute(mode: str) -> str:
    """Choose how fp32 tensors are computed ("fp32", "fp16" or "bf16", see above); returns the previous setting."""
    global _FP32_COMPUTE
    assert mode in ("fp32", "fp16", "bf16"), f"unknown fp32 compute mode {mode!r}"
    _lib.host().set_fp32_compute({"fp32": _lib.FP32, "fp16": _lib.FP16, "bf16": _lib.BF16}[mode])
    previous, _FP32_COMPUTE = _FP32_COMPUTE, mode
    return previous


# Query rows per chunk of the chunk-visible variant when the caller does not
# say: the value the reference hard-wires in its launchers (moda_v16.py:581-585).
DEFAULT_CHUNK_ROWS = 64


class PackedBatch(NamedTuple):
    """A variable-length batch on one packed token axis, as the kernels take it."""
    cu: torch.Tensor  # int32 [n + 1] on the device: first base token of each sequence, then the total
    n: int            # sequences
    max_len: int      # base tokens of the longest sequence
    total: int        # base tokens in the packed axis
    host: object = None  # ctypes int32 array [n + 1]: the offsets again, in host memory (the library checks them and
                         # can launch per sequence where it has no packed kernel)


def _packed(cu_seqlens, q: torch.Tensor, rows_per_token: int) -> Optional[PackedBatch]:
    """``cu_seqlens`` as a caller passes it (fla's convention: cumulative sequence lengths, first entry 0,
    tensors of batch size 1 holding all sequences back to back) -> PackedBatch.  The offsets count BASE
    TOKENS, i.e. rows of k/v; sequence i owns query rows ``cu[i]*G .. cu[i+1]*G`` and depth rows
    ``cu[i]*L .. cu[i+1]*L``.  The reference carries the argument but asserts it away
    (moda_v14.py:2672-2673); its dormant kernel code reads the offsets in query rows (moda_v14.py:83-101),
    which is the same thing for ``moda_group_num == 1``.  Costs one device-to-host copy of the offsets
    (the longest sequence sizes the launch); pass the returned PackedBatch instead of the tensor to reuse it."""
    if cu_seqlens is None or isinstance(cu_seqlens, PackedBatch):
        return cu_seqlens
    p = _lib.host().pack(cu_seqlens, q, rows_per_token)
    return PackedBatch(p.cu, p.n, p.max_len, p.total, (ctypes.c_int32 * (p.n + 1))(*p.host))


def _native_packed(p: Optional[PackedBatch]):
    if p is None:
        return None
    return _lib.host().Packed(p.cu, p.n, p.max_len, p.total, list(p.host) if p.host is not None else [])


def _offsets(cu_seqlens):
    """``cu_seqlens`` of a public call -> the two arguments the native call takes it as: a tensor, or a PackedBatch."""
    if cu_seqlens is None:
        return None, None
    if isinstance(cu_seqlens, PackedBatch):
        return None, _native_packed(cu_seqlens)
    return cu_seqlens, None


def _ptr(x: Optional[torch.Tensor]):
    return ctypes.c_void_p(x.data_ptr()) if x is not None else ctypes.c_void_p(0)


def _stream(x: torch.Tensor):
    return ctypes.c_void_p(torch.cuda.current_stream(x.device).cuda_stream)


def _matrix_core_path(q: torch.Tensor, val: torch.Tensor, packed: Optional["PackedBatch"] = None) -> bool:
    """Whether the call runs on the matrix-core kernels, whose rows must be 16-byte aligned.  The rule is the
    library's own (``moda_hip_uses_matrix_cores``): it is asked with a descriptor that carries what the rule reads
    -- dtype, head dims, whether the batch is packed and has host offsets."""
    if q.dtype not in _DTYPES:
        raise TypeError(f"unsupported dtype {q.dtype}; expected bf16, fp16 or fp32")
    d = Desc()
    d.struct_size = ctypes.sizeof(Desc)
    d.dtype = _DTYPES[q.dtype]
    d.mode = _lib.NONCAUSAL
    d.B = d.T = d.H = d.G = 1
    d.D, d.Dv = q.shape[3], val.shape[3]
    d.scale = 1.0
    if packed is not None:
        d.B, d.T, d.total_tokens = packed.n, packed.max_len, packed.total
        d.cu_seqlens = packed.cu.data_ptr()
        if packed.host is not None:
            d.cu_seqlens_host = ctypes.cast(packed.host, ctypes.c_void_p)
    rc = _lib.load().moda_hip_uses_matrix_cores(ctypes.byref(d))
    if rc < 0:  # a head dim the library rejects: the launch itself will report it
        return False
    return rc == 1


def _strides(x: Optional[torch.Tensor]) -> Strides:
    if x is None:
        return Strides(0, 0, 0)
    return Strides(x.stride(0), x.stride(1), x.stride(2))


def _check_device(x: torch.Tensor):
    if not x.is_cuda:
        raise RuntimeError(
            "moda_amd operators run only on an MI355X (gfx950) device tensor; there is no CPU path"
        )


def _desc(mode, q, k, v, kd, vd, G, L, chunk_tokens, scale, o=None, do=None, dq=None, dk=None, dv=None, dkd=None,
          dvd=None, depth_valid=None, packed: Optional[PackedBatch] = None, accumulate_depth=False) -> Desc:
    d = Desc()
    d.struct_size = ctypes.sizeof(Desc)
    if q.dtype not in _DTYPES:
        raise TypeError(f"unsupported dtype {q.dtype}; expected bf16, fp16 or fp32")
    d.dtype = _DTYPES[q.dtype]
    d.mode = mode
    src = kd if mode == _lib.DEPTH_ONLY else k
    d.B = q.shape[0]
    d.H = src.shape[2]
    d.G = G
    d.D = q.shape[3]
    val = vd if mode == _lib.DEPTH_ONLY else v
    d.Dv = val.shape[3]
    d.L = L
    if depth_valid is not None and L > 0:
        assert 1 <= depth_valid <= L, f"depth_valid must be in [1, {L}], got {depth_valid}"
        d.L_valid = int(depth_valid)
    if mode == _lib.DEPTH_ONLY:
        d.T = q.shape[1] // G
    else:
        d.T = k.shape[1]
    if packed is not None:
        d.B, d.T = packed.n, packed.max_len
        d.cu_seqlens = packed.cu.data_ptr()
        d.total_tokens = packed.total
        if packed.host is not None:
            d.cu_seqlens_host = ctypes.cast(packed.host, ctypes.c_void_p)
    d.chunk_tokens = chunk_tokens
    d.flags = _lib.FLAG_ACCUMULATE_DEPTH_GRADS if accumulate_depth else 0
    d.scale = float(scale)
    d.q, d.k, d.v, d.kd, d.vd = _strides(q), _strides(k), _strides(v), _strides(kd), _strides(vd)
    d.o, d.d_o = _strides(o), _strides(do)
    d.dq, d.dk, d.dv, d.dkd, d.dvd = _strides(dq), _strides(dk), _strides(dv), _strides(dkd), _strides(dvd)
    return d


def _check_shapes(mode, q, k, v, kd, vd, G, o=None, do=None, lse=None):
    """Every extent the kernels derive from ``k`` (or ``q``), ``G`` and the depth row count, checked against what the
    tensors hold.  Returns ``(T, L)``."""
    return _lib.host().check_shapes(mode, q, k, v, kd, vd, G, o, do, lse)


def _raw_fwd(mode, q, k, v, kd, vd, scale, G, chunk_tokens=0, depth_valid=None, packed=None):
    """Launch the forward kernels. Returns (o, lse)."""
    return _lib.host().forward(mode, q, k, v, kd, vd, scale, G, chunk_tokens, depth_valid, _native_packed(packed))


def _raw_bwd(mode, q, k, v, kd, vd, o, lse, do, scale, G, chunk_tokens=0, stages=_lib.STAGE_ALL, out=None, ws=None,
             depth_valid=None, packed=None, accumulate_depth=False):
    """Launch the backward kernels. Returns (dq, dk, dv, dkd, dvd).

    ``stages`` selects a subset of {delta, dq, dk/dv}; ``out`` (a previous return
    value) and ``ws`` (a workspace tensor) let the caller reuse buffers across calls.
    ``accumulate_depth``: the depth gradients are ADDED to the ``dkd, dvd`` given in ``out`` (slots
    ``>= depth_valid`` untouched) instead of overwriting them."""
    return _lib.host().backward(mode, q, k, v, kd, vd, o, lse, do, scale, G, chunk_tokens, depth_valid,
                                _native_packed(packed), int(stages), out, ws, accumulate_depth)


def bwd_workspace(mode, q, k, v, kd, vd, G, chunk_tokens=0, packed=None) -> torch.Tensor:
    """A workspace tensor of the size the backward asks for, for callers that reuse one across calls (``ws=``)."""
    T, L = _check_shapes(mode, q, k, v, kd, vd, G)
    kd_a, vd_a = (kd, vd) if L > 0 else (None, None)
    d = _desc(mode, q, k, v, kd_a, vd_a, G, L, chunk_tokens, 1.0, packed=packed)
    nbytes = _lib.load().moda_hip_bwd_workspace_bytes(ctypes.byref(d))
    return torch.empty(max(int(nbytes), 4), dtype=torch.uint8, device=q.device)


# ---------------------------------------------------------------------------
# MoDA (causal / non-causal)  -- moda_v14.py
# ---------------------------------------------------------------------------
def _assert_group_tile(moda_group_num: int, rows: int = 128):
    assert (
        rows % moda_group_num == 0
    ), "To keep depth alignment consistent with backward, BT % moda_group_num must be 0"


def parallel_moda_fwd(q, k, v, g_cumsum, scale, cu_seqlens=None, cached_k=None, cached_v=None, moda_group_num=1,
                      is_causal=True, customized_BT=None, customized_BS=None, customized_BK=None, customized_BV=None,
                      customized_num_warps=None, depth_valid=None):
    """moda_v14.py:381-522.  Returns ``(o, lse)``; tile-size knobs are accepted and ignored.
    ``depth_valid`` (not in the reference): only the first ``depth_valid`` of the ``L`` slots per token
    of ``cached_k/v`` are visible."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    assert q.shape[2] == k.shape[2], (
        "Implicit head-dimension GQA is not allowed. "
        "Please fold grouping only into `moda_group_num`: "
        "use q.shape[2] == k.shape[2] and set T_q = T_kv * moda_group_num."
    )
    _assert_group_tile(moda_group_num)
    mode = _lib.CAUSAL if is_causal else _lib.NONCAUSAL
    return _raw_fwd(mode, q, k, v, cached_k, cached_v, scale, moda_group_num, depth_valid=depth_valid,
                    packed=_packed(cu_seqlens, q, moda_group_num))


def parallel_moda_bwd(q, k, v, o, g_cumsum, lse, do, scale=None, chunk_size=128, cu_seqlens=None, cached_k=None,
                      cached_v=None, moda_group_num=1, is_causal=True, customized_BT=None, customized_BS=None,
                      customized_BK=None, customized_BV=None, customized_num_warps=None, group_bs=None,
                      group_warps=None, depth_bs=None, depth_warps=None, depth_valid=None):
    """moda_v14.py:1470-1842.  Returns ``(dq, dk, dv, dg_cumsum=None, d_cached_k, d_cached_v)``."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    assert q.shape[2] == k.shape[2], (
        "Implicit head-dimension GQA is not allowed. "
        "Please fold grouping only into `moda_group_num`: "
        "use q.shape[2] == k.shape[2] and set T_q = T_kv * moda_group_num."
    )
    if scale is None:
        scale = q.shape[-1] ** -0.5
    _assert_group_tile(moda_group_num)
    mode = _lib.CAUSAL if is_causal else _lib.NONCAUSAL
    dq, dk, dv, dkd, dvd = _raw_bwd(mode, q, k, v, cached_k, cached_v, o, lse, do, scale, moda_group_num,
                                    depth_valid=depth_valid, packed=_packed(cu_seqlens, q, moda_group_num))
    return dq, dk, dv, None, dkd, dvd


def _refuse_decay(g, q):
    """``g`` (the reference's decay) is part of the signatures and unsupported, like there."""
    assert g.shape[:3] == q.shape[:3], "g must be [B,T_q,HQ]"
    assert g is None, "g is not supported in this version"


class _AttentionFunction(torch.autograd.Function):
    """What the four operators' autograd Functions share.  ``apply`` of one of them builds the native node of the same
    computation (csrc/host.cpp, Attend), which costs a tenth of the host time; a class derived from one of them runs
    its own ``forward`` and ``backward`` as any Function does.  So do all of them while ``torch.jit.trace`` records: a
    Function is recorded as one operation that runs again on replay, of the native node only its empty output
    tensors would be.  The gradient into ``lse`` is ignored."""

    @classmethod
    def apply(cls, *args, **kwargs):
        if cls in _NATIVE_FUNCTIONS and not _tracing():
            return cls._attend(*args, **kwargs)
        return super().apply(*args, **kwargs)

    @staticmethod
    def _run(ctx, mode, q, k, v, cached_k, cached_v, scale, moda_group_num, chunk_tokens, depth_valid, cu_seqlens):
        if cached_k is None or cached_v is None:
            cached_k = cached_v = None
        packed = _packed(cu_seqlens, q, 1 if mode == _lib.PLAIN_GQA else moda_group_num)
        scale = q.shape[-1] ** -0.5 if scale is None else scale
        o, lse = _raw_fwd(mode, q, k, v, cached_k, cached_v, scale, moda_group_num, chunk_tokens, depth_valid, packed)
        ctx.save_for_backward(q, k, v, cached_k, cached_v, o, lse)
        ctx.call = (mode, scale, moda_group_num, chunk_tokens, depth_valid, packed)
        ctx.set_materialize_grads(False)
        return o, lse

    @staticmethod
    def _gradients(ctx, do):
        if do is None:
            return (None,) * 5
        mode, scale, G, chunk_tokens, depth_valid, packed = ctx.call
        q, k, v, cached_k, cached_v, o, lse = ctx.saved_tensors
        return _raw_bwd(mode, q, k, v, cached_k, cached_v, o, lse, do.to(o.dtype), scale, G, chunk_tokens,
                        depth_valid=depth_valid, packed=packed)


class ParallelMixtureOfDepthAttentionFunction(_AttentionFunction):
    """moda_v14.py:2649-2789: differentiable in q, k, v, cached_k, cached_v."""

    @staticmethod
    def _attend(q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, is_causal=True,
                group_bs=None, group_warps=None, depth_bs=None, depth_warps=None, depth_valid=None):
        assert g is None, "g is not supported in this version"
        cu, packed = _offsets(cu_seqlens)
        return _lib.host().attend(_lib.CAUSAL if is_causal else _lib.NONCAUSAL, q, k, v, cached_k, cached_v, scale,
                                  moda_group_num, 0, depth_valid, cu, packed, False, 128)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda")
    def forward(ctx, q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, is_causal=True,
                group_bs=None, group_warps=None, depth_bs=None, depth_warps=None, depth_valid=None):
        assert g is None, "g is not supported in this version"
        _assert_group_tile(moda_group_num)
        o, lse = _AttentionFunction._run(ctx, _lib.CAUSAL if is_causal else _lib.NONCAUSAL, q, k, v, cached_k, cached_v,
                                         scale, moda_group_num, 0, depth_valid, cu_seqlens)
        ctx.mark_non_differentiable(lse)
        return o, lse

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, do, dlse):
        dq, dk, dv, dkd, dvd = _AttentionFunction._gradients(ctx, do)
        return dq, dk, dv, None, None, None, dkd, dvd, None, None, None, None, None, None, None


def _head_last(*xs):
    return tuple(x if x is None else x.transpose(1, 2) for x in xs)


def _warn_layout(api_name, q):
    warnings.warn(
        f"[{api_name}] detected seq_len({q.shape[1]}) < num_heads({q.shape[2]}). "
        "input may be in head_first format while head_first=True is not set.", stacklevel=3
    )


def _warn_depth_grads(cached_k, cached_v):
    if cached_k is not None and cached_v is not None and (cached_k.requires_grad or cached_v.requires_grad):
        warnings.warn(
            "cached_k/v requires gradients, but return_depth_grads=False. "
            "Gradients are still computed and returned.", stacklevel=3
        )


def parallel_moda(q, k, v, g=None, cached_k=None, cached_v=None, scale=None, cu_seqlens=None, moda_group_num=1,
                  is_causal=True, head_first=False, need_lse=False, return_depth_grads=True, warn_shape=True,
                  customized_BT=None, customized_BS=None, customized_BT_backward=None, customized_BS_backward=None,
                  group_bs=None, group_warps=None, depth_bs=None, depth_warps=None, depth_valid=None):
    """Fused sequence+depth attention; signature of moda_v14.py:2792-2815, plus ``depth_valid``.

    q ``[B, T*G, H, D]``; k, v ``[B, T, H, D]``; cached_k/v ``[B, T*L, H, D]`` or
    None.  Returns ``o`` (q.dtype) or ``(o, lse)`` with ``lse`` fp32 in base-2
    units.  The ``customized_*``, ``group_*`` and ``depth_*`` knobs tune the
    reference's Triton launches and have no meaning here; they are accepted and
    ignored.  ``depth_valid`` (an extension): ``cached_k/v`` keep ``L`` slots per token
    but only the first ``depth_valid`` are visible -- the result equals that for the
    compacted ``[B, T*depth_valid, H, D]`` tensors, the gradients of the other slots are
    zero, and a preallocated cache (``DepthCache``) need not be rebuilt per layer.  The other slots are
    never read: they may hold anything (an uninitialised ``torch.empty`` buffer included).
    """
    if head_first:
        q, k, v, g, cached_k, cached_v = _head_last(q, k, v, g, cached_k, cached_v)
    elif warn_shape and q.shape[1] < q.shape[2]:
        _warn_layout("parallel_moda", q)
    if not return_depth_grads:
        _warn_depth_grads(cached_k, cached_v)
    if g is not None:
        _refuse_decay(g, q)
    mode = _lib.CAUSAL if is_causal else _lib.NONCAUSAL
    if _tracing():
        _lib.host().check_folded_contract(mode, q, k, cached_k, cached_v, moda_group_num)
        out = ParallelMixtureOfDepthAttentionFunction.apply(q, k, v, None, scale, cu_seqlens, cached_k, cached_v, moda_group_num,
                                                            is_causal, None, None, None, None, depth_valid)
    else:
        cu, packed = _offsets(cu_seqlens)
        out = _lib.host().attend(mode, q, k, v, cached_k, cached_v, scale, moda_group_num, 0, depth_valid, cu, packed, True, 128)
    return out if need_lse else out[0]


# ---------------------------------------------------------------------------
# chunk-visible MoDA -- moda_v16.py
# ---------------------------------------------------------------------------
def _chunk_tokens(moda_group_num: int, chunk_rows: Optional[int]) -> int:
    """Base tokens per chunk.  The reference's launchers take ``customized_BT`` but overwrite it with 64 rows on
    every device (moda_v16.py:545-584), so a chunk is always 64 query rows there; ``chunk_rows`` (an argument
    the reference does not have) is the way to ask for another chunk size here."""
    rows = chunk_rows if chunk_rows is not None else DEFAULT_CHUNK_ROWS
    assert (
        rows % moda_group_num == 0
    ), "BT must be divisible by moda_group_num to keep chunk-visible base_t aligned"
    return rows // moda_group_num


def parallel_moda_chunk_visible_fwd(q, k, v, g_cumsum, scale, cu_seqlens=None, cached_k=None, cached_v=None,
                                    moda_group_num=1, customized_BT=None, customized_BS=None, customized_BK=None,
                                    customized_BV=None, customized_num_warps=None, chunk_rows=None, depth_valid=None):
    """moda_v16.py:498-633.  The tile-size knobs are accepted and ignored, ``customized_BT`` included (the
    reference overwrites it with 64, moda_v16.py:581-585); ``chunk_rows`` sets the chunk size in query rows,
    ``depth_valid`` is that of ``parallel_moda``."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    assert q.shape[2] == k.shape[2], "Implicit head-dimension GQA is not allowed."
    cb = _chunk_tokens(moda_group_num, chunk_rows)
    return _raw_fwd(_lib.CHUNK_VISIBLE, q, k, v, cached_k, cached_v, scale, moda_group_num, cb,
                    depth_valid=depth_valid, packed=_packed(cu_seqlens, q, moda_group_num))


def parallel_moda_chunk_visible_bwd(q, k, v, o, g_cumsum, lse, do, scale=None, chunk_size=128, cu_seqlens=None,
                                    cached_k=None, cached_v=None, moda_group_num=1, customized_BT=None,
                                    customized_BS=None, customized_BK=None, customized_BV=None,
                                    customized_num_warps=None, chunk_rows=None, depth_valid=None):
    """moda_v16.py:2099-2343 (``customized_BT`` ignored as there, ``chunk_rows``, ``depth_valid`` as in the forward)."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    if scale is None:
        scale = q.shape[-1] ** -0.5
    cb = _chunk_tokens(moda_group_num, chunk_rows)
    dq, dk, dv, dkd, dvd = _raw_bwd(_lib.CHUNK_VISIBLE, q, k, v, cached_k, cached_v, o, lse, do, scale,
                                    moda_group_num, cb, depth_valid=depth_valid,
                                    packed=_packed(cu_seqlens, q, moda_group_num))
    return dq, dk, dv, None, dkd, dvd


class ParallelMixtureOfDepthAttentionChunkVisibleFunction(_AttentionFunction):
    """moda_v16.py:3456-3493."""

    @staticmethod
    def _attend(q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, chunk_rows=None,
                depth_valid=None):
        assert g is None, "g is not supported in this version"
        cu, packed = _offsets(cu_seqlens)
        return _lib.host().attend(_lib.CHUNK_VISIBLE, q, k, v, cached_k, cached_v, scale, moda_group_num,
                                  _chunk_tokens(moda_group_num, chunk_rows), depth_valid, cu, packed, False, 0)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda")
    def forward(ctx, q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, chunk_rows=None,
                depth_valid=None):
        assert g is None, "g is not supported in this version"
        o, lse = _AttentionFunction._run(ctx, _lib.CHUNK_VISIBLE, q, k, v, cached_k, cached_v, scale, moda_group_num,
                                         _chunk_tokens(moda_group_num, chunk_rows), depth_valid, cu_seqlens)
        ctx.mark_non_differentiable(lse)
        return o, lse

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, do, dlse):
        dq, dk, dv, dkd, dvd = _AttentionFunction._gradients(ctx, do)
        return dq, dk, dv, None, None, None, dkd, dvd, None, None, None


def parallel_moda_chunk_visible(q, k, v, g=None, cached_k=None, cached_v=None, scale=None, cu_seqlens=None,
                                moda_group_num=1, head_first=False, need_lse=False, return_depth_grads=True,
                                warn_shape=True, customized_BT=None, customized_BS=None, customized_BT_backward=None,
                                customized_BS_backward=None, chunk_rows=None, depth_valid=None):
    """Chunk-visible MoDA; signature of moda_v16.py:3614-3632 plus ``chunk_rows`` and ``depth_valid`` (the latter
    as in ``parallel_moda``: only the first ``depth_valid`` slots of every token hold data).  A query of base
    token ``t`` additionally sees the depth slots of tokens ``floor(t/Cb)*Cb .. t`` with
    ``Cb = 64 // moda_group_num``.  The four ``customized_*`` arguments are accepted and dropped exactly as the
    reference's wrapper drops them (moda_v16.py:3646-3650: a chunk is 64 query rows whatever they say);
    ``chunk_rows``, which the reference does not have, selects another chunk size in query rows."""
    if head_first:
        q, k, v, g, cached_k, cached_v = _head_last(q, k, v, g, cached_k, cached_v)
    elif warn_shape and q.shape[1] < q.shape[2]:
        _warn_layout("parallel_moda_chunk_visible", q)
    if not return_depth_grads:
        _warn_depth_grads(cached_k, cached_v)
    if g is not None:
        _refuse_decay(g, q)
    if _tracing():
        _lib.host().check_folded_contract(_lib.CHUNK_VISIBLE, q, k, cached_k, cached_v, moda_group_num)
        out = ParallelMixtureOfDepthAttentionChunkVisibleFunction.apply(q, k, v, None, scale, cu_seqlens, cached_k, cached_v,
                                                                        moda_group_num, chunk_rows, depth_valid)
    else:
        cu, packed = _offsets(cu_seqlens)
        out = _lib.host().attend(_lib.CHUNK_VISIBLE, q, k, v, cached_k, cached_v, scale, moda_group_num,
                                 _chunk_tokens(moda_group_num, chunk_rows), depth_valid, cu, packed, True, 0)
    return out if need_lse else out[0]


# ---------------------------------------------------------------------------
# FDA (depth-only) -- fda_v12.py
# ---------------------------------------------------------------------------
def parallel_fda_fwd(q, g_cumsum, scale, cu_seqlens=None, cached_k=None, cached_v=None, moda_group_num=1,
                     customized_BT=None, customized_BS=None, customized_BK=None, customized_BV=None,
                     customized_num_warps=None):
    """fda_v12.py:261-400.  Returns ``(o, lse)``."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    assert cached_k is not None and cached_v is not None, "Flash Depth Attention requires cached_k/cached_v"
    _assert_group_tile(moda_group_num)
    return _raw_fwd(_lib.DEPTH_ONLY, q, None, None, cached_k, cached_v, scale, moda_group_num,
                    packed=_packed(cu_seqlens, q, moda_group_num))


def parallel_fda_bwd(q, o, g_cumsum, lse, do, scale=None, chunk_size=128, cu_seqlens=None, cached_k=None,
                     cached_v=None, moda_group_num=1, customized_BT=None, customized_BS=None, customized_BK=None,
                     customized_BV=None, customized_num_warps=None, group_bs=None, group_warps=None, depth_bs=None,
                     depth_warps=None):
    """fda_v12.py:881-1135.  Returns ``(dq, dg_cumsum=None, d_cached_k, d_cached_v)``."""
    assert g_cumsum is None, "g_cumsum is not supported in this version"
    if scale is None:
        scale = q.shape[-1] ** -0.5
    dq, _, _, dkd, dvd = _raw_bwd(_lib.DEPTH_ONLY, q, None, None, cached_k, cached_v, o, lse, do, scale,
                                  moda_group_num, packed=_packed(cu_seqlens, q, moda_group_num))
    return dq, None, dkd, dvd


class ParallelFlashDepthAttentionFunction(_AttentionFunction):
    """fda_v12.py:1207-1338 (the k, v slots must be None)."""

    @staticmethod
    def _check(k, v, g, cached_k, cached_v):
        assert g is None, "g is not supported in this version"
        assert k is None and v is None, "Flash Depth Attention does not accept legacy k/v; pass None"
        assert cached_k is not None and cached_v is not None, "Flash Depth Attention requires cached_k/cached_v"

    @staticmethod
    def _attend(q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, group_bs=None,
                group_warps=None, depth_bs=None, depth_warps=None):
        ParallelFlashDepthAttentionFunction._check(k, v, g, cached_k, cached_v)
        cu, packed = _offsets(cu_seqlens)
        return _lib.host().attend(_lib.DEPTH_ONLY, q, None, None, cached_k, cached_v, scale, moda_group_num, 0, None,
                                  cu, packed, False, 128)

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda")
    def forward(ctx, q, k, v, g, scale, cu_seqlens, cached_k=None, cached_v=None, moda_group_num=1, group_bs=None,
                group_warps=None, depth_bs=None, depth_warps=None):
        ParallelFlashDepthAttentionFunction._check(k, v, g, cached_k, cached_v)
        _assert_group_tile(moda_group_num)
        o, lse = _AttentionFunction._run(ctx, _lib.DEPTH_ONLY, q, None, None, cached_k, cached_v, scale, moda_group_num,
                                         0, None, cu_seqlens)
        ctx.mark_non_differentiable(lse)
        return o, lse

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, do, dlse):
        dq, _, _, dkd, dvd = _AttentionFunction._gradients(ctx, do)
        return dq, None, None, None, None, None, dkd, dvd, None, None, None, None, None


def parallel_fda(q, k=None, v=None, g=None, cached_k=None, cached_v=None, scale=None, cu_seqlens=None,
                 moda_group_num=1, head_first=False, need_lse=False, return_depth_grads=True, warn_shape=True,
                 customized_BT=None, customized_BS=None, customized_BT_backward=None, customized_BS_backward=None,
                 group_bs=None, group_warps=None, depth_bs=None, depth_warps=None):
    """Depth-only attention; signature of fda_v12.py:1346-1368."""
    assert k is None and v is None, "Flash Depth Attention does not accept legacy k/v; pass None"
    if head_first:
        q, g, cached_k, cached_v = _head_last(q, g, cached_k, cached_v)
    elif warn_shape and q.shape[1] < q.shape[2]:
        _warn_layout("parallel_fda", q)
    if not return_depth_grads:
        _warn_depth_grads(cached_k, cached_v)
    if g is not None:
        _refuse_decay(g, q)
    if _tracing():
        _lib.host().check_folded_contract(_lib.DEPTH_ONLY, q, None, cached_k, cached_v, moda_group_num)
        out = ParallelFlashDepthAttentionFunction.apply(q, None, None, None, scale, cu_seqlens, cached_k, cached_v, moda_group_num)
    else:
        cu, packed = _offsets(cu_seqlens)
        out = _lib.host().attend(_lib.DEPTH_ONLY, q, None, None, cached_k, cached_v, scale, moda_group_num, 0, None, cu,
                                 packed, True, 128)
    return out if need_lse else out[0]


# ---------------------------------------------------------------------------
# head-dim GQA <-> the folded layout of the depth modes
# ---------------------------------------------------------------------------
def fold_gqa_heads(x: torch.Tensor, num_kv_heads: int, head_order: str = "group_major") -> torch.Tensor:
    """``[B, T, Hq, D]`` (one query head per head-dim slot) -> the folded ``[B, T*G, Hkv, D]`` that
    ``parallel_moda`` / ``parallel_moda_chunk_visible`` / ``parallel_fda`` take with ``moda_group_num = G``,
    ``G = Hq // Hkv``: the G query heads that share a kv head become G consecutive rows of the token.

    Which query heads share a kv head is a convention of the model, so it is an explicit argument:
    ``"group_major"`` -- query head ``g*Hkv + hkv`` reads kv head ``hkv`` (the fold of the reference's vision
    model, vision_tasks/deit/models.py:248-250); a free view of a contiguous ``x``.
    ``"kv_major"`` -- query head ``hkv*G + g`` reads kv head ``hkv`` (``repeat_interleave`` models and the plain
    comparator, fla/ops/attn/parallel.py:48-49); needs one copy."""
    B, T, Hq, D = x.shape
    assert Hq % num_kv_heads == 0, "query heads must be a multiple of kv heads"
    G = Hq // num_kv_heads
    if head_order == "group_major":
        return x.reshape(B, T, G, num_kv_heads, D).reshape(B, T * G, num_kv_heads, D)
    assert head_order == "kv_major", "head_order must be 'group_major' or 'kv_major'"
    return x.reshape(B, T, num_kv_heads, G, D).transpose(2, 3).reshape(B, T * G, num_kv_heads, D)


def unfold_gqa_heads(x: torch.Tensor, moda_group_num: int, head_order: str = "group_major") -> torch.Tensor:
    """Inverse of :func:`fold_gqa_heads`: ``[B, T*G, Hkv, D]`` -> ``[B, T, G*Hkv, D]``."""
    B, TG, Hkv, D = x.shape
    G = moda_group_num
    assert TG % G == 0, "rows must be a multiple of moda_group_num"
    if head_order == "group_major":
        return x.reshape(B, TG // G, G * Hkv, D)
    assert head_order == "kv_major", "head_order must be 'group_major' or 'kv_major'"
    return x.reshape(B, TG // G, G, Hkv, D).transpose(2, 3).reshape(B, TG // G, Hkv * G, D)


# ---------------------------------------------------------------------------
# plain causal attention with head-dim GQA -- fla/ops/attn/parallel.py
# ---------------------------------------------------------------------------
def parallel_attn_fwd(q, k, v, g_cumsum=None, scale=None, cu_seqlens=None):
    """fla/ops/attn/parallel.py:443-503.  q ``[B,T,HQ,D]``, k/v ``[B,T,H,D]``; returns ``(o, lse)``."""
    assert g_cumsum is None
    assert q.shape[2] % k.shape[2] == 0, "HQ must be a multiple of H"
    assert q.shape[1] == k.shape[1]
    if scale is None:
        scale = k.shape[-1] ** -0.5
    return _raw_fwd(_lib.PLAIN_GQA, q, k, v, None, None, scale, q.shape[2] // k.shape[2],
                    packed=_packed(cu_seqlens, q, 1))


def parallel_attn_bwd(q, k, v, o, g_cumsum, lse, do, scale=None, chunk_size=128, cu_seqlens=None):
    """fla/ops/attn/parallel.py:522-629.  Returns ``(dq, dk, dv, dg=None)``."""
    assert g_cumsum is None
    if scale is None:
        scale = k.shape[-1] ** -0.5
    dq, dk, dv, _, _ = _raw_bwd(_lib.PLAIN_GQA, q, k, v, None, None, o, lse, do, scale, q.shape[2] // k.shape[2],
                                packed=_packed(cu_seqlens, q, 1))
    return dq, dk, dv, None


class ParallelAttentionFunction(_AttentionFunction):
    """fla/ops/attn/parallel.py:632-675."""

    @staticmethod
    def _check(q, k, g):
        assert g is None, "g is not supported"
        assert q.shape[2] % k.shape[2] == 0, "HQ must be a multiple of H"
        assert q.shape[1] == k.shape[1]

    @staticmethod
    def _attend(q, k, v, g, scale, cu_seqlens):
        ParallelAttentionFunction._check(q, k, g)
        cu, packed = _offsets(cu_seqlens)
        return _lib.host().attend(_lib.PLAIN_GQA, q, k, v, None, None, scale, q.shape[2] // k.shape[2], 0, None, cu,
                                  packed, False, 0)[0]

    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda")
    def forward(ctx, q, k, v, g, scale, cu_seqlens):
        ParallelAttentionFunction._check(q, k, g)
        return _AttentionFunction._run(ctx, _lib.PLAIN_GQA, q, k, v, None, None, scale, q.shape[2] // k.shape[2], 0, None,
                                       cu_seqlens)[0]

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, do):
        return *_AttentionFunction._gradients(ctx, do)[:3], None, None, None


_NATIVE_FUNCTIONS = frozenset((ParallelMixtureOfDepthAttentionFunction, ParallelMixtureOfDepthAttentionChunkVisibleFunction,
                               ParallelFlashDepthAttentionFunction, ParallelAttentionFunction))


def parallel_attn(q, k, v, g=None, scale=None, cu_seqlens=None, head_first=False):
    """Plain causal attention with head-dim GQA; signature of fla/ops/attn/parallel.py:678-686."""
    if head_first:
        raise DeprecationWarning(
            "head_first is deprecated and will be removed in a future version. "
            "Please use head_first=False for now instead."
        )
    if q.shape[1] < q.shape[2]:
        warnings.warn(
            f"Input tensor shape suggests potential format mismatch: seq_len ({q.shape[1]}) < num_heads ({q.shape[2]}). "
        )
    return ParallelAttentionFunction.apply(q, k, v, g, scale, cu_seqlens)
