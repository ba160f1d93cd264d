"""CPU-side checks of the drop-in boundary: the C-ABI library loads and exports
every symbol the header declares, the ctypes mirror of the descriptor matches,
and the host functions keep the reference's argument contract
(moda_v14.py:2834-2871, fda_v12.py:1370-1437).  No kernel is launched here."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_functions():
    text = open(os.path.join(ROOT, "include", "moda_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(moda_hip_[a-z_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from moda_amd import _lib

    lib = _lib.load()
    names = _header_functions()
    assert set(names) == set(_lib.EXPORTS)
    for n in names:
        assert getattr(lib, n) is not None


def test_descriptor_layout_and_version():
    from moda_amd import _lib

    lib = _lib.load()
    assert lib.moda_hip_version() == 105
    assert ctypes.sizeof(_lib.Desc) == 16 + 7 * 8 + 8 + 12 * 24 + 24 + 8
    assert _lib.Desc.cu_seqlens.offset == 80 + 12 * 24
    assert _lib.Desc.q.offset == 80
    # a descriptor with the wrong struct_size is rejected without touching any device
    d = _lib.Desc()
    d.struct_size = 12
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(d)) == 0
    assert lib.moda_hip_fwd(ctypes.byref(d), None, None, None, None, None, None, None, None) == -1
    assert b"invalid" in lib.moda_hip_strerror(-1)


def test_descriptor_validation_codes():
    from moda_amd import _lib

    lib = _lib.load()

    def desc(**kw):
        d = _lib.Desc()
        d.struct_size = ctypes.sizeof(_lib.Desc)
        d.dtype, d.mode = _lib.BF16, _lib.CAUSAL
        d.B, d.T, d.H, d.G, d.D, d.L = 1, 8, 1, 1, 64, 0
        d.scale = 1.0
        for k, v in kw.items():
            setattr(d, k, v)
        return d

    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(desc())) == 8 * 4
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(desc(G=4, H=2, B=3))) == 3 * 2 * 32 * 4
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(desc(mode=_lib.PLAIN_GQA, G=4, H=2))) == 8 * 8 * 4
    # packed variable-length batch: the workspace covers the packed row axis once, not B x longest sequence
    assert lib.moda_hip_bwd_workspace_bytes(
        ctypes.byref(desc(B=3, T=8, G=2, H=2, cu_seqlens=0x1000, total_tokens=13))) == 2 * 13 * 2 * 4
    # ... the longest sequence cannot exceed the packed axis; the offsets must be 4-byte aligned
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(desc(B=3, T=8, cu_seqlens=0x1000, total_tokens=7))) == 0
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(desc(B=3, T=8, cu_seqlens=0x1002, total_tokens=9))) == 0
    null = None
    # missing q pointer
    assert lib.moda_hip_fwd(ctypes.byref(desc()), null, null, null, null, null, null, null, null) == -1
    # unsupported head dim
    assert lib.moda_hip_fwd(ctypes.byref(desc(D=512)), null, null, null, null, null, null, null, null) == -2
    # depth-only without depth slots, plain GQA with depth slots, chunk-visible without chunk size
    assert lib.moda_hip_fwd(ctypes.byref(desc(mode=_lib.DEPTH_ONLY)), null, null, null, null, null, null, null, null) == -1
    assert lib.moda_hip_fwd(ctypes.byref(desc(mode=_lib.PLAIN_GQA, L=2)), null, null, null, null, null, null, null, null) == -1
    assert lib.moda_hip_fwd(ctypes.byref(desc(mode=_lib.CHUNK_VISIBLE, L=2)), null, null, null, null, null, null, null, null) == -1
    # value head dim: negative is invalid, beyond 256 or not a multiple of 4 unsupported
    assert lib.moda_hip_fwd(ctypes.byref(desc(Dv=-4)), null, null, null, null, null, null, null, null) == -1
    assert lib.moda_hip_fwd(ctypes.byref(desc(Dv=512)), null, null, null, null, null, null, null, null) == -2
    assert lib.moda_hip_fwd(ctypes.byref(desc(Dv=30)), null, null, null, null, null, null, null, null) == -2
    # empty problem is a successful no-op
    assert lib.moda_hip_fwd(ctypes.byref(desc(T=0)), null, null, null, null, null, null, null, null) == 0
    # misaligned pointer (never dereferenced: alignment is checked first)
    bogus = ctypes.c_void_p(0x1008)
    ok = ctypes.c_void_p(0x1000)
    assert lib.moda_hip_fwd(ctypes.byref(desc()), bogus, ok, ok, null, null, ok, ok, null) == -3
    # reorg argument checks
    arr = (ctypes.c_void_p * 1)(0x1000)
    assert lib.moda_hip_depth_reorg_fwd(arr, 1, 3, 3, 1, 4, 1, 64, _lib.BF16, ok, null) == -1  # slot out of range
    assert lib.moda_hip_depth_reorg_fwd(arr, 0, 0, 3, 1, 4, 1, 64, _lib.BF16, ok, null) == 0   # nothing to do


def test_matrix_core_routing_rule_is_the_librarys():
    """The host wrapper asks the library which kernels a call runs on (rows must be 16-byte aligned for the
    matrix kernels): every combination of dtype, head dims and packing, against the rule stated in the header."""
    from moda_amd import _lib, ops

    lib = _lib.load()
    host = (ctypes.c_int32 * 3)(0, 5, 13)
    for dtype, tdt in ((_lib.BF16, torch.bfloat16), (_lib.FP16, torch.float16), (_lib.FP32, torch.float32)):
        for D in (8, 36, 64, 100, 128, 136, 192, 256):
            for Dv in (D, 64 if D != 64 else 32):
                for packed in (None, "device_only", "with_host"):
                    d = _lib.Desc()
                    d.struct_size = ctypes.sizeof(_lib.Desc)
                    d.dtype, d.mode = dtype, _lib.CAUSAL
                    d.B, d.T, d.H, d.G, d.D, d.Dv, d.L = 1, 8, 1, 1, D, Dv, 0
                    d.scale = 1.0
                    pb = None
                    if packed:
                        d.B, d.T, d.total_tokens, d.cu_seqlens = 2, 8, 13, 0x1000
                        cu = torch.tensor([0, 5, 13], dtype=torch.int32)
                        pb = ops.PackedBatch(cu, 2, 8, 13, host if packed == "with_host" else None)
                        if packed == "with_host":
                            d.cu_seqlens_host = ctypes.cast(host, ctypes.c_void_p)
                    want = (dtype != _lib.FP32 and D % 8 == 0 and Dv % 8 == 0
                            and not (max(D, Dv) > 128 and packed == "device_only"))
                    assert lib.moda_hip_uses_matrix_cores(ctypes.byref(d)) == int(want), (dtype, D, Dv, packed)
                    q, v = torch.zeros(1, 8, 1, D, dtype=tdt), torch.zeros(1, 8, 1, Dv, dtype=tdt)
                    assert ops._matrix_core_path(q, v, pb) == want, (dtype, D, Dv, packed)
    bad = _lib.Desc()
    bad.struct_size = 4
    assert lib.moda_hip_uses_matrix_cores(ctypes.byref(bad)) == -1


def test_host_offsets_are_validated():
    from moda_amd import _lib

    lib = _lib.load()

    def desc(offsets, T, total, with_device=True):
        d = _lib.Desc()
        d.struct_size = ctypes.sizeof(_lib.Desc)
        d.dtype, d.mode = _lib.BF16, _lib.CAUSAL
        d.B, d.T, d.H, d.G, d.D, d.L = len(offsets) - 1, T, 1, 1, 64, 0
        d.scale = 1.0
        d.total_tokens = total
        if with_device:
            d.cu_seqlens = 0x1000
        arr = (ctypes.c_int32 * len(offsets))(*offsets)
        d.cu_seqlens_host = ctypes.cast(arr, ctypes.c_void_p)
        return d, arr

    d, keep = desc([0, 5, 13], 8, 13)
    assert lib.moda_hip_bwd_workspace_bytes(ctypes.byref(d)) == 13 * 4
    for offsets, T, total in (([1, 5, 13], 8, 13),   # does not start at 0
                              ([0, 9, 5, 13], 9, 13),  # decreases
                              ([0, 5, 12], 8, 13),    # does not end at total_tokens
                              ([0, 4, 13], 8, 13)):   # a sequence longer than T
        d, keep = desc(offsets, T, total)
        assert lib.moda_hip_uses_matrix_cores(ctypes.byref(d)) == -1, offsets
    d, keep = desc([0, 5, 13], 8, 13, with_device=False)  # host offsets without the device array
    assert lib.moda_hip_uses_matrix_cores(ctypes.byref(d)) == -1


def test_workspace_alignment_codes():
    from moda_amd import _lib

    lib = _lib.load()
    d = _lib.Desc()
    d.struct_size = ctypes.sizeof(_lib.Desc)
    d.dtype, d.mode = _lib.BF16, _lib.CAUSAL
    d.B, d.T, d.H, d.G, d.D, d.L = 1, 8, 1, 1, 64, 0
    d.scale = 1.0
    for f in ("q", "k", "v", "o", "d_o", "dq", "dk", "dv"):
        getattr(d, f).b, getattr(d, f).t, getattr(d, f).h = 512, 64, 64
    ok = ctypes.c_void_p(0x1000)
    args = [ok] * 3 + [None, None] + [ok] * 6 + [None, None]
    # a workspace pointer that is not 4-byte aligned is refused before anything is launched or dereferenced
    assert lib.moda_hip_bwd(ctypes.byref(d), *args, ctypes.c_void_p(0x1002), 64, None) == -3
    assert lib.moda_hip_bwd(ctypes.byref(d), *args, None, 64, None) == -4
    assert lib.moda_hip_bwd(ctypes.byref(d), *args, ok, 8, None) == -4


def test_import_shim_names_and_reference_loops():
    import os
    import sys

    root = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moda_amd", "compat")
    sys.path.insert(0, root)
    try:
        for m in [m for m in sys.modules if m == "fla" or m.startswith("fla.")]:
            del sys.modules[m]
        import fla.ops.moda as shim
        import moda_amd

        assert shim.parallel_moda is moda_amd.parallel_moda
        assert shim.parallel_moda_chunk_visible_bwd is moda_amd.parallel_moda_chunk_visible_bwd
        # the reference package also exports its torch loops; here that is an ImportError that says where to look
        with pytest.raises(ImportError, match="oracle/moda_oracle.py"):
            from fla.ops.moda import naive_mixture_of_depth_causal_ref  # noqa: F401
        with pytest.raises(ImportError, match="reference's torch loops"):
            shim.naive_mixture_of_depth_causal_chunk_visible_ref
        with pytest.raises(AttributeError):
            shim.no_such_name
    finally:
        sys.path.remove(root)
        for m in [m for m in sys.modules if m == "fla" or m.startswith("fla.")]:
            del sys.modules[m]


def test_missing_library_fails_loudly(monkeypatch):
    from moda_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libmoda_hip.so")
    with pytest.raises(_lib.MissingLibraryError):
        _lib.load()


def test_cpu_tensors_are_rejected():
    import moda_amd

    q = torch.zeros(1, 8, 1, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        moda_amd.parallel_moda(q, q, q)


def test_argument_contract_matches_reference():
    import moda_amd

    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    # implicit head-dim GQA is refused (moda_v14.py:2839-2843)
    with pytest.raises(AssertionError, match="Implicit head-dimension GQA"):
        moda_amd.parallel_moda(z(1, 8, 4, 64), z(1, 8, 2, 64), z(1, 8, 2, 64))
    # T_q must be T_kv * G (moda_v14.py:2847-2852)
    with pytest.raises(AssertionError, match="T_q must equal T_kv"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), moda_group_num=2)
    with pytest.raises(AssertionError, match="moda_group_num=1"):
        moda_amd.parallel_moda(z(1, 16, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64))
    # depth cache shape checks (moda_v14.py:2856-2862)
    with pytest.raises(AssertionError, match="T_kv \\* L"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), cached_k=z(1, 12, 2, 64),
                               cached_v=z(1, 12, 2, 64))
    with pytest.raises(AssertionError, match="head count"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), cached_k=z(1, 16, 1, 64),
                               cached_v=z(1, 16, 1, 64))
    # g is unsupported (moda_v14.py:2672); cu_seqlens, which the reference asserts away in the next line,
    # is accepted here and validated on the host
    with pytest.raises(AssertionError, match="g is not supported"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), g=torch.zeros(1, 8, 2))
    with pytest.raises(AssertionError, match="batch size must be 1"):
        moda_amd.parallel_moda(z(2, 8, 2, 64), z(2, 8, 2, 64), z(2, 8, 2, 64), cu_seqlens=torch.tensor([0, 8]))
    with pytest.raises(AssertionError, match="start at 0 and not decrease"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), cu_seqlens=torch.tensor([0, 5, 3, 8]))
    with pytest.raises(AssertionError, match="ends at 7 base tokens"):
        moda_amd.parallel_moda(z(1, 16, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), moda_group_num=2,
                               cu_seqlens=torch.tensor([0, 3, 7]))
    with pytest.raises(RuntimeError, match="no CPU path"):
        moda_amd.parallel_moda(z(1, 8, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), cu_seqlens=torch.tensor([0, 3, 8]))
    # group size must divide the query tile (moda_v14.py:476-478)
    with pytest.raises(AssertionError, match="BT % moda_group_num"):
        moda_amd.parallel_moda(z(1, 24, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64), moda_group_num=3)
    # FDA (fda_v12.py:1370-1372, 1391-1393)
    with pytest.raises(AssertionError, match="does not accept legacy k/v"):
        moda_amd.parallel_fda(z(1, 8, 2, 64), k=z(1, 8, 2, 64), v=z(1, 8, 2, 64), cached_k=z(1, 16, 2, 64),
                              cached_v=z(1, 16, 2, 64))
    with pytest.raises(AssertionError, match="requires cached_k/cached_v"):
        moda_amd.parallel_fda(z(1, 8, 2, 64))
    # seq_len < num_heads warning (moda_v14.py:2828-2832)
    with pytest.warns(UserWarning, match="head_first"):
        with pytest.raises(RuntimeError):
            moda_amd.parallel_moda(z(1, 2, 4, 64), z(1, 2, 4, 64), z(1, 2, 4, 64))


def test_low_level_entry_points_check_every_extent_before_launching():
    """The C ABI takes bare pointers and derives all extents from k, G and the depth row count; a tensor that
    does not match would be read or written out of bounds on the device.  The host refuses such calls before
    anything is launched (these run on CPU tensors: the shape check comes before the device check)."""
    import moda_amd
    from moda_amd import _lib, ops

    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    q, k, v = z(1, 16, 2, 64), z(1, 8, 2, 64), z(1, 8, 2, 64)
    kd, vd = z(1, 24, 2, 64), z(1, 24, 2, 64)
    lse, o, do = torch.zeros(1, 16, 2), z(1, 16, 2, 64), z(1, 16, 2, 64)
    # a wrong moda_group_num: q rows != T * G
    with pytest.raises(AssertionError, match="expected T\\*moda_group_num"):
        moda_amd.parallel_moda_fwd(q, k, v, None, 0.125, cached_k=kd, cached_v=vd, moda_group_num=1)
    with pytest.raises(AssertionError, match="expected T\\*moda_group_num"):
        moda_amd.parallel_moda_bwd(q, k, v, o, None, lse, do, 0.125, cached_k=kd, cached_v=vd, moda_group_num=4)
    with pytest.raises(AssertionError, match="expected T\\*moda_group_num"):
        moda_amd.parallel_moda_chunk_visible_fwd(q, k, v, None, 0.125, cached_k=kd, cached_v=vd, moda_group_num=1)
    # depth rows that are not T * L, depth v shorter than depth k
    with pytest.raises(AssertionError, match="depth rows must be T \\* L"):
        moda_amd.parallel_moda_fwd(q, k, v, None, 0.125, cached_k=z(1, 20, 2, 64), cached_v=z(1, 20, 2, 64),
                                   moda_group_num=2)
    with pytest.raises(AssertionError, match="same number of rows"):
        moda_amd.parallel_moda_fwd(q, k, v, None, 0.125, cached_k=kd, cached_v=z(1, 16, 2, 64), moda_group_num=2)
    with pytest.raises(AssertionError, match="k and v must agree"):
        moda_amd.parallel_moda_fwd(q, k, z(1, 4, 2, 64), None, 0.125, moda_group_num=2)
    # backward: o / do / lse of the wrong size
    with pytest.raises(AssertionError, match="do must be"):
        moda_amd.parallel_moda_bwd(q, k, v, o, None, lse, z(1, 8, 2, 64), 0.125, moda_group_num=2)
    with pytest.raises(AssertionError, match="lse must be"):
        moda_amd.parallel_moda_bwd(q, k, v, o, None, torch.zeros(1, 8, 2), do, 0.125, moda_group_num=2)
    # depth-only: rows not a multiple of G, depth rows not T * L
    with pytest.raises(AssertionError, match="multiple of moda_group_num"):
        moda_amd.parallel_fda_fwd(z(1, 15, 2, 64), None, 0.125, cached_k=kd, cached_v=vd, moda_group_num=2)
    with pytest.raises(AssertionError, match="depth rows must be T \\* L"):
        moda_amd.parallel_fda_fwd(q, None, 0.125, cached_k=z(1, 20, 2, 64), cached_v=z(1, 20, 2, 64), moda_group_num=2)
    # a consistent call gets as far as the device check
    with pytest.raises(RuntimeError, match="no CPU path"):
        moda_amd.parallel_moda_fwd(q, k, v, None, 0.125, cached_k=kd, cached_v=vd, moda_group_num=2)
    assert ops._check_shapes(_lib.CAUSAL, q, k, v, kd, vd, 2, o=o, do=do, lse=lse) == (8, 3)


def test_depth_cache_append_checks_the_layer_against_the_cache():
    import moda_amd

    cache = moda_amd.DepthCache(2, 8, 3, 2, 64, torch.bfloat16, "cpu")
    z = lambda *s, dt=torch.bfloat16: torch.zeros(*s, dtype=dt)
    with pytest.raises(AssertionError, match="like the cache"):
        cache.append(z(2, 9, 2, 64), z(2, 9, 2, 64))       # more tokens than the cache has
    with pytest.raises(AssertionError, match="like the cache"):
        cache.append(z(2, 8, 2, 128), z(2, 8, 2, 128))     # wider head dim
    with pytest.raises(AssertionError, match="like the cache"):
        cache.append(z(2, 8, 2, 64), z(2, 8, 4, 64))       # v with more heads
    with pytest.raises(AssertionError, match="dtype"):
        cache.append(z(2, 8, 2, 64, dt=torch.float16), z(2, 8, 2, 64, dt=torch.float16))
    assert cache.n == 0
    with pytest.raises(RuntimeError, match="no CPU path"):  # a matching layer reaches the device check
        cache.append(z(2, 8, 2, 64), z(2, 8, 2, 64))
    with pytest.raises(AssertionError, match="cache must be a contiguous"):
        moda_amd.depth_cache._reorg_fwd([z(2, 8, 2, 64)], z(2, 16, 2, 64), 0, 3)


def test_gqa_head_folds_match_the_two_head_conventions():
    """fold_gqa_heads turns head-dim GQA queries into the folded layout of the depth modes.  Pinned on the oracle:
    kv_major folding + the folded operator == the plain comparator (query head hq reads kv head hq // G, the
    repeat_interleave convention); group_major folding == the reference caller's reshape; both invert exactly."""
    import moda_amd
    import oracle

    gen = torch.Generator().manual_seed(3)
    B, T, Hkv, G, D = 2, 9, 2, 3, 8
    q = torch.randn(B, T, Hkv * G, D, generator=gen, dtype=torch.float64)
    k = torch.randn(B, T, Hkv, D, generator=gen, dtype=torch.float64)
    v = torch.randn(B, T, Hkv, D, generator=gen, dtype=torch.float64)
    ref, _ = oracle.plain_gqa_dense(q, k, v, dtype=torch.float64)
    qf = moda_amd.fold_gqa_heads(q, Hkv, "kv_major")
    o, _ = oracle.moda_dense(qf, k, v, None, None, None, G, "causal", dtype=torch.float64)
    assert torch.allclose(moda_amd.unfold_gqa_heads(o, G, "kv_major"), ref, atol=1e-12)
    # group-major: query head g*Hkv + hkv reads kv head hkv, i.e. the caller's q.reshape(B, N, G, Hkv, D)
    qg = moda_amd.fold_gqa_heads(q, Hkv, "group_major")
    assert torch.equal(qg, q.reshape(B, T, G, Hkv, D).reshape(B, T * G, Hkv, D))
    assert qg.data_ptr() == q.data_ptr()  # a view, no copy
    o, _ = oracle.moda_dense(qg, k, v, None, None, None, G, "causal", dtype=torch.float64)
    kk = torch.cat([k] * G, dim=2)  # kv head of query head g*Hkv + hkv is hkv
    vv = torch.cat([v] * G, dim=2)
    ref_g, _ = oracle.plain_gqa_dense(q, kk, vv, dtype=torch.float64)  # one kv head per query head
    assert torch.allclose(moda_amd.unfold_gqa_heads(o, G, "group_major"), ref_g, atol=1e-12)
    for order in ("group_major", "kv_major"):
        assert torch.equal(moda_amd.unfold_gqa_heads(moda_amd.fold_gqa_heads(q, Hkv, order), G, order), q)


def test_compat_package_reexports():
    import sys

    sys.path.insert(0, os.path.join(ROOT, "moda_amd", "compat"))
    try:
        from fla.ops.moda import parallel_moda, parallel_moda_chunk_visible  # noqa: F401
        import moda_amd

        assert parallel_moda is moda_amd.parallel_moda
    finally:
        sys.path.pop(0)
        for m in [m for m in sys.modules if m == "fla" or m.startswith("fla.")]:
            del sys.modules[m]


def test_attention_module_mirrors_reference_parameters():
    """Parameter names and shapes of vision_tasks/deit/models.py:224-243 (a reference state_dict loads
    unchanged); an empty depth stream yields no cache."""
    import moda_amd

    m = moda_amd.MoDAAttention(384, num_heads=6, num_kv_heads=3, qkv_bias=True)
    shapes = {n: tuple(p.shape) for n, p in m.state_dict().items()}
    assert shapes == {"q.weight": (384, 384), "q.bias": (384,), "kv.weight": (384, 384), "kv.bias": (384,),
                      "proj.weight": (384, 384), "proj.bias": (384,)}
    assert m.moda_group_num == 2 and m.head_dim == 64 and m.scale == 64 ** -0.5
    with pytest.raises(ValueError, match="divisible by num_kv_heads"):
        moda_amd.MoDAAttention(384, num_heads=6, num_kv_heads=4)
    s = moda_amd.DepthStream(4)
    assert s.context() == (None, None, None) and len(s) == 0
    with pytest.raises(RuntimeError, match="no CPU path"):
        m(torch.zeros(1, 8, 384))


def test_fp32_compute_setting():
    import moda_amd

    assert moda_amd.set_fp32_compute("fp16") == "fp32"
    assert moda_amd.set_fp32_compute("fp32") == "fp16"
    with pytest.raises(AssertionError):
        moda_amd.set_fp32_compute("tf32")
    assert moda_amd.set_fp32_compute("fp32") == "fp32"


def _function_calls():
    """The operators' autograd Functions with arguments of a small call each, and which of them are tensors."""
    import moda_amd

    g = torch.Generator().manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)
    q, k, v, kd, vd = r(1, 8, 2, 4), r(1, 4, 2, 4), r(1, 4, 2, 4), r(1, 12, 2, 4), r(1, 12, 2, 4)
    return [(moda_amd.ParallelMixtureOfDepthAttentionFunction, [q, k, v, None, 0.5, None, kd, vd, 2]),
            (moda_amd.ParallelMixtureOfDepthAttentionChunkVisibleFunction, [q, k, v, None, 0.5, None, kd, vd, 2]),
            (moda_amd.ParallelFlashDepthAttentionFunction, [q, None, None, None, 0.5, None, kd, vd, 2]),
            (moda_amd.ParallelAttentionFunction, [r(1, 4, 4, 4), k, v, None, 0.5, None])]


def _stub_kernels(monkeypatch):
    """Stand-ins for the launches: an output that depends on every input, a gradient that names the input it is of."""
    from moda_amd import ops

    def fwd(mode, q, k, v, kd, vd, scale, G, chunk_tokens=0, depth_valid=None, packed=None):
        o = q * scale + sum(x.sum() for x in (k, v, kd, vd) if x is not None)
        return o, o.sum(-1)

    def bwd(mode, q, k, v, kd, vd, o, lse, do, scale, G, chunk_tokens=0, **kw):
        return tuple(None if x is None else torch.full_like(x, 10.0 * (i + 1)) for i, x in enumerate((q, k, v, kd, vd)))

    monkeypatch.setattr(ops, "_raw_fwd", fwd)
    monkeypatch.setattr(ops, "_raw_bwd", bwd)


def test_operator_functions_are_autograd_functions(monkeypatch):
    """The Functions the reference's modules export are torch.autograd.Functions with a forward and a backward of their
    own, which a class derived from one of them runs; every gradient arrives at the input it belongs to."""
    _stub_kernels(monkeypatch)
    for cls, args in _function_calls():
        assert issubclass(cls, torch.autograd.Function)
        assert "forward" in cls.__dict__ and "backward" in cls.__dict__
        xs = [x.clone().requires_grad_() if isinstance(x, torch.Tensor) else x for x in args]
        out = type("Derived", (cls,), {}).apply(*xs)
        o = out[0] if isinstance(out, tuple) else out
        assert o.grad_fn is not None and (not isinstance(out, tuple) or not out[1].requires_grad)
        o.sum().backward()
        order = [xs[i] for i in (0, 1, 2, 6, 7) if i < len(xs)]
        for i, x in enumerate(order):
            assert x is None or (x.grad == 10.0 * (i + 1)).all(), (cls.__name__, i)


def test_a_traced_operator_is_recorded_as_an_operation(monkeypatch):
    """torch.jit.trace records an operator as one operation, which runs again on replay (the native node's launches
    write through bare pointers: of it only the empty output tensors would be recorded)."""
    import moda_amd
    from moda_amd import _lib, ops

    _stub_kernels(monkeypatch)
    real, replays = _lib.host(), []

    class Host:  # the native call of a replay, on the stand-ins
        def attend(self, mode, q, k, v, kd, vd, scale, G, *_):
            replays.append(mode)
            return ops._raw_fwd(mode, q, k, v, kd, vd, q.shape[-1] ** -0.5 if scale is None else scale, G)

        def __getattr__(self, name):
            return getattr(real, name)

    monkeypatch.setattr(_lib, "host", lambda host=Host(): host)
    r = lambda *s: torch.randn(*s, dtype=torch.float64)
    for f, shapes in (
            (lambda q, k, v, kd, vd: moda_amd.parallel_moda(q, k, v, cached_k=kd, cached_v=vd, moda_group_num=2), "qkvde"),
            (lambda q, k, v, kd, vd: moda_amd.parallel_moda_chunk_visible(q, k, v, cached_k=kd, cached_v=vd, moda_group_num=2,
                                                                          need_lse=True), "qkvde"),
            (lambda q, kd, vd: moda_amd.parallel_fda(q, cached_k=kd, cached_v=vd, moda_group_num=2), "qde"),
            (lambda q, k, v: moda_amd.parallel_attn(q, k, v), "kkv")):
        dims = {"q": (1, 8, 2, 4), "k": (1, 4, 2, 4), "v": (1, 4, 2, 4), "d": (1, 12, 2, 4), "e": (1, 12, 2, 4)}
        traced = torch.jit.trace(f, tuple(r(*dims[s]) for s in shapes), check_trace=False)
        assert "^Parallel" in str(traced.graph)
        xs = [r(*dims[s]) for s in shapes]
        del replays[:]
        got, want = traced(*xs), f(*xs)
        assert len(replays) == 2  # the replay and the eager call
        for a, b in zip(*((x if isinstance(x, tuple) else (x,)) for x in (got, want))):
            assert torch.equal(a, b)
    with pytest.raises(AssertionError, match="T_q must equal T_kv"):  # the argument contract holds while recording
        torch.jit.trace(lambda q, k: moda_amd.parallel_moda(q, k, k), (r(1, 8, 2, 4), r(1, 4, 2, 4)))


def test_a_traced_depth_stream_is_rebuilt_not_written_in_place(monkeypatch):
    import moda_amd
    from moda_amd import modules

    monkeypatch.setattr(modules, "stack_depth", lambda xs: torch.stack(xs, 2).flatten(1, 2))
    monkeypatch.setattr(modules, "parallel_moda", lambda q, k, v, cached_k=None, cached_v=None, **kw:
                        q + k + v + (0 if cached_k is None else (cached_k + cached_v).sum(1, keepdim=True)))

    def f(q, k, v):
        s = moda_amd.DepthStream(3)
        for _ in range(3):
            q = s.attend(q, k, v)
            s.push(k, v)
        return q

    r = lambda: torch.randn(1, 4, 2, 4, dtype=torch.float64, requires_grad=True)
    traced = torch.jit.trace(f, (r(), r(), r()), check_trace=False)
    q, k, v = r(), r(), r()
    d = (k + v).sum(1, keepdim=True)
    assert torch.allclose(traced(q, k, v), q + 3 * (k + v) + 3 * d)
    outer = moda_amd.DepthStream(2)  # began in place, outside
    outer._mode = "train"
    with pytest.raises(RuntimeError, match="cannot be traced"):
        torch.jit.trace(lambda q: outer.attend(q, q, q), (r(),))


def _native_stack(monkeypatch):
    """A small stack of blocks whose native forward pass answers with a mark instead of launching anything."""
    import moda_amd
    from moda_amd import _lib

    real, mark = _lib.host(), torch.zeros(1)

    class Host:
        def stack_forward(self, *_):
            return mark

        def __getattr__(self, name):
            return getattr(real, name)

    monkeypatch.setattr(_lib, "host", lambda host=Host(): host)
    return moda_amd.MoDAStack(64, 2, 2, 1).eval(), torch.zeros(1, 4, 64), mark


def _runs_modules(model, x):
    with torch.no_grad(), pytest.raises(RuntimeError, match="no CPU path"):  # the modules' attention says so
        model(x)


def test_stack_of_dual_tensors_is_left_to_the_modules(monkeypatch):
    """no_grad leaves forward-mode differentiation on: the native forward pass has no tangents, the modules refuse them."""
    import torch.autograd.forward_ad as fwAD

    model, x, mark = _native_stack(monkeypatch)
    with torch.no_grad():
        assert model(x) is mark
    with fwAD.dual_level():
        _runs_modules(model, fwAD.make_dual(x, torch.ones_like(x)))
    with torch.no_grad():
        assert model(x) is mark


def test_stack_under_a_dispatch_mode_is_left_to_the_modules(monkeypatch):
    """A dispatch mode is there to see the framework's operations, which the native forward pass does not issue."""
    from torch.utils._python_dispatch import TorchDispatchMode

    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    model, x, mark = _native_stack(monkeypatch)
    with Watch():
        _runs_modules(model, x)
    assert any("addmm" in s or "linear" in s for s in seen)
    with torch.no_grad():
        assert model(x) is mark


def test_dense_entry_points_refuse_what_their_kernels_cannot_take():
    """Codes of moda_hip_linear and moda_hip_layer_norm, all returned before a device is looked at (nothing is read)."""
    from moda_amd import _lib

    lib = _lib.load()
    i64, ptr = ctypes.c_int64, ctypes.c_void_p

    class Part(ctypes.Structure):
        _fields_ = [("w", ptr), ("bias", ptr), ("y", ptr), ("ldy", i64), ("n", i64)]

    def linear(dtype=0, rows=4, K=64, x=0x1000, ldx=64, n_parts=1, residual=None, ld_res=64, gelu=0, **part):
        p = dict(w=0x2000, bias=0x3000, y=0x4000, ldy=64, n=64)
        p.update(part)
        parts = (Part * 3)(*(Part(*(p[k] for k in ("w", "bias", "y", "ldy", "n"))) for _ in range(3)))
        return lib.moda_hip_linear(dtype, i64(rows), i64(K), ptr(x), i64(ldx), parts, n_parts, ptr(residual), i64(ld_res), gelu, None)

    def norm(dtype=0, rows=4, dim=64, x=0x1000, w=0x2000, b=0x3000, y=0x4000):
        return lib.moda_hip_layer_norm(dtype, i64(rows), i64(dim), ptr(x), ptr(w), ptr(b), ctypes.c_float(1e-6), ptr(y), None)

    assert linear(rows=0) == 0 and norm(rows=0) == 0
    for bad in (dict(dtype=2), dict(dtype=-1), dict(rows=-1), dict(K=0), dict(n_parts=0), dict(n_parts=4), dict(x=None), dict(w=None),
                dict(y=None), dict(n=0), dict(residual=0x5000, n_parts=2), dict(residual=0x5000, gelu=1)):
        assert linear(**bad) == -1, bad
    for bad in (dict(K=96, ldx=96), dict(n=60), dict(rows=1 << 30), dict(ldx=1 << 22)):
        assert linear(**bad) == -2, bad
    for bad in (dict(x=0x1008), dict(ldx=68), dict(ldx=56), dict(w=0x2008), dict(y=0x4002), dict(ldy=68), dict(bias=0x3004),
                dict(residual=0x5008), dict(residual=0x5000, ld_res=68)):
        assert linear(**bad) == -3, bad
    for bad in (dict(dtype=2), dict(rows=-1), dict(dim=0), dict(x=None), dict(w=None), dict(b=None), dict(y=None)):
        assert norm(**bad) == -1, bad
    for bad in (dict(dim=60), dict(dim=4104), dict(rows=1 << 31)):
        assert norm(**bad) == -2, bad
    for bad in (dict(x=0x1008), dict(w=0x2008), dict(b=0x3008), dict(y=0x4008)):
        assert norm(**bad) == -3, bad


def test_block_tail_and_weight_packing_refuse_what_their_kernels_cannot_take():
    """Codes of moda_hip_block_tail and moda_hip_pack_weights, all returned before a device is looked at (nothing is read)."""
    from moda_amd import _lib

    lib = _lib.load()
    i32, i64, ptr = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p
    biases, pointers = ("proj_b", "fc1_b", "fc2_b"), ("attention", "residual", "x", "proj_w", "fc1_w", "fc2_w", "mid_norm_w", "mid_norm_b")

    class Part(ctypes.Structure):
        _fields_ = [("w", ptr), ("bias", ptr), ("y", ptr), ("ldy", i64), ("n", i64)]

    class Tail(ctypes.Structure):
        _fields_ = [("struct_size", i32), ("dtype", i32), ("rows", i64), ("width", i64), ("hidden", i64), ("attention", ptr),
                    ("residual", ptr), ("x", ptr), ("proj_w", ptr), ("proj_b", ptr), ("fc1_w", ptr), ("fc1_b", ptr), ("fc2_w", ptr),
                    ("fc2_b", ptr), ("mid_norm_w", ptr), ("mid_norm_b", ptr), ("end_norm_w", ptr), ("end_norm_b", ptr),
                    ("gelu_table", ptr), ("mid_norm_eps", ctypes.c_float), ("end_norm_eps", ctypes.c_float), ("post_norm", i32),
                    ("n_parts", i32), ("parts", Part * 3)]

    class Weight(ctypes.Structure):
        _fields_ = [("w", ptr), ("packed", ptr), ("n", i64), ("k", i64)]

    def tail(joined=None, **given):
        v = dict(struct_size=ctypes.sizeof(Tail), dtype=0, rows=4, width=256, hidden=1024, post_norm=0, n_parts=1, gelu_table=0x1000,
                 end_norm_w=0x1000, end_norm_b=0x1000, **{n: 0x1000 for n in pointers + biases})
        part = dict(w=0x2000, bias=0x3000, y=0x4000, ldy=64, n=64)
        part.update({n: given.pop("part_" + n) for n in list(part) if "part_" + n in given})
        t = Tail(**{**v, **given})
        for i in range(3):
            t.parts[i] = Part(*(part[n] for n in ("w", "bias", "y", "ldy", "n")))
        if joined is None:
            return lib.moda_hip_block_tail(ctypes.byref(t), None)
        d = _lib.Desc()
        d.struct_size, d.mode, d.B, d.T, d.H, d.G, d.D, d.scale = ctypes.sizeof(d), 1, 2, 2, 1, 4, 64, 1.0
        at = dict(q=0x1000, k=0x1000, v=0x1000, kd=None, vd=None)
        at.update({n: joined[n] for n in at if n in joined})
        for n, x in joined.items():
            if n not in at:
                setattr(d, n, x)
        for n in ("q", "k", "v", "kd", "vd", "o"):
            setattr(d, n, _lib.Strides(1024, 64, 64))
        return lib.moda_hip_attend_block_tail(ctypes.byref(d), *(at[n] for n in ("q", "k", "v", "kd", "vd")), ctypes.byref(t), None)

    def pack(n=1, table=0x1000, **given):
        w = dict(w=0x2000, packed=0x3000, n=32, k=64)
        w.update({f: given[f] for f in w if f in given})
        if "rows" in given:
            w["n"] = given["rows"]
        return lib.moda_hip_pack_weights((Weight * 2)(*(Weight(w["w"], w["packed"], w["n"], w["k"]) for _ in range(2))), n, ptr(table), None)

    assert tail(rows=0) == 0 and lib.moda_hip_block_tail(None, None) == -1 and lib.moda_hip_pack_weights(None, 1, None, None) == -1
    for bad in (dict(struct_size=8), dict(dtype=2), dict(rows=-1), dict(width=0), dict(hidden=0), dict(n_parts=-1), dict(n_parts=4),
                dict(gelu_table=None), dict(end_norm_w=None), dict(end_norm_b=None), dict(n_parts=0, post_norm=1, end_norm_w=None),
                dict(part_w=None), dict(part_y=None), dict(part_n=0), *({n: None} for n in pointers)):
        assert tail(**bad) == -1, bad
    for bad in (dict(width=64), dict(width=640), dict(hidden=64), dict(hidden=1 << 20), dict(rows=1 << 30), dict(part_n=40), dict(part_n=1 << 20)):
        assert tail(**bad) == -2, bad
    for bad in (dict(gelu_table=0x1008), dict(end_norm_w=0x1008), dict(part_w=0x2008), dict(part_y=0x4008), dict(part_ldy=68),
                dict(part_bias=0x3004), *({n: 0x1008} for n in pointers), *({n: 0x1004} for n in biases)):
        assert tail(**bad) == -3, bad
    # the same with the attention before it, whose output is not asked for
    assert tail({"B": 0}, rows=0) == 0 and tail({}, attention=None) == tail({})
    for bad in (dict(rows=5), dict(dtype=1), dict(residual=None), *({"joined": {n: None}} for n in "qkv"), dict(joined=dict(L=3))):
        assert tail(**{"joined": {}, **bad}) == -1, bad
    for bad in (dict(joined=dict(G=2)), dict(joined=dict(G=1), width=128), dict(joined=dict(G=8), width=512), dict(joined=dict(H=2)),
                dict(joined=dict(D=32)), dict(joined=dict(D=128)), dict(joined=dict(Dv=32)), dict(width=384)):
        assert tail(**{"joined": {}, **bad}) == -2, bad
    for bad in (*({"joined": {n: 0x1008}} for n in "qkv"), dict(joined=dict(L=3, kd=0x1008, vd=0x1000)), dict(x=0x1008)):
        assert tail(**{"joined": {}, **bad}) == -3, bad
    for bad in (dict(n=0), dict(w=None), dict(packed=None), dict(rows=0), dict(k=0)):
        assert pack(**bad) == -1, bad
    for bad in (dict(rows=24), dict(k=48), dict(rows=1 << 20), dict(k=1 << 20), dict(rows=1 << 16, k=1 << 15)):
        assert pack(**bad) == -2, bad
    for bad in (dict(table=0x1008), dict(w=0x2008), dict(packed=0x3008)):
        assert pack(**bad) == -3, bad

    class Norm(ctypes.Structure):
        _fields_ = [("x", ptr), ("weight", ptr), ("bias", ptr), ("y", ptr), ("rows", i64), ("dim", i64), ("eps", ctypes.c_float), ("dtype", i32)]

    def both(n=1, **given):
        v = dict(x=0x1000, weight=0x1000, bias=0x1000, y=0x1000, rows=4, dim=256, eps=1e-6, dtype=0)
        return lib.moda_hip_pack_weights_and_norm((Weight * 1)(Weight(0x2000, 0x3000, 32, 64)), n, ptr(0x1000), ctypes.byref(Norm(**{**v, **given})), None)

    assert lib.moda_hip_pack_weights_and_norm((Weight * 1)(Weight(0x2000, 0x3000, 32, 64)), 1, ptr(0x1000), None, None) == -1
    for want, bads in ((-1, [dict(n=0), dict(dtype=2), dict(rows=-1), dict(dim=0), *({n: None} for n in ("x", "weight", "bias", "y"))]),
                       (-2, [dict(dim=100), dict(dim=520), dict(dim=4104), dict(rows=1 << 31)]), (-3, [{n: 0x1008} for n in ("x", "weight", "bias", "y")])):
        for bad in bads:
            assert both(**bad) == want, bad
    # what need not be there is not asked for: no parts and no norm behind them, no biases, no table in fp16; here no device
    # either, which is the next thing to be looked at
    fine = (dict(n_parts=0, end_norm_w=None, end_norm_b=None), dict(proj_b=None, fc1_b=None, fc2_b=None, part_bias=None),
            dict(dtype=1, gelu_table=None))
    if not torch.cuda.is_available():
        assert [tail(**f) for f in fine] == [pack(table=None)] * 3 and pack() not in (0, -1, -2, -3)


@pytest.mark.parametrize("way", ["forward hook", "forward pre-hook", "global hook", "dropout", "replaced activation", "tanh GELU",
                                 "derived linear", "patched forward", "derived attention", "swapped parameter", "blocks that differ",
                                 "another scale", "autocast", "gradients", "derived tensor", "rebuilt cache"])
def test_ways_back_from_the_native_stack_to_its_modules(monkeypatch, way):
    """What the native forward pass does not do, the modules do: a stack runs them as soon as one is not what the
    constructor made, is hooked, drops out, or the call asks for more than values."""
    import moda_amd

    model, x, mark = _native_stack(monkeypatch)
    with torch.no_grad():
        assert model(x) is mark
    blk, nn = model.blocks[1], torch.nn
    if way == "forward hook":
        blk.norm2.register_forward_hook(lambda *a: None)
    elif way == "forward pre-hook":
        blk.attn.kv.register_forward_pre_hook(lambda *a: None)
    elif way == "dropout":
        blk.attn.proj_drop.p = 0.1
        with torch.no_grad():
            assert model(x) is mark  # not active in evaluation
        model.train()
    elif way == "replaced activation":
        blk.mlp[1] = nn.SiLU()
    elif way == "tanh GELU":
        blk.mlp[1] = nn.GELU(approximate="tanh")
    elif way == "derived linear":
        class Linear(nn.Linear):
            pass
        blk.attn.q = Linear(64, 64)
    elif way == "patched forward":
        blk.mlp[2].forward = lambda h: h[..., :64]
    elif way == "derived attention":
        class Attention(moda_amd.MoDAAttention):
            pass
        blk.attn = Attention(64, 2, 1, qkv_bias=True)
    elif way == "swapped parameter":
        blk.norm1._parameters["weight"] = torch.ones(64)
    elif way == "blocks that differ":
        blk.attn.is_causal = True
    elif way == "another scale":
        for b in model.blocks:
            b.attn.scale = 1.0
    if way == "global hook":
        handle = nn.modules.module.register_module_forward_pre_hook(lambda *a: None)
        try:
            _runs_modules(model, x)
        finally:
            handle.remove()
    elif way == "autocast":
        monkeypatch.setattr(torch, "is_autocast_enabled", lambda device: device == "cuda")  # (off on a host without a GPU)
        _runs_modules(model, x)
    elif way == "gradients":
        with pytest.raises(RuntimeError, match="no CPU path"):
            model(x)
    elif way == "derived tensor":
        _runs_modules(model, nn.Parameter(x))
    elif way == "rebuilt cache":
        with torch.no_grad(), pytest.raises(RuntimeError, match="no CPU path"):
            model(x, inplace_cache=False)
    else:
        _runs_modules(model, x)


@pytest.mark.parametrize("way", ["wrapped block", "wrapped attention", "replicas", "plain tensors"])
def test_a_stack_whose_modules_are_wrapped_runs_them(monkeypatch, way):
    """What training and sharding wrappers make of a model: a module that stands in front of a block, replicas and flattened
    parameters, which are attributes and no longer entries of the module's parameters."""

    class Wrapper(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *args, **kwargs):
            return self.inner(*args, **kwargs)

        def __getattr__(self, name):
            try:
                return super().__getattr__(name)
            except AttributeError:
                return getattr(self.inner, name)

    model, x, _ = _native_stack(monkeypatch)
    if way == "wrapped block":
        model.blocks[0] = Wrapper(model.blocks[0])
    elif way == "wrapped attention":
        model.blocks[1].attn = Wrapper(model.blocks[1].attn)
    else:
        attn = model.blocks[1].attn
        linear = attn.q._replicate_for_data_parallel() if way == "replicas" else attn.q
        for name in ("weight", "bias"):
            value = getattr(attn.q, name).detach().clone()
            linear._parameters.pop(name, None)
            setattr(linear, name, value)
        attn._modules["q"] = linear
    _runs_modules(model, x)
