"""Every global-memory access of the matrix-core kernels, replayed on the CPU.

``tests/address_walker.cpp`` is compiled for the host (hipcc, host pass only: no GPU needed) together with the
kernels' own index arithmetic (``moda_amd/csrc/geometry.h``, ``kargs.h``, ``tile.h``, ``tile16.h``, ``tuning.h``)
and walks every (workgroup, wave, lane, trip) of a forward + backward launch: register operand loads, every tile
descriptor with each lane's vector and scalar offset (the lanes that fetch past the tensors' head dim included),
the row-statistics loads, the LDS targets against the launch's dynamic LDS size, and all stores; every output
element must be written exactly once.  The fp32 matrix kernels, the launches that dQ and dK/dV share, the linear, layer-norm and
depth-slot kernels, a stack's block tail, the attention that joins it and the packing of its weights are walked the same way.

The first case is the packed batch that once ended in a GPU memory fault on the packed instantiations of the
256-wide kernels (switched off since).  The walk finds every access of it inside its tensor: the fault is not an
error of the kernels' index arithmetic.
"""
import os
import shutil
import subprocess

import pytest

from cases import ONE_LAUNCH

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MODES = {"causal": 0, "noncausal": 1, "chunk_visible": 2, "depth_only": 3, "plain": 4}


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("walker") / "address_walker")
    # host pass only, under AddressSanitizer (the walker's own tables and the kernels' index code run checked)
    checked = ["-fsanitize=address", "-fno-gpu-sanitize", "-fno-omit-frame-pointer"]  # host code only
    subprocess.run(["hipcc", "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-g", *checked,
                    os.path.join(ROOT, "tests", "address_walker.cpp"), "-o", out], check=True,
                   stdout=subprocess.PIPE, stderr=subprocess.PIPE)
    return out


def tile_width(D):
    return 64 if D <= 64 else 128 if D <= 128 else 256


def run(walker, lengths, H, D, L, G, mode, cb=0, packed=True, B=1, Lv=0, split=1, env=None, Dv=None):
    n = len(lengths) if packed else B
    Dv = D if Dv is None else Dv
    args = [walker, tile_width(max(D, Dv)), D, Dv, H, G, L, Lv, MODES[mode], cb, split, int(packed), n] + list(lengths)
    e = dict(os.environ)
    e.update(env or {})
    r = subprocess.run([str(x) for x in args], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, env=e,
                       timeout=600)
    return r.returncode, r.stdout.strip() + r.stderr.strip()


FAULTED = dict(lengths=(70, 200, 33), H=1, D=192, L=5, G=4, mode="chunk_visible", cb=8)

PACKED = [
    # the packed cases of the GPU parity tests (tests/test_parity_gpu.py: PACKED), 16-bit head dims that are a
    # multiple of 8: lengths, H, D, L, G, mode, chunk tokens
    ((300, 1, 0, 129, 64, 700), 2, 128, 3, 4, "causal", 0),
    ((197, 197, 50), 3, 64, 12, 1, "noncausal", 0),
    ((5, 260, 33), 2, 64, 2, 2, "noncausal", 0),
    ((130, 17, 400), 1, 128, 6, 4, "chunk_visible", 16),
    ((64, 0, 65, 3), 2, 64, 5, 2, "chunk_visible", 32),
    ((100, 7, 260), 2, 128, 7, 2, "depth_only", 0),
    ((1100,), 1, 128, 2, 1, "causal", 0),
    ((3, 2, 1, 1, 40), 2, 64, 0, 2, "causal", 0),
    ((40, 55), 1, 96, 2, 1, "noncausal", 0),
    ((70, 200, 33), 1, 128, 5, 4, "chunk_visible", 8),
    ((130, 17, 400), 2, 64, 3, 4, "chunk_visible", 32),
    # the packed instantiations of the 256-wide kernels (not launched by the library)
    ((130, 1, 0, 300, 65), 2, 256, 3, 2, "causal", 0),
    ((100, 7, 260), 2, 160, 4, 1, "depth_only", 0),
    ((70, 200, 33), 2, 136, 3, 8, "chunk_visible", 4),
    ((333, 1, 64), 1, 248, 2, 2, "noncausal", 0),
]

FIXED = [
    # B, T, H, D, L, G, mode, chunk tokens, Lv
    (2, 150, 2, 64, 5, 2, "causal", 0, 0),
    (1, 197, 3, 128, 4, 1, "noncausal", 0, 0),
    (1, 300, 2, 128, 6, 4, "chunk_visible", 16, 0),
    (1, 260, 1, 64, 3, 4, "chunk_visible", 40, 0),
    (2, 60, 2, 128, 3, 1, "depth_only", 0, 0),
    (1, 333, 2, 128, 0, 4, "plain", 0, 0),
    (1, 200, 2, 120, 3, 4, "causal", 0, 0),
    (1, 90, 1, 8, 2, 2, "causal", 0, 0),
    (2, 64, 2, 64, 4, 2, "causal", 0, 2),          # partially filled depth stream: tile loads through the slot mapping
    (1, 150, 2, 128, 7, 4, "noncausal", 0, 3),
    (2, 100, 1, 64, 5, 1, "depth_only", 0, 1),
    (1, 300, 2, 128, 6, 4, "chunk_visible", 16, 4),  # ... chunks within one query tile (chunk kernel)
    (1, 260, 1, 64, 3, 4, "chunk_visible", 40, 2),   # ... and above it (ring depth tiles, depth column tiles)
    (1, 200, 2, 192, 5, 2, "chunk_visible", 16, 3),  # ... on the 256-wide tiles
    (2, 130, 2, 256, 12, 1, "causal", 0, 5),
    (2, 130, 2, 192, 6, 4, "chunk_visible", 16, 0),
    (1, 700, 1, 256, 3, 2, "chunk_visible", 64, 0),
    (1, 197, 3, 160, 12, 1, "noncausal", 0, 0),
    (1, 100, 2, 256, 7, 4, "depth_only", 0, 0),
    (1, 1, 1, 256, 1, 1, "causal", 0, 0),
    (3, 2100, 1, 128, 2, 2, "causal", 0, 0),       # the throughput launch shape (256 rows per workgroup)
    # query groups that fill a wave's 32 rows, or do not divide them (a token's rows then straddle waves and tiles)
    (1, 77, 2, 128, 5, 8, "causal", 0, 0),
    (1, 40, 1, 64, 3, 32, "noncausal", 0, 2),
    (2, 90, 2, 128, 4, 3, "causal", 0, 0),
    (1, 50, 1, 64, 6, 5, "depth_only", 0, 4),
    (2, 1500, 1, 128, 3, 4, "causal", 0, 2),       # ... in the throughput launch shape, partially filled
    # 64-wide tiles, more than 512 query rows, three sequence column tiles per compute unit: the four-wave dK/dV kernel
    (12, 1024, 8, 64, 2, 2, "causal", 0, 0),
    # what the per-sequence route launches for the packed case above: one fixed-length problem per sequence
    (1, 70, 1, 192, 5, 4, "chunk_visible", 8, 0),
    (1, 200, 1, 192, 5, 4, "chunk_visible", 8, 0),
    (1, 33, 1, 192, 5, 4, "chunk_visible", 8, 0),
]


def test_the_packed_wide_case_that_faulted_stays_inside_its_tensors(walker):
    rc, out = run(walker, **FAULTED)
    assert rc == 0 and "OK checked" in out, out
    # ... and the walk is not vacuous: the same launch over tensors that are one row short is reported, whichever
    # tensor it is (a read through a tile descriptor, a register load, a store)
    for name, cut in (("kd", 192 * 2), ("q", 192 * 2), ("dvd", 192 * 2), ("lse", 4), ("delta", 4), ("do", 16), ("o", 8)):
        rc, out = run(walker, env={"WALKER_SHRINK": f"{name}:{cut}"}, **FAULTED)
        assert rc == 1 and "VIOLATION" in out, (name, out)


@pytest.mark.parametrize("n", [64, 65, 256, 257])
@pytest.mark.parametrize("shape", [(1, 64, 2, 2, "causal", 0), (2, 128, 2, 1, "noncausal", 0), (1, 96, 2, 4, "chunk_visible", 40)],
                         ids=lambda s: f"{s[4]}-D{s[1]}")
def test_packed_batches_of_many_sequences(walker, shape, n):
    """Every tile of every sequence has one workgroup, in the list of all tiles and (above 256 sequences) in the grid of
    the longest one."""
    H, D, L, G, mode, cb = shape
    rc, out = run(walker, [i * 37 % 50 + (300 if i == 40 else 0) for i in range(n)], H, D, L, G, mode, cb, split=-1)
    assert rc == 0 and "OK checked" in out, out


@pytest.mark.parametrize("case", [
    # lengths, H, D, L, G, mode, chunk tokens: more than 256 workgroups in the longest sequence's grid, so that rows and columns
    # are taken from the list; row segments, depth tiles behind the sequence tiles, an empty and a one-token sequence
    ((700, 0, 65, 1, 130), 8, 64, 2, 4, "causal", 0),
    ((700, 33, 300), 16, 64, 0, 2, "noncausal", 0),
    ((900, 100), 16, 64, 2, 8, "chunk_visible", 40),
    ((600, 1, 0, 129), 16, 128, 3, 4, "causal", 0),
], ids=lambda c: f"{c[5]}-{'_'.join(map(str, c[0]))}-D{c[2]}")
def test_packed_batches_in_the_list_of_all_tiles(walker, case):
    lengths, H, D, L, G, mode, cb = case
    rc, out = run(walker, lengths, H, D, L, G, mode, cb, split=-1)
    assert rc == 0 and "OK checked" in out, out


@pytest.mark.parametrize("case", [
    # lengths, H, G, mode, rows in list or grid, columns, most work of an XCD and of a compute unit's turn over the mean
    ((2667, 2000, 1798), 8, 1, "causal", "list", "list", 1.05, 1.85),        # in tile order, segments side by side: 1.00, 1.97
    ((3825, 3400, 3362), 1, 4, "causal", "list", "list", 1.05, 2.5),         # 1.40, 2.11
    ((1497, 1400, 1300, 1200, 1094), 2, 4, "causal", "list", "list", 1.05, 2.0),   # 1.34, 2.12
    ((1332, 1300, 1200, 1100, 1050, 1007, 1000, 1000, 950, 950, 900, 900), 4, 1, "causal", "list", "list", 1.05, 1.7),  # 1.45, 1.93
    ((5909, 433), 4, 1, "causal", "list", "list", 1.05, 1.5),                # 1.10, 1.83
    ((262, 150, 100, 60, 30, 25, 20, 14), 4, 2, "noncausal", "grid", "grid", 9, 99),  # a compute unit for every workgroup
    ((2600, 133), 4, 1, "noncausal", "grid", "list", 1.05, 2.0),             # rows 168, columns in segments 672
], ids=lambda c: f"{c[3]}-{c[0][0]}-H{c[1]}")
def test_packed_launches_take_the_list_where_it_pays_and_spread_their_work(walker, case):
    lengths, H, G, mode, rows, columns, xcd, place = case
    rc, out = run(walker, lengths, H, 64, 0, G, mode, split=-1, env={"WALKER_ORDER": "1"})
    w = out.split()
    got = dict(zip(w[-8::2], w[-7::2]))
    assert rc == 0 and (got["rows"], got["columns"]) == (rows, columns), out
    assert float(got["xcd"]) <= xcd and float(got["place"]) <= place, out


@pytest.mark.parametrize("case", PACKED, ids=lambda c: f"{c[5]}-{'_'.join(map(str, c[0]))}-D{c[2]}")
def test_packed_batches(walker, case):
    lengths, H, D, L, G, mode, cb = case
    rc, out = run(walker, lengths, H, D, L, G, mode, cb)
    assert rc == 0 and "OK checked" in out, out


@pytest.mark.parametrize("case", FIXED, ids=lambda c: f"{c[6]}-B{c[0]}T{c[1]}H{c[2]}D{c[3]}L{c[4]}G{c[5]}")
def test_fixed_length_batches(walker, case):
    B, T, H, D, L, G, mode, cb, Lv = case
    rc, out = run(walker, (T,), H, D, L, G, mode, cb, packed=False, B=B, Lv=Lv)
    assert rc == 0 and "OK checked" in out, out


@pytest.mark.parametrize("case", [
    # B, T, H, D, Dv, L, G, mode, chunk tokens, Lv: value head dim different from the key head dim (one tile width)
    (2, 150, 2, 64, 32, 5, 2, "causal", 0, 0),
    (1, 197, 3, 64, 128, 4, 1, "noncausal", 0, 0),
    (1, 300, 2, 128, 96, 6, 4, "chunk_visible", 16, 0),
    (1, 260, 1, 40, 64, 3, 4, "chunk_visible", 40, 2),
    (2, 60, 2, 128, 256, 3, 1, "depth_only", 0, 0),
    (1, 333, 2, 192, 64, 0, 4, "plain", 0, 0),
    (1, 2100, 1, 128, 64, 2, 2, "causal", 0, 1),
], ids=lambda c: f"{c[7]}-D{c[3]}-Dv{c[4]}")
def test_value_head_dim_differs(walker, case):
    B, T, H, D, Dv, L, G, mode, cb, Lv = case
    rc, out = run(walker, (T,), H, D, L, G, mode, cb, packed=False, B=B, Lv=Lv, Dv=Dv)
    assert rc == 0 and "OK checked" in out, out


def test_row_split_launch(walker):
    """Light launches cut every key tile's query rows into segments (one workgroup each): the tile loads of every
    segment stay inside q, do, lse and the row sums."""
    for split in (2, 4, 8):
        rc, out = run(walker, (4096,), 1, 128, 0, 2, "causal", packed=False, B=1, split=split)
        assert rc == 0 and "OK checked" in out, out


@pytest.mark.parametrize("case", [
    # lengths, H, D, L, G, mode, chunk tokens, packed, B, segments expected
    ((2048,), 2, 128, 2, 4, "causal", 0, False, 1, True),
    ((1100,), 2, 64, 0, 4, "causal", 0, False, 1, True),        # 64-wide tiles, ragged last tile
    ((1000,), 3, 64, 2, 2, "noncausal", 0, False, 1, True),     # more than 1024 query rows: no row waves
    ((3000, 1, 300, 0, 777), 1, 128, 2, 4, "causal", 0, True, 1, False),  # packed on the wider tiles: one pass
    ((3000, 130, 64, 0, 1), 1, 64, 2, 4, "causal", 0, True, 1, True),
    ((1500, 700), 1, 96, 0, 8, "plain", 0, True, 1, False),     # head-dim GQA, padded head dim
    ((1500, 700), 1, 48, 0, 8, "plain", 0, True, 1, True),      # ... on the 64-wide tiles
    ((900, 100), 1, 128, 2, 8, "chunk_visible", 40, True, 1, False),
    ((900, 100), 1, 64, 2, 8, "chunk_visible", 40, True, 1, True),   # sequence segments and depth column tiles in one launch
    ((197,), 1, 64, 3, 4, "noncausal", 0, False, 5, False),     # row waves
    ((250,), 2, 64, 0, 4, "causal", 0, False, 3, False),        # ... with a diagonal
    ((33,), 1, 40, 2, 3, "noncausal", 0, False, 2, False),      # ... one short query tile, padded head dim
], ids=lambda c: f"{c[5]}-{'_'.join(map(str, c[0]))}-D{c[2]}G{c[4]}")
def test_balanced_row_segments_and_row_waves(walker, case):
    """The rule that cuts long column tiles into segments (tiles of one segment write their gradients themselves), and
    the short launches whose waves share their columns: every access in bounds, every gradient row written once."""
    lengths, H, D, L, G, mode, cb, packed, B, split = case
    rc, out = run(walker, lengths, H, D, L, G, mode, cb, packed=packed, B=B, split=-1)
    assert rc == 0 and "OK" in out, out
    assert (int(out.split("segments=")[1].split()[0]) > 1) == split, out


@pytest.mark.parametrize("case", [
    # B, T, H, D, L, G, mode, launches of the forward and dQ kernels on the 64-wide tiles
    (257, 33, 1, 64, 2, 1, "noncausal", "fwd_kernel(short) dq_kernel(short)"),            # one 64-row tile a head
    (130, 70, 2, 40, 0, 2, "causal", "fwd_kernel(short) dq_kernel(short)"),
    (1100, 20, 1, 64, 1, 1, "noncausal", "fwd_kernel(small) dq_kernel(short, three stages)"),
    (300, 50, 2, 64, 3, 2, "noncausal", "fwd_kernel(small) dq_kernel(short, three stages)"),
    (2, 300, 2, 64, 3, 4, "causal", "fwd_kernel(small) dq_kernel(small)"),
], ids=lambda c: f"{c[6]}-B{c[0]}T{c[1]}")
def test_launch_shapes_of_the_narrow_tiles(walker, case):
    B, T, H, D, L, G, mode, shapes = case
    rc, out = run(walker, (T,), H, D, L, G, mode, packed=False, B=B)
    assert rc == 0 and out.startswith(shapes + " OK"), out


def test_slot_arithmetic(walker):
    """Token and slot of a column of a partially filled stream, by a reciprocal and a correction."""
    p = subprocess.run([walker, "slots"], capture_output=True, text=True)
    assert p.returncode == 0 and "OK checked" in p.stdout, p.stdout + p.stderr


@pytest.mark.parametrize("case", [
    # T, H, D, L, Lv, G, B: a backward that adds slot Lv of the depth gradients: row waves, row segments
    (197, 1, 64, 3, 1, 4, 3),
    (1100, 2, 40, 4, 2, 4, 1),
])
def test_own_slot_rows(walker, case):
    T, H, D, L, Lv, G, B = case
    args = dict(lengths=(T,), H=H, D=D, L=L, G=G, mode="noncausal", packed=False, B=B, Lv=Lv, split=-1)
    rc, out = run(walker, env={"WALKER_OWN_SLOT": "1"}, **args)
    assert rc == 0 and "OK checked" in out, out
    rc, out = run(walker, env={"WALKER_OWN_SLOT": "1", "WALKER_SHRINK": f"dkd:{2 * H * D * L}"}, **args)
    assert rc == 1 and "VIOLATION" in out, out


@pytest.mark.parametrize("case", ONE_LAUNCH, ids=lambda c: "-".join(map(str, c[0])))
def test_backward_passes_in_one_launch(walker, case):
    """The rule takes the cases of the GPU test the way that they are meant to test, and the shared launch stays inside its
    tensors and writes every gradient once."""
    (B, T, H, G, D, L, Lv, mode, dtype), one = case
    args = dict(lengths=(T,), H=H, D=D, L=L, G=G, mode=mode.lower(), cb=16 // G, packed=False, B=B, Lv=Lv if Lv != L else 0, split=-1)
    env = {"WALKER_FP32": "1"} if dtype == "fp32" else {}
    rc, out = run(walker, env={"WALKER_ROUTE": "1", **env}, **args)
    assert rc == 0 and out.endswith("one launch" if one else "two launches"), out
    if B * T * H * G > 13000:
        return
    rc, out = run(walker, env=env, **args)
    assert rc == 0 and "OK checked" in out and (("bwd_short_kernel" in out) or ("fp32_bwd_kernel" in out)) == one, out


def test_long_rows_without_room_for_segments_take_two_launches(walker):
    for T, one in ((1024, True), (1025, False), (1100, False)):
        rc, out = run(walker, (T,), 2, 64, 3, 1, "causal", packed=False, B=1, split=1, env={"WALKER_ROUTE": "1"})
        assert rc == 0 and out.endswith("one launch" if one else "two launches"), out


FP32 = [
    # lengths, H, D, Dv, L, Lv, G, mode, chunk tokens, packed, B
    ((1,), 1, 64, 64, 3, 0, 2, "causal", 0, False, 1),
    ((15,), 2, 64, 64, 0, 0, 1, "causal", 0, False, 2),
    ((17,), 3, 4, 4, 7, 0, 3, "causal", 0, False, 1),
    ((129,), 2, 60, 68, 9, 4, 2, "noncausal", 0, False, 2),
    ((300,), 2, 128, 128, 12, 0, 4, "causal", 0, False, 1),
    ((145,), 1, 124, 36, 4, 3, 8, "causal", 0, False, 1),
    ((70,), 2, 64, 64, 70, 0, 1, "depth_only", 0, False, 1),
    ((200,), 2, 64, 64, 3, 2, 2, "chunk_visible", 32, False, 1),
    ((83,), 2, 64, 64, 0, 0, 3, "plain", 0, False, 2),
    ((40, 0, 1, 133), 2, 64, 64, 3, 0, 2, "causal", 0, True, 1),
    ((17, 90), 1, 128, 64, 5, 2, 4, "chunk_visible", 16, True, 1),
    ((50, 3), 1, 100, 100, 2, 0, 1, "depth_only", 0, True, 1),
]


@pytest.mark.parametrize("case", FP32, ids=lambda c: f"{c[7]}-{'_'.join(map(str, c[0]))}-D{c[2]}-Dv{c[3]}-L{c[4]}")
def test_fp32_kernels(walker, case):
    lengths, H, D, Dv, L, Lv, G, mode, cb, packed, B = case
    args = dict(lengths=lengths, H=H, D=D, Dv=Dv, L=L, G=G, mode=mode, cb=cb, packed=packed, B=B, Lv=Lv)
    rc, out = run(walker, env={"WALKER_FP32": "1"}, **args)
    assert rc == 0 and "OK checked" in out, out
    for name, cut in (("q", 16), ("lse", 4), ("do", 16), *((("kd", 16),) if L else (("k", 16),))):
        rc, out = run(walker, env={"WALKER_FP32": "1", "WALKER_SHRINK": f"{name}:{cut}"}, **args)
        if Lv and name == "kd":
            continue  # the last slot holds no data: nobody reads it
        assert rc == 1 and "VIOLATION" in out, (name, out)


@pytest.mark.parametrize("case", [
    # which: arguments, what the rule has to choose
    (("linear", 1, 64, 0, 8), "64x64"),
    (("linear", 65, 192, 0, 72, 24, 136), "64x64"),
    (("linear", 4999, 64, 1, 1000), "128x128"),
    (("linear", 8187, 64, 0, 504), "128x64 "),
    (("linear", 8187, 576, 1, 184, 120), "128x64,3"),
    *((("norm", rows, dim), "") for dim in (8, 136, 512, 520, 1032, 4096) for rows in (1, 37)),
    *((("slot", 2, 33, 3, 40, 4, 2, wide, to_cache), "") for wide in (0, 1) for to_cache in (0, 1)),
], ids=lambda c: "-".join(map(str, c[0])) if isinstance(c, tuple) and isinstance(c[0], tuple) else None)
def test_dense_and_slot_kernels(walker, case):
    args, chosen = case
    for shrink, want in ((None, 0), (f"{'y' if args[0] == 'norm' else 'y0' if args[0] == 'linear' else 'cache_v' if args[-1] else 'v'}:8", 1)):
        e = dict(os.environ)
        if shrink:
            e["WALKER_SHRINK"] = shrink
        if shrink and args[0] == "slot" and args[-1]:
            e["WALKER_SHRINK"] = f"cache_v:{2 * 3 * 40 * 2}"  # behind the slot that is written lies one more
        r = subprocess.run([walker, *map(str, args)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, env=e, timeout=600)
        out = r.stdout + r.stderr
        assert r.returncode == want and out.startswith(chosen) and ("VIOLATION" if want else "OK checked") in out, out


@pytest.mark.parametrize("case", [
    # dtype, rows, width, hidden, post-norm, features of each part: 32 rows a workgroup and 64, a last chunk of the hidden
    # width that leaves waves without features, 2, 3 and 4 feature blocks a wave, more than one turn, no part
    ("bf16", 1, 128, 128, 0, 128, 16, 16),
    ("bf16", 45, 256, 640, 1, 256, 64, 64),
    ("fp16", 8195, 128, 384, 0, 128),
    ("bf16", 8251, 256, 256, 0, 256, 128, 128),
    ("bf16", 8200, 384, 128, 1, 384, 16),
    ("bf16", 70, 512, 1024, 1),
    ("fp16", 8193, 512, 256, 0, 512, 128, 128),
], ids=lambda c: "-".join(map(str, c)))
def test_block_tail(walker, case):
    cuts = [None, "x:2", "attention:2", "residual:2", "fc2_w:2", "end_b:2" if case[4] or len(case) > 5 else "mid_b:2"]
    for shrink in cuts + (["y0:2", f"w{len(case) - 6}:2", "bias0:2"] if len(case) > 5 else []) + (["gelu_table:2"] if case[0] == "bf16" else []):
        e = dict(os.environ, **({"WALKER_SHRINK": shrink} if shrink else {}))
        out = subprocess.run([walker, "tail", *map(str, case)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=e, timeout=600)
        assert out.returncode == (1 if shrink else 0) and ("VIOLATION" if shrink else "OK checked") in out.stdout, (shrink, out.stdout)


@pytest.mark.parametrize("case", [
    # dtype, sequences, tokens, width, hidden, post-norm, features of each part: 32 tokens a workgroup and 64; one token, whole
    # workgroups, a last one of one token
    ("bf16", 1, 1, 128, 128, 0, 128, 16, 16),
    ("bf16", 3, 33, 256, 256, 1, 256, 64, 64),
    ("fp16", 65, 129, 128, 128, 0, 128, 64, 64),
    ("bf16", 129, 64, 256, 256, 0, 256, 64, 64),
    ("bf16", 3, 33, 512, 256, 0, 512, 128, 128),
], ids=lambda c: "-".join(map(str, c)))
def test_attention_with_block_tail(walker, case):
    """The rows of the dense part where the attention joins it; the attention's own accesses are the forward kernel's."""
    for shrink in (None, "x:2", "residual:2", "y0:2", "end_w:2"):
        e = dict(os.environ, **({"WALKER_SHRINK": shrink} if shrink else {}))
        out = subprocess.run([walker, "attend_tail", *map(str, case)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=e, timeout=600)
        assert out.returncode == (1 if shrink else 0) and ("VIOLATION" if shrink else "OK checked") in out.stdout, (shrink, out.stdout)


@pytest.mark.parametrize("case", [
    # dtype, sequences, tokens, key/value heads, query heads on each, slots, filled ones, mode, chunk tokens: the cases of the GPU test of
    # the joined launch; 32 tokens a workgroup and 64, waves that only load, one and two heads, none to many private tiles, rings of depth
    ("bf16", 1, 1, 1, 4, 0, 0, "noncausal", 0),
    ("bf16", 3, 1, 1, 2, 3, 2, "causal", 0),
    ("fp16", 2, 31, 1, 4, 12, 11, "noncausal", 0),
    ("bf16", 5, 33, 1, 2, 12, 1, "noncausal", 0),
    ("bf16", 3, 64, 1, 4, 5, 5, "causal", 0),
    ("bf16", 2, 65, 1, 4, 40, 21, "noncausal", 0),
    ("fp16", 2, 300, 1, 2, 6, 4, "causal", 0),
    ("bf16", 2, 261, 1, 4, 0, 0, "causal", 0),
    ("bf16", 2, 100, 1, 4, 12, 7, "chunk_visible", 16),
    ("bf16", 2, 150, 1, 2, 3, 2, "chunk_visible", 48),
    ("bf16", 65, 129, 1, 4, 12, 11, "noncausal", 0),
    ("fp16", 65, 129, 1, 2, 4, 3, "causal", 0),
    ("bf16", 84, 100, 1, 4, 6, 5, "chunk_visible", 16),
    ("bf16", 84, 100, 1, 2, 3, 2, "chunk_visible", 48),
    ("bf16", 3, 33, 2, 2, 12, 11, "noncausal", 0),
    ("fp16", 2, 261, 2, 4, 6, 2, "causal", 0),
    ("bf16", 1, 1, 2, 4, 0, 0, "noncausal", 0),
    ("bf16", 64, 129, 2, 2, 4, 3, "noncausal", 0),
    ("bf16", 85, 100, 2, 2, 6, 5, "chunk_visible", 16),
    ("bf16", 2, 150, 2, 4, 3, 2, "chunk_visible", 48),
], ids=lambda c: "-".join(map(str, c)))
def test_attention_of_the_joined_launch(walker, case):
    """What test_attention_with_block_tail leaves out: the attention before the dense part, whose shapes no forward launch has."""
    args = [walker, "attention", *map(str, case[:7]), str(MODES[case[7]]), str(case[8])]
    small = case[1] * case[2] <= 600
    for shrink in (None, "q:2", "k:2", "v:2", "kd:2", "vd:2") if small else (None, "q:2"):
        in_cache = 0 < case[6] < case[5]
        if shrink and (shrink[0] in "kv" and (case[5] == 0 if shrink[1] == "d" else in_cache)):
            continue  # a tensor that the case does without
        e = dict(os.environ, **({"WALKER_SHRINK": shrink} if shrink else {}))
        out = subprocess.run(args, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=e, timeout=600)
        if shrink and shrink[1] == "d" and in_cache and case[6] + 1 < case[5]:
            assert "OK checked" in out.stdout, (shrink, out.stdout)  # the last slot holds nothing
        else:
            assert out.returncode == (1 if shrink else 0) and ("VIOLATION" if shrink else "OK checked") in out.stdout, (shrink, out.stdout)


@pytest.mark.parametrize("case", [
    # sequences, tokens, width, heads, key/value heads, compute units: rounds of workgroups by sequences against those of all rows;
    # six blocks, us apart / joined
    (64, 197, 256, 4, 1, 256, "joins"),   # 281 / 256
    (36, 197, 256, 4, 1, 256, "joins"),   # 218 / 193: 252 workgroups of 32 tokens
    (37, 197, 256, 4, 1, 256, "apart"),   # 259 of them
    (64, 257, 256, 4, 1, 256, "joins"),   # 462 / 464: two rounds either way
    (100, 145, 256, 4, 1, 256, "apart"),  # 300 workgroups of 64 tokens, 227 of 64 rows
    (64, 50, 128, 2, 1, 256, "joins"),    # 130 / 108
    (64, 197, 256, 4, 2, 256, "joins"),
    (36, 197, 512, 8, 2, 256, "joins"),
    (64, 197, 512, 8, 2, 256, "apart"),   # what the kernel does not take: 64 tokens of eight heads
    (64, 197, 128, 2, 2, 256, "apart"),
    (64, 197, 256, 2, 1, 256, "apart"),
    (64, 197, 512, 8, 1, 256, "apart"),
    (64, 197, 384, 6, 1, 256, "apart"),
], ids=lambda c: "-".join(map(str, c[:6])))
def test_when_a_blocks_attention_joins_its_tail(walker, case):
    out = subprocess.run([walker, "attend_tail_rule", *map(str, case[:-1])], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out.strip() == case[-1]


@pytest.mark.parametrize("case", [
    # sequences, tokens, heads, key/value heads, causal; us of six blocks apart / joined on 256 compute units
    (1, 16384, 2, 1, False, "joins"),  # 1284 / 1256: one round of one wave a SIMD, as apart
    (16, 1024, 2, 1, True, "joins"),   # 235 / 200
    (1, 16384, 2, 1, True, "joins"),   # 1275 / 1239
    (64, 512, 2, 1, False, "apart"),   # 303 / 313: two rounds of one wave, apart one of two
    (96, 197, 2, 1, False, "joins"),   # 270 / 259
    (4, 6144, 2, 1, True, "joins"),    # 666 / 550: apart the unit with the longest row has two more
    (4, 16384, 2, 1, False, "apart"),  # 3836 / 4959
    (1, 65536, 2, 1, True, "apart"),   # 7509 / 9688
    (192, 256, 2, 1, True, "apart"),   # 369 / 395: three rounds
    (1, 16384, 4, 1, False, "joins"),  # 2022 / 1991: one round of two waves, as apart
    (32, 512, 4, 1, True, "joins"),    # 303 / 286
    (8, 2048, 4, 1, True, "apart"),    # 416 / 434: ends with its longest row, where apart the others make room
    (1, 16384, 4, 1, True, "apart"),   # 1475 / 1854
    (1, 8192, 4, 1, True, "joins"),    # 755 / 703: 32 tokens, one wave
    (64, 512, 4, 1, False, "joins"),   # 578 / 556
    (4, 8192, 4, 1, False, "apart"),   # 2147 / 2172
    (32, 1024, 4, 1, True, "joins"),   # 589 / 554
    (1, 65536, 4, 1, True, "apart"),   # 13 993 / 15 286
    (8, 512, 4, 2, True, "joins"),     # 231 / 218: 32 tokens, the halves' waves on the same SIMDs
    (2, 2048, 4, 2, False, "apart"),   # 331 / 382
    (4, 4096, 4, 2, False, "joins"),   # 716 / 703
    (4, 4096, 4, 2, True, "apart"),    # 579 / 656
    (8, 1024, 8, 2, True, "joins"),    # 563 / 506
    (1, 8192, 8, 2, True, "apart"),    # 1090 / 1235
], ids=lambda c: "-".join(map(str, c[:5])))
def test_what_length_mask_and_heads_say_of_joining(walker, case):
    sequences, tokens, heads, kv_heads, causal, want = case
    out = subprocess.run([walker, "attend_tail_rule", *map(str, (sequences, tokens, 64 * heads, heads, kv_heads, 256, 6, int(causal)))], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out.strip() == want


@pytest.mark.parametrize("sequences, tokens, of_a_workgroup", [(1, 1, 32), (3, 64, 32), (8, 197, 64), (1, 8257, 64), (5, 33, 32)])
def test_order_of_the_joined_launch(walker, sequences, tokens, of_a_workgroup):
    """Every tile of every sequence once; where they differ in cost (causal), those with the most keys first."""
    tiles = -(-tokens // of_a_workgroup)
    for causal in (0, 1):
        out = subprocess.run([walker, "attend_tail_order", *map(str, (sequences, tokens, of_a_workgroup, causal))], stdout=subprocess.PIPE, text=True, check=True).stdout
        places = [tuple(map(int, p.split(":"))) for p in out.split()]
        assert sorted(places) == [(b, t) for b in range(sequences) for t in range(tiles)]
        assert [t for _, t in places] == sorted((t for _, t in places), reverse=bool(causal))


@pytest.mark.parametrize("case", [
    # tokens, heads, key/value heads, slots: one sequence on either side of 2 GiB a slice (tokens x slots x key/value features)
    (16384, 2, 1, 1024, "apart"),
    (16384, 2, 1, 1023, "joins"),
    (8192, 4, 1, 2048, "apart"),
    (8192, 4, 1, 2047, "joins"),
    (8192, 8, 2, 1024, "apart"),
    (65536, 4, 2, 128, "apart"),
    (87382, 4, 2, 96, "apart"),
    (349526, 4, 2, 24, "apart"),
    (16777216, 4, 1, 1, "apart"),
], ids=lambda c: "-".join(map(str, c[:4])))
def test_a_blocks_attention_joins_only_what_the_joined_launch_takes(walker, case):
    """Chunk-visible stacks of one sequence, as long as attention could join or longer.  Slices of 2 GiB and more go apart: the joined call
    refuses them, the forward call takes them, as far as can be seen without a device."""
    import ctypes

    import torch

    from moda_amd import _lib

    tokens, heads, kv_heads, slots, want = case
    width, kv = 64 * heads, 64 * kv_heads
    out = subprocess.run([walker, "attend_tail_rule", "1", *map(str, (tokens, width, heads, kv_heads, 256, slots))], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out.strip() == want
    if torch.cuda.is_available():
        return  # made-up addresses

    i32, i64, f32, ptr = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p
    named = ("attention", "residual", "x", "proj_w", "proj_b", "fc1_w", "fc1_b", "fc2_w", "fc2_b", "mid_norm_w", "mid_norm_b", "end_norm_w", "end_norm_b", "gelu_table")

    class Tail(ctypes.Structure):  # moda_hip_block_tail_args, without parts
        _fields_ = [("struct_size", i32), ("dtype", i32), ("rows", i64), ("width", i64), ("hidden", i64), *((n, ptr) for n in named),
                    ("mid_norm_eps", f32), ("end_norm_eps", f32), ("post_norm", i32), ("n_parts", i32), ("parts", i64 * 15)]

    t = Tail(struct_size=ctypes.sizeof(Tail), rows=tokens, width=width, hidden=4 * width, **{n: 0x1000 for n in named})
    d = _lib.Desc()
    d.struct_size, d.mode, d.chunk_tokens, d.scale = ctypes.sizeof(d), _lib.CHUNK_VISIBLE, 16, 0.125
    d.B, d.T, d.H, d.G, d.D, d.Dv = 1, tokens, kv_heads, heads // kv_heads, 64, 64
    d.q = d.o = _lib.Strides(tokens * width, kv, 64)
    d.k = d.v = _lib.Strides(tokens * slots * kv, slots * kv, 64)
    d.kd = d.vd = _lib.Strides(tokens * slots * kv, kv, 64)
    p, lib, refused, no_device = ptr(0x1000), _lib.load(), -2, -6
    for filled in {0, 1, slots // 2}:  # a stack's first block, and later ones
        d.L, d.L_valid = (slots, filled) if filled else (0, 0)
        assert lib.moda_hip_fwd(ctypes.byref(d), p, p, p, p, p, p, p, None) == no_device
        got = lib.moda_hip_attend_block_tail(ctypes.byref(d), p, p, p, p, p, ctypes.byref(t), None)
        assert got == (no_device if want == "joins" else refused), filled


@pytest.mark.parametrize("case", [
    # rows, rows a workgroup, packing workgroups of the widest matrix, matrices (and the table); workgroups of one launch, 0: two
    (12608, 8, 128, 61, 1576 + 128 * 61),
    (1, 16, 1, 2, 3),
    ((1 << 26) - 4 * 97, 4, 1, 96, (1 << 24) - 1),
    ((1 << 26) - 4 * 97 + 1, 4, 1, 97, 0),
    (4, 4, 1 << 18, 64, 0),  # 64 matrices of 2^29 elements
    (4, 4, 1 << 20, 97, 0),  # (as many as a launch takes, the largest there are)
    ((1 << 30) - 1, 4, 1 << 20, 97, 0),
], ids=str)
def test_weights_and_norm_in_one_grid(walker, case):
    """A dimension of a grid ends below 2^32 threads, which 256 a workgroup reach at 2^24."""
    out = subprocess.run([walker, "pack_and_norm", *map(str, case[:4])], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert int(out) == case[4]


def test_packed_weights(walker):
    out = subprocess.run([walker, "pack", "7"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=600)
    assert out.returncode == 0 and "OK checked" in out.stdout, out.stdout


@pytest.mark.parametrize("case", [
    # dtype, rows, width, MLP, K/V width, compute units, what has to be chosen: points on both sides of the rule that measured
    # at least 5 % apart (256 compute units), times of a block in one launch / in pieces
    ("bf16", 200, 256, 1024, 64, 256, "one launch, 32 rows"),      # 45 / 64 us
    ("bf16", 16, 256, 4096, 64, 256, "pieces, 32 rows"),           # 67 / 56
    ("bf16", 2320, 256, 4096, 64, 256, "one launch, 32 rows"),     # 74 / 80
    ("fp16", 580, 256, 4096, 64, 256, "pieces, 32 rows"),          # 82 / 68
    ("bf16", 1160, 256, 16384, 64, 256, "pieces, 32 rows"),        # 230 / 182
    ("bf16", 200, 128, 8192, 64, 256, "pieces, 32 rows"),          # 100 / 85
    ("fp16", 1160, 128, 8192, 64, 256, "pieces, 32 rows"),         # 115 / 107
    ("fp16", 4728, 128, 2048, 64, 256, "one launch, 32 rows"),
    ("bf16", 8128, 384, 1536, 192, 256, "one launch, 32 rows"),    # 63 / 87
    ("fp16", 200, 384, 384, 192, 256, "one launch, 32 rows"),      # 36 / 39
    ("bf16", 200, 384, 1536, 192, 256, "pieces, 32 rows"),         # 55 / 48
    ("fp16", 8128, 384, 6144, 192, 256, "one launch, 32 rows"),    # 151 / 196
    ("bf16", 8128, 512, 2048, 128, 256, "one launch, 32 rows"),    # 86 / 107
    ("fp16", 16, 512, 512, 128, 256, "pieces, 32 rows"),           # 41 / 37
    ("fp16", 8128, 512, 512, 128, 256, "one launch, 32 rows"),     # 55 / 73
    ("bf16", 16448, 256, 1024, 64, 256, "one launch, 64 rows"),    # 80 / 94
    ("bf16", 16448, 384, 1536, 192, 256, "pieces, 64 rows"),       # 161 / 151
    ("fp16", 9280, 384, 1536, 192, 256, "one launch, 64 rows"),    # 90 / 101
    ("bf16", 9280, 512, 2048, 128, 256, "one launch, 64 rows"),    # 121 / 126
    ("fp16", 9280, 512, 512, 128, 256, "pieces, 64 rows"),         # 95 / 85
    ("fp16", 12608, 512, 2048, 128, 256, "one launch, 64 rows"),   # 154 / 160
    # a partition with fewer compute units: a round holds fewer rows
    ("bf16", 2048, 384, 1536, 192, 64, "one launch, 32 rows"),
    ("bf16", 4097, 384, 1536, 192, 64, "pieces, 64 rows"),
], ids=lambda c: "-".join(map(str, c[:4])))
def test_a_blocks_dense_part_takes_the_faster_way(walker, case):
    out = subprocess.run([walker, "tail_rule", *map(str, case[:-1])], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out.strip() == case[-1]
