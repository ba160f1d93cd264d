// Host-side address walker for the matrix-core attention kernels (test infrastructure, built and run by
// tests/test_address_model_cpu.py; needs no GPU).
//
// For one problem description it replays, on the CPU, every global-memory access the kernels of a forward and a
// backward launch would make -- per workgroup, wave, lane and trip: the register operand loads, every buffer
// descriptor of the global->LDS tile loads with each lane's vector and scalar offset, the row statistics, and all
// stores -- and checks each one against the extent of the tensor it belongs to.  The index arithmetic is not
// restated here: it is the kernels' own (moda_amd/csrc/geometry.h, kargs.h: enter_sequence, tile.h: Tile,
// AsyncTileLoader, WaveTileLoader, tile16.h: slot_base, tuning.h), compiled for the host; what this file adds is
// the kernels' control flow around it (which tile is issued when, which lanes are guarded by what).
//
// Checked per access:
//   * register loads and stores: [address, address + bytes) inside the tensor;
//   * tile loads: the descriptor's base inside the tensor and every lane the range check lets through inside it
//     (lanes whose offset + 16 exceeds num_records receive zeros and touch no memory); the lane's offset
//     voffset + soffset does not wrap 32 bits (the range check the kernels rely on compares that sum with
//     num_records); a lane whose chunk lies past the tensors' head dim is out of range; the 64 LDS slots the load
//     fills lie inside the launch's dynamic LDS allocation;
//   * coverage: every element of o, lse, dq, dk, dv, dkd, dvd and of the row-sum workspace is written exactly once;
//     every partial sum of a row segment that is read was written once, and every one that was written is read.
//
// usage: address_walker HD D Dv H G L Lv mode(0..4) chunk_tokens row_segments packed B_or_n len0 [len1 ...]
//   packed = 0: a fixed-length batch of B sequences of len0 tokens; packed = 1: n sequences on one packed axis.
//   environment: WALKER_FP32=1 walks the fp32 matrix kernels instead; WALKER_OWN_SLOT=1 a backward that leaves the slots
//   without data alone and adds slot Lv of the depth gradients to dk, dv; instead of a walk, WALKER_ORDER=1 prints
//   the order of a packed batch's launches, WALKER_ROUTE=1 whether a backward pass is one launch.
// usage: address_walker linear rows K gelu n0 [n1 n2]   |   norm rows dim   |   slot B T H D L slot wide to_cache
//   |   tail bf16|fp16 rows width hidden post_norm [n0 [n1 [n2]]]   |   pack matrices
//   |   attention bf16|fp16 sequences tokens heads group slots filled mode chunk_tokens
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../include/moda_hip.h"
#include "../moda_amd/csrc/block.h"
#include "../moda_amd/csrc/geometry.h"
#include "../moda_amd/csrc/kargs.h"
#include "../moda_amd/csrc/tile.h"
#include "../moda_amd/csrc/tile16.h"
#include "../moda_amd/csrc/tuning.h"

using namespace moda;

namespace {

struct Region {
  std::string name;
  uint64_t base = 0, bytes = 0;
  std::vector<uint8_t> writes;  // per 2-byte (or 4-byte for fp32 regions) unit: number of writes
  int unit = 2;
  bool track = false;
};

std::map<std::string, Region> g_regions;
long long g_checked = 0, g_dma_in = 0, g_dma_out = 0;
bool g_fp32 = false, g_own_slot = false;
struct Where {  // put into words when there is something to say
  const char* kernel;
  int block, wave, lane;
  const char* what;
} g_where = {"", 0, 0, 0, ""};

[[noreturn]] void fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  fprintf(stdout, "VIOLATION [%s block %d wave %d lane %d: %s] ", g_where.kernel, g_where.block, g_where.wave, g_where.lane, g_where.what);
  vfprintf(stdout, fmt, ap);
  fprintf(stdout, "\n");
  va_end(ap);
  exit(1);
}

Region& region(const char* name) { return g_regions.at(name); }

const uint16_t* add_region(const char* name, int idx, uint64_t bytes, int unit, bool track) {
  // self-test hook: WALKER_SHRINK=<tensor>:<bytes> makes one tensor smaller than the kernels are told, which the
  // walk must report
  if (const char* e = getenv("WALKER_SHRINK")) {
    const char* colon = strchr(e, ':');
    if (colon && std::string(e, colon - e) == name) {
      const uint64_t cut = strtoull(colon + 1, nullptr, 10);
      bytes = bytes > cut ? bytes - cut : 0;
      track = false;
    }
  }
  Region r;
  r.name = name;
  r.base = ((uint64_t)(idx + 1)) << 40;  // far apart: an offset error cannot land in a neighbour
  r.bytes = bytes;
  r.unit = unit;
  r.track = track;
  if (track) r.writes.assign(bytes / unit, 0);
  g_regions[name] = r;
  return (const uint16_t*)r.base;
}

void check_access(const char* name, const void* p, uint64_t n, bool write) {
  Region& r = region(name);
  const uint64_t a = (uint64_t)p;
  g_checked++;
  if (a < r.base || a + n > r.base + r.bytes)
    fail("%s of %llu bytes at %s%+lld (tensor holds %llu bytes)", write ? "store" : "load", (unsigned long long)n, name,
         (long long)(a - r.base), (unsigned long long)r.bytes);
  if (write && r.track)
    for (uint64_t i = (a - r.base) / r.unit; i < (a - r.base + n) / r.unit; i++)
      if (++r.writes[i] > 1) fail("%s unit %llu written twice", name, (unsigned long long)i);
}

// one lane of a global->LDS load
void check_dma(const char* name, const void* desc_base, uint32_t num_records, int voff, int soff, int bytes,
               uint32_t lds_byte, uint32_t lds_limit, bool lane_is_pad) {
  Region& r = region(name);
  const uint64_t b = (uint64_t)desc_base;
  g_checked++;
  // The descriptor of a (batch, head) slice starts at the slice's first row and covers whole row strides, so behind
  // the tensor's last row it may reach into the other heads' share of one more stride; no lane offset does (each
  // in-range lane is checked against the tensor below).  The base itself must lie inside the tensor.
  if (num_records > 0 && (b < r.base || b >= r.base + r.bytes))
    fail("descriptor of %s: base %+lld, %u bytes (tensor holds %llu)", name, (long long)(b - r.base), num_records,
         (unsigned long long)r.bytes);
  if (voff < 0 || soff < 0) fail("negative offset into %s: voffset %d soffset %d", name, voff, soff);
  const uint64_t off = (uint64_t)(uint32_t)voff + (uint64_t)(uint32_t)soff;
  if (off + bytes > 0xffffffffull) fail("offset into %s wraps 32 bits: voffset %d soffset %d", name, voff, soff);
  const bool in_range = off + bytes <= num_records;
  if (lane_is_pad && in_range) fail("padding lane of %s in range: voffset %d soffset %d records %u", name, voff, soff, num_records);
  if (in_range) {
    g_dma_in++;
    check_access(name, (const char*)desc_base + off, bytes, false);
  } else {
    g_dma_out++;
  }
  if ((uint64_t)lds_byte + 64ull * bytes > lds_limit)
    fail("LDS target %u (+%d) beyond the %u bytes of dynamic LDS", lds_byte, 64 * bytes, lds_limit);
}

// partial sums of row segments: written once before they are read, and then marked so that the rest can be found
long long g_partials_read = 0;
void read_partials(const float* p, int n) {
  check_access("part", p, 4ull * n, false);
  Region& r = region("part");
  for (uint64_t i = ((uint64_t)p - r.base) / 4; i < ((uint64_t)p - r.base) / 4 + n; i++) {
    if (r.writes[i] != 1) fail("partial sum %llu read %s", (unsigned long long)i, r.writes[i] ? "twice" : "that no segment wrote");
    r.writes[i] = 2;
    g_partials_read++;
  }
}

struct Case {
  int HD, D, Dv, H, G, L, Lv, mode, cb, packed, nseq;
  std::vector<int> len;
  std::vector<int32_t> cu;
  int total, Tmax;
};

KArgs make_args(const Case& c) {
  KArgs a;
  memset(&a, 0, sizeof(a));
  const bool plain = c.mode == 4;
  const int Bt = c.packed ? 1 : c.nseq;  // batch extent of the tensors
  const int T = c.packed ? c.total : c.Tmax;
  a.B = c.nseq;
  a.T = c.Tmax;
  a.Hkv = c.H;
  a.D = c.D;
  a.Dv = c.Dv;
  a.Tq = plain ? c.Tmax : c.Tmax * c.G;
  a.Gf = plain ? 1 : c.G;
  a.Hq = plain ? c.H * c.G : c.H;
  a.hdiv = plain ? c.G : 1;
  a.L = c.L;
  a.Lv = c.Lv > 0 ? c.Lv : c.L;
  a.Cb = c.mode == 2 ? (c.cb > 0 ? c.cb : 1) : 1;
  a.has_seq = c.mode != 3;
  a.causal = c.mode == 0 || c.mode == 2 || plain;
  a.chunk = c.mode == 2;
  a.scale = 1.f;
  a.dkv_split = 1;
  a.compute_units = 256;
  const int64_t qrows = plain ? T : (int64_t)T * c.G;
  a.delta_pitch = c.packed ? (int)qrows : a.Tq;
  a.own_delta = 1;  // a whole backward: the dQ kernel forms the row sums (the delta kernel is walked as well)
  auto strides = [&](int64_t rows, int heads, int dim) { return Str3{rows * heads * dim, (int64_t)heads * dim, (int64_t)dim}; };
  a.own_slot = a.keep_slots = g_own_slot ? 1 : 0;
  // a dense [Bt, rows, heads, dim] tensor
  const int es = g_fp32 ? 4 : 2;
  auto bytes = [&](int64_t rows, int heads, int dim) { return (uint64_t)Bt * rows * heads * dim * es; };
  int idx = 0;
  a.q = add_region("q", idx++, bytes(qrows, a.Hq, c.D), es, false);
  a.o = add_region("o", idx++, bytes(qrows, a.Hq, c.Dv), es, true);
  a.out_o = (uint16_t*)a.o;
  a.d_o = add_region("do", idx++, bytes(qrows, a.Hq, c.Dv), es, false);
  a.dq = (uint16_t*)add_region("dq", idx++, bytes(qrows, a.Hq, c.D), es, true);
  a.k = add_region("k", idx++, bytes(T, c.H, c.D), es, false);
  a.v = add_region("v", idx++, bytes(T, c.H, c.Dv), es, false);
  a.dk = (uint16_t*)add_region("dk", idx++, bytes(T, c.H, c.D), es, true);
  a.dv = (uint16_t*)add_region("dv", idx++, bytes(T, c.H, c.Dv), es, true);
  a.kd = add_region("kd", idx++, bytes((int64_t)T * c.L, c.H, c.D), es, false);
  a.vd = add_region("vd", idx++, bytes((int64_t)T * c.L, c.H, c.Dv), es, false);
  a.dkd = (uint16_t*)add_region("dkd", idx++, bytes((int64_t)T * c.L, c.H, c.D), es, true);
  a.dvd = (uint16_t*)add_region("dvd", idx++, bytes((int64_t)T * c.L, c.H, c.Dv), es, true);
  a.lse = (float*)add_region("lse", idx++, (uint64_t)Bt * qrows * a.Hq * 4, 4, true);
  a.delta = (float*)add_region("delta", idx++, (uint64_t)(c.packed ? 1 : c.nseq) * a.Hq * a.delta_pitch * 4, 4, true);
  if (!g_fp32 && depth_scores_from_dq(a, c.HD)) {  // P and dS of the (query row, slot) pairs, handed from dQ to the depth-gradient kernel
    const uint64_t n = (uint64_t)(c.packed ? 1 : c.nseq) * a.Hq * a.delta_pitch * a.Lv * 2;
    a.depth_p = (uint16_t*)add_region("hand_p", idx++, n, 2, true);
    a.depth_ds = (uint16_t*)add_region("hand_ds", idx++, n, 2, true);
  }
  a.sq = a.sdq = strides(qrows, a.Hq, c.D);
  a.so = a.sdo = strides(qrows, a.Hq, c.Dv);
  a.sk = a.sdk = strides(T, c.H, c.D);
  a.sv = a.sdv = strides(T, c.H, c.Dv);
  a.skd = a.sdkd = strides((int64_t)T * c.L, c.H, c.D);
  a.svd = a.sdvd = strides((int64_t)T * c.L, c.H, c.Dv);
  if (c.packed) a.cu = c.cu.data();
  return a;
}

// what a place says of its sequence is what the offsets say
template <typename Place>
void check_place(const KArgs& a, const Place& p) {
  if (p.t0 != a.cu[p.b] || p.T != a.cu[p.b + 1] - a.cu[p.b]) fail("place of sequence %d: tokens %d + %d", p.b, p.t0, p.T);
}

// argument block of the workgroup: rebased on its sequence for a packed batch
KArgs seq_args(const KArgs& in, int& b) {
  KArgs a = in;
  enter_sequence(a, b);
  return a;
}

void ctx(const char* kernel, int block, int wave, int lane, const char* what) {
  g_where = {kernel, block, wave, lane, what};
}

// One tile of the workgroup's ring, this lane's loads: sequence rows (of the tensors `k_name`, `v_name`) or depth columns from row0 on
template <int HD, int NT, bool WIDE_ADDR>
void ring_tile_loads(const KArgs& a, int b, int hkv, const AsyncTileLoader<HD, 64, NT>& ld, const typename AsyncTileLoader<HD, 64, NT>::Source& srcK,
                     const typename AsyncTileLoader<HD, 64, NT>::Source& srcV, int row0, bool dep, bool mapped, uint32_t kt, uint32_t lds_bytes,
                     const char* k_name, const char* v_name) {
  typedef AsyncTileLoader<HD, 64, NT> Loader;
  constexpr int BN = 64;
  for (int i = 0; i < Loader::N; i++) {
    const uint32_t ldsK = kt + (uint32_t)ld.lds_elems(i) * 2, ldsV = ldsK + BN * HD * 2;
    if (dep && mapped) {  // partially filled stream: one descriptor anchored at the first column's token
      const int w0 = row0 / a.Lv, l0 = row0 - w0 * a.Lv;
      const int64_t anchor = (int64_t)w0 * a.L, rows_total = (int64_t)a.T * a.L;
      check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + anchor * a.skd.t,
                mapped_bytes(anchor, rows_total, (uint32_t)a.skd.t * 2u),
                ld.mapped_offset(i, l0, a.L, a.Lv, (int)a.skd.t * 2, a.D), 0, 16, ldsK, lds_bytes, ld.pads(a.D));
      check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + anchor * a.svd.t,
                mapped_bytes(anchor, rows_total, (uint32_t)a.svd.t * 2u),
                ld.mapped_offset(i, l0, a.L, a.Lv, (int)a.svd.t * 2, a.Dv), 0, 16, ldsV, lds_bytes, ld.pads(a.Dv));
      // a lane in range must have fetched a slot that holds data
      const int rel = mapped_row(l0, Loader::rows_before(i) + ld.row_in_pass, a.L, a.Lv);
      if ((anchor + rel) % a.L >= a.Lv) fail("mapped depth tile reads slot %d of %d filled", (int)((anchor + rel) % a.L), a.Lv);
    } else if (WIDE_ADDR) {
      const int row_end = dep ? a.T * a.L : a.T;
      const uint16_t* kb = dep ? a.kd + b * a.skd.b + hkv * a.skd.h : a.k + b * a.sk.b + hkv * a.sk.h;
      const uint16_t* vb = dep ? a.vd + b * a.svd.b + hkv * a.svd.h : a.v + b * a.sv.b + hkv * a.sv.h;
      const int64_t ks = dep ? a.skd.t : a.sk.t, vs = dep ? a.svd.t : a.sv.t;
      check_dma(dep ? "kd" : k_name, kb + (int64_t)row0 * ks, Loader::anchored_bytes(ks, row0, row_end),
                ld.lane_offset((int)ks * 2, a.D), Loader::rows_before(i) * (int)ks * 2, 16, ldsK, lds_bytes, ld.pads(a.D));
      check_dma(dep ? "vd" : v_name, vb + (int64_t)row0 * vs, Loader::anchored_bytes(vs, row0, row_end),
                ld.lane_offset((int)vs * 2, a.Dv), Loader::rows_before(i) * (int)vs * 2, 16, ldsV, lds_bytes, ld.pads(a.Dv));
    } else {
      check_dma(dep ? "kd" : k_name, srcK.base, srcK.nbytes, srcK.voff, Loader::source_soffset(srcK, row0, i), 16, ldsK,
                lds_bytes, ld.pads(a.D));
      check_dma(dep ? "vd" : v_name, srcV.base, srcV.nbytes, srcV.voff, Loader::source_soffset(srcV, row0, i), 16, ldsV,
                lds_bytes, ld.pads(a.Dv));
    }
  }
}
// Load i of a wave's own K and V tile of depth columns [col0, col0 + nrows)
template <int HD>
void own_tile_load(const KArgs& a, int b, int hkv, const WaveTileLoader<HD>& own, int i, int col0, int nrows, bool mapped, uint32_t kt, uint32_t vt,
                   uint32_t lds_bytes) {
  if (mapped) {
    const int w0 = col0 / a.Lv, l0 = col0 - w0 * a.Lv;
    const int64_t anchor = (int64_t)w0 * a.L, rows_total = (int64_t)a.T * a.L;
    const int vk = own.mapped_offset(i, l0, a.L, a.Lv, nrows, (int)a.skd.t * 2, a.D);
    const int vv = own.mapped_offset(i, l0, a.L, a.Lv, nrows, (int)a.svd.t * 2, a.Dv);
    check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + anchor * a.skd.t,
              nrows > 0 ? mapped_bytes(anchor, rows_total, (uint32_t)a.skd.t * 2u) : 0u, vk, 0, 16, kt + i * 1024,
              lds_bytes, vk == kPadOffset);
    check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + anchor * a.svd.t,
              nrows > 0 ? mapped_bytes(anchor, rows_total, (uint32_t)a.svd.t * 2u) : 0u, vv, 0, 16, vt + i * 1024,
              lds_bytes, vv == kPadOffset);
    return;
  }
  const int voffk = own.lane_offset(i, (int)a.skd.t * 2, a.D), voffv = own.lane_offset(i, (int)a.svd.t * 2, a.Dv);
  check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + (int64_t)col0 * a.skd.t,
            nrows > 0 ? (uint32_t)nrows * (uint32_t)a.skd.t * 2u : 0u, voffk, 0, 16, kt + i * 1024, lds_bytes,
            voffk == kPadOffset);
  check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + (int64_t)col0 * a.svd.t,
            nrows > 0 ? (uint32_t)nrows * (uint32_t)a.svd.t * 2u : 0u, voffv, 0, 16, vt + i * 1024, lds_bytes,
            voffv == kPadOffset);
}

// ---------------------------------------------------------------------------------------------------------------
// forward / dQ: the ring of K+V tiles and the waves' own depth tiles.  `dq`: also dO, lse, delta reads, dq stores.
// ROWS_PER_WAVE: 32 (forward on 32x32x16) or 16 * NB.
// ---------------------------------------------------------------------------------------------------------------
template <int HD, typename Shape, bool WIDE_ADDR>
void walk_row_kernel(const KArgs& a_in, bool dq, int rows_per_wave, bool own_possible, uint32_t lds_bytes,
                     const char* kname) {
  constexpr int BN = 64, NT = 64 * Shape::W, NST = Shape::NST, DIST = Shape::DIST;
  const int BM = rows_per_wave * Shape::W;
  const bool varlen = a_in.cu != nullptr;
  const int64_t nblk = row_kernel_blocks(a_in, BM);
  typedef AsyncTileLoader<HD, BN, NT> Loader;
  for (int64_t block = 0; block < nblk; block++) {
    const RowPlace place = varlen ? row_place<true>(a_in, (int)block, BM) : row_place<false>(a_in, (int)block, BM);
    if (varlen && !place.active) continue;
    if (varlen) check_place(a_in, place);
    int b = place.b;
    const int hq = place.hq, hkv = hq / a_in.hdiv, qt = place.qt;
    const KArgs a = seq_args(a_in, b);
    const int Ld = a.L;
    const int nqt = (a.Tq + BM - 1) / BM;
    if (qt < 0 || qt >= nqt) fail("%s: query tile %d of %d", kname, qt, nqt);
    const bool own_depth = own_possible && waves_own_depth(a, Ld);
    const RowTilePlan plan = row_tile_plan(a, qt, BM, BN, Ld > 0 && !own_depth);
    const int ntiles = plan.n_seq + plan.n_dep;
    for (int tid = 0; tid < NT; tid++) {
      const int lane = tid & 63, wave = tid >> 6;
      // register operands, statistics, stores: lane owns row(s) r, 16-byte pieces of the head dim
      const int rpl = rows_per_wave == 32 ? 1 : rows_per_wave / 16;  // rows per lane
      for (int nb = 0; nb < rpl; nb++) {
        const int r = rows_per_wave == 32 ? qt * BM + wave * 32 + (lane & 31) : qt * BM + wave * rows_per_wave + 16 * nb + (lane & 15);
        if (r >= a.Tq) continue;
        const int piece = rows_per_wave == 32 ? 8 * (lane >> 5) : 8 * (lane >> 4);  // first element of this lane's pieces
        const int step = rows_per_wave == 32 ? 16 : 32;
        ctx(kname, (int)block, wave, lane, "Q / dO register rows");
        for (int e = piece; e < HD; e += step) {
          if (e < a.D) check_access("q", a.q + b * a.sq.b + hq * a.sq.h + (int64_t)r * a.sq.t + e, 16, false);
          if (dq && e < a.Dv) check_access("do", a.d_o + b * a.sdo.b + hq * a.sdo.h + (int64_t)r * a.sdo.t + e, 16, false);
          if (dq && a.own_delta && e < a.Dv) check_access("o", a.o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t + e, 16, false);
        }
        const bool stat_lane = rows_per_wave == 32 ? (lane >> 5) == 0 : (lane >> 4) == 0;
        ctx(kname, (int)block, wave, lane, "row statistics and result rows");
        if (dq) {
          check_access("lse", a.lse + ((int64_t)b * a.Tq + r) * a.Hq + hq, 4, false);
          // the row sum: read, or formed here and left for the later kernels by the first of the row's four lanes
          if (!a.own_delta || stat_lane)
            check_access("delta", a.delta + ((int64_t)b * a.Hq + hq) * (varlen ? a.delta_pitch : a.Tq) + r, 4, a.own_delta != 0);
        } else if (stat_lane) {
          check_access("lse", a.lse + ((int64_t)b * a.Tq + r) * a.Hq + hq, 4, true);
        }
        // result row: 8-byte stores, lane group g / q4 owns elements 4g + 8j (32x32) or 4q + 16j (16x16)
        const int first = rows_per_wave == 32 ? 4 * (lane >> 5) : 4 * (lane >> 4), stride = rows_per_wave == 32 ? 8 : 16;
        for (int e = first; e < HD; e += stride) {
          if (dq && e < a.D) check_access("dq", a.dq + b * a.sdq.b + hq * a.sdq.h + (int64_t)r * a.sdq.t + e, 8, true);
          if (!dq && e < a.Dv) check_access("o", a.out_o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t + e, 8, true);
        }
      }
      // ring tiles: every tile 0 .. ntiles-1 is issued once, stages in turn
      Loader ld;
      ld.init(tid);
      typename Loader::Source srcK{}, srcV{};
      if (a.has_seq && plan.n_seq > 0) {
        srcK = ld.source(a.k + b * a.sk.b + hkv * a.sk.h, a.sk.t, 0, a.T, a.D);
        srcV = ld.source(a.v + b * a.sv.b + hkv * a.sv.h, a.sv.t, 0, a.T, a.Dv);
      }
      for (int it = 0; it < ntiles; it++) {
        const int st = it % NST;
        const uint32_t kt = (uint32_t)st * 2 * BN * HD * 2;
        const bool dep = it >= plan.n_seq;
        if (Ld > 0 && it == plan.n_seq) {
          srcK = ld.source(a.kd + b * a.skd.b + hkv * a.skd.h, a.skd.t, plan.dep0, a.T * a.L, a.D);
          srcV = ld.source(a.vd + b * a.svd.b + hkv * a.svd.h, a.svd.t, plan.dep0, a.T * a.L, a.Dv);
        }
        const int row0 = ring_tile_row0(plan, it, BN);
        ctx(kname, (int)block, wave, lane, dep ? "ring depth tile" : "ring sequence tile");
        ring_tile_loads<HD, NT, WIDE_ADDR>(a, b, hkv, ld, srcK, srcV, row0, dep, a.Lv != a.L, kt, lds_bytes, "k", "v");
      }
      // the wave's own depth columns, 32 at a time through a private K tile and V tile
      if (own_depth) {
        typedef WaveTileLoader<HD> Own;
        uint32_t kt = (uint32_t)wave * (2 * 32 * HD) * 2, vt = kt + 32 * HD * 2;
        // forward on the 64-wide tiles: the first tiles go to the stage that is free while the last, masked sequence tile
        // is worked on; two sets a stage apart for two waves, else K in that stage and V in the other
        const bool early = !dq && HD <= 64 && NST == 2, two_sets = early && Shape::W <= 2;
        const bool fused = dq && depth_grads_in_dq(a, HD), beside = plan.n_full < ntiles;  // (a masked tile to travel beside)
        const int last = beside ? (ntiles - 1) % NST : 0;
        const uint32_t stage = 2 * BN * HD * 2, first = beside ? (uint32_t)fwd_first_private_set(last) : 0u;
        if (early && !two_sets) {
          kt = first * stage + (uint32_t)wave * 32 * HD * 2;
          vt = (first ^ 1) * stage + (uint32_t)wave * 32 * HD * 2;
        }
        const int rw0 = qt * BM + wave * rows_per_wave;
        if (rw0 < a.Tq) {
          const DepthSpan span = own_depth_span(a, rw0, rows_per_wave);
          const int nh = (span.c_end - span.c_beg + 31) / 32;
          Own own;
          own.init(lane);
          ctx(kname, (int)block, wave, lane, "own depth tile");
          for (int j = 0; j < nh; j++) {
            const int col0 = span.c_beg + 32 * j;
            const int nrows = imin(32, span.c_end - col0);
            // where the dQ kernel forms the depth gradients it alternates between two sets of private tiles
            const uint32_t fused_first = beside ? (uint32_t)dq_first_private_set(Shape::W, last) : 0u;
            const uint32_t set = two_sets ? (first ^ (uint32_t)(j & 1)) * stage
                                          : fused ? (fused_first ^ (uint32_t)(j & 1)) * Shape::W * 64 * HD * 2 : 0u;
            if (j == 0 && beside && (early || fused)) {  // other waves may still read the last ring tile
              const auto clear = [&](uint32_t at) { return at + 32 * HD * 2 <= last * stage || at >= (last + 1) * stage; };
              if (!clear(kt + set)) fail("%s: first private K tile in the stage of the last ring tile", kname);
              if ((two_sets || fused) && !clear(vt + set)) fail("%s: first private V tile in the stage of the last ring tile", kname);
            }
            for (int i = 0; i < Own::N; i++) {
              if (fused) {  // rows of the tile and of its gradients, from slot 0 of the first column's token or the column itself
                const int tok = col0 / a.Lv, slot = col0 - tok * a.Lv, row = i * Own::RPW + own.prow;
                const int64_t row0 = a.Lv != a.L ? (int64_t)tok * a.L : (int64_t)col0, rows_total = (int64_t)a.T * a.L;
                const int rel = row < nrows ? (a.Lv != a.L ? mapped_row(slot, row, a.L, a.Lv) : row) : -1;
                const bool pad_k = own.chunk(i) * 8 >= a.D, pad_v = own.chunk(i) * 8 >= a.Dv;
                const int vk = own.row_offset(i, rel, (int)a.skd.t * 2, pad_k), vv = own.row_offset(i, rel, (int)a.svd.t * 2, pad_v);
                check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + row0 * a.skd.t, mapped_bytes(row0, rows_total, (uint32_t)a.skd.t * 2u), vk, 0,
                          16, kt + set + i * 1024, lds_bytes, vk == kPadOffset);
                check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + row0 * a.svd.t, mapped_bytes(row0, rows_total, (uint32_t)a.svd.t * 2u), vv, 0,
                          16, vt + set + i * 1024, lds_bytes, vv == kPadOffset);
                const int gk = own.row_offset(i, rel, (int)a.sdkd.t * 2, pad_k), gv = own.row_offset(i, rel, (int)a.sdvd.t * 2, pad_v);
                ctx(kname, (int)block, wave, lane, "own depth gradients");
                if (rel >= 0 && (row0 + rel) / a.L >= a.T) fail("%s: depth column %d outside the stream", kname, col0 + row);
                if (rel >= 0 && (row0 + rel) % a.L >= a.Lv) fail("%s: gradient of slot %d of %d filled", kname, (int)((row0 + rel) % a.L), a.Lv);
                if (gk < 0 || gv < 0) fail("%s: gradient row offset past 31 bits", kname);
                if (gk != kPadOffset) check_access("dkd", a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + row0 * a.sdkd.t + gk / 2, 16, true);
                if (gv != kPadOffset) check_access("dvd", a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + row0 * a.sdvd.t + gv / 2, 16, true);
                ctx(kname, (int)block, wave, lane, "own depth tile");
                continue;
              }
              own_tile_load<HD>(a, b, hkv, own, i, col0, nrows, a.Lv != a.L, kt + set, vt + set, lds_bytes);
            }
          }
          // dQ kernel handing P and dS of its rows' visible depth columns to the depth-gradient kernel: lane (n, q4)
          // holds, per 16-column block, the columns slot_base(q4) .. +3 of rows 16*nb + n
          if (dq && a.depth_p && !depth_grads_in_dq(a, HD)) {
            const int n = lane & 15, q4 = lane >> 4;
            ctx(kname, (int)block, wave, lane, "depth scores for the depth-gradient kernel");
            for (int nb = 0; nb < rows_per_wave / 16; nb++) {
              const int r = rw0 + 16 * nb + n;
              const RowVis vis = row_visibility(a, r, Ld);
              const int t = r / a.Gf;  // slot l of row r: element l * Gf + (r - t * Gf) of token t's block
              const int64_t at = (((int64_t)b * a.Hq + hq) * (varlen ? a.delta_pitch : a.Tq) + (int64_t)t * a.Gf) * a.Lv + (r - t * a.Gf);
              for (int j = 0; j < nh; j++)
                for (int mb = 0; mb < 2; mb++)
                  for (int i = 0; i < 4; i++) {
                    const int c = span.c_beg + 32 * j + 16 * mb + slot_base(q4) + i;
                    if (c < vis.dlo || c >= vis.dhi) continue;
                    check_access("hand_p", a.depth_p + at + (int64_t)(c - vis.dlo) * a.Gf, 2, true);
                    check_access("hand_ds", a.depth_ds + at + (int64_t)(c - vis.dlo) * a.Gf, 2, true);
                  }
            }
          }
          // dQ kernel outside chunk-visible mode: the same pass forms dK and dV of the wave's own depth columns.
          // The gradient rows leave through the tile's own blocks; behind the two sets lies the block through which dS crosses.
          if (dq && depth_grads_in_dq(a, HD)) {
            if (rows_per_wave != 32) fail("%s: depth gradients need 32 rows per wave", kname);
            const uint32_t block_at = 2u * Shape::W * 64 * HD * 2 + (uint32_t)wave * 16 * HD * 2;
            if (block_at + 32 * 32 * 2 > lds_bytes || 16 * HD * 2 < 32 * 32 * 2) fail("%s: dS block past its LDS", kname);
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// row sums: o * do -> workspace
// ---------------------------------------------------------------------------------------------------------------
template <int HD>
void walk_delta(const KArgs& a_in) {
  constexpr int TPR = HD / 8, RPB = 256 / TPR;
  const int nrb = (a_in.Tq + RPB - 1) / RPB;
  const int64_t nblk = delta_kernel_blocks(a_in, RPB);
  for (int64_t block = 0; block < nblk; block++)
    for (int tid = 0; tid < 256; tid++) {
      const int bh = (int)(block / nrb), rb = (int)(block - (int64_t)bh * nrb);
      int b = bh / a_in.Hq;
      const int hq = bh % a_in.Hq;
      const KArgs a = seq_args(a_in, b);
      const int r = rb * RPB + tid / TPR, c = (tid % TPR) * 8;
      ctx("delta_kernel", (int)block, tid >> 6, tid & 63, "o, do rows and the row sum");
      if (r < a.Tq && c < a.Dv) {
        check_access("o", a.o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t + c, 16, false);
        check_access("do", a.d_o + b * a.sdo.b + hq * a.sdo.h + (int64_t)r * a.sdo.t + c, 16, false);
      }
      if (r < a.Tq && (tid % TPR) == 0)
        check_access("delta", a.delta + ((int64_t)b * a.Hq + hq) * a.delta_pitch + r, 4, true);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// dK/dV column tiles (sequence keys, and depth columns in chunk-visible mode when not done by whole chunks)
// ---------------------------------------------------------------------------------------------------------------
template <int HD>
void walk_dkv(const KArgs& a_in) {
  constexpr int NB = HD > 128 ? 1 : 2, BM = HD > 128 ? 32 : 64, MBLK = BM / 16, BN = 4 * 16 * NB, KS = HD / 32, MB = HD / 16,
                NST = 3, NP = (MBLK / 2) * NB, SP = 64;
  const uint32_t lds_bytes = 3 * 2 * BM * HD * 2 + 2 * 4 * (BM / 32) * NB * 64 * 16 + 3 * 2 * 64 * 4;
  const uint32_t stat_byte = NST * 2 * BM * HD * 2 + 2 * 4 * NP * 64 * 16;
  const bool varlen = a_in.cu != nullptr;
  const int nseg = a_in.dkv_split;
  const int64_t nblk = col_kernel_blocks(a_in, HD, BN, nseg);
  typedef AsyncTileLoader<HD, BM, 512> Loader;
  for (int64_t block = 0; block < nblk; block++) {
    const ColPlace place = varlen ? col_place<true>(a_in, (int)block, BN, nseg) : col_place<false>(a_in, (int)block, BN, nseg);
    if (varlen && !place.active) continue;
    if (varlen) check_place(a_in, place);
    int b = place.b;
    const int ct = place.ct, hkv = place.hkv, first = varlen ? a_in.cu[b] : 0;
    const KArgs a = seq_args(a_in, b);
    const ColTilePlan plan = col_tile_plan(a_in, a, ct, BN, BM, varlen, nseg);
    if (!plan.active) {
      if (!varlen && nseg == 1) fail("dkv_kernel: inactive column tile in a fixed-length launch");
      continue;
    }
    const bool dep = plan.dep;
    for (int tid = 0; tid < 512; tid++) {
      const int lane = tid & 63, n = lane & 15, q4 = lane >> 4, wave = tid >> 6, kblk = wave & 3;
      const bool role_b = wave >= 4;
      for (int nb = 0; nb < NB; nb++) {
        const int c = plan.c_first + kblk * (16 * NB) + 16 * nb + n;
        const bool valid = c < plan.ncols;
        const int64_t crow = dep ? depth_row_of(a, c) : c;
        ctx("dkv_kernel", (int)block, wave, lane, "stationary K / V rows");
        const uint16_t* src = role_b ? (dep ? a.vd + b * a.svd.b + hkv * a.svd.h : a.v + b * a.sv.b + hkv * a.sv.h)
                                     : (dep ? a.kd + b * a.skd.b + hkv * a.skd.h : a.k + b * a.sk.b + hkv * a.sk.h);
        const int64_t st = role_b ? (dep ? a.svd.t : a.sv.t) : (dep ? a.skd.t : a.sk.t);
        const char* sname = role_b ? (dep ? "vd" : "v") : (dep ? "kd" : "k");
        for (int ks = 0; ks < KS; ks++)
          if (valid && 32 * ks + 8 * q4 < (role_b ? a.Dv : a.D)) check_access(sname, src + crow * st + 32 * ks + 8 * q4, 16, false);
        if (!valid) continue;
        ctx("dkv_kernel", (int)block, wave, lane, "gradient rows");
        if (plan.nsegs > 1 && !dep) {  // a row segment: fp32 partial sums, all HD columns of the tile width
          const int64_t pitch = part_rows(a), plane = (int64_t)(varlen ? 1 : a.B) * a.Hkv * pitch * HD;
          float* pp = a.dkv_part + ((int64_t)(role_b ? 0 : 1) * nseg + plan.seg) * plane +
                      (((int64_t)b * a.Hkv + hkv) * pitch + first + c) * HD;
          for (int d = 0; d < MB; d++) check_access("part", pp + 16 * d + 4 * q4, 16, true);
          continue;
        }
        const char* oname = role_b ? (dep ? "dkd" : "dk") : (dep ? "dvd" : "dv");
        uint16_t* outp = !role_b ? (dep ? a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + crow * a.sdvd.t
                                        : a.dv + b * a.sdv.b + hkv * a.sdv.h + crow * a.sdv.t)
                                 : (dep ? a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + crow * a.sdkd.t
                                        : a.dk + b * a.sdk.b + hkv * a.sdk.h + crow * a.sdk.t);
        for (int d = 0; d < MB; d++)
          if (16 * d + 4 * q4 < (role_b ? a.D : a.Dv)) check_access(oname, outp + 16 * d + 4 * q4, 8, true);
      }
      // the streamed query tiles: per query head, from the top tile down, stages in turn
      Loader ld;
      ld.init(tid);
      const uint32_t q_row_bytes = (uint32_t)a.sq.t * 2u, do_row_bytes = (uint32_t)a.sdo.t * 2u;
      const int voff_q = ld.lane_offset((int)q_row_bytes, a.D), voff_do = ld.lane_offset((int)do_row_bytes, a.Dv);
      const int voff_stat = wave == 0 ? lane * a.Hq * 4 : lane * 4;
      const uint32_t stat_row_bytes = wave == 0 ? (uint32_t)a.Hq * 4u : 4u;
      int ld_st = 0;
      for (int gh = 0; gh < a.hdiv; gh++) {
        const int hq = hkv * a.hdiv + gh;
        int f_q0 = (plan.qt0 + plan.nqt - 1) * BM;
        for (int t = 0; t < plan.nqt; t++, f_q0 -= BM) {
          if (f_q0 < 0) fail("dkv_kernel: query tile row %d", f_q0);
          const uint32_t rows = (uint32_t)query_tile_rows(a, f_q0, BM);
          if (rows == 0) fail("dkv_kernel: empty query tile at row %d (Tq %d)", f_q0, a.Tq);
          const uint16_t* qp = a.q + b * a.sq.b + hq * a.sq.h + (int64_t)f_q0 * a.sq.t;
          const uint16_t* dop = a.d_o + b * a.sdo.b + hq * a.sdo.h + (int64_t)f_q0 * a.sdo.t;
          const uint32_t lds_q = (uint32_t)(ld_st * 2 * BM * HD + wave * 512) * 2;
          ctx("dkv_kernel", (int)block, wave, lane, "query tile (Q, dO)");
          for (int k = 0; k < Loader::N; k++) {
            check_dma("q", qp, rows * q_row_bytes, voff_q, k * 8 * Loader::RPW * (int)q_row_bytes, 16, lds_q + k * 8 * 1024,
                      lds_bytes, ld.pads(a.D));
            check_dma("do", dop, rows * do_row_bytes, voff_do, k * 8 * Loader::RPW * (int)do_row_bytes, 16,
                      lds_q + BM * HD * 2 + k * 8 * 1024, lds_bytes, ld.pads(a.Dv));
          }
          if (wave < 2) {
            ctx("dkv_kernel", (int)block, wave, lane, wave == 0 ? "query tile lse" : "query tile row sums");
            const float* sp = wave == 0 ? a.lse + ((int64_t)b * a.Tq + f_q0) * a.Hq + hq
                                        : a.delta + ((int64_t)b * a.Hq + hq) * (varlen ? a.delta_pitch : a.Tq) + f_q0;
            check_dma(wave == 0 ? "lse" : "delta", sp, (rows - 1) * stat_row_bytes + 4u, voff_stat, 0, 4,
                      stat_byte + (uint32_t)(ld_st * 2 * SP + (wave == 0 ? 0 : SP)) * 4, lds_bytes, false);
          }
          ld_st = (ld_st + 1) % NST;
        }
      }
    }
  }
}

// dkv_flat_kernel: four waves, a wave's 32 columns with K and V in registers, query tiles of 32 rows; or (RW = 4) the
// waves on the same 32 columns, 32 rows each of a query tile of 128
// OWN_DELTA: beside the dQ workgroups of a launch (bwd_short_kernel): the waves read o instead of the row sums
template <int HD, int RW, bool OWN_DELTA = false>
void walk_dkv_flat(const KArgs& a_in) {
  constexpr int NB = 2, BM = 32 * RW, BN = 4 / RW * 16 * NB, KS = HD / 32, MB = HD / 16, NST = RW == 1 ? 3 : 2, SP = RW == 1 ? 64 : BM;
  const uint32_t lds_bytes = NST * 2 * BM * HD * 2 + NST * 2 * SP * 4 + (OWN_DELTA ? 4 * 32 * 4 : 0);
  const int nseg = a_in.dkv_split;
  if (RW > 1 && nseg > 1) fail("dkv_flat_kernel: row waves and segments");
  const uint32_t stat_byte = NST * 2 * BM * HD * 2;
  const bool varlen = a_in.cu != nullptr;
  const int64_t nblk = dkv_flat_blocks(a_in, BN, nseg);
  typedef AsyncTileLoader<HD, BM, 256> Loader;
  for (int64_t block = 0; block < nblk; block++) {
    const ColPlace place = varlen ? col_place<true>(a_in, (int)block, BN, nseg) : col_place<false>(a_in, (int)block, BN, nseg);
    if (varlen && !place.active) continue;
    if (varlen) check_place(a_in, place);
    int b = place.b;
    const int ct = place.ct, hkv = place.hkv, first = varlen ? a_in.cu[b] : 0;
    const KArgs a = seq_args(a_in, b);
    const ColTilePlan plan = col_tile_plan(a_in, a, ct, BN, BM, varlen, nseg);
    if (!plan.active) {
      if (!varlen && nseg == 1) fail("dkv_flat_kernel: inactive column tile in a fixed-length launch");
      continue;
    }
    if (plan.dep) fail("dkv_flat_kernel: column tile %d is not a sequence tile", ct);
    for (int tid = 0; tid < 256; tid++) {
      const int lane = tid & 63, n = lane & 15, q4 = lane >> 4, wave = tid >> 6;
      for (int nb = 0; nb < NB; nb++) {
        const int c = plan.c_first + (RW == 1 ? wave : 0) * (16 * NB) + 16 * nb + n;
        if (c >= a.T) continue;
        ctx("dkv_flat_kernel", (int)block, wave, lane, "stationary K and V rows");
        for (int ks = 0; ks < KS; ks++) {
          if (32 * ks + 8 * q4 < a.D) check_access("k", a.k + b * a.sk.b + hkv * a.sk.h + 8 * q4 + (int64_t)c * a.sk.t + 32 * ks, 16, false);
          if (32 * ks + 8 * q4 < a.Dv) check_access("v", a.v + b * a.sv.b + hkv * a.sv.h + 8 * q4 + (int64_t)c * a.sv.t + 32 * ks, 16, false);
        }
        ctx("dkv_flat_kernel", (int)block, wave, lane, "gradient rows");
        uint16_t* dkp = a.dk + b * a.sdk.b + hkv * a.sdk.h + (int64_t)c * a.sdk.t + 4 * q4;
        uint16_t* dvp = a.dv + b * a.sdv.b + hkv * a.sdv.h + (int64_t)c * a.sdv.t + 4 * q4;
        if (plan.nsegs > 1) {
          const int64_t pitch = part_rows(a), plane = (int64_t)(varlen ? 1 : a.B) * a.Hkv * pitch * HD;
          float* kp = a.dkv_part + plan.seg * plane + (((int64_t)b * a.Hkv + hkv) * pitch + first + c) * HD + 4 * q4;
          for (int d = 0; d < MB; d++) {
            check_access("part", kp + 16 * d, 16, true);
            check_access("part", kp + nseg * plane + 16 * d, 16, true);
          }
          continue;
        }
        const int64_t slot = (int64_t)c * a.L + a.Lv;  // the layer's own, joined where the launch has been asked to
        if (a.own_slot && RW == 1 && nseg == 1) fail("dkv_flat_kernel: the long launches' kernel does not add an own slot");
        for (int d = 0; d < MB; d++) {
          if (RW > 1 && d / (MB / 2) != (wave & 1)) continue;  // waves 0, 1 write dk, waves 2, 3 dv, half the blocks each
          if (a.own_slot && (RW == 1 || wave < 2) && 16 * d + 4 * q4 < a.D)
            check_access("dkd", a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + slot * a.sdkd.t + 4 * q4 + 16 * d, 8, false);
          if (a.own_slot && (RW == 1 || wave >= 2) && 16 * d + 4 * q4 < a.Dv)
            check_access("dvd", a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + slot * a.sdvd.t + 4 * q4 + 16 * d, 8, false);
          if ((RW == 1 || wave < 2) && 16 * d + 4 * q4 < a.D) check_access("dk", dkp + 16 * d, 8, true);
          if ((RW == 1 || wave >= 2) && 16 * d + 4 * q4 < a.Dv) check_access("dv", dvp + 16 * d, 8, true);
        }
      }
      Loader ld;
      ld.init(tid);
      const bool st_lse = OWN_DELTA || (wave & 1) == 0;
      const char* stb = st_lse ? (const char*)(a.lse + (int64_t)b * a.Tq * a.Hq + hkv) : (const char*)(a.delta + ((int64_t)b * a.Hq + hkv) * (varlen ? a.delta_pitch : a.Tq));
      const uint32_t st_row = st_lse ? (uint32_t)a.Hq * 4u : 4u;
      int ld_st = 0;
      for (int it = 0; it < plan.nqt; it++) {
        const int f_q0 = (plan.qt0 + plan.nqt - 1 - it) * BM;
        if (f_q0 < 0) fail("dkv_flat_kernel: query tile row %d", f_q0);
        const uint32_t Qt = (uint32_t)(ld_st * 2 * BM * HD) * 2;
        ctx("dkv_flat_kernel", (int)block, wave, lane, "query tile (Q, dO)");
        for (int i = 0; i < Loader::N; i++) {
          check_dma("q", a.q + b * a.sq.b + hkv * a.sq.h + (int64_t)f_q0 * a.sq.t, Loader::anchored_bytes(a.sq.t, f_q0, a.Tq),
                    ld.lane_offset((int)a.sq.t * 2, a.D), Loader::rows_before(i) * (int)a.sq.t * 2, 16,
                    Qt + (uint32_t)ld.lds_elems(i) * 2, lds_bytes, ld.pads(a.D));
          check_dma("do", a.d_o + b * a.sdo.b + hkv * a.sdo.h + (int64_t)f_q0 * a.sdo.t, Loader::anchored_bytes(a.sdo.t, f_q0, a.Tq),
                    ld.lane_offset((int)a.sdo.t * 2, a.Dv), Loader::rows_before(i) * (int)a.sdo.t * 2, 16,
                    Qt + (uint32_t)(BM * HD + ld.lds_elems(i)) * 2, lds_bytes, ld.pads(a.Dv));
        }
        const int rows = imax(imin(a.Tq - f_q0, BM), 0), st_first = RW == 1 ? 0 : (wave >> 1) * 64;
        if (rows == 0) fail("dkv_flat_kernel: empty query tile at row %d (Tq %d)", f_q0, a.Tq);
        if (OWN_DELTA) {  // two lanes a row, four pieces each; the sums lie behind the statistics
          ctx("bwd_short_kernel", (int)block, wave, lane, "pieces of o");
          const int r = imin(f_q0 + (RW == 1 ? 0 : wave) * 32 + (lane >> 1), a.Tq - 1);
          for (int c = 0; c < 4; c++) {
            const int chunk = 2 * (lane & 1) + (c >> 1) + 4 * (c & 1);
            check_access("o", a.o + b * a.so.b + hkv * a.so.h + (int64_t)r * a.so.t + (chunk * 8 < a.Dv ? chunk * 8 : 0), 16, false);
          }
          if (stat_byte + (uint32_t)(NST * 2 * SP + wave * 32 + (lane >> 1) + 1) * 4 > lds_bytes) fail("row sums past the LDS allocation");
        }
        ctx("dkv_flat_kernel", (int)block, wave, lane, st_lse ? "query tile lse" : "query tile row sums");
        check_dma(st_lse ? "lse" : "delta", stb + (int64_t)f_q0 * st_row, (uint32_t)(rows - 1) * st_row + 4u,
                  (st_first + lane) * (int)st_row, 0, 4, stat_byte + (uint32_t)(ld_st * 2 * SP + (st_lse ? 0 : SP) + st_first) * 4,
                  lds_bytes, false);
        ld_st = (ld_st + 1) % NST;
      }
    }
  }
}

// the partial sums of the row segments -> dk, dv
template <int HD>
void walk_reduce(const KArgs& a_in, int BN, int BM) {
  constexpr int TPR = HD / 8, RPB = 256 / TPR;
  const int BHk = a_in.B * a_in.Hkv;
  const int64_t nblk = ((int64_t)a_in.T + RPB - 1) / RPB * BHk;
  for (int64_t block = 0; block < nblk; block++)
    for (int tid = 0; tid < 256; tid++) {
      const int bh = (int)(block % BHk), hkv = bh % a_in.Hkv, sub = tid % TPR, c = (int)(block / BHk) * RPB + tid / TPR;
      int b = bh / a_in.Hkv;
      const int first = a_in.cu ? a_in.cu[b] : 0;
      const KArgs a = seq_args(a_in, b);
      if (c >= a.T) continue;
      const int row0 = a.causal ? c / BN * BN * a.Gf : 0;
      const int nsegs = tile_segments(a, (a.Tq + BM - 1) / BM - row0 / BM, a.dkv_split);
      if (nsegs == 1) continue;
      const int64_t pitch = part_rows(a), plane = (int64_t)(a.cu ? 1 : a.B) * a.Hkv * pitch * HD;
      const int64_t row = ((int64_t)b * a.Hkv + hkv) * pitch + first + c;
      ctx("dkv_reduce_kernel", (int)block, tid >> 6, tid & 63, "partial sums and dk, dv rows");
      for (int which = 0; which < 2; which++) {
        const float* src = a.dkv_part + (int64_t)which * a.dkv_split * plane + row * HD + 8 * sub;
        for (int sg = 0; sg < nsegs; sg++) read_partials(src + sg * plane, 8);
        uint16_t* outp = which == 0 ? a.dk + b * a.sdk.b + hkv * a.sdk.h + (int64_t)c * a.sdk.t
                                    : a.dv + b * a.sdv.b + hkv * a.sdv.h + (int64_t)c * a.sdv.t;
        if (a.own_slot && 8 * sub < (which == 0 ? a.D : a.Dv)) {
          const int64_t slot = (int64_t)c * a.L + a.Lv;
          if (which == 0)
            check_access("dkd", a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + slot * a.sdkd.t + 8 * sub, 16, false);
          else
            check_access("dvd", a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + slot * a.sdvd.t + 8 * sub, 16, false);
        }
        if (8 * sub < (which == 0 ? a.D : a.Dv)) check_access(which == 0 ? "dk" : "dv", outp + 8 * sub, 16, true);
      }
    }
}

// chunk-visible depth columns by whole chunks (tile widths up to 128)
template <int HD>
void walk_chunk_depth(const KArgs& a_in) {
  constexpr int BM = 64, CH = HD / 8, RPW = 64 / CH, NPASS = 32 / RPW;
  const uint32_t lds_bytes = (2 * 64 + 4 * 32) * HD * 2 + 2 * 64 * 4;
  const bool varlen = a_in.cu != nullptr;
  const int BHk = a_in.B * a_in.Hkv;
  const int64_t nx = (((int64_t)a_in.T + a_in.Cb - 1) / a_in.Cb) * BHk;
  typedef AsyncTileLoader<HD, BM, 256> Loader;
  for (int64_t block = 0; block < nx; block++) {
    const int bh = (int)(block % BHk), chunk = (int)(block / BHk);
    int b = bh / a_in.Hkv;
    const int hkv = bh % a_in.Hkv;
    const KArgs a = seq_args(a_in, b);
    const int t0 = chunk * a.Cb;
    if (t0 >= a.T) continue;
    const int t1 = imin(a.T, t0 + a.Cb), r0 = t0 * a.Gf, r_end = t1 * a.Gf, c_end = t1 * a.Lv;
    if (r_end - r0 > BM) fail("chunk_depth_kernel: a chunk of %d query rows", r_end - r0);
    for (int tid = 0; tid < 256; tid++) {
      const int lane = tid & 63, wave = tid >> 6;
      Loader ld;
      ld.init(tid);
      ctx("chunk_depth_kernel", (int)block, wave, lane, "the chunk's Q, dO, lse, row sums");
      for (int i = 0; i < Loader::N; i++) {
        check_dma("q", a.q + b * a.sq.b + hkv * a.sq.h + (int64_t)r0 * a.sq.t, Loader::anchored_bytes(a.sq.t, r0, r_end),
                  ld.lane_offset((int)a.sq.t * 2, a.D), Loader::rows_before(i) * (int)a.sq.t * 2, 16, (uint32_t)ld.lds_elems(i) * 2,
                  lds_bytes, ld.pads(a.D));
        check_dma("do", a.d_o + b * a.sdo.b + hkv * a.sdo.h + (int64_t)r0 * a.sdo.t, Loader::anchored_bytes(a.sdo.t, r0, r_end),
                  ld.lane_offset((int)a.sdo.t * 2, a.Dv), Loader::rows_before(i) * (int)a.sdo.t * 2, 16,
                  (uint32_t)(BM * HD + ld.lds_elems(i)) * 2, lds_bytes, ld.pads(a.Dv));
      }
      if (tid < BM && r0 + tid < r_end) {
        check_access("lse", a.lse + ((int64_t)b * a.Tq + r0 + tid) * a.Hq + hkv, 4, false);
        check_access("delta", a.delta + ((int64_t)b * a.Hq + hkv) * (varlen ? a.delta_pitch : a.Tq) + r0 + tid, 4, false);
      }
      const int prow = lane / CH, pch = lane % CH;
      const uint32_t wt = (uint32_t)(2 * BM * HD + wave * 32 * HD) * 2;
      WaveTileLoader<HD> own;
      own.init(lane);
      for (int cb = t0 * a.Lv + wave * 32; cb < c_end; cb += 128) {
        const int nrows = imin(32, c_end - cb);
        for (int i = 0; i < NPASS; i++) {
          const int row = i * RPW + prow, lch = pch ^ Tile<HD>::swz(row);
          const bool pad_k = !(lch * 8 < a.D), pad_v = !(lch * 8 < a.Dv);
          ctx("chunk_depth_kernel", (int)block, wave, lane, "depth K / V rows");
          if (a.Lv != a.L) {
            const int w0 = cb / a.Lv, l0 = cb - w0 * a.Lv;
            const int64_t anchor = (int64_t)w0 * a.L, rows_total = (int64_t)a.T * a.L;
            const int vk = own.mapped_offset(i, l0, a.L, a.Lv, nrows, (int)a.skd.t * 2, a.D);
            const int vv = own.mapped_offset(i, l0, a.L, a.Lv, nrows, (int)a.svd.t * 2, a.Dv);
            check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + anchor * a.skd.t,
                      mapped_bytes(anchor, rows_total, (uint32_t)a.skd.t * 2u), vk, 0, 16, wt + i * 1024, lds_bytes, vk == kPadOffset);
            check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + anchor * a.svd.t,
                      mapped_bytes(anchor, rows_total, (uint32_t)a.svd.t * 2u), vv, 0, 16, wt + i * 1024, lds_bytes, vv == kPadOffset);
          } else {
            const int vk = own.lane_offset(i, (int)a.skd.t * 2, a.D), vv = own.lane_offset(i, (int)a.svd.t * 2, a.Dv);
            check_dma("kd", a.kd + b * a.skd.b + hkv * a.skd.h + (int64_t)cb * a.skd.t, (uint32_t)nrows * (uint32_t)a.skd.t * 2u,
                      vk, 0, 16, wt + i * 1024, lds_bytes, pad_k);
            check_dma("vd", a.vd + b * a.svd.b + hkv * a.svd.h + (int64_t)cb * a.svd.t, (uint32_t)nrows * (uint32_t)a.svd.t * 2u,
                      vv, 0, 16, wt + i * 1024, lds_bytes, pad_v);
          }
          ctx("chunk_depth_kernel", (int)block, wave, lane, "depth gradient rows");
          if (cb + row < c_end) {
            const int64_t prow_t = depth_row_of(a, cb + row);
            if (!pad_k) check_access("dkd", a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + prow_t * a.sdkd.t + lch * 8, 16, true);
            if (!pad_v) check_access("dvd", a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + prow_t * a.sdvd.t + lch * 8, 16, true);
          }
        }
      }
    }
  }
}

// the gradient rows of the slots without data of a partially filled stream (launched where the kernels that form
// the depth gradients only visit the slots that hold data)
template <int HD>
void walk_zero_unfilled(const KArgs& a) {
  constexpr int TPR = HD / 8;
  const int64_t rows = a.cu ? (int64_t)(a.delta_pitch / a.Gf) * a.L : (int64_t)a.T * a.L;
  const int batches = a.cu ? 1 : a.B;
  const int64_t nthreads = rows * batches * a.Hkv * TPR;
  for (int64_t gid = 0; gid < (nthreads + 255) / 256 * 256; gid++) {
    const int sub = (int)(gid % TPR);
    int64_t rest = gid / TPR;
    const int h = (int)(rest % a.Hkv);
    rest /= a.Hkv;
    const int64_t row = rest % rows, b = rest / rows;
    if (b >= batches || (int)(row % a.L) < a.Lv) continue;
    ctx("zero_unfilled_slots_kernel", (int)(gid / 256), (int)(gid % 256) >> 6, (int)(gid & 63), "gradient rows of empty slots");
    if (8 * sub < a.D) check_access("dkd", a.dkd + b * a.sdkd.b + h * a.sdkd.h + row * a.sdkd.t + 8 * sub, 16, true);
    if (8 * sub < a.Dv) check_access("dvd", a.dvd + b * a.sdvd.b + h * a.sdvd.h + row * a.sdvd.t + 8 * sub, 16, true);
  }
}

// depth columns outside chunk-visible mode: one column per HD/8 lanes
template <int HD>
void walk_depth_cols(const KArgs& launch) {
  const KArgs a_in = packed_as_one(launch);
  constexpr int LPC = HD / 8, CPW = 64 / LPC, CPB = 4 * CPW;
  const int BHk = a_in.B * a_in.Hkv;
  const int64_t nx = (((int64_t)a_in.T * a_in.L + CPB - 1) / CPB) * BHk;
  for (int64_t block = 0; block < nx; block++)
    for (int tid = 0; tid < 256; tid++) {
      const int lane = tid & 63, wave = tid >> 6, sub = lane % LPC;
      const int bh = (int)(block % BHk);
      int b = bh / a_in.Hkv;
      const int hkv = bh % a_in.Hkv;
      const KArgs a = seq_args(a_in, b);
      const int64_t c = (int64_t)(block / BHk) * CPB + wave * CPW + lane / LPC;
      if (c >= (int64_t)a.T * a.L) continue;
      const int w = (int)(c / a.L), slot = (int)(c - (int64_t)w * a.L);
      const bool in_k = 8 * sub < a.D, in_v = 8 * sub < a.Dv;
      ctx("depth_cols_kernel", (int)block, wave, lane, "depth column");
      uint16_t* dk_out = a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + c * a.sdkd.t + 8 * sub;
      uint16_t* dv_out = a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + c * a.sdvd.t + 8 * sub;
      if (slot >= a.Lv) {
        if (!a.keep_slots) {
          if (in_k) check_access("dkd", dk_out, 16, true);
          if (in_v) check_access("dvd", dv_out, 16, true);
        }
        continue;
      }
      const bool handed = a.depth_p != nullptr;  // depth_cols_handed_kernel: P and dS from the dQ kernel, no kd, vd, statistics
      if (!handed && in_k) check_access("kd", a.kd + b * a.skd.b + hkv * a.skd.h + c * a.skd.t + 8 * sub, 16, false);
      if (!handed && in_v) check_access("vd", a.vd + b * a.svd.b + hkv * a.svd.h + c * a.svd.t + 8 * sub, 16, false);
      for (int gq = 0; gq < a.Gf; gq++) {
        const int64_t r = (int64_t)w * a.Gf + gq;
        if (in_k) check_access("q", a.q + b * a.sq.b + hkv * a.sq.h + 8 * sub + r * a.sq.t, 16, false);
        if (in_v) check_access("do", a.d_o + b * a.sdo.b + hkv * a.sdo.h + 8 * sub + r * a.sdo.t, 16, false);
        if (handed) {
          const int64_t at = (((int64_t)b * a.Hq + hkv) * a.delta_pitch + (int64_t)w * a.Gf) * a.Lv + (int64_t)slot * a.Gf + gq;
          check_access("hand_p", a.depth_p + at, 2, false);
          check_access("hand_ds", a.depth_ds + at, 2, false);
          continue;
        }
        check_access("lse", a.lse + ((int64_t)b * a.Tq + r) * a.Hq + hkv, 4, false);
        check_access("delta", a.delta + ((int64_t)b * a.Hq + hkv) * a.delta_pitch + r, 4, false);
      }
      if (in_k) check_access("dkd", dk_out, 16, true);
      if (in_v) check_access("dvd", dv_out, 16, true);
    }
}

// the same organised by token (query groups of up to four rows with the depth scores handed over by the dQ kernel)
template <int HD>
void walk_depth_tokens(const KArgs& launch) {
  const KArgs a_in = packed_as_one(launch);
  constexpr int LPT = HD / 8, TPW = 64 / LPT, TPB = 4 * TPW;
  const int BHk = a_in.B * a_in.Hkv;
  const int64_t nt = (((int64_t)a_in.T + TPB - 1) / TPB) * BHk;
  for (int64_t block = 0; block < nt; block++)
    for (int tid = 0; tid < 256; tid++) {
      const int lane = tid & 63, wave = tid >> 6, sub = lane % LPT;
      const int bh = (int)(block % BHk);
      int b = bh / a_in.Hkv;
      const int hkv = bh % a_in.Hkv;
      const KArgs a = seq_args(a_in, b);
      const int w = (int)(block / BHk) * TPB + wave * TPW + lane / LPT;
      if (w >= a.T) continue;
      const bool in_k = 8 * sub < a.D, in_v = 8 * sub < a.Dv;
      ctx("depth_token_handed_kernel", (int)block, wave, lane, "token");
      for (int g = 0; g < a.Gf; g++) {
        const int64_t r = (int64_t)w * a.Gf + g;
        if (in_k) check_access("q", a.q + b * a.sq.b + hkv * a.sq.h + 8 * sub + r * a.sq.t, 16, false);
        if (in_v) check_access("do", a.d_o + b * a.sdo.b + hkv * a.sdo.h + 8 * sub + r * a.sdo.t, 16, false);
      }
      const int64_t blk = (((int64_t)b * a.Hq + hkv) * a.delta_pitch + (int64_t)w * a.Gf) * a.Lv;
      for (int slot = 0; slot < a.L; slot++) {
        if (slot >= a.Lv && a.keep_slots) continue;
        if (slot < a.Lv)
          for (int g = 0; g < a.Gf; g++) {
            check_access("hand_p", a.depth_p + blk + (int64_t)slot * a.Gf + g, 2, false);
            check_access("hand_ds", a.depth_ds + blk + (int64_t)slot * a.Gf + g, 2, false);
          }
        const int64_t c = (int64_t)w * a.L + slot;
        if (in_k) check_access("dkd", a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + c * a.sdkd.t + 8 * sub, 16, true);
        if (in_v) check_access("dvd", a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + c * a.sdvd.t + 8 * sub, 16, true);
      }
    }
}

// The order of a packed batch's launches on the 64-wide tiles: which grid each takes, and the query tiles that the dK/dV
// workgroups of the fullest XCD (block % 8) and of the fullest place of one (32 compute units in turn) have, over the mean.
void packed_launch_order(const KArgs& a) {
  constexpr int BN = 128, BM = 32;
  const int nseg = a.dkv_split;
  std::vector<double> xcd(8, 0.), place(256, 0.);
  double all = 0.;
  for (int64_t block = 0; block < dkv_flat_blocks(a, BN, nseg); block++) {
    const ColPlace p = col_place<true>(a, (int)block, BN, nseg);
    if (!p.active) continue;
    int b = p.b;
    const KArgs one = seq_args(a, b);
    const ColTilePlan plan = col_tile_plan(a, one, p.ct, BN, BM, true, nseg);
    if (!plan.active) continue;
    xcd[block % 8] += plan.nqt;
    place[block % 256] += plan.nqt;
    all += plan.nqt;
  }
  const auto name = [&](int64_t grid) { return packed_order(a, grid) ? "list" : "grid"; };
  printf("rows %s columns %s xcd %.2f place %.2f\n", name(longest_row_grid(a, 128)), name(longest_col_grid(a, BN, nseg)),
         8 * *std::max_element(xcd.begin(), xcd.end()) / all, 256 * *std::max_element(place.begin(), place.end()) / all);
}

void reset_writes(const char* name) {
  Region& r = region(name);
  std::fill(r.writes.begin(), r.writes.end(), 0);
}
// every element of the rows that exist must have been written exactly once (elements of a row past the head dim do
// not exist: the regions are dense [rows, heads, D])
void require_full(const char* name) {
  Region& r = region(name);
  if (!r.track) return;
  for (size_t i = 0; i < r.writes.size(); i++)
    if (r.writes[i] != 1) fail("%s unit %zu written %d times after the launch", name, i, (int)r.writes[i]);
}
// the depth gradients: rows of slots that hold data once, the others once or (keep_slots) not at all
void require_depth_rows(const char* name, const KArgs& a, int dim) {
  Region& r = region(name);
  if (!r.track) return;
  for (size_t i = 0; i < r.writes.size(); i++) {
    const int want = a.keep_slots && (int)(i / ((size_t)a.Hkv * dim) % a.L) >= a.Lv ? 0 : 1;
    if (r.writes[i] != want) fail("%s unit %zu written %d times after the launch, not %d", name, i, (int)r.writes[i], want);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// fp32 matrix kernels: 16-row (or 16-column) tiles, operands straight from global memory
// ---------------------------------------------------------------------------------------------------------------
template <int HD>
void walk_fp32(const KArgs& a_in) {
  constexpr int KS = HD / 16, H4 = HD / 64, W = 8, CW = HD <= 64 ? 8 : 4, PART = 16 * (HD + 4);
  const bool full = a_in.D == HD && a_in.Dv == HD;
  auto f = [](const uint16_t* p) { return (const float*)p; };
  // the 16-byte pieces of one row as a score operand (lane group q) and as a second product's operand (lane n)
  auto score = [&](const char* name, const float* row, int q, int d) {
    for (int s = 0; s < KS; s++) check_access(name, row + (full || 16 * s + 4 * q < d ? 16 * s + 4 * q : 0), 16, false);
  };
  auto sum = [&](const char* name, const float* row, int n, int d) {
    for (int h = 0; h < H4; h++) check_access(name, row + (full || 64 * h + 4 * n < d ? 64 * h + 4 * n : 0), 16, false);
  };
  auto partial = [&](int first, uint32_t lds_bytes) {  // a wave's accumulators on their way to LDS
    for (int n = 0; n < 16; n++)
      if ((uint32_t)(first + n * (HD + 4) + HD) * 4 > lds_bytes) fail("partial results past the LDS allocation");
  };
  for (int which = 0; which < 3; which++) {  // forward, row sums alone, dQ
    const char* kname = which == 0 ? "fp32_fwd_kernel" : which == 1 ? "fp32_delta_kernel" : "fp32_dq_kernel";
    const uint32_t lds_bytes = W * PART * 4 + (which == 0 ? W * 32 * 4 : 0);
    const int64_t nblk = (int64_t)((a_in.Tq + 15) / 16) * a_in.B * a_in.Hq;
    const int BH = a_in.B * a_in.Hq;
    for (int64_t block = 0; block < nblk; block++) {
      int b = (int)(block % BH) / a_in.Hq;
      const int hq = (int)(block % BH) % a_in.Hq, hkv = hq / a_in.hdiv;
      KArgs a = a_in;
      enter_sequence(a, b, 2);
      const int qt = which == 1 ? (int)(block / BH) : query_tile_of((int)block, BH, 16, a_in.Tq);
      if (which != 1 && qt * 16 >= a.Tq) continue;
      if (a.Tq == 0) continue;
      const RowTilePlan plan = row_tile_plan(a, qt, 16, 16, a.L > 0);
      const int nblocks = which == 1 ? 0 : plan.n_seq + plan.n_dep;
      for (int tid = 0; tid < (which == 1 ? 64 : 64 * W); tid++) {
        const int lane = tid & 63, n = lane & 15, q = lane >> 4, wave = tid >> 6;
        const int r = qt * 16 + n, rc = imin(r, a.Tq - 1);
        ctx(kname, (int)block, wave, lane, "rows of q, do, o and their statistics");
        if (which != 1) score("q", f(a.q) + b * a.sq.b + hq * a.sq.h + (int64_t)rc * a.sq.t, q, a.D);
        if (which != 0) {
          score("do", f(a.d_o) + b * a.sdo.b + hq * a.sdo.h + (int64_t)rc * a.sdo.t, q, a.Dv);
          score("o", f(a.o) + b * a.so.b + hq * a.so.h + (int64_t)rc * a.so.t, q, a.Dv);
        }
        if (which == 2) check_access("lse", a.lse + ((int64_t)b * a.Tq + rc) * a.Hq + hq, 4, false);
        if (which != 0 && wave == 0 && q == 0 && r < a.Tq)
          check_access("delta", a.delta + ((int64_t)b * a.Hq + hq) * a.delta_pitch + r, 4, true);
        for (int blk = wave; blk < nblocks; blk += W) {
          const bool dep = blk >= plan.n_seq;
          const int col0 = dep ? plan.dep0 + (blk - plan.n_seq) * 16 : blk * 16, ncols = dep ? a.T * a.Lv : a.T;
          auto row_of = [&](int c) { return dep ? depth_row_of(a, imin(c, ncols - 1)) : (int64_t)imin(c, ncols - 1); };
          const char *kn = dep ? "kd" : "k", *vn = dep ? "vd" : "v";
          const float* kp = dep ? f(a.kd) + b * a.skd.b + hkv * a.skd.h : f(a.k) + b * a.sk.b + hkv * a.sk.h;
          const float* vp = dep ? f(a.vd) + b * a.svd.b + hkv * a.svd.h : f(a.v) + b * a.sv.b + hkv * a.sv.h;
          const int64_t ks = dep ? a.skd.t : a.sk.t, vs = dep ? a.svd.t : a.sv.t;
          ctx(kname, (int)block, wave, lane, dep ? "depth columns" : "sequence columns");
          if (dep && row_of(col0 + n) % a.L >= a.Lv) fail("depth row of a slot without data");
          score(kn, kp + row_of(col0 + n) * ks, q, a.D);
          if (which == 2) score(vn, vp + row_of(col0 + n) * vs, q, a.Dv);
          for (int i = 0; i < 4; i++) {
            if (which == 0)
              sum(vn, vp + row_of(col0 + 4 * q + i) * vs, n, a.Dv);
            else
              sum(kn, kp + row_of(col0 + 4 * q + i) * ks, n, a.D);
          }
        }
        if (which == 1) continue;
        if (lane == 0) partial(wave * PART, W * PART * 4);
        if (which == 0 && (uint32_t)(W * PART + (wave * 16 + n) * 2 + 2) * 4 > lds_bytes) fail("row statistics past the LDS allocation");
        const int row = tid / (HD / 4), d = (tid % (HD / 4)) * 4;
        ctx(kname, (int)block, wave, lane, "result row");
        if (tid >= 16 * HD / 4 || qt * 16 + row >= a.Tq) continue;
        const int64_t ro = qt * 16 + row;
        if (which == 0 && d < a.Dv) check_access("o", f(a.out_o) + b * a.so.b + hq * a.so.h + ro * a.so.t + d, 16, true);
        if (which == 0 && d == 0) check_access("lse", a.lse + ((int64_t)b * a.Tq + ro) * a.Hq + hq, 4, true);
        if (which == 2 && d < a.D) check_access("dq", f(a.dq) + b * a.sdq.b + hq * a.sdq.h + ro * a.sdq.t + d, 16, true);
      }
    }
    if (which == 0) {
      require_full("o");
      require_full("lse");
    } else {
      require_full("delta");
      if (which == 1) reset_writes("delta");
    }
    if (which == 2) require_full("dq");
  }
  // dK/dV: as a launch of its own, and beside the dQ workgroups, where it reads o instead of the row sums
  const bool one_launch = HD == 64 && fp32_one_launch(a_in);
  if (one_launch) printf("fp32_bwd_kernel ");
  for (int own_delta = 0; own_delta <= (one_launch ? 1 : 0); own_delta++) {
    for (const char* name : {"dk", "dv", "dkd", "dvd"}) reset_writes(name);
    const int BHk = a_in.B * a_in.Hkv, n_seq_tiles = a_in.has_seq ? (a_in.T + 15) / 16 : 0;
    const int64_t ndep = ((int64_t)a_in.T * a_in.Lv + 16 * CW - 1) / (16 * CW), nblk = (n_seq_tiles + ndep) * BHk;
    for (int64_t block = 0; block < nblk; block++) {
      const int hkv = (int)(block % BHk) % a_in.Hkv, tile = (int)(block / BHk);
      int b = (int)(block % BHk) / a_in.Hkv;
      KArgs a = a_in;
      enter_sequence(a, b, 2);
      const bool dep = tile >= n_seq_tiles;
      const int ncols = dep ? a.T * a.Lv : a.T;
      for (int tid = 0; tid < 64 * CW; tid++) {
        const int lane = tid & 63, n = lane & 15, q = lane >> 4, wave = tid >> 6;
        const int c0 = dep ? ((tile - n_seq_tiles) * CW + wave) * 16 : tile * 16;
        if (c0 >= ncols) continue;
        const int c = c0 + n, cc = imin(c, ncols - 1);
        const int64_t crow = dep ? depth_row_of(a, cc) : (int64_t)cc;
        ctx("fp32_dkv_kernel", (int)block, wave, lane, "stationary K and V rows");
        score(dep ? "kd" : "k", dep ? f(a.kd) + b * a.skd.b + hkv * a.skd.h + crow * a.skd.t : f(a.k) + b * a.sk.b + hkv * a.sk.h + crow * a.sk.t, q, a.D);
        score(dep ? "vd" : "v", dep ? f(a.vd) + b * a.svd.b + hkv * a.svd.h + crow * a.svd.t : f(a.v) + b * a.sv.b + hkv * a.sv.h + crow * a.sv.t, q, a.Dv);
        int lo, hi, unused;
        q_interval(a, dep, c0, lo, unused);
        q_interval(a, dep, imin(ncols, c0 + 16) - 1, unused, hi);
        const int r_first = lo / 16 * 16, nrb = (hi - r_first + 15) / 16, nb = nrb * a.hdiv;
        ctx("fp32_dkv_kernel", (int)block, wave, lane, "query rows and their statistics");
        for (int blk = dep ? 0 : wave; blk < nb; blk += dep ? 1 : CW) {
          const int hq = hkv * a.hdiv + blk / nrb, r0 = r_first + blk % nrb * 16;
          const float *qp = f(a.q) + b * a.sq.b + hq * a.sq.h, *dop = f(a.d_o) + b * a.sdo.b + hq * a.sdo.h;
          const int64_t r = imin(r0 + n, a.Tq - 1);
          score("q", qp + r * a.sq.t, q, a.D);
          score("do", dop + r * a.sdo.t, q, a.Dv);
          if (own_delta) score("o", f(a.o) + b * a.so.b + hq * a.so.h + r * a.so.t, q, a.Dv);
          for (int i = 0; i < 4; i++) {
            const int64_t ri = imin(r0 + 4 * q + i, a.Tq - 1);
            check_access("lse", a.lse + ((int64_t)b * a.Tq + ri) * a.Hq + hq, 4, false);
            if (!own_delta) check_access("delta", a.delta + ((int64_t)b * a.Hq + hq) * a.delta_pitch + ri, 4, false);
            sum("q", qp + ri * a.sq.t, n, a.D);
            sum("do", dop + ri * a.sdo.t, n, a.Dv);
          }
        }
        ctx("fp32_dkv_kernel", (int)block, wave, lane, "gradient rows");
        if (dep) {
          if (c >= ncols) continue;
          const float *dkp = f(a.dkd) + b * a.sdkd.b + hkv * a.sdkd.h + crow * a.sdkd.t, *dvp = f(a.dvd) + b * a.sdvd.b + hkv * a.sdvd.h + crow * a.sdvd.t;
          for (int h = 0; h < H4; h++)
            for (int i = 0; i < 4; i++) {
              const int d = 64 * h + 16 * q + 4 * i;
              if (d < a.D) check_access("dkd", dkp + d, 16, true);
              if (d < a.Dv) check_access("dvd", dvp + d, 16, true);
            }
          if (a.Lv != a.L && !a.keep_slots && c % a.Lv == a.Lv - 1)
            for (int slot = a.Lv; slot < a.L; slot++) {
              dkp += a.sdkd.t;
              dvp += a.sdvd.t;
              for (int d = 4 * q; d < a.D; d += 16) check_access("dkd", dkp + d, 16, true);
              for (int d = 4 * q; d < a.Dv; d += 16) check_access("dvd", dvp + d, 16, true);
            }
          continue;
        }
        if (lane == 0) partial((CW + wave) * PART, 2 * CW * PART * 4);
        for (int e = tid; e < 2 * 16 * HD / 4; e += 64 * CW) {
          const int w = e / (16 * HD / 4), row = e % (16 * HD / 4) / (HD / 4), d = (e % (HD / 4)) * 4;
          if (c0 + row >= ncols || d >= (w ? a.Dv : a.D)) continue;
          if (w)
            check_access("dv", f(a.dv) + b * a.sdv.b + hkv * a.sdv.h + (int64_t)(c0 + row) * a.sdv.t + d, 16, true);
          else
            check_access("dk", f(a.dk) + b * a.sdk.b + hkv * a.sdk.h + (int64_t)(c0 + row) * a.sdk.t + d, 16, true);
        }
      }
    }
    if (a_in.has_seq) {
      require_full("dk");
      require_full("dv");
    }
    if (a_in.L > 0) {
      require_depth_rows("dkd", a_in, a_in.D);
      require_depth_rows("dvd", a_in, a_in.Dv);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// linear layers, layer norm, depth slots
// ---------------------------------------------------------------------------------------------------------------
template <int BM, int BN, int NST>
void walk_linear_tiles(int rows, int K, const std::vector<int>& parts, bool residual) {
  constexpr int MB = BN / 32, NB = BM / 32;
  const uint32_t lds_bytes = NST * (BM + BN) * 64 * 2;
  const int64_t ldx = K + 8, ldy_pad = 16;
  int idx = 0;
  const uint16_t* x = add_region("x", idx++, ((int64_t)(rows - 1) * ldx + K) * 2, 2, false);  // nothing behind the last row
  std::vector<const uint16_t*> w, bias, y;
  std::vector<int> end;
  std::vector<std::string> names;
  for (size_t i = 0; i < parts.size(); i++) {
    const std::string k = std::to_string(i);
    w.push_back(add_region(("w" + k).c_str(), idx++, (int64_t)parts[i] * K * 2, 2, false));
    bias.push_back(add_region(("bias" + k).c_str(), idx++, (int64_t)parts[i] * 2, 2, false));
    y.push_back(add_region(("y" + k).c_str(), idx++, ((int64_t)(rows - 1) * (parts[i] + ldy_pad) + parts[i]) * 2, 2, true));
    end.push_back((end.empty() ? 0 : end.back()) + (parts[i] + BN - 1) / BN);
  }
  const uint16_t* res = add_region("residual", idx++, residual ? (int64_t)rows * parts[0] * 2 : 0, 2, false);
  const int m_tiles = (rows + BM - 1) / BM, n_tiles = end.back();
  typedef AsyncTileLoader<64, BM, 256> LoadX;
  typedef AsyncTileLoader<64, BN, 256> LoadW;
  for (int64_t block = 0; block < linear_blocks(m_tiles, n_tiles); block++) {
    const int mt = linear_row_tile((unsigned)block, n_tiles);
    int nt = linear_feature_tile((unsigned)block, n_tiles), pi = 0;
    if (mt >= m_tiles) continue;
    while (nt >= end[pi]) pi++;
    const int n = parts[pi], ldy = n + (int)ldy_pad;
    if (pi > 0) nt -= end[pi - 1];
    const int r0 = mt * BM, f0 = nt * BN;
    const std::string wn = "w" + std::to_string(pi), bn = "bias" + std::to_string(pi), yn = "y" + std::to_string(pi);
    for (int tid = 0; tid < 256; tid++) {
      const int lane = tid & 63, ln = lane & 15, q4 = lane >> 4, wave = tid >> 6, wm = wave >> 1, wf = wave & 1;
      LoadX lx;
      LoadW lw;
      lx.init(tid);
      lw.init(tid);
      ctx("linear_kernel", (int)block, wave, lane, "operand tiles");
      for (int it = 0; it < K / 64; it++) {
        const uint32_t xs = (uint32_t)(it % NST) * (BM + BN) * 64 * 2;
        for (int i = 0; i < LoadX::N; i++)
          check_dma("x", x + it * 64 + (int64_t)r0 * ldx, LoadX::anchored_bytes(ldx, r0, rows), lx.lane_offset((int)ldx * 2, 64),
                    LoadX::rows_before(i) * (int)ldx * 2, 16, xs + (uint32_t)lx.lds_elems(i) * 2, lds_bytes, false);
        for (int i = 0; i < LoadW::N; i++)
          check_dma(wn.c_str(), w[pi] + it * 64 + (int64_t)f0 * K, LoadW::anchored_bytes(K, f0, n), lw.lane_offset(K * 2, 64),
                    LoadW::rows_before(i) * K * 2, 16, xs + BM * 64 * 2 + (uint32_t)lw.lds_elems(i) * 2, lds_bytes, false);
      }
      ctx("linear_kernel", (int)block, wave, lane, "results");
      for (int mb = 0; mb < MB; mb++) {
        const int f = f0 + wf * (BN / 2) + 16 * mb + slot_base(q4);
        if (f >= n) continue;
        check_access(bn.c_str(), bias[pi] + f, 8, false);
        for (int nb = 0; nb < NB; nb++) {
          const int r = r0 + wm * (BM / 2) + 16 * nb + slot_base(ln >> 2) + (ln & 3);
          if (r >= rows) continue;
          if (residual) check_access("residual", res + (int64_t)r * n + f, 8, false);
          check_access(yn.c_str(), y[pi] + (int64_t)r * ldy + f, 8, true);
        }
      }
    }
  }
  for (size_t i = 0; i < parts.size(); i++) {
    Region& r = region(("y" + std::to_string(i)).c_str());
    for (size_t u = 0; r.track && u < r.writes.size(); u++) {
      const int want = (int)(u % (size_t)(parts[i] + ldy_pad)) < parts[i] ? 1 : 0;
      if (r.writes[u] != want) fail("%s unit %zu written %d times, not %d", r.name.c_str(), u, (int)r.writes[u], want);
    }
  }
}
void walk_linear(int rows, int K, bool gelu, const std::vector<int>& parts) {
  const bool residual = parts.size() == 1 && !gelu;
  switch (pick_linear_tile(rows, K, parts.data(), (int)parts.size(), 256)) {
    case LinearTile::k128x128: printf("128x128 "); return walk_linear_tiles<128, 128, 2>(rows, K, parts, residual);
    case LinearTile::k128x64: printf("128x64 "); return walk_linear_tiles<128, 64, 2>(rows, K, parts, residual);
    case LinearTile::k128x64ThreeStages: printf("128x64,3 "); return walk_linear_tiles<128, 64, 3>(rows, K, parts, residual);
    default: printf("64x64 "); return walk_linear_tiles<64, 64, 2>(rows, K, parts, residual);
  }
}

void walk_norm(int rows, int dim) {
  const int lpr = dim <= 128 ? 16 : dim <= 256 ? 32 : 64, ch = dim <= 512 ? 1 : dim <= 1024 ? 2 : dim <= 2048 ? 4 : 8;
  const uint16_t* x = add_region("x", 0, (int64_t)rows * dim * 2, 2, false);
  const uint16_t* w = add_region("weight", 1, (int64_t)dim * 2, 2, false);
  const uint16_t* b = add_region("bias", 2, (int64_t)dim * 2, 2, false);
  const uint16_t* y = add_region("y", 3, (int64_t)rows * dim * 2, 2, true);
  const int rpb = 256 / lpr;
  for (int block = 0; block < (rows + rpb - 1) / rpb; block++)
    for (int tid = 0; tid < 256; tid++) {
      const int row = block * rpb + tid / lpr;
      if (row >= rows) continue;
      ctx("layer_norm_kernel", block, tid >> 6, tid & 63, "row, weight, bias");
      for (int c = 0; c < ch; c++) {
        const int e = (c * lpr + tid % lpr) * 8;
        if (e >= dim) continue;
        check_access("x", x + (int64_t)row * dim + e, 16, false);
        check_access("weight", w + e, 16, false);
        check_access("bias", b + e, 16, false);
        check_access("y", y + (int64_t)row * dim + e, 16, true);
      }
    }
  require_full("y");
}

// The attention of attend_tail_kernel: the forward kernel's body on RowBlock shapes.  Query rows, the ring of each key/value head (half the
// waves and half the ring each where there are two), both private sets of depth tiles, the rows left for the dense part; who has which
// part of LDS while the ring is in use (first set beside it) and after its last tile (second set over it).
template <int C, int NB, int KV_HEADS>
void walk_attention(bool fp16, const KArgs& a, const char* k_name, const char* v_name) {
  constexpr int BM = 16 * NB, G = C / 64 / KV_HEADS, WORK = BM * G / 32, HD = 64, BN = 64;
  typedef RowBlock<KV_HEADS, WORK> Shape;
  constexpr int W = Shape::W, NT = 64 * W, NST = Shape::NST, DIST = Shape::DIST, ROWS = 32 * WORK;
  static_assert(ROWS == BM * G && W * KV_HEADS == 8 && Shape::APART, "a head's query rows of the workgroup's tokens");
  const char* kname = "attend_tail_kernel";
  const uint32_t table = fp16 ? 0 : MODA_HIP_GELU_TABLE_BYTES, X = table, H = X + BM * C * 2;  // bytes
  const uint32_t behind = H + attend_ring<Shape, BM>() * 2, lds_bytes = behind + KV_HEADS * WORK * 32 * HD * 2;
  if (lds_bytes > 160 * 1024) fail("%u bytes of LDS", lds_bytes);
  typedef AsyncTileLoader<HD, BN, NT> Loader;
  typedef WaveTileLoader<HD> Own;
  const bool own_depth = waves_own_depth(a, a.L);
  for (int block = 0; block < attend_tail_blocks(a, BM); block++) {
    const AttendTailPlace place = attend_tail_place(a, block, BM);
    const int b = place.b, qt = place.tile;
    if (place.first_row != b * a.T + qt * BM || qt < 0 || qt * BM >= a.T) fail("%s: tile %d of sequence %d", kname, qt, b);
    const RowTilePlan plan = row_tile_plan(a, qt, ROWS, BN, a.L > 0 && !own_depth);
    const int ntiles = plan.n_seq + plan.n_dep;
    // owners of LDS, 16 bytes each: while the ring is in use, and after it; times an element of the attention rows was written
    static std::vector<int> during, after;  // (static: a walk may end in the middle)
    static std::vector<uint8_t> left;
    during.assign(lds_bytes / 16, -1);
    after.assign(lds_bytes / 16, -1);
    left.assign(BM * C / 4, 0);
    const auto take = [lds_bytes, kname](std::vector<int>& lds, uint32_t from, uint32_t bytes, int who) {
      for (uint32_t i = from / 16; i < (from + bytes) / 16; i++) {
        if (from + bytes > lds_bytes || (lds[i] != -1 && lds[i] != who)) fail("%s: byte %u of LDS is another's", kname, 16 * i);
        lds[i] = who;
      }
    };
    for (int tid = 0; tid < 512; tid++) {
      const int lane = tid & 63, head = tid / NT, wave = tid % NT / 64, who = tid / 64;  // (wave: of the head's)
      const bool idle = wave >= WORK;
      const uint32_t ring = H + (uint32_t)head * NST * 2 * BN * HD * 2;
      const int r = qt * ROWS + wave * 32 + (lane & 31);
      ctx(kname, block, who, lane, "Q register rows");
      if (!idle && r < a.Tq)
        for (int e = 8 * (lane >> 5); e < HD; e += 16) check_access("q", a.q + b * a.sq.b + head * a.sq.h + (int64_t)r * a.sq.t + e, 16, false);
      Loader ld;
      ld.init(tid % NT);
      auto srcK = ld.source(a.k + b * a.sk.b + head * a.sk.h, a.sk.t, 0, a.T, a.D), srcV = ld.source(a.v + b * a.sv.b + head * a.sv.h, a.sv.t, 0, a.T, a.Dv);
      for (int it = 0; it < ntiles; it++) {
        const bool dep = it >= plan.n_seq;
        ctx(kname, block, who, lane, dep ? "ring depth tile" : "ring sequence tile");
        for (int ahead = 1; ahead <= DIST; ahead++)
          if ((it + ahead) % NST == it % NST) fail("%s: a tile on its way into the stage that is read", kname);
        const uint32_t kt = ring + (uint32_t)(it % NST) * 2 * BN * HD * 2;
        ring_tile_loads<HD, NT, false>(a, b, head, ld, srcK, srcV, ring_tile_row0(plan, it, BN), dep, true, kt, lds_bytes, k_name, v_name);
        if (lane == 0)
          for (int i = 0; i < Loader::N; i++)
            for (uint32_t v : {0u, (uint32_t)BN * HD * 2}) take(during, kt + v + (uint32_t)ld.lds_elems(i) * 2, 1024, 100 + head);
      }
      const int rw0 = qt * ROWS + wave * 32;
      if (own_depth && !idle && rw0 < a.Tq) {
        const DepthSpan span = own_depth_span(a, rw0, 32);
        Own own;
        own.init(lane);
        ctx(kname, block, who, lane, "own depth tile");
        for (int j = 0; 32 * j < span.c_end - span.c_beg; j++) {
          const int col0 = span.c_beg + 32 * j, nrows = imin(32, span.c_end - col0);
          const uint32_t tile = 32 * HD * 2, kt = j % 2 ? ring + (uint32_t)wave * 2 * tile : X + (uint32_t)(head * WORK + wave) * tile;
          const uint32_t vt = j % 2 ? kt + tile : behind + (uint32_t)(head * WORK + wave) * tile;
          for (int i = 0; i < Own::N; i++) own_tile_load<HD>(a, b, head, own, i, col0, nrows, true, kt, vt, lds_bytes);
          if (lane == 0)
            for (uint32_t at : {kt, vt}) {
              take(after, at, tile, who);
              if (j == 0) take(during, at, tile, who);
              if (j % 2 && (at < ring || at + tile > ring + NST * 2 * BN * HD * 2)) fail("%s: second private set outside of the head's ring", kname);
            }
        }
      }
      ctx(kname, block, who, lane, "attention rows");
      for (int chunk = 0; !idle && chunk < HD / 8; chunk++) {
        const int row = wave * 32 + (lane & 31), at = RowLayout<C>::off(row / G, (row % G * KV_HEADS + head) * 8 + chunk) + 4 * (lane >> 5);
        if (at < 0 || at + 4 > BM * C || left[at / 4]++) fail("%s: element %d of the attention rows", kname, at);
      }
    }
    for (size_t i = 0; i < left.size(); i++)
      if (!left[i]) fail("%s: attention rows %zu of workgroup %d not written", kname, 4 * i, block);
  }
}
void walk_attention(bool fp16, const KArgs& a, const char* k_name, const char* v_name) {
  const int kv = a.Hkv, width = 64 * kv * a.Gf, bm = block_tail_rows((int64_t)a.B * a.T, a.compute_units);
  if (!attend_tail_takes(width, kv * a.Gf, kv, bm)) fail("heads that the joined launch does not take");
  if (width == 128) return bm == 32 ? walk_attention<128, 2, 1>(fp16, a, k_name, v_name) : walk_attention<128, 4, 1>(fp16, a, k_name, v_name);
  if (width == 256 && kv == 1) return bm == 32 ? walk_attention<256, 2, 1>(fp16, a, k_name, v_name) : walk_attention<256, 4, 1>(fp16, a, k_name, v_name);
  if (width == 256) return bm == 32 ? walk_attention<256, 2, 2>(fp16, a, k_name, v_name) : walk_attention<256, 4, 2>(fp16, a, k_name, v_name);
  walk_attention<512, 2, 2>(fp16, a, k_name, v_name);
}

// A block's dense part in one launch: rows in and out, every product's weights, biases, norms and parts; what LDS holds.
// Weights are read through their packed copies, each piece against the order that pack_weights_kernel leaves.
// `tokens` > 0: with the attention before it (attend_tail_kernel), workgroups of BM tokens of one of rows / tokens sequences.
template <int C, int NB>
void walk_tail_of(bool fp16, int rows, int hidden, bool post, const std::vector<int>& parts, int tokens) {
  constexpr int BM = 16 * NB, MB2 = C / 128, MB1 = 2, HC = 256, CH = C / 8, TPR = 512 / BM, NL = CH / TPR;
  const uint32_t table = fp16 ? 0 : MODA_HIP_GELU_TABLE_BYTES, X = table / 2, H = X + BM * C;  // elements
  KArgs att = {};
  att.B = tokens ? rows / tokens : 0;
  att.T = tokens;
  const uint32_t ring = std::max(4 * 2 * 64 * 64, BM * 2 * HC), apart = BM * (C / 64);  // elements; 64 a query row, K or V
  if (tokens && BM * (C / 64) > 256) fail("more query rows than eight waves take");
  const uint32_t lds_bytes = table + (tokens ? (BM * C + ring + 64 * apart) * 2 : (uint32_t)BM * (C + std::max(C, 2 * HC)) * 2);
  if (tokens && (X + 64 * apart > H || H + ring + 64 * apart > lds_bytes / 2)) fail("private K and V tiles of the attention");
  int idx = 0;
  const auto region2 = [&](const char* name, int64_t n, bool track = false) { return add_region(name, idx++, n * 2, 2, track); };
  const uint16_t *h = region2("attention", (int64_t)rows * C), *res = region2("residual", (int64_t)rows * C), *x = region2("x", (int64_t)rows * C, true);
  const uint16_t *proj_w = region2("proj_w", C * C), *proj_b = region2("proj_b", C), *fc1_w = region2("fc1_w", (int64_t)hidden * C);
  const uint16_t *fc1_b = region2("fc1_b", hidden), *fc2_w = region2("fc2_w", (int64_t)hidden * C), *fc2_b = region2("fc2_b", C);
  const uint16_t *mid_w = region2("mid_w", C), *mid_b = region2("mid_b", C), *end_w = region2("end_w", C), *end_b = region2("end_b", C);
  const uint16_t* gelu_table = region2("gelu_table", table / 2);
  std::vector<const uint16_t*> w, bias, y;
  std::vector<int> end;
  std::vector<std::string> wn, bn, yn;
  for (size_t i = 0; i < parts.size(); i++) {
    const std::string k = std::to_string(i);
    wn.push_back("w" + k);
    bn.push_back("bias" + k);
    yn.push_back("y" + k);
    w.push_back(region2(wn[i].c_str(), (int64_t)parts[i] * C));
    bias.push_back(region2(bn[i].c_str(), parts[i]));
    y.push_back(region2(yn[i].c_str(), (int64_t)(rows - 1) * (parts[i] + 8) + parts[i], true));
    end.push_back((end.empty() ? 0 : end.back()) + parts[i] / 16);
  }
  const auto lds = [&](uint32_t first, int64_t off, int elems, uint32_t limit, const char* what) {  // [first, limit) elements
    if (off < 0 || first + off + elems > limit || limit * 2 > lds_bytes) fail("%s at element %lld of LDS", what, (long long)off);
  };
  const int nblk = tokens ? (int)attend_tail_blocks(att, BM) : (rows + BM - 1) / BM;
  for (int block = 0; block < nblk; block++)
    for (int tid = 0; tid < 512; tid++) {
      const AttendTailPlace place = tokens ? attend_tail_place(att, block, BM) : AttendTailPlace{0, block, block * BM, rows};
      const int rows_end = place.rows_end;
      if (place.first_row >= rows_end) fail("a workgroup without rows");
      const int lane = tid & 63, n = lane & 15, q4 = lane >> 4, wave = tid >> 6, r0 = place.first_row, sigma = slot_base(n >> 2) + (n & 3);
      const int f2 = wave * 16 * MB2, lrow = tid / TPR, lsub = tid % TPR;
      const uint32_t all = lds_bytes / 2;
      // one product: `mb` blocks of 16 features from f on (packed [features][width]), steps first .. first + nk - 1 of 32
      const auto product = [&](const char* name, const uint16_t* packed, int f, int mbs, int width, int first, int nk, int ahead) {
        ctx("block_tail_kernel", block, wave, lane, name);
        if (nk % 4 || ahead > nk) fail("%d steps", nk);
        for (int mb = 0; mb < mbs; mb++)
          for (int ks = 0; ks < nk; ks++) {
            const char* at = (const char*)(packed + (size_t)(f + 16 * mb) * width + first * 512) + lane * 16 + (size_t)ks * 1024;
            if (at != (const char*)(packed + packed_piece((int64_t)((f + 16 * mb) / 16) * (width / 32) + first + ks, lane))) fail("a piece that is not where it was packed");
            check_access(name, at, 16, false);
          }
      };
      const auto operand = [&](auto layout, uint32_t base, uint32_t limit, int nk) {
        typedef decltype(layout) L;
        for (int ks = 0; ks < nk; ks++)
          for (int nb = 0; nb < NB; nb++)
            lds(base, L::off(sigma, 4 * (ks & 3) + q4) + 16 * nb * L::kWidth + (ks >> 2) * 128, 8, limit, "row operand");
      };
      const auto pieces = [&](const char* name, const uint16_t* b, int f, int mbs) {
        for (int mb = 0; mb < mbs; mb++) check_access(name, b + f + 16 * mb + 4 * q4, 8, false);
      };
      const auto norm = [&](const char* wn, const uint16_t* weight, const char* bn, const uint16_t* b, bool normalise, bool store) {
        ctx("block_tail_kernel", block, wave, lane, "layer norm");
        for (int j = 0; j < NL; j++) {
          lds(X, RowLayout<C>::off(lrow, lsub + TPR * j), 8, H, "row");
          if (normalise) {
            check_access(wn, weight + (lsub + TPR * j) * 8, 16, false);
            check_access(bn, b + (lsub + TPR * j) * 8, 16, false);
          }
          if (store && r0 + lrow < rows_end) check_access("x", x + (int64_t)(r0 + lrow) * C + (lsub + TPR * j) * 8, 16, true);
        }
      };
      ctx("block_tail_kernel", block, wave, lane, "rows in");
      for (int j = 0; j < BM * CH / 512; j++) {
        const int at = (tid + 512 * j) / CH, row = std::min(r0 + at, rows_end - 1), ch = (tid + 512 * j) % CH;
        if (!tokens) check_access("attention", h + (int64_t)row * C + ch * 8, 16, false);
        check_access("residual", res + (int64_t)row * C + ch * 8, 16, false);
        lds(X, RowLayout<C>::off(at, ch), 8, H, "residual row");
        lds(H, RowLayout<C>::off(at, ch), 8, all, "attention row");
      }
      const int nt = table / 16;
      for (int j = 0; j < (nt + 511) / 512; j++) check_access("gelu_table", gelu_table + (tid + 512 * j < nt ? tid + 512 * j : 0) * 8, 16, false);
      product("proj_w", proj_w, f2, MB2, C, 0, C / 32, MB2 <= 3 ? 4 : 2);
      operand(RowLayout<C>{}, H, all, C / 32);
      pieces("proj_b", proj_b, f2, MB2);
      for (int mb = 0; mb < MB2; mb++)
        for (int nb = 0; nb < NB; nb++) lds(X, RowLayout<C>::off(sigma, (f2 >> 3) + 2 * mb + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * C, 4, H, "own piece");
      norm("mid_w", mid_w, "mid_b", mid_b, true, false);
      for (int c0 = 0, stage = 0; c0 < hidden; c0 += HC, stage ^= 1) {
        // (a wave without features of a short last chunk may read others', see the kernel, but leaves nothing)
        const bool mine = c0 + wave * 16 * MB1 < hidden;
        const int f1 = mine ? c0 + wave * 16 * MB1 : c0, left = std::min(hidden - c0, HC);
        const uint32_t Hs = H + stage * BM * HC, Hs_end = Hs + BM * HC;
        product("fc1_w", fc1_w, f1, MB1, C, 0, C / 32, 4);
        operand(RowLayout<C>{}, X, H, C / 32);
        pieces("fc1_b", fc1_b, f1, MB1);
        if (mine) {
          for (int mb = 0; mb < MB1; mb++)
            for (int nb = 0; nb < NB; nb++)
              lds(Hs, RowLayout<HC>::off(sigma, wave * 2 * MB1 + 2 * mb + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * HC, 4, Hs_end, "hidden piece");
        }
        product("fc2_w", fc2_w, f2, MB2, hidden, c0 / 32, left / 32, MB2 <= 3 ? 4 : 2);
        operand(RowLayout<HC>{}, Hs, Hs_end, left / 32);
      }
      pieces("fc2_b", fc2_b, f2, MB2);
      norm("end_w", end_w, "end_b", end_b, post || !parts.empty(), true);
      if (parts.empty()) continue;
      const int blocks = end.back();
      const auto projections = [&](auto side_by_side) {
        constexpr int MBQ = decltype(side_by_side)::value, W = 128 * MBQ;
        for (int first = 0; first < blocks; first += 8 * MBQ) {
          for (int mb = 0; mb < MBQ; mb++) {
            const int blk = std::min(first + wave * MBQ + mb, blocks - 1);
            size_t pi = 0;
            while (blk >= end[pi]) pi++;
            const int f = 16 * (blk - (pi ? end[pi - 1] : 0));
            product(wn[pi].c_str(), w[pi], f, 1, C, 0, C / 32, MBQ <= 3 ? 4 : 2);
            pieces(bn[pi].c_str(), bias[pi], f, 1);
            for (int nb = 0; nb < NB; nb++)
              lds(H, RowLayout<W>::off(sigma, 2 * (wave * MBQ + mb) + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * W, 4, all, "projected piece");
          }
          ctx("block_tail_kernel", block, wave, lane, "projected rows out");
          const int chunks = 2 * std::min(blocks - first, 8 * MBQ);
          for (int ch = lsub; ch < chunks && r0 + lrow < rows_end; ch += TPR) {
            const int blk = first + (ch >> 1);
            size_t pi = 0;
            while (blk >= end[pi]) pi++;
            lds(H, RowLayout<W>::off(lrow, ch), 8, all, "projected row");
            check_access(yn[pi].c_str(), y[pi] + (int64_t)(r0 + lrow) * (parts[pi] + 8) + 8 * (2 * first + ch) - (pi ? 16 * end[pi - 1] : 0), 16, true);
          }
        }
      };
      if (blocks <= 16)
        projections(std::integral_constant<int, 2>{});
      else if (blocks <= 24)
        projections(std::integral_constant<int, 3>{});
      else
        projections(std::integral_constant<int, 4>{});
    }
  require_full("x");
  for (size_t i = 0; i < parts.size(); i++) {
    Region& r = region(("y" + std::to_string(i)).c_str());
    for (size_t u = 0; r.track && u < r.writes.size(); u++) {
      const int want = (int)(u % (size_t)(parts[i] + 8)) < parts[i] ? 1 : 0;
      if (r.writes[u] != want) fail("%s unit %zu written %d times, not %d", r.name.c_str(), u, (int)r.writes[u], want);
    }
  }
}
void walk_tail(bool fp16, int rows, int width, int hidden, bool post, const std::vector<int>& parts, int tokens = 0) {
  const auto go = [&](auto c) {
    constexpr int C = decltype(c)::value;
    block_tail_rows(rows, 256) == 32 ? walk_tail_of<C, 2>(fp16, rows, hidden, post, parts, tokens)
                                     : walk_tail_of<C, 4>(fp16, rows, hidden, post, parts, tokens);
  };
  switch (width) {
    case 128: return go(std::integral_constant<int, 128>{});
    case 256: return go(std::integral_constant<int, 256>{});
    case 384: return go(std::integral_constant<int, 384>{});
    default: return go(std::integral_constant<int, 512>{});
  }
}

// weights [n][k] into their packed order: matrices of alternating sizes, as many as given
void walk_pack(int matrices) {
  const int sizes[3][2] = {{16, 32}, {48, 128}, {128, 96}};
  int64_t most = 0;
  for (const auto& s : sizes) most = std::max(most, (int64_t)(s[0] / 16) * (s[1] / 32));
  for (int m = 0; m < matrices; m++) {
    const int n = sizes[m % 3][0], k = sizes[m % 3][1], blocks = n / 16, steps = k / 32;
    const uint16_t *from = add_region("w", 0, (int64_t)n * k * 2, 2, true), *to = add_region("packed", 1, (int64_t)n * k * 2, 2, true);
    for (int block = 0; block < (most + 3) / 4; block++)
      for (int tid = 0; tid < 256; tid++) {
        const int lane = tid & 63, item = block * 4 + (tid >> 6);
        if (item >= blocks * steps) continue;
        ctx("pack_weights_kernel", block, tid >> 6, lane, "piece");
        check_access("w", from + weight_piece(item / steps, item % steps, steps, lane), 16, true);  // (read, each element once)
        check_access("packed", to + packed_piece(item, lane), 16, true);
      }
    require_full("w");
    require_full("packed");
  }
}

// one layer's K and V (views of one projection: rows 2 H D + 8 elements apart) against slot `slot` of the caches
void walk_slot(int64_t B, int64_t T, int64_t H, int64_t D, int64_t L, int64_t slot, bool wide, bool to_cache) {
  const int64_t st = 2 * H * D + 8, sb = T * st, piece = wide ? 16 : 2, per_row = D * 2 / piece, units = B * T * H * per_row;
  for (int i = 0; i < 2; i++) {
    const uint16_t* layer = add_region(i ? "v" : "k", 2 * i, (((B - 1) * T + T - 1) * st + H * D) * 2, 2, !to_cache);
    const uint16_t* cache = add_region(i ? "cache_v" : "cache_k", 2 * i + 1, B * T * L * H * D * 2, 2, to_cache);
    for (int64_t u = 0; u < (units + 255) / 256 * 256; u++) {
      if (u >= units) continue;
      const int64_t w = u % per_row, row = u / per_row, tok = row / H, h = row - tok * H, b = tok / T, t = tok - b * T;
      ctx("slot_kernel", (int)(u / 256), (int)(u % 256) >> 6, (int)(u & 63), to_cache ? "layer into its slot" : "slot onto its layer");
      check_access(i ? "v" : "k", (const char*)layer + (b * sb + t * st + h * D) * 2 + w * piece, piece, !to_cache);
      check_access(i ? "cache_v" : "cache_k", (const char*)cache + (slot + tok * L) * H * D * 2 + (h * per_row + w) * piece, piece, to_cache);
    }
    Region& c = region(to_cache ? (i ? "cache_v" : "cache_k") : (i ? "v" : "k"));
    for (size_t u = 0; u < c.writes.size(); u++) {
      const int want = to_cache ? (int64_t)u / (H * D) % L == slot : (int64_t)u % st < H * D;
      if (c.writes[u] != want) fail("%s unit %zu written %d times, not %d", c.name.c_str(), u, (int)c.writes[u], want);
    }
  }
}

template <int HD>
void walk_all(const Case& c, const KArgs& a) {
  if (!narrow_slices(a)) fail("slices beyond 2 GiB are not walked (the fake tensors would not fit the walker's write maps)");
  const bool small = a.cu ? use_small_rows(a.delta_pitch, a.Hq, a.compute_units) : use_small_rows(a.Tq, (long long)a.B * a.Hq, a.compute_units);
  const ShortRows rows = a.cu ? ShortRows::kNone : pick_short_rows(a.Tq, (long long)a.B * a.Hq, a.causal, a.compute_units);
  // ---- forward
  const auto ring = [](int NST) { return (uint32_t)NST * 2 * 64 * HD * 2; };
  const auto fwd = [&](auto shape, const char* name) {
    typedef decltype(shape) Shape;
    printf("%s ", name);
    walk_row_kernel<HD, Shape, false>(a, false, HD > 128 ? 16 : 32, HD <= 128, ring(Shape::NST), name);
  };
  if constexpr (HD > 128) {
    fwd(RowWide{}, "fwd_wide_kernel");
  } else if constexpr (HD <= 64) {
    if (rows == ShortRows::kTwoStages)
      fwd(RowShort{}, "fwd_kernel(short)");
    else
      fwd(RowSmall<HD>{}, "fwd_kernel(small)");
  } else {
    if (small)
      fwd(RowSmall<HD>{}, "fwd_kernel(small)");
    else
      fwd(RowLargePP{}, "fwd_kernel");
  }
  require_full("o");
  require_full("lse");
  // ---- backward
  // the row sums: by the delta kernel when that stage is run alone, else inside the dQ kernel
  walk_delta<HD>(a);
  require_full("delta");
  reset_writes("delta");
  const auto dq = [&](auto shape, const char* name) {
    typedef decltype(shape) Shape;
    const uint32_t own = (uint32_t)Shape::W * (HD <= kDepthGradsInDqMaxWidth ? 2 * 64 + 16 : 64) * HD * 2;
    const bool own_fits = a.L > 0 && (uint32_t)Shape::W * 64 * HD * 2 <= 128 * 1024;
    printf("%s ", name);
    walk_row_kernel<HD, Shape, false>(a, true, HD > 128 ? 16 : 32, HD <= 128, own_fits ? std::max(ring(Shape::NST), own) : ring(Shape::NST), name);
  };
  if constexpr (HD > 128) {
    dq(RowWide{}, "dq_kernel(wide)");
  } else if constexpr (HD <= 64) {
    if (rows == ShortRows::kTwoStages)
      dq(RowShort{}, "dq_kernel(short)");
    else if (rows == ShortRows::kThreeStages)
      dq(RowShort3{}, "dq_kernel(short, three stages)");
    else
      dq(RowSmall<HD>{}, "dq_kernel(small)");
  } else {
    if (small)
      dq(RowSmall<HD>{}, "dq_kernel(small)");
    else
      dq(RowLarge{}, "dq_kernel");
  }
  require_full("dq");
  require_full("delta");
  if (a.depth_p) {
    require_full("hand_p");
    require_full("hand_ds");
  }
  const bool flat = takes_dkv_flat(a, HD);
  if (a.own_slot && !flat) fail("only dkv_flat_kernel's launches add an own slot");
  if (flat) {
    if constexpr (HD == 64) {
      if (dkv_flat_row_waves(a))
        walk_dkv_flat<HD, 4>(a);
      else
        walk_dkv_flat<HD, 1>(a);
    }
  } else {
    walk_dkv<HD>(a);
  }
  if (a.dkv_split > 1 && a.has_seq) {
    walk_reduce<HD>(a, HD > 128 ? 64 : 128, flat || HD > 128 ? 32 : 64);
    for (uint8_t w : region("part").writes)  // (short tiles have fewer segments, or none: their places stay empty)
      if (w == 1) fail("a partial sum that no column adds up");
    if (g_partials_read == 0) fail("row segments without partial sums");
  }
  if (a.has_seq) {
    require_full("dk");
    require_full("dv");
  }
  if (a.L > 0) {
    if ((a.chunk || depth_grads_in_dq(a, HD)) && a.Lv != a.L && !a.keep_slots) walk_zero_unfilled<HD>(a);
    if (a.chunk) {
      if constexpr (HD <= 128) {
        if (depth_by_chunks(a, HD)) walk_chunk_depth<HD>(a);
      }
    } else if (!depth_grads_in_dq(a, HD)) {
      if (a.depth_p && a.Gf <= 4)
        walk_depth_tokens<HD>(a);
      else
        walk_depth_cols<HD>(a);
    }
    require_depth_rows("dkd", a, a.D);
    require_depth_rows("dvd", a, a.Dv);
  }
  // ---- the whole backward where dQ and dK/dV share a launch (the stages apart are what is walked above)
  if constexpr (HD == 64)
    if (bwd_one_launch(a, HD)) {
      printf("bwd_short_kernel ");
      if (row_kernel_blocks(a, kBwdShortRows) + dkv_flat_blocks(a, 32) > 2 * a.compute_units) fail("more workgroups than run at once");
      for (const char* name : {"delta", "dq", "dk", "dv", "dkd", "dvd"}) reset_writes(name);
      if (a.depth_p)
        for (const char* name : {"hand_p", "hand_ds"}) reset_writes(name);
      const uint32_t own = (uint32_t)RowSmall<64>::W * (2 * 64 + 16) * HD * 2;
      walk_row_kernel<HD, RowSmall<64>, false>(a, true, 32, true, a.L > 0 ? std::max(ring(RowSmall<64>::NST), own) : ring(RowSmall<64>::NST), "bwd_short_kernel");
      walk_dkv_flat<HD, 4, true>(a);
      for (const char* name : {"delta", "dq", "dk", "dv"}) require_full(name);
      if (a.L > 0 && depth_grads_in_dq(a, HD)) {
        if (a.Lv != a.L && !a.keep_slots) walk_zero_unfilled<HD>(a);
        require_depth_rows("dkd", a, a.D);
        require_depth_rows("dvd", a, a.Dv);
      }
    }
  (void)c;
}

}  // namespace

int main(int argc, char** argv) {
  const auto arg = [&](int i) { return i < argc ? atoi(argv[i]) : 0; };
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "tail_rule") {  // dtype rows width hidden kv compute_units
    printf("%s, %d rows\n", block_tail_pays(std::string(argv[2]) == "fp16", arg(3), arg(4), arg(5), arg(6), arg(7)) ? "one launch" : "pieces",
           block_tail_rows(arg(3), arg(7)));
    return 0;
  }
  if (what == "tail") {  // dtype rows width hidden post_norm n0 [n1 n2]
    std::vector<int> parts;
    for (int i = 7; i < argc; i++) parts.push_back(arg(i));
    walk_tail(std::string(argv[2]) == "fp16", arg(3), arg(4), arg(5), arg(6) != 0, parts);
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  if (what == "attend_tail") {  // dtype sequences tokens width hidden post_norm n0 [n1 n2]
    std::vector<int> parts;
    for (int i = 8; i < argc; i++) parts.push_back(arg(i));
    walk_tail(std::string(argv[2]) == "fp16", arg(3) * arg(4), arg(5), arg(6), arg(7) != 0, parts, arg(4));
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  if (what == "attention") {  // dtype sequences tokens heads group slots filled mode chunk_tokens
    Case c = {64, 64, 64, arg(5), arg(6), arg(7), arg(8), arg(9), arg(10), 0, arg(3), {}, {}, arg(4), arg(4)};
    KArgs a = make_args(c);
    const bool in_cache = c.Lv > 0 && c.Lv < c.L;  // k and v in the first free slot, as a stack has them
    if (in_cache) {
      a.k = a.kd + c.Lv * c.H * 64;
      a.v = a.vd + c.Lv * c.H * 64;
      a.sk = a.sv = Str3{a.skd.b, (int64_t)c.L * c.H * 64, 64};
    }
    walk_attention(std::string(argv[2]) == "fp16", a, in_cache ? "kd" : "k", in_cache ? "vd" : "v");
    printf("OK checked=%lld dma_in_range=%lld dma_zero_filled=%lld\n", g_checked, g_dma_in, g_dma_out);
    return 0;
  }
  if (what == "attend_tail_rule") {  // sequences tokens width heads kv_heads compute_units [slots [causal]]
    printf("%s\n", attention_joins_tail(arg(2), arg(3), arg(4), arg(5), arg(6), argc > 8 ? arg(8) : 12, arg(9) != 0, arg(7)) ? "joins" : "apart");
    return 0;
  }
  if (what == "pack_and_norm") {  // rows rows_of_a_workgroup packing_workgroups parts
    printf("%lld\n", (long long)pack_and_norm_blocks(atoll(argv[2]), arg(3), atoll(argv[4]), arg(5)));
    return 0;
  }
  if (what == "attend_tail_order") {  // sequences tokens tokens_of_a_workgroup causal: sequence and tile of every workgroup
    KArgs a = {};
    a.B = arg(2);
    a.T = arg(3);
    a.causal = arg(5);
    for (int block = 0; block < attend_tail_blocks(a, arg(4)); block++) {
      const AttendTailPlace p = attend_tail_place(a, block, arg(4));
      if (p.first_row != p.b * a.T + p.tile * arg(4) || p.rows_end != (p.b + 1) * a.T) fail("rows of workgroup %d", block);
      printf("%d:%d ", p.b, p.tile);
    }
    printf("\n");
    return 0;
  }
  if (what == "slots") {  // the slot arithmetic of partially filled streams against the division it stands for
    for (int Lv : {1, 2, 3, 5, 7, 11, 12, 24, 31, 33, 63, 64, 65, 72, 127, 1000, 65537, (1 << 24) + 3, (1 << 30) + 1})
      for (int l0 : {0, 1, Lv / 2, Lv - 2, Lv - 1})
        for (int rho = 0; rho <= 64; rho++) {
          if (l0 < 0 || l0 >= Lv) continue;
          const SlotStep s = slot_step(l0, rho, Lv);
          if (s.tokens != (l0 + rho) / Lv || s.slot != (l0 + rho) % Lv) fail("slot %d + %d of %d: token %d, slot %d", l0, rho, Lv, s.tokens, s.slot);
          g_checked++;
        }
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  if (what == "pack") {
    walk_pack(arg(2));
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  if (what == "linear" || what == "norm" || what == "slot") {
    std::vector<int> parts;
    for (int i = 5; i < argc; i++) parts.push_back(arg(i));
    if (what == "linear") walk_linear(arg(2), arg(3), arg(4) != 0, parts);
    if (what == "norm") walk_norm(arg(2), arg(3));
    if (what == "slot") walk_slot(arg(2), arg(3), arg(4), arg(5), arg(6), arg(7), arg(8) != 0, arg(9) != 0);
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  g_fp32 = getenv("WALKER_FP32") != nullptr;
  g_own_slot = getenv("WALKER_OWN_SLOT") != nullptr;
  if (argc < 14) {
    fprintf(stderr, "usage: %s HD D Dv H G L Lv mode chunk_tokens split packed n len0 [len1 ...]\n", argv[0]);
    return 2;
  }
  Case c;
  int i = 1;
  c.HD = atoi(argv[i++]);
  c.D = atoi(argv[i++]);
  c.Dv = atoi(argv[i++]);
  c.H = atoi(argv[i++]);
  c.G = atoi(argv[i++]);
  c.L = atoi(argv[i++]);
  c.Lv = atoi(argv[i++]);
  c.mode = atoi(argv[i++]);
  c.cb = atoi(argv[i++]);
  const int split = atoi(argv[i++]);
  c.packed = atoi(argv[i++]);
  c.nseq = atoi(argv[i++]);
  for (; i < argc; i++) c.len.push_back(atoi(argv[i]));
  c.cu.push_back(0);
  c.Tmax = 0;
  if (c.packed) {
    if ((int)c.len.size() != c.nseq) return 2;
    for (int n : c.len) {
      c.cu.push_back(c.cu.back() + n);
      c.Tmax = std::max(c.Tmax, n);
    }
    c.total = c.cu.back();
  } else {
    c.Tmax = c.len[0];
    c.total = c.Tmax;
  }
  KArgs a = make_args(c);
  a.dkv_split = split > 0 && !c.packed ? split : 1;
  if (split < 0) {  // the library's own rule
    const DkvSplit plan = dkv_split_plan(a, c.HD);
    a.dkv_split = plan.nseg;
    a.dkv_seg_tiles = plan.seg_tiles;
    printf("segments=%d ", plan.nseg);
  }
  if (a.dkv_split > 1)
    a.dkv_part = (float*)add_region("part", 20, (uint64_t)2 * a.dkv_split * (a.cu ? 1 : a.B) * a.Hkv * part_rows(a) * c.HD * 4, 4, true);
  if (getenv("WALKER_ROUTE")) {  // of a whole backward pass; split 1: a workspace without room for segments
    const bool one = g_fp32 ? c.HD == 64 && fp32_one_launch(a) : bwd_one_launch(a, c.HD);
    printf("%s\n", one ? "one launch" : "two launches");
    return 0;
  }
  if (getenv("WALKER_ORDER")) {
    packed_launch_order(a);
    return 0;
  }
  if (g_fp32) {
    if (c.HD > 128) return 2;
    c.HD == 64 ? walk_fp32<64>(a) : walk_fp32<128>(a);
    printf("OK checked=%lld\n", g_checked);
    return 0;
  }
  switch (c.HD) {
    case 64: walk_all<64>(c, a); break;
    case 128: walk_all<128>(c, a); break;
    case 256: walk_all<256>(c, a); break;
    default: return 2;
  }
  printf("OK checked=%lld dma_in_range=%lld dma_zero_filled=%lld\n", g_checked, g_dma_in, g_dma_out);
  return 0;
}
