// C ABI of libmoda_hip.so (see include/moda_hip.h): descriptor validation and
// dispatch to the gfx950 kernels.  No tensor-library types cross this file.
#include <hip/hip_runtime.h>

#include <atomic>
#include <initializer_list>
#include <string.h>

#include "../../include/moda_hip.h"
#include "geometry.h"
#include "kargs.h"
#include "tuning.h"

namespace moda {
hipError_t launch_fwd(const KArgs& a, int dtype, int hd, hipStream_t stream);
hipError_t launch_delta(const KArgs& a, int dtype, int hd, hipStream_t stream);
hipError_t launch_dq(const KArgs& a, int dtype, int hd, hipStream_t stream);
hipError_t launch_dkv(const KArgs& a, int dtype, int hd, hipStream_t stream);
hipError_t launch_bwd_short(const KArgs& a, int dtype, hipStream_t stream);
hipError_t launch_generic(const KArgs& a, int dtype, int D, int Dv, int which, hipStream_t stream);
hipError_t launch_fp32(const KArgs& a, int which, hipStream_t stream);
hipError_t launch_reorg(void* const* layers, int64_t n_layers, int64_t slot0, int64_t L_total, int64_t n_tokens,
                        int64_t row_bytes, void* cache, bool to_cache, hipStream_t stream);
hipError_t launch_slot(void* const (&layer)[2], const int64_t (&strides)[2][3], void* const (&cache)[2], int64_t slot, int64_t L_total,
                       int64_t B, int64_t T, int64_t H, int64_t D, int dtype, bool to_cache, hipStream_t stream);
hipError_t launch_linear(int dtype, int64_t rows, int64_t K, const void* x, int64_t ldx, const moda_hip_linear_part* parts, int n_parts,
                         const void* residual, int64_t ld_res, bool gelu, int compute_units, hipStream_t stream);
hipError_t launch_layer_norm(int dtype, int64_t rows, int64_t dim, const void* x, const void* weight, const void* bias, float eps, void* y,
                             hipStream_t stream);
hipError_t launch_pack_weights(const moda_hip_weight* w, int n, float* gelu_table, const moda_hip_norm_rows* norm, hipStream_t stream);
hipError_t launch_block_tail(const moda_hip_block_tail_args* args, int compute_units, hipStream_t stream);
hipError_t launch_attend_tail(const moda_hip_block_tail_args* args, const KArgs& attention, hipStream_t stream);
}  // namespace moda

using moda::KArgs;
using moda::Str3;

namespace {

int elem_size(int dtype) { return dtype == MODA_HIP_FP32 ? 4 : 2; }

Str3 cvt(const moda_hip_strides& s) { return Str3{s.b, s.t, s.h}; }

// The MFMA kernels move rows with 16-byte accesses; the vector-ALU kernels load element by element and
// need element alignment only.
bool aligned(const void* p, const moda_hip_strides& s, int esize, bool vec16) {
  if (!vec16) return (uintptr_t)p % esize == 0;
  const int64_t m = 16 / esize;
  return ((uintptr_t)p % 16 == 0) && (s.b % m == 0) && (s.t % m == 0) && (s.h % m == 0);
}

// The streaming kernels address rows inside a tile with 32-bit byte offsets: a row stride must stay
// below 16 MiB (tiles have at most 64 rows per pass).
bool row_stride_ok(const moda_hip_strides& s, int esize) { return s.t >= 0 && s.t * esize < (1ll << 24); }

// A partially filled depth stream is read through one descriptor per tile, anchored at the first column's token:
// the byte offsets of a tile's 64 columns from that anchor -- up to 64 / Lv + 2 tokens of L rows -- must fit 31 bits.
bool mapped_span_ok(const KArgs& a, const moda_hip_strides& s, int esize) {
  if (a.L == 0 || a.Lv == a.L) return true;
  return (int64_t)(64 / a.Lv + 2) * a.L * s.t * esize < (1ll << 31);
}

// The fp32 matrix kernels move 16-byte pieces of rows; fp32 tensors that are not laid out for that run on the vector-ALU
// kernels, which ask for element alignment only (the host therefore does not copy fp32 views).
struct TensorAt {
  const void* p;
  const moda_hip_strides& s;
};
bool fp32_matrix(const moda_hip_desc* d, const KArgs& a, std::initializer_list<TensorAt> tensors) {
  if (d->dtype != MODA_HIP_FP32 || a.D > 128 || a.Dv > 128) return false;
  for (const TensorAt& t : tensors)
    if (t.p && !aligned(t.p, t.s, 4, true)) return false;
  return true;
}

int value_dim(const moda_hip_desc* d) { return (int)(d->Dv > 0 ? d->Dv : d->D); }

// The matrix-core kernels exist for tile widths 64, 128 and 256; any 16-bit head dim that is a multiple of 8 (whole
// 16-byte chunks) up to 256 runs on the next width, zero-padded inside the kernels.
bool mfma_shape(const moda_hip_desc* d) {
  return (d->dtype == MODA_HIP_BF16 || d->dtype == MODA_HIP_FP16) && d->D % 8 == 0 && d->D <= 256 &&
         value_dim(d) % 8 == 0 && value_dim(d) <= 256;
}
// Packed variable-length batches with head dims above 128 do not run the packed instantiations of the 256-wide
// kernels: that combination (with chunk-visible mode) once ended in a GPU memory fault whose cause was never
// found, so those instantiations stay switched off.  With a host copy of the offsets the batch runs as one launch
// per sequence on the fixed-length 256-wide kernels (per_sequence below); without it, on the vector-ALU kernels.
int widest_dim(const moda_hip_desc* d) { return (int)(d->D > value_dim(d) ? d->D : value_dim(d)); }
bool packed_wide(const moda_hip_desc* d) { return widest_dim(d) > 128 && d->cu_seqlens; }
bool per_sequence(const moda_hip_desc* d) { return mfma_shape(d) && packed_wide(d) && d->cu_seqlens_host; }
bool use_mfma(const moda_hip_desc* d) { return mfma_shape(d) && !packed_wide(d); }
// keys and values share one tile width: that of the wider of the two head dims
int tile_width(const moda_hip_desc* d) { return widest_dim(d) <= 64 ? 64 : widest_dim(d) <= 128 ? 128 : 256; }

// Validates the descriptor and fills the geometry part of KArgs.
int fill_geometry(const moda_hip_desc* d, KArgs& a) {
  if (!d || d->struct_size != (int32_t)sizeof(moda_hip_desc)) return MODA_HIP_EINVAL;
  if (d->dtype < MODA_HIP_BF16 || d->dtype > MODA_HIP_FP32) return MODA_HIP_EINVAL;
  if (d->mode < MODA_HIP_CAUSAL || d->mode > MODA_HIP_PLAIN_GQA) return MODA_HIP_EINVAL;
  if (d->B < 0 || d->T < 0 || d->H <= 0 || d->G <= 0 || d->D <= 0 || d->L < 0) return MODA_HIP_EINVAL;
  if (d->D > 256 || d->D % 4 != 0) return MODA_HIP_EUNSUPPORTED;
  if (d->Dv < 0) return MODA_HIP_EINVAL;
  if (d->Dv > 256 || d->Dv % 4 != 0) return MODA_HIP_EUNSUPPORTED;
  if (d->mode == MODA_HIP_PLAIN_GQA && d->L != 0) return MODA_HIP_EINVAL;
  if (d->mode == MODA_HIP_DEPTH_ONLY && d->L == 0) return MODA_HIP_EINVAL;
  if (d->mode == MODA_HIP_CHUNK_VISIBLE && d->L > 0 && d->chunk_tokens <= 0) return MODA_HIP_EINVAL;
  if (d->L_valid < 0 || d->L_valid > d->L) return MODA_HIP_EINVAL;
  if (d->flags & ~(int32_t)(MODA_HIP_FLAG_ACCUMULATE_DEPTH_GRADS | MODA_HIP_FLAG_KEEP_DEPTH_SLOTS | MODA_HIP_FLAG_ADD_OWN_SLOT))
    return MODA_HIP_EINVAL;
  // 32-bit index space used for rows and flattened depth columns inside the kernels
  if (d->T * d->G >= (1ll << 30) || d->T * (d->L > 0 ? d->L : 1) >= (1ll << 30) || d->B * d->H * d->G >= (1ll << 20))
    return MODA_HIP_EUNSUPPORTED;
  memset(&a, 0, sizeof(a));
  const bool plain = d->mode == MODA_HIP_PLAIN_GQA;
  a.B = (int)d->B;
  a.T = (int)d->T;
  a.Hkv = (int)d->H;
  a.D = (int)d->D;
  a.Dv = value_dim(d);
  a.Tq = plain ? (int)d->T : (int)(d->T * d->G);
  a.Gf = plain ? 1 : (int)d->G;
  a.Hq = plain ? (int)(d->H * d->G) : (int)d->H;
  a.hdiv = plain ? (int)d->G : 1;
  a.L = (int)d->L;
  a.Lv = d->L_valid > 0 ? (int)d->L_valid : (int)d->L;
  if (a.Lv == 0) a.Lv = a.L = 0;
  a.Cb = d->mode == MODA_HIP_CHUNK_VISIBLE ? (int)(d->chunk_tokens > 0 ? d->chunk_tokens : 1) : 1;
  a.has_seq = d->mode != MODA_HIP_DEPTH_ONLY;
  a.causal = d->mode == MODA_HIP_CAUSAL || d->mode == MODA_HIP_CHUNK_VISIBLE || plain;
  a.chunk = d->mode == MODA_HIP_CHUNK_VISIBLE;
  a.own_slot = (d->flags & MODA_HIP_FLAG_ADD_OWN_SLOT) ? 1 : 0;
  a.accum_depth = (d->flags & MODA_HIP_FLAG_ACCUMULATE_DEPTH_GRADS) ? 1 : 0;
  a.keep_slots = (d->flags & (MODA_HIP_FLAG_ACCUMULATE_DEPTH_GRADS | MODA_HIP_FLAG_KEEP_DEPTH_SLOTS)) ? 1 : 0;
  // The dQ kernel that forms the depth gradients stores a tile's rows in the same way as it reads them; of a full stream 32 rows in
  // a row, which row_stride_ok keeps within 512 MiB.
  a.far_depth_grads = !mapped_span_ok(a, d->dkd, elem_size(d->dtype)) || !mapped_span_ok(a, d->dvd, elem_size(d->dtype));
  a.nqt = (a.Tq + 127) / 128;
  a.scale = d->scale;
  a.delta_pitch = a.Tq;
  a.dkv_split = 1;
  if (d->cu_seqlens) {
    // packed batch: T is the longest sequence, the row axes hold total_tokens tokens
    if (d->total_tokens < d->T || ((uintptr_t)d->cu_seqlens % 4) != 0) return MODA_HIP_EINVAL;
    if (d->total_tokens * d->G >= (1ll << 30) || d->total_tokens * (d->L > 0 ? d->L : 1) >= (1ll << 30))
      return MODA_HIP_EUNSUPPORTED;
    if (d->cu_seqlens_host) {  // the host copy can be checked: offsets start at 0, do not decrease, fit T and total
      const int32_t* h = d->cu_seqlens_host;
      if (h[0] != 0 || h[d->B] != d->total_tokens) return MODA_HIP_EINVAL;
      for (int64_t i = 0; i < d->B; i++)
        if (h[i + 1] < h[i] || h[i + 1] - h[i] > d->T) return MODA_HIP_EINVAL;
    }
    a.cu = d->cu_seqlens;
    a.delta_pitch = (int)(plain ? d->total_tokens : d->total_tokens * d->G);
  } else if (d->cu_seqlens_host) {
    return MODA_HIP_EINVAL;
  }
  return MODA_HIP_OK;
}

// Bytes of the row-sum part of the backward workspace, rounded up so that what follows stays aligned.
size_t delta_bytes_exact(const KArgs& a) {
  const size_t n = (a.cu ? (size_t)1 : (size_t)a.B) * a.Hq * a.delta_pitch * sizeof(float);
  return n ? n : sizeof(float);
}
size_t delta_bytes(const KArgs& a) { return (delta_bytes_exact(a) + 255) / 256 * 256; }

// Row segments of the sequence dK/dV launch (geometry.h: dkv_split_plan).
moda::DkvSplit desired_dkv_split(const moda_hip_desc* d, const KArgs& a) {
  if (!use_mfma(d)) return {1, 0};
  return moda::dkv_split_plan(a, tile_width(d));
}

// P and dS of the (query row, depth slot) pairs, handed from the dQ kernel to the depth-gradient kernel (see
// KArgs::depth_p): two 16-bit arrays indexed like the row sums, times the slots that hold data.
size_t depth_handover_bytes(const moda_hip_desc* d, const KArgs& a) {
  if (!use_mfma(d) || !moda::depth_scores_from_dq(a, tile_width(d))) return 0;
  const size_t n = (a.cu ? (size_t)1 : (size_t)a.B) * a.Hq * a.delta_pitch * a.Lv * sizeof(uint16_t);
  return 2 * ((n + 255) / 256 * 256);
}

size_t dkv_part_bytes(const moda_hip_desc* d, const KArgs& a, int split) {
  return split > 1 ? (size_t)2 * split * (a.cu ? 1 : a.B) * a.Hkv * moda::part_rows(a) * tile_width(d) * sizeof(float) : 0;
}

// The current device must be a gfx950; reports its compute-unit count.  One entry per device is cached.
int check_device(int* compute_units = nullptr) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return MODA_HIP_EDEVICE;
  struct Entry {
    std::atomic<int> state{0};  // 0 unknown, 1 gfx950, -1 something else
    int cus = 0;
  };
  static Entry cache[64];
  Entry local;
  Entry& e = (dev >= 0 && dev < 64) ? cache[dev] : local;
  int st = e.state.load(std::memory_order_acquire);
  if (st == 0) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, dev) != hipSuccess) return MODA_HIP_EDEVICE;
    e.cus = p.multiProcessorCount;
    st = strncmp(p.gcnArchName, "gfx950", 6) == 0 ? 1 : -1;
    e.state.store(st, std::memory_order_release);
  }
  if (compute_units) *compute_units = e.cus;
  return st == 1 ? MODA_HIP_OK : MODA_HIP_EDEVICE;
}

// Workspace of moda_hip_bwd_static: lives in the code object, one copy per device the library is loaded on, for as
// long as the process runs.  In host code the array's name is only a handle for hipGetSymbolAddress; the
// device address is looked up once per device and kept.
static __device__ __align__(256) unsigned char scratch[MODA_HIP_STATIC_WORKSPACE_BYTES];

int static_workspace(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return MODA_HIP_EDEVICE;
  static std::atomic<void*> table[64];
  if (dev < 0 || dev >= 64) return MODA_HIP_EDEVICE;
  void* p = table[dev].load(std::memory_order_acquire);
  if (!p) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MODA_HIP_ELAUNCH;
    table[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return MODA_HIP_OK;
}


// Sequence i of a packed batch as a fixed-length problem of batch size 1: the descriptor, and the element offsets
// of its first query row, key row and depth row on the packed row axes.
struct SeqView {
  moda_hip_desc d;
  int64_t q_row, k_row, d_row;
};
SeqView sequence_view(const moda_hip_desc* d, int64_t i) {
  SeqView v;
  v.d = *d;
  const int64_t t0 = d->cu_seqlens_host[i];
  v.d.B = 1;
  v.d.T = d->cu_seqlens_host[i + 1] - t0;
  v.d.cu_seqlens = nullptr;
  v.d.cu_seqlens_host = nullptr;
  v.d.total_tokens = 0;
  v.q_row = d->mode == MODA_HIP_PLAIN_GQA ? t0 : t0 * d->G;
  v.k_row = t0;
  v.d_row = t0 * d->L;
  return v;
}
const void* at(const void* p, int64_t row, int64_t stride, int esize) {
  return p ? (const char*)p + row * stride * esize : nullptr;
}
void* at(void* p, int64_t row, int64_t stride, int esize) { return p ? (char*)p + row * stride * esize : nullptr; }

#define MODA_REQ_PTR(p) \
  if (!(p)) return MODA_HIP_EINVAL
#define MODA_REQ_ALIGN(p, s)                                    \
  if (!aligned((p), (s), es, vec16)) return MODA_HIP_EALIGN; \
  if (vec16 && !row_stride_ok((s), es)) return MODA_HIP_EUNSUPPORTED

}  // namespace

extern "C" {

int moda_hip_fwd(const moda_hip_desc* d, const void* q, const void* k, const void* v, const void* kd,
                 const void* vd, void* o, float* lse, void* stream) {
  KArgs a;
  int rc = fill_geometry(d, a);
  if (rc) return rc;
  if ((int64_t)a.B * a.Tq * a.Hq == 0) return MODA_HIP_OK;
  const int es = elem_size(d->dtype);
  if (per_sequence(d)) {
    MODA_REQ_PTR(lse);
    for (int64_t i = 0; i < d->B; i++) {
      const SeqView s = sequence_view(d, i);
      if (s.d.T == 0) continue;
      rc = moda_hip_fwd(&s.d, at(q, s.q_row, d->q.t, es), at(k, s.k_row, d->k.t, es), at(v, s.k_row, d->v.t, es),
                        at(kd, s.d_row, d->kd.t, es), at(vd, s.d_row, d->vd.t, es), at(o, s.q_row, d->o.t, es),
                        lse + s.q_row * a.Hq, stream);
      if (rc) return rc;
    }
    return MODA_HIP_OK;
  }
  const bool vec16 = use_mfma(d);
  MODA_REQ_PTR(q);
  MODA_REQ_PTR(o);
  MODA_REQ_PTR(lse);
  MODA_REQ_ALIGN(q, d->q);
  MODA_REQ_ALIGN(o, d->o);
  if (a.has_seq) {
    MODA_REQ_PTR(k);
    MODA_REQ_PTR(v);
    MODA_REQ_ALIGN(k, d->k);
    MODA_REQ_ALIGN(v, d->v);
  }
  if (a.L > 0) {
    MODA_REQ_PTR(kd);
    MODA_REQ_PTR(vd);
    MODA_REQ_ALIGN(kd, d->kd);
    MODA_REQ_ALIGN(vd, d->vd);
    if (vec16 && !(mapped_span_ok(a, d->kd, es) && mapped_span_ok(a, d->vd, es))) return MODA_HIP_EUNSUPPORTED;
  }
  if ((rc = check_device(&a.compute_units))) return rc;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.v = (const uint16_t*)v;
  a.kd = (const uint16_t*)kd;
  a.vd = (const uint16_t*)vd;
  a.out_o = (uint16_t*)o;
  a.lse = lse;
  a.sq = cvt(d->q);
  a.sk = cvt(d->k);
  a.sv = cvt(d->v);
  a.skd = cvt(d->kd);
  a.svd = cvt(d->vd);
  a.so = cvt(d->o);
  hipError_t e;
  if (use_mfma(d))
    e = moda::launch_fwd(a, d->dtype, tile_width(d), (hipStream_t)stream);
  else if (fp32_matrix(d, a, {{q, d->q}, {k, d->k}, {v, d->v}, {kd, d->kd}, {vd, d->vd}, {o, d->o}}))
    e = moda::launch_fp32(a, 0, (hipStream_t)stream);
  else
    e = moda::launch_generic(a, d->dtype, (int)d->D, value_dim(d), 0, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

size_t moda_hip_bwd_workspace_bytes(const moda_hip_desc* d) {
  KArgs a;
  if (fill_geometry(d, a)) return 0;
  const size_t part = dkv_part_bytes(d, a, desired_dkv_split(d, a).nseg);
  const size_t hand = depth_handover_bytes(d, a);
  // the row sums, then (each optional) the handed-over depth scores and the partial sums of the row split
  return (part || hand) ? delta_bytes(a) + hand + part : delta_bytes_exact(a);
}

int moda_hip_bwd(const moda_hip_desc* d, const void* q, const void* k, const void* v, const void* kd,
                 const void* vd, const void* o, const float* lse, const void* d_o, void* dq, void* dk, void* dv,
                 void* dkd, void* dvd, void* workspace, size_t workspace_bytes, void* stream) {
  return moda_hip_bwd_stages(d, q, k, v, kd, vd, o, lse, d_o, dq, dk, dv, dkd, dvd, workspace, workspace_bytes,
                             MODA_HIP_STAGE_ALL, stream);
}

int moda_hip_bwd_static(const moda_hip_desc* d, const void* q, const void* k, const void* v, const void* kd,
                        const void* vd, const void* o, const float* lse, const void* d_o, void* dq, void* dk,
                        void* dv, void* dkd, void* dvd, void* stream) {
  KArgs g;
  const int grc = fill_geometry(d, g);
  if (grc) return grc;
  if (delta_bytes_exact(g) > (size_t)MODA_HIP_STATIC_WORKSPACE_BYTES) return MODA_HIP_ESTATIC;
  void* ws = nullptr;
  const int rc = static_workspace(&ws);
  if (rc) return rc;
  return moda_hip_bwd_stages(d, q, k, v, kd, vd, o, lse, d_o, dq, dk, dv, dkd, dvd, ws,
                             (size_t)MODA_HIP_STATIC_WORKSPACE_BYTES, MODA_HIP_STAGE_ALL, stream);
}

int moda_hip_bwd_stages(const moda_hip_desc* d, const void* q, const void* k, const void* v, const void* kd,
                        const void* vd, const void* o, const float* lse, const void* d_o, void* dq, void* dk,
                        void* dv, void* dkd, void* dvd, void* workspace, size_t workspace_bytes, int stages,
                        void* stream) {
  KArgs a;
  int rc = fill_geometry(d, a);
  if (rc) return rc;
  if (stages < 0 || stages > MODA_HIP_STAGE_ALL) return MODA_HIP_EINVAL;
  if (a.own_slot) {
    if (a.L == 0 || a.Lv >= a.L || !a.keep_slots) return MODA_HIP_EINVAL;
    if (!use_mfma(d) || a.cu || !moda::takes_dkv_flat(a, tile_width(d))) return MODA_HIP_EUNSUPPORTED;
  }
  const int es = elem_size(d->dtype);
  if (per_sequence(d) && (int64_t)a.B * a.Tq * a.Hq > 0) {
    MODA_REQ_PTR(lse);
    if (!workspace || workspace_bytes < delta_bytes_exact(a)) return MODA_HIP_EWORKSPACE;
    for (int64_t i = 0; i < d->B; i++) {
      const SeqView s = sequence_view(d, i);
      if (s.d.T == 0) continue;
      // every sequence keeps its own part of the row-sum workspace ([heads][its query rows]), so the stages of
      // one backward may still be issued as separate calls
      const size_t ws_off = (size_t)a.Hq * s.q_row * sizeof(float);
      const size_t ws_len = (size_t)a.Hq * (d->mode == MODA_HIP_PLAIN_GQA ? s.d.T : s.d.T * d->G) * sizeof(float);
      rc = moda_hip_bwd_stages(&s.d, at(q, s.q_row, d->q.t, es), at(k, s.k_row, d->k.t, es),
                               at(v, s.k_row, d->v.t, es), at(kd, s.d_row, d->kd.t, es), at(vd, s.d_row, d->vd.t, es),
                               at(o, s.q_row, d->o.t, es), lse + s.q_row * a.Hq, at(d_o, s.q_row, d->d_o.t, es),
                               at(dq, s.q_row, d->dq.t, es), at(dk, s.k_row, d->dk.t, es), at(dv, s.k_row, d->dv.t, es),
                               at(dkd, s.d_row, d->dkd.t, es), at(dvd, s.d_row, d->dvd.t, es),
                               (char*)workspace + ws_off, ws_len, stages, stream);
      if (rc) return rc;
    }
    return MODA_HIP_OK;
  }
  const bool vec16 = use_mfma(d);
  const bool have_rows = (int64_t)a.B * a.Tq * a.Hq > 0;
  if (have_rows) {
    MODA_REQ_PTR(q);
    MODA_REQ_PTR(o);
    MODA_REQ_PTR(lse);
    MODA_REQ_PTR(d_o);
    MODA_REQ_PTR(dq);
    MODA_REQ_ALIGN(q, d->q);
    MODA_REQ_ALIGN(o, d->o);
    MODA_REQ_ALIGN(d_o, d->d_o);
    MODA_REQ_ALIGN(dq, d->dq);
    if (a.has_seq) {
      MODA_REQ_PTR(k);
      MODA_REQ_PTR(v);
      MODA_REQ_PTR(dk);
      MODA_REQ_PTR(dv);
      MODA_REQ_ALIGN(k, d->k);
      MODA_REQ_ALIGN(v, d->v);
      MODA_REQ_ALIGN(dk, d->dk);
      MODA_REQ_ALIGN(dv, d->dv);
    }
    if (a.L > 0) {
      MODA_REQ_PTR(kd);
      MODA_REQ_PTR(vd);
      MODA_REQ_PTR(dkd);
      MODA_REQ_PTR(dvd);
      MODA_REQ_ALIGN(kd, d->kd);
      MODA_REQ_ALIGN(vd, d->vd);
      MODA_REQ_ALIGN(dkd, d->dkd);
      MODA_REQ_ALIGN(dvd, d->dvd);
      if (vec16 && !(mapped_span_ok(a, d->kd, es) && mapped_span_ok(a, d->vd, es))) return MODA_HIP_EUNSUPPORTED;
    }
    if (!workspace || workspace_bytes < delta_bytes_exact(a)) return MODA_HIP_EWORKSPACE;
    if ((uintptr_t)workspace % sizeof(float) != 0) return MODA_HIP_EALIGN;
    // the row split of light launches uses what the workspace offers beyond the row sums: a caller that gives
    // less than moda_hip_bwd_workspace_bytes asks for (moda_hip_bwd_static) gets fewer segments or none
    // ... and likewise the hand-over of the depth scores from the dQ kernel to the depth-gradient kernel, which sits
    // between the row sums and the partial sums
    size_t hand = depth_handover_bytes(d, a);
    if (delta_bytes(a) + hand > workspace_bytes) hand = 0;
    moda::DkvSplit split = desired_dkv_split(d, a);
    const int most = split.nseg;
    while (split.nseg > 1 && delta_bytes(a) + hand + dkv_part_bytes(d, a, split.nseg) > workspace_bytes) split.nseg /= 2;
    if ((uintptr_t)workspace % 16 != 0) split.nseg = 1;  // the partial sums are written and read 16 bytes at a time
    a.dkv_split = split.nseg;
    if (a.own_slot && split.nseg == 1 && !moda::dkv_flat_row_waves(a)) return MODA_HIP_EUNSUPPORTED;
    a.dkv_seg_tiles = (split.seg_tiles * most + split.nseg - 1) / split.nseg;  // fewer segments: longer ones
    a.dkv_part = (float*)((char*)workspace + delta_bytes(a) + hand);
    if (hand) {
      a.depth_p = (uint16_t*)((char*)workspace + delta_bytes(a));
      a.depth_ds = (uint16_t*)((char*)workspace + delta_bytes(a) + hand / 2);
    }
  } else {
    return MODA_HIP_OK;
  }
  if ((rc = check_device(&a.compute_units))) return rc;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.v = (const uint16_t*)v;
  a.kd = (const uint16_t*)kd;
  a.vd = (const uint16_t*)vd;
  a.o = (const uint16_t*)o;
  a.d_o = (const uint16_t*)d_o;
  a.lse = const_cast<float*>(lse);
  a.delta = (float*)workspace;
  a.dq = (uint16_t*)dq;
  a.dk = (uint16_t*)dk;
  a.dv = (uint16_t*)dv;
  a.dkd = (uint16_t*)dkd;
  a.dvd = (uint16_t*)dvd;
  a.sq = cvt(d->q);
  a.sk = cvt(d->k);
  a.sv = cvt(d->v);
  a.skd = cvt(d->kd);
  a.svd = cvt(d->vd);
  a.so = cvt(d->o);
  a.sdo = cvt(d->d_o);
  a.sdq = cvt(d->dq);
  a.sdk = cvt(d->dk);
  a.sdv = cvt(d->dv);
  a.sdkd = cvt(d->dkd);
  a.sdvd = cvt(d->dvd);
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = hipSuccess;
  // Launches one after the other let dk, dv take the place of k, v (a dK/dV workgroup reads its own rows of them first, and the
  // dQ launch is done) and dq that of o; side by side they would overwrite what the other half still reads.
  bool in_place = false;
  for (const void* out : {dq, dk, dv})
    for (const void* in : {q, k, v, o, d_o}) in_place = in_place || (out && out == in);
  if (use_mfma(d)) {
    // with both stages asked for, the dQ kernel forms the row sums itself (one launch and one pass over o, do less)
    a.own_delta = (stages & MODA_HIP_STAGE_DELTA) && (stages & MODA_HIP_STAGE_DQ) ? 1 : 0;
    if ((stages & MODA_HIP_STAGE_DELTA) && !a.own_delta) e = moda::launch_delta(a, d->dtype, tile_width(d), s);
    if ((stages & MODA_HIP_STAGE_DKV) && !in_place && moda::bwd_one_launch(a, tile_width(d))) {
      e = moda::launch_bwd_short(a, d->dtype, s);
      a.seq_done = 1;
    } else if (e == hipSuccess && (stages & MODA_HIP_STAGE_DQ)) {
      e = moda::launch_dq(a, d->dtype, tile_width(d), s);
    }
    if (e == hipSuccess && (stages & MODA_HIP_STAGE_DKV)) e = moda::launch_dkv(a, d->dtype, tile_width(d), s);
  } else if (fp32_matrix(d, a, {{q, d->q}, {k, d->k}, {v, d->v}, {kd, d->kd}, {vd, d->vd}, {o, d->o}, {d_o, d->d_o}, {dq, d->dq},
                                {dk, d->dk}, {dv, d->dv}, {dkd, d->dkd}, {dvd, d->dvd}})) {
    // the dQ kernel forms the row sums for the dK/dV kernel; a dK/dV stage that runs alone has them formed first
    const bool rows = stages & MODA_HIP_STAGE_DQ, dkv = stages & MODA_HIP_STAGE_DKV;
    if (rows && dkv && !in_place && moda::fp32_one_launch(a)) {
      e = moda::launch_fp32(a, 4, s);
    } else {
      if (rows) e = moda::launch_fp32(a, 1, s);
      if (e == hipSuccess && !rows && stages) e = moda::launch_fp32(a, 3, s);
      if (e == hipSuccess && dkv) e = moda::launch_fp32(a, 2, s);
    }
  } else {
    // the generic kernels recompute delta inline; the DELTA stage is a no-op for them
    if (stages & MODA_HIP_STAGE_DQ) e = moda::launch_generic(a, d->dtype, (int)d->D, value_dim(d), 1, s);
    if (e == hipSuccess && (stages & MODA_HIP_STAGE_DKV)) e = moda::launch_generic(a, d->dtype, (int)d->D, value_dim(d), 2, s);
  }
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

int moda_hip_depth_reorg_fwd(const void* const* layers, int64_t n_layers, int64_t slot0, int64_t L_total, int64_t B,
                             int64_t T, int64_t H, int64_t D, int32_t dtype, void* cache, void* stream) {
  if (n_layers < 0 || slot0 < 0 || slot0 + n_layers > L_total || B < 0 || T < 0 || H <= 0 || D <= 0)
    return MODA_HIP_EINVAL;
  if (dtype < MODA_HIP_BF16 || dtype > MODA_HIP_FP32) return MODA_HIP_EINVAL;
  if (B * T == 0 || n_layers == 0) return MODA_HIP_OK;
  if (!layers || !cache) return MODA_HIP_EINVAL;
  for (int64_t i = 0; i < n_layers; i++)
    if (!layers[i]) return MODA_HIP_EINVAL;
  if (B * T >= (1ll << 31)) return MODA_HIP_EUNSUPPORTED;
  hipError_t e = moda::launch_reorg(const_cast<void* const*>(layers), n_layers, slot0, L_total, B * T,
                                    H * D * elem_size(dtype), cache, true, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

int moda_hip_depth_reorg_bwd(const void* d_cache, int64_t n_layers, int64_t slot0, int64_t L_total, int64_t B,
                             int64_t T, int64_t H, int64_t D, int32_t dtype, void* const* d_layers, void* stream) {
  if (n_layers < 0 || slot0 < 0 || slot0 + n_layers > L_total || B < 0 || T < 0 || H <= 0 || D <= 0)
    return MODA_HIP_EINVAL;
  if (dtype < MODA_HIP_BF16 || dtype > MODA_HIP_FP32) return MODA_HIP_EINVAL;
  if (B * T == 0 || n_layers == 0) return MODA_HIP_OK;
  if (!d_layers || !d_cache) return MODA_HIP_EINVAL;
  for (int64_t i = 0; i < n_layers; i++)
    if (!d_layers[i]) return MODA_HIP_EINVAL;
  if (B * T >= (1ll << 31)) return MODA_HIP_EUNSUPPORTED;
  hipError_t e = moda::launch_reorg(d_layers, n_layers, slot0, L_total, B * T, H * D * elem_size(dtype),
                                    const_cast<void*>(d_cache), false, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

static int depth_slot(void* k, void* v, const moda_hip_strides* sk, const moda_hip_strides* sv, int64_t slot, int64_t L_total, int64_t B,
                      int64_t T, int64_t H, int64_t D, int32_t dtype, void* cache_k, void* cache_v, bool to_cache, void* stream) {
  if (slot < 0 || slot >= L_total || B < 0 || T < 0 || H <= 0 || D <= 0 || B * T >= (1ll << 31) || H >= (1ll << 31) || D >= (1ll << 31))
    return MODA_HIP_EINVAL;
  if (dtype < MODA_HIP_BF16 || dtype > MODA_HIP_FP32) return MODA_HIP_EINVAL;
  if (B * T == 0) return MODA_HIP_OK;
  if (!k || !v || !sk || !sv || !cache_k || !cache_v) return MODA_HIP_EINVAL;
  void* const layer[2] = {k, v};
  void* const cache[2] = {cache_k, cache_v};
  const int64_t strides[2][3] = {{sk->b, sk->t, sk->h}, {sv->b, sv->t, sv->h}};
  const hipError_t e = moda::launch_slot(layer, strides, cache, slot, L_total, B, T, H, D, dtype, to_cache, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}
int moda_hip_depth_push(const void* k, const void* v, const moda_hip_strides* sk, const moda_hip_strides* sv, int64_t slot,
                        int64_t L_total, int64_t B, int64_t T, int64_t H, int64_t D, int32_t dtype, void* cache_k, void* cache_v,
                        void* stream) {
  return depth_slot(const_cast<void*>(k), const_cast<void*>(v), sk, sv, slot, L_total, B, T, H, D, dtype, cache_k, cache_v, true, stream);
}
int moda_hip_depth_slot_add(void* dk, void* dv, const moda_hip_strides* sdk, const moda_hip_strides* sdv, int64_t slot, int64_t L_total,
                            int64_t B, int64_t T, int64_t H, int64_t D, int32_t dtype, const void* d_cache_k, const void* d_cache_v,
                            void* stream) {
  return depth_slot(dk, dv, sdk, sdv, slot, L_total, B, T, H, D, dtype, const_cast<void*>(d_cache_k), const_cast<void*>(d_cache_v), false,
                    stream);
}

int moda_hip_linear(int32_t dtype, int64_t rows, int64_t K, const void* x, int64_t ldx, const moda_hip_linear_part* parts, int32_t n_parts,
                    const void* residual, int64_t ld_res, int32_t gelu, void* stream) {
  if ((dtype != MODA_HIP_BF16 && dtype != MODA_HIP_FP16) || rows < 0 || K <= 0 || n_parts < 1 || n_parts > 3 || !parts) return MODA_HIP_EINVAL;
  if (rows == 0) return MODA_HIP_OK;
  if (!x || (residual && (n_parts != 1 || gelu))) return MODA_HIP_EINVAL;
  if (K % 64 != 0 || rows >= (1ll << 30) || ldx >= (1ll << 22) || K >= (1ll << 22)) return MODA_HIP_EUNSUPPORTED;
  if ((uintptr_t)x % 16 != 0 || ldx % 8 != 0 || ldx < K || (residual && ((uintptr_t)residual % 16 != 0 || ld_res % 8 != 0)))
    return MODA_HIP_EALIGN;
  for (int i = 0; i < n_parts; i++) {
    const moda_hip_linear_part& p = parts[i];
    if (!p.w || !p.y || p.n <= 0 || p.n >= (1ll << 24)) return MODA_HIP_EINVAL;
    if (p.n % 8 != 0) return MODA_HIP_EUNSUPPORTED;
    if ((uintptr_t)p.w % 16 != 0 || (uintptr_t)p.y % 16 != 0 || p.ldy % 8 != 0 || (uintptr_t)p.bias % 8 != 0) return MODA_HIP_EALIGN;
  }
  int cus = 0;
  const int rc = check_device(&cus);
  if (rc) return rc;
  const hipError_t e = moda::launch_linear(dtype, rows, K, x, ldx, parts, n_parts, residual, ld_res, gelu != 0, cus, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

namespace {
int check_norm(int32_t dtype, int64_t rows, int64_t dim, std::initializer_list<const void*> pointers) {
  if ((dtype != MODA_HIP_BF16 && dtype != MODA_HIP_FP16) || rows < 0 || dim <= 0) return MODA_HIP_EINVAL;
  if (rows == 0) return MODA_HIP_OK;
  for (const void* p : pointers)
    if (!p) return MODA_HIP_EINVAL;
  if (dim % 8 != 0 || dim > 4096 || rows >= (1ll << 31)) return MODA_HIP_EUNSUPPORTED;
  for (const void* p : pointers)
    if ((uintptr_t)p % 16 != 0) return MODA_HIP_EALIGN;
  return MODA_HIP_OK;
}
}  // namespace

int moda_hip_layer_norm(int32_t dtype, int64_t rows, int64_t dim, const void* x, const void* weight, const void* bias, float eps, void* y,
                        void* stream) {
  const int rc = check_norm(dtype, rows, dim, {x, weight, bias, y});
  if (rc || rows == 0) return rc;
  const hipError_t e = moda::launch_layer_norm(dtype, rows, dim, x, weight, bias, eps, y, (hipStream_t)stream);
  return e == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

namespace {
int pack(const moda_hip_weight* w, int32_t n, void* gelu_table, const moda_hip_norm_rows* norm, void* stream) {
  if (!w || n < 1) return MODA_HIP_EINVAL;
  if ((uintptr_t)gelu_table % 16 != 0) return MODA_HIP_EALIGN;
  for (int i = 0; i < n; i++) {
    if (!w[i].w || !w[i].packed || w[i].n <= 0 || w[i].k <= 0) return MODA_HIP_EINVAL;
    if (w[i].n % 16 != 0 || w[i].k % 32 != 0 || w[i].n >= (1 << 20) || w[i].k >= (1 << 20) || w[i].n * w[i].k >= (1ll << 31))
      return MODA_HIP_EUNSUPPORTED;
    if ((uintptr_t)w[i].w % 16 != 0 || (uintptr_t)w[i].packed % 16 != 0) return MODA_HIP_EALIGN;
  }
  const int rc = check_device();
  if (rc) return rc;
  return moda::launch_pack_weights(w, n, (float*)gelu_table, norm, (hipStream_t)stream) == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}
}  // namespace

int moda_hip_pack_weights(const moda_hip_weight* w, int32_t n, void* gelu_table, void* stream) { return pack(w, n, gelu_table, nullptr, stream); }

int moda_hip_pack_weights_and_norm(const moda_hip_weight* w, int32_t n, void* gelu_table, const moda_hip_norm_rows* norm, void* stream) {
  if (!norm) return MODA_HIP_EINVAL;
  const int rc = check_norm(norm->dtype, norm->rows, norm->dim, {norm->x, norm->weight, norm->bias, norm->y});
  if (rc) return rc;
  if (norm->dim > 512) return MODA_HIP_EUNSUPPORTED;
  return pack(w, n, gelu_table, norm, stream);
}

namespace {
// what both launches ask of a block tail's arguments; `attention`: with the attention output
int check_tail(const moda_hip_block_tail_args* t, bool attention) {
  if (!t || t->struct_size != (int32_t)sizeof(*t) || (t->dtype != MODA_HIP_BF16 && t->dtype != MODA_HIP_FP16)) return MODA_HIP_EINVAL;
  if (t->rows < 0 || t->width <= 0 || t->hidden <= 0 || t->n_parts < 0 || t->n_parts > 3) return MODA_HIP_EINVAL;
  if (t->rows == 0) return MODA_HIP_OK;
  if (t->dtype == MODA_HIP_BF16 && !t->gelu_table) return MODA_HIP_EINVAL;
  if ((uintptr_t)t->gelu_table % 16 != 0) return MODA_HIP_EALIGN;
  const bool end_norm = t->post_norm || t->n_parts > 0;
  for (const void* p : {attention ? t->attention : t->residual, t->residual, (const void*)t->x, t->proj_w, t->fc1_w, t->fc2_w, t->mid_norm_w,
                        t->mid_norm_b, end_norm ? t->end_norm_w : t->x, end_norm ? t->end_norm_b : t->x})
    if (!p) return MODA_HIP_EINVAL;
  if ((t->width != 128 && t->width != 256 && t->width != 384 && t->width != 512) || t->hidden % 128 != 0 || t->hidden >= (1 << 20) ||
      t->rows >= (1ll << 30))
    return MODA_HIP_EUNSUPPORTED;
  for (const void* p : {attention ? t->attention : t->residual, t->residual, (const void*)t->x, t->proj_w, t->fc1_w, t->fc2_w, t->mid_norm_w,
                        t->mid_norm_b, end_norm ? t->end_norm_w : t->x, end_norm ? t->end_norm_b : t->x})
    if ((uintptr_t)p % 16 != 0) return MODA_HIP_EALIGN;
  for (const void* p : {t->proj_b, t->fc1_b, t->fc2_b})
    if ((uintptr_t)p % 8 != 0) return MODA_HIP_EALIGN;
  for (int i = 0; i < t->n_parts; i++) {
    const moda_hip_linear_part& p = t->parts[i];
    if (!p.w || !p.y || p.n <= 0) return MODA_HIP_EINVAL;
    if (p.n % 16 != 0 || p.n >= (1 << 20)) return MODA_HIP_EUNSUPPORTED;
    if ((uintptr_t)p.w % 16 != 0 || (uintptr_t)p.y % 16 != 0 || p.ldy % 8 != 0 || (uintptr_t)p.bias % 8 != 0) return MODA_HIP_EALIGN;
  }
  return MODA_HIP_OK;
}
}  // namespace

int moda_hip_block_tail(const moda_hip_block_tail_args* t, void* stream) {
  int cus = 0, rc = check_tail(t, true);
  if (rc || t->rows == 0) return rc;
  if ((rc = check_device(&cus))) return rc;
  return moda::launch_block_tail(t, cus, (hipStream_t)stream) == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

int moda_hip_attend_block_tail(const moda_hip_desc* d, const void* q, const void* k, const void* v, const void* kd, const void* vd,
                               const moda_hip_block_tail_args* t, void* stream) {
  KArgs a;
  int rc = fill_geometry(d, a);
  if (rc || (rc = check_tail(t, false))) return rc;
  if (t->rows != (int64_t)a.B * a.T || t->dtype != d->dtype) return MODA_HIP_EINVAL;
  if (a.D != 64 || a.Dv != 64 || a.hdiv != 1 || !a.has_seq || a.cu || !moda::attend_tail_takes(t->width, (int64_t)a.Hkv * a.Gf, a.Hkv, 32))
    return MODA_HIP_EUNSUPPORTED;
  if (t->rows == 0) return MODA_HIP_OK;
  const int es = elem_size(d->dtype);
  const bool vec16 = true;
  MODA_REQ_PTR(q);
  MODA_REQ_PTR(k);
  MODA_REQ_PTR(v);
  MODA_REQ_ALIGN(q, d->q);
  MODA_REQ_ALIGN(k, d->k);
  MODA_REQ_ALIGN(v, d->v);
  if (a.L > 0) {
    MODA_REQ_PTR(kd);
    MODA_REQ_PTR(vd);
    MODA_REQ_ALIGN(kd, d->kd);
    MODA_REQ_ALIGN(vd, d->vd);
    if (!(mapped_span_ok(a, d->kd, es) && mapped_span_ok(a, d->vd, es))) return MODA_HIP_EUNSUPPORTED;
  }
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.v = (const uint16_t*)v;
  a.kd = (const uint16_t*)kd;
  a.vd = (const uint16_t*)vd;
  a.sq = cvt(d->q);
  a.sk = cvt(d->k);
  a.sv = cvt(d->v);
  a.skd = cvt(d->kd);
  a.svd = cvt(d->vd);
  if (!moda::narrow_slices(a)) return MODA_HIP_EUNSUPPORTED;
  if ((rc = check_device(&a.compute_units))) return rc;
  if (!moda::attend_tail_takes(t->width, (int64_t)a.Hkv * a.Gf, a.Hkv, moda::block_tail_rows(t->rows, a.compute_units))) return MODA_HIP_EUNSUPPORTED;
  return moda::launch_attend_tail(t, a, (hipStream_t)stream) == hipSuccess ? MODA_HIP_OK : MODA_HIP_ELAUNCH;
}

int moda_hip_uses_matrix_cores(const moda_hip_desc* d) {
  KArgs a;
  const int rc = fill_geometry(d, a);
  if (rc) return rc;
  return (use_mfma(d) || per_sequence(d)) ? 1 : 0;
}

const char* moda_hip_strerror(int code) {
  switch (code) {
    case MODA_HIP_OK: return "ok";
    case MODA_HIP_EINVAL: return "invalid descriptor field or missing tensor pointer";
    case MODA_HIP_EUNSUPPORTED: return "unsupported head dim / dtype / size";
    case MODA_HIP_EALIGN: return "tensor pointer or stride is not 16-byte aligned";
    case MODA_HIP_EWORKSPACE: return "workspace missing or too small";
    case MODA_HIP_ELAUNCH: return "HIP kernel launch failed";
    case MODA_HIP_EDEVICE: return "current device is not an MI355X-class (gfx950) GPU";
    case MODA_HIP_ESTATIC: return "problem needs more than the MODA_HIP_STATIC_WORKSPACE_BYTES of moda_hip_bwd_static";
    default: return "unknown error";
  }
}

int moda_hip_version(void) { return MODA_HIP_VERSION; }

}  // extern "C"
