// The operators' host path on torch tensors: argument contract, descriptor, output and workspace allocation, launch,
// and the autograd nodes.  A call of a small problem is bounded by this code (its kernels take 45 us forward and
// backward, the same steps written in Python took 270 us), so it is native: one call from Python per operator, the
// backward enters the kernels straight from the autograd engine.  Python module moda_amd._host.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <atomic>
#include <cmath>
#include <memory>
#include <optional>
#include <sstream>
#include <vector>

#include "../../include/moda_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptTensor;

namespace {

// a violated argument contract: AssertionError in Python
struct ContractError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
template <typename... A>
[[noreturn]] void refuse(const A&... parts) {
  std::ostringstream s;
  (s << ... << parts);
  throw ContractError(s.str());
}
#define CONTRACT(cond, ...) \
  if (!(cond)) refuse(__VA_ARGS__)

std::string shape_text(std::initializer_list<int64_t> dims) {
  std::ostringstream s;
  s << '(';
  bool first = true;
  for (int64_t d : dims) {
    if (!first) s << ", ";
    first = false;
    s << d;
  }
  s << ')';
  return s.str();
}
bool has_shape(const Tensor& x, std::initializer_list<int64_t> dims) {
  return x.sizes() == c10::IntArrayRef(dims.begin(), dims.size());
}

// ------------------------------------------------------------------------------------------------------------------
// settings and arguments
// ------------------------------------------------------------------------------------------------------------------

// how fp32 tensors are computed: in fp32, or rounded to fp16 / bf16 (moda_amd.set_fp32_compute)
std::atomic<int> fp32_compute{MODA_HIP_FP32};

bool narrows(const Tensor& q) { return q.scalar_type() == at::kFloat && fp32_compute.load() != MODA_HIP_FP32; }
at::ScalarType narrow_type() { return fp32_compute.load() == MODA_HIP_FP16 ? at::kHalf : at::kBFloat16; }
Tensor narrowed(const Tensor& x) { return x.defined() ? x.to(narrow_type()) : x; }

// A packed variable-length batch (cu_seqlens): device offsets, what the launch is sized by, optional host offsets.
struct Packed {
  Tensor cu;
  int64_t n, max_len, total;
  std::vector<int32_t> host;  // empty: the library gets the device offsets only
};

// cu_seqlens as a caller passes it -> Packed.  One device-to-host copy: the longest sequence sizes the launch.
std::shared_ptr<Packed> pack(const Tensor& cu_seqlens, const Tensor& q, int64_t rows_per_token) {
  CONTRACT(q.size(0) == 1, "with cu_seqlens all sequences share one packed row axis: batch size must be 1");
  CONTRACT(cu_seqlens.dim() == 1 && cu_seqlens.numel() >= 1, "cu_seqlens must be a vector of n+1 offsets");
  const Tensor host = cu_seqlens.detach().to(at::kCPU, at::kLong).contiguous();
  const int64_t* h = host.const_data_ptr<int64_t>();
  auto p = std::make_shared<Packed>();
  p->n = host.numel() - 1;
  p->max_len = 0;
  bool sorted = h[0] == 0;
  for (int64_t i = 0; i < p->n; i++) {
    sorted = sorted && h[i + 1] >= h[i];
    p->max_len = std::max(p->max_len, h[i + 1] - h[i]);
  }
  CONTRACT(sorted, "cu_seqlens must start at 0 and not decrease");
  p->total = h[p->n];
  CONTRACT(p->total * rows_per_token == q.size(1), "cu_seqlens ends at ", p->total, " base tokens but q holds ", q.size(1),
           " rows (", rows_per_token, " per token)");
  p->host.assign(h, h + p->n + 1);
  p->cu = cu_seqlens.detach().to(q.device(), at::kInt).contiguous();
  return p;
}

// What a call is besides its tensors.
struct Call : torch::CustomClassHolder {
  int mode = 0;
  double scale = 1.0;
  int64_t G = 1, chunk_tokens = 0;
  std::optional<int64_t> depth_valid;  // none: every slot
  std::shared_ptr<Packed> packed;
};

int dtype_code(const Tensor& x) {
  switch (x.scalar_type()) {
    case at::kBFloat16: return MODA_HIP_BF16;
    case at::kHalf: return MODA_HIP_FP16;
    case at::kFloat: return MODA_HIP_FP32;
    default: {
      std::ostringstream s;
      s << "unsupported dtype " << x.scalar_type() << "; expected bf16, fp16 or fp32";
      throw py::type_error(s.str());
    }
  }
}

void check_rc(int rc, const char* what) {
  if (rc != 0) {
    std::ostringstream s;
    s << what << " failed: " << moda_hip_strerror(rc) << " (code " << rc << ")";
    throw std::runtime_error(s.str());
  }
}

void check_device(const Tensor& x) {
  if (!x.is_cuda())
    throw std::runtime_error("moda_amd operators run only on an MI355X (gfx950) device tensor; there is no CPU path");
}

void same_dtype(std::initializer_list<const Tensor*> xs) {
  const Tensor* first = nullptr;
  for (const Tensor* x : xs) {
    if (!x->defined()) continue;
    if (!first) first = x;
    if (x->scalar_type() != first->scalar_type()) {
      std::ostringstream s;
      s << "all tensors must share one dtype, got " << first->scalar_type() << " and " << x->scalar_type();
      throw py::type_error(s.str());
    }
  }
}

struct Extent {
  int64_t T, L;
};

// The C ABI takes bare pointers: it derives every extent from k (or q), G and the depth row count and cannot see what
// the buffers really hold.  A mismatch would be an out-of-bounds access on the device, so every extent is checked
// here, before any launch.
Extent check_shapes(int mode, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& kd, const Tensor& vd, int64_t G,
                    const Tensor& o, const Tensor& d_o, const Tensor& lse) {
  CONTRACT(q.dim() == 4, "q must be [B, rows, heads, D]");
  const int64_t B = q.size(0);
  CONTRACT(G >= 1, "moda_group_num must be positive");
  Extent e{0, 0};
  int64_t H;
  if (mode == MODA_HIP_DEPTH_ONLY) {
    CONTRACT(!k.defined() && !v.defined(), "depth-only attention takes no sequence k/v");
    CONTRACT(kd.defined() && vd.defined(), "depth-only attention needs the depth k/v");
    CONTRACT(q.size(1) % G == 0, "query rows must be a multiple of moda_group_num");
    CONTRACT(kd.dim() == 4, "depth k/v must be [B, T*L, H, D]");
    e.T = q.size(1) / G;
    H = kd.size(2);
    CONTRACT(q.size(2) == H, "q and depth k/v must have the same number of heads");
  } else {
    CONTRACT(k.defined() && v.defined() && k.dim() == 4 && v.dim() == 4, "k, v must be [B, T, H, D]");
    e.T = k.size(1);
    H = k.size(2);
    CONTRACT(k.size(0) == B && v.size(0) == B, "batch sizes of q, k, v differ");
    CONTRACT(v.size(1) == e.T && v.size(2) == H, "k and v must agree in tokens and heads");
    CONTRACT(k.size(3) == q.size(3), "q and k must share the head dim");
    if (mode == MODA_HIP_PLAIN_GQA) {
      CONTRACT(q.size(1) == e.T && q.size(2) == H * G, "plain GQA: q must be [B, T, H*G, D]");
    } else {
      CONTRACT(q.size(2) == H, "folded layout: q and k must have the same number of heads");
      CONTRACT(q.size(1) == e.T * G, "q holds ", q.size(1), " rows, expected T*moda_group_num = ", e.T * G);
    }
  }
  if (kd.defined() || vd.defined()) {
    CONTRACT(kd.defined() && vd.defined(), "depth k and v must be given together");
    CONTRACT(kd.dim() == 4 && vd.dim() == 4, "depth k/v must be [B, T*L, H, D]");
    CONTRACT(kd.size(0) == B && vd.size(0) == B, "depth k/v batch size differs from q");
    CONTRACT(kd.size(2) == H && vd.size(2) == H, "depth k/v head count mismatch");
    CONTRACT(kd.size(3) == q.size(3), "depth k must share q's head dim");
    CONTRACT(vd.size(1) == kd.size(1), "depth k and v must have the same number of rows");
    if (e.T > 0) {
      CONTRACT(kd.size(1) % e.T == 0, "depth rows must be T * L");
      e.L = kd.size(1) / e.T;
    } else {
      CONTRACT(kd.size(1) == 0, "depth rows must be T * L");
    }
    if (v.defined()) CONTRACT(vd.size(3) == v.size(3), "v and depth v must share the value head dim");
  }
  const int64_t Dv = (mode == MODA_HIP_DEPTH_ONLY ? vd : v).size(3);
  const Tensor* outs[2] = {&o, &d_o};
  for (int i = 0; i < 2; i++)
    if (outs[i]->defined())
      CONTRACT(has_shape(*outs[i], {B, q.size(1), q.size(2), Dv}), i == 0 ? "o" : "do", " must be ",
               shape_text({B, q.size(1), q.size(2), Dv}));
  if (lse.defined())
    CONTRACT(has_shape(lse, {B, q.size(1), q.size(2)}) && lse.scalar_type() == at::kFloat, "lse must be fp32 [B, rows, heads]");
  return e;
}

// `x` if the kernels can read it in place (unit inner stride, and for the matrix kernels 16-byte aligned rows), else a
// contiguous copy -- the reference's @contiguous (fla/utils.py:130-164) copied every non-contiguous input.
// vec16 = false: the vector-ALU kernels, which load element by element and take any non-negative strides.
Tensor usable(const Tensor& x, bool vec16) {
  if (!x.defined()) return x;
  bool ok = x.dim() == 4 && (x.stride(3) == 1 || x.size(3) == 1);
  const int64_t es = x.element_size(), m = 16 / es;
  for (int i = 0; ok && i < 3; i++) ok = x.stride(i) >= 0 && (!vec16 || x.stride(i) % m == 0);
  if (ok && vec16)
    ok = (uintptr_t)x.const_data_ptr() % 16 == 0 && x.stride(1) * es < (1 << 24);  // row offsets inside a tile are 32-bit
  return ok ? x : x.contiguous();
}

moda_hip_strides strides_of(const Tensor& x) {
  return x.defined() ? moda_hip_strides{x.stride(0), x.stride(1), x.stride(2)} : moda_hip_strides{0, 0, 0};
}
const void* in_ptr(const Tensor& x) { return x.defined() ? x.const_data_ptr() : nullptr; }
void* out_ptr(const Tensor& x) { return x.defined() ? x.mutable_data_ptr() : nullptr; }
void* stream_of(const Tensor& x) { return (void*)c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

// the geometry part of the descriptor (no strides)
moda_hip_desc geometry(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& kd, const Tensor& vd,
                       const Extent& e) {
  moda_hip_desc d = {};
  const bool depth_only = c.mode == MODA_HIP_DEPTH_ONLY;
  d.struct_size = sizeof(d);
  d.dtype = dtype_code(q);
  d.mode = c.mode;
  d.B = q.size(0);
  d.T = e.T;
  d.H = (depth_only ? kd : k).size(2);
  d.G = c.G;
  d.D = q.size(3);
  d.Dv = (depth_only ? vd : v).size(3);
  d.L = e.L;
  if (c.depth_valid.has_value() && e.L > 0) {
    CONTRACT(*c.depth_valid >= 1 && *c.depth_valid <= e.L, "depth_valid must be in [1, ", e.L, "], got ", *c.depth_valid);
    d.L_valid = (int32_t)*c.depth_valid;
  }
  if (c.packed) {
    d.B = c.packed->n;
    d.T = c.packed->max_len;
    d.cu_seqlens = c.packed->cu.const_data_ptr<int32_t>();
    d.total_tokens = c.packed->total;
    d.cu_seqlens_host = c.packed->host.empty() ? nullptr : c.packed->host.data();
  }
  d.chunk_tokens = c.chunk_tokens;
  d.scale = (float)c.scale;
  return d;
}

// ------------------------------------------------------------------------------------------------------------------
// forward and backward
// ------------------------------------------------------------------------------------------------------------------

std::pair<Tensor, Tensor> forward(const Call& c, Tensor q, Tensor k, Tensor v, Tensor kd, Tensor vd) {
  if (narrows(q)) {
    auto r = forward(c, narrowed(q), narrowed(k), narrowed(v), narrowed(kd), narrowed(vd));
    return {r.first.to(at::kFloat), r.second};
  }
  const Extent e = check_shapes(c.mode, q, k, v, kd, vd, c.G, {}, {}, {});
  check_device(q);
  same_dtype({&q, &k, &v, &kd, &vd});
  moda_hip_desc d = geometry(c, q, k, v, kd, vd, e);
  const bool vec16 = moda_hip_uses_matrix_cores(&d) == 1;
  for (Tensor* x : {&q, &k, &v, &kd, &vd}) *x = usable(*x, vec16);
  if (e.L == 0) kd = vd = Tensor();
  Tensor o = at::empty({q.size(0), q.size(1), q.size(2), d.Dv}, q.options());
  Tensor lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  d.q = strides_of(q);
  d.k = strides_of(k);
  d.v = strides_of(v);
  d.kd = strides_of(kd);
  d.vd = strides_of(vd);
  d.o = strides_of(o);
  c10::OptionalDeviceGuard guard(q.device());
  check_rc(moda_hip_fwd(&d, in_ptr(q), in_ptr(k), in_ptr(v), in_ptr(kd), in_ptr(vd), out_ptr(o), (float*)out_ptr(lse),
                        stream_of(q)),
           "moda_hip_fwd");
  return {o, lse};
}

typedef std::array<Tensor, 5> Grads;  // dq, dk, dv, dkd, dvd

// `out`: gradient buffers to write to (undefined entries where the input is), else allocated here; `ws`: workspace to
// use, else allocated here; `accumulate`: dkd, dvd of `out` are added to (slots >= depth_valid untouched).
Grads backward(const Call& c, Tensor q, Tensor k, Tensor v, Tensor kd, Tensor vd, Tensor o, Tensor lse, Tensor d_o, int stages,
               const Grads* out, Tensor ws, bool accumulate) {
  CONTRACT(!accumulate || (out && (*out)[3].defined() && (*out)[4].defined()), "accumulate_depth needs the gradient buffers to add to");
  if (narrows(q)) {
    // 16-bit gradients from the matrix kernels (without the accumulate flag: the slots without data come back as
    // zeros), widened into the caller's fp32 buffers or added to them
    Grads g = backward(c, narrowed(q), narrowed(k), narrowed(v), narrowed(kd), narrowed(vd), narrowed(o), lse, narrowed(d_o), stages,
                       nullptr, Tensor(), false);
    for (int i = 0; i < 5; i++) {
      if (!out) {
        if (g[i].defined()) g[i] = g[i].to(at::kFloat);
      } else if ((*out)[i].defined()) {
        if (accumulate && i >= 3)
          (*out)[i].add_(g[i]);
        else
          (*out)[i].copy_(g[i]);
        g[i] = (*out)[i];
      }
    }
    return g;
  }
  const Extent e = check_shapes(c.mode, q, k, v, kd, vd, c.G, o, d_o, lse);
  check_device(q);
  same_dtype({&q, &k, &v, &kd, &vd, &o, &d_o});
  moda_hip_desc d = geometry(c, q, k, v, kd, vd, e);
  const bool vec16 = moda_hip_uses_matrix_cores(&d) == 1;
  for (Tensor* x : {&q, &k, &v, &kd, &vd, &o, &d_o}) *x = usable(*x, vec16);
  lse = lse.contiguous();
  const Tensor* ins[5] = {&q, &k, &v, &kd, &vd};
  Grads g;
  for (int i = 0; i < 5; i++) {
    if (out) {
      g[i] = (*out)[i];
      CONTRACT(g[i].defined() == ins[i]->defined() &&
                   (!g[i].defined() || (g[i].sizes() == ins[i]->sizes() && g[i].scalar_type() == ins[i]->scalar_type())),
               "reused gradient buffers must match their inputs in shape and dtype");
    } else if (ins[i]->defined()) {
      g[i] = at::empty(ins[i]->sizes(), ins[i]->options());
    }
  }
  Grads to = g;  // what the library sees: no depth gradients of an empty stream
  if (e.L == 0) kd = vd = to[3] = to[4] = Tensor();
  if (accumulate && e.L > 0) d.flags = MODA_HIP_FLAG_ACCUMULATE_DEPTH_GRADS;
  d.q = strides_of(q);
  d.k = strides_of(k);
  d.v = strides_of(v);
  d.kd = strides_of(kd);
  d.vd = strides_of(vd);
  d.o = strides_of(o);
  d.d_o = strides_of(d_o);
  d.dq = strides_of(to[0]);
  d.dk = strides_of(to[1]);
  d.dv = strides_of(to[2]);
  d.dkd = strides_of(to[3]);
  d.dvd = strides_of(to[4]);
  c10::OptionalDeviceGuard guard(q.device());
  if (!ws.defined())
    ws = at::empty({std::max<int64_t>((int64_t)moda_hip_bwd_workspace_bytes(&d), 4)}, q.options().dtype(at::kByte));
  check_rc(moda_hip_bwd_stages(&d, in_ptr(q), in_ptr(k), in_ptr(v), in_ptr(kd), in_ptr(vd), in_ptr(o), (const float*)in_ptr(lse),
                               in_ptr(d_o), out_ptr(to[0]), out_ptr(to[1]), out_ptr(to[2]), out_ptr(to[3]), out_ptr(to[4]),
                               out_ptr(ws), (size_t)ws.nbytes(), stages, stream_of(q)),
           "moda_hip_bwd");
  return g;
}

Tensor value(const OptTensor& x) { return x.has_value() ? *x : Tensor(); }
OptTensor optional(const Tensor& x) { return x.defined() ? OptTensor(x) : OptTensor(); }

// The autograd node of every operator (moda_v14.py:2649-2789, moda_v16.py:3456-3493, fda_v12.py:1207-1338,
// fla/ops/attn/parallel.py:632-675): gradient into lse ignored.
struct Attend : torch::autograd::Function<Attend> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd,
                               const OptTensor& vd, const c10::intrusive_ptr<Call>& call) {
    auto r = ::forward(*call, q, value(k), value(v), value(kd), value(vd));
    ctx->save_for_backward({q, value(k), value(v), value(kd), value(vd), r.first, r.second});
    ctx->saved_data["call"] = c10::IValue::make_capsule(call);
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({r.second});
    return {r.first, r.second};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
    if (!grads[0].defined()) return variable_list(6);
    Grads g = ::backward(*call, s[0], s[1], s[2], s[3], s[4], s[5], s[6], grads[0].to(s[5].scalar_type()), MODA_HIP_STAGE_ALL,
                         nullptr, Tensor(), false);
    return {g[0], g[1], g[2], g[3], g[4], Tensor()};
  }
};

c10::intrusive_ptr<Call> make_call(int mode, double scale, int64_t G, int64_t chunk_tokens, std::optional<int64_t> depth_valid,
                                   std::shared_ptr<Packed> packed) {
  auto c = c10::make_intrusive<Call>();
  c->mode = mode;
  c->scale = scale;
  c->G = G;
  c->chunk_tokens = chunk_tokens;
  c->depth_valid = depth_valid;
  c->packed = std::move(packed);
  return c;
}

// The argument contract of the folded operators (moda_v14.py:2817-2871, moda_v16.py:3496-3565; depth-only:
// fda_v12.py:1370-1437), which comes before the extents are looked at one by one.
void check_folded_contract(int mode, const Tensor& q, const Tensor& k, const Tensor& cached_k, const Tensor& cached_v, int64_t G) {
  const bool depth_only = mode == MODA_HIP_DEPTH_ONLY, has_depth = cached_k.defined() && cached_v.defined();
  const Tensor& keys = depth_only ? cached_k : k;
  CONTRACT(!depth_only || has_depth, "Flash Depth Attention requires cached_k/cached_v");
  CONTRACT(q.dim() == 4 && keys.dim() == 4, "q and ", depth_only ? "cached_k" : "k", " must be 4-dimensional");
  const int64_t B = q.size(0), T_q = q.size(1), H = keys.size(2);
  if (depth_only) {
    CONTRACT(G > 0, "moda_group_num must be positive");
    CONTRACT(T_q % G == 0, "T_q must be divisible by moda_group_num");
  }
  CONTRACT(q.size(2) == H,
           "Implicit head-dimension GQA is not allowed. Please fold grouping only into `moda_group_num`: use q.shape[2] == ",
           depth_only ? "cached_k" : "k", ".shape[2] and set T_q = T_kv * moda_group_num.");
  const int64_t T = depth_only ? T_q / G : k.size(1);
  if (!depth_only) {
    CONTRACT(G <= 1 || T_q == T * G, "When moda_group_num > 1, T_q must equal T_kv * moda_group_num");
    CONTRACT(G > 1 || T_q == T, "When moda_group_num=1, T_q must equal T_kv");
  }
  if (!has_depth) return;
  CONTRACT(cached_k.dim() == 4 && cached_v.dim() == 4 && cached_k.size(0) == B && cached_v.size(0) == B,
           "cached_k/v must be [B, T_kv * L, H, D] with q's batch size");
  CONTRACT(cached_k.size(2) == H && cached_v.size(2) == H, "cached_k/v head count mismatch");
  if (T == 0) return;
  CONTRACT(cached_k.size(1) % T == 0, "cached_k time dimension must be T_kv * L");
  CONTRACT(!depth_only || cached_k.size(1) > 0, "Flash Depth Attention requires at least one depth slot per token");
  CONTRACT(cached_v.size(1) == cached_k.size(1), "cached_v shape mismatch");
}

// One operator call from Python: (o, lse), differentiable in q, k, v, kd, vd.  `folded`: check the contract of the
// folded operators first; `group_rows`: rows that G must divide (0: no such rule); `scale` none: D ** -0.5.
py::tuple attend(int mode, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd, const OptTensor& vd,
                 std::optional<double> scale, int64_t G, int64_t chunk_tokens, std::optional<int64_t> depth_valid,
                 const OptTensor& cu_seqlens, std::shared_ptr<Packed> packed, bool folded, int64_t group_rows) {
  variable_list r;
  {
    py::gil_scoped_release nogil;
    if (folded) check_folded_contract(mode, q, value(k), value(kd), value(vd), G);
    if (cu_seqlens.has_value()) packed = pack(*cu_seqlens, q, mode == MODA_HIP_PLAIN_GQA ? 1 : G);
    CONTRACT(group_rows == 0 || group_rows % G == 0,
             "To keep depth alignment consistent with backward, BT % moda_group_num must be 0");
    const bool has_depth = kd.has_value() && vd.has_value();  // one without the other counts as none
    const double sc = scale.has_value() ? *scale : 1.0 / std::sqrt((double)q.size(-1));
    r = Attend::apply(q, k, v, has_depth ? kd : OptTensor(), has_depth ? vd : OptTensor(),
                      make_call(mode, sc, G, chunk_tokens, depth_valid, std::move(packed)));
  }
  return py::make_tuple(r[0], r[1]);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const ContractError& e) {
      PyErr_SetString(PyExc_AssertionError, e.what());
    }
  });
  py::class_<Packed, std::shared_ptr<Packed>>(m, "Packed")
      .def(py::init([](const Tensor& cu, int64_t n, int64_t max_len, int64_t total, std::vector<int32_t> host) {
        return std::make_shared<Packed>(Packed{cu, n, max_len, total, std::move(host)});
      }))
      .def_readonly("cu", &Packed::cu)
      .def_readonly("n", &Packed::n)
      .def_readonly("max_len", &Packed::max_len)
      .def_readonly("total", &Packed::total)
      .def_readonly("host", &Packed::host);
  m.def("set_fp32_compute", [](int code) { fp32_compute.store(code); });
  m.def("pack", &pack);
  m.def("check_shapes", [](int mode, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd, const OptTensor& vd,
                           int64_t G, const OptTensor& o, const OptTensor& d_o, const OptTensor& lse) {
    const Extent e = check_shapes(mode, q, value(k), value(v), value(kd), value(vd), G, value(o), value(d_o), value(lse));
    return py::make_tuple(e.T, e.L);
  });
  m.def("attend", &attend);
  m.def("forward", [](int mode, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd, const OptTensor& vd,
                      double scale, int64_t G, int64_t chunk_tokens, std::optional<int64_t> depth_valid,
                      std::shared_ptr<Packed> packed) {
    std::pair<Tensor, Tensor> r;
    {
      py::gil_scoped_release nogil;
      r = forward(*make_call(mode, scale, G, chunk_tokens, depth_valid, std::move(packed)), q, value(k), value(v), value(kd), value(vd));
    }
    return py::make_tuple(r.first, r.second);
  });
  m.def("backward", [](int mode, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd, const OptTensor& vd,
                       const Tensor& o, const Tensor& lse, const Tensor& d_o, double scale, int64_t G, int64_t chunk_tokens,
                       std::optional<int64_t> depth_valid, std::shared_ptr<Packed> packed, int stages,
                       std::optional<std::array<OptTensor, 5>> out, const OptTensor& ws, bool accumulate) {
    std::array<OptTensor, 5> r;
    {
      py::gil_scoped_release nogil;
      Grads buffers;
      if (out.has_value())
        for (int i = 0; i < 5; i++) buffers[i] = value((*out)[i]);
      const Grads g = backward(*make_call(mode, scale, G, chunk_tokens, depth_valid, std::move(packed)), q, value(k), value(v),
                               value(kd), value(vd), o, lse, d_o, stages, out.has_value() ? &buffers : nullptr, value(ws), accumulate);
      for (int i = 0; i < 5; i++) r[i] = optional(g[i]);
    }
    return py::make_tuple(r[0], r[1], r[2], r[3], r[4]);
  });
}
