// The operators' host path on torch tensors: argument contract, descriptor, output and workspace allocation, launch,
// and the autograd nodes.  A call of a small problem is bounded by this code (its kernels take 45 us forward and
// backward, the same steps written in Python took 270 us), so it is native: one call from Python per operator, the
// backward enters the kernels straight from the autograd engine.  Python module moda_amd._host.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <atomic>
#include <cmath>
#include <memory>
#include <optional>
#include <sstream>
#include <vector>

#include "../../include/moda_hip.h"
#include "tuning.h"

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
struct Call : c10::intrusive_ptr_target {
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
// what happens to dkd, dvd: overwritten; added to, slots >= depth_valid untouched; overwritten, those slots untouched
enum DepthGrads { kOverwrite = 0, kAccumulate = MODA_HIP_FLAG_ACCUMULATE_DEPTH_GRADS, kKeepSlots = MODA_HIP_FLAG_KEEP_DEPTH_SLOTS };

// `out`: gradient buffers to write to (an undefined entry is allocated here like all of them without `out`); `ws`:
// workspace to use, else allocated here.  `add_own_slot`: in, dk and dv are to have slot depth_valid of dkd, dvd added; out,
// whether they have.
Grads backward(const Call& c, Tensor q, Tensor k, Tensor v, Tensor kd, Tensor vd, Tensor o, Tensor lse, Tensor d_o, int stages,
               const Grads* out, Tensor ws, DepthGrads depth_grads, bool* add_own_slot = nullptr) {
  const bool accumulate = depth_grads == kAccumulate;
  CONTRACT(!accumulate || (out && (*out)[3].defined() && (*out)[4].defined()), "accumulate_depth needs the gradient buffers to add to");
  const bool own_slot = add_own_slot && *add_own_slot && !narrows(q);
  if (add_own_slot) *add_own_slot = false;
  if (narrows(q)) {
    // 16-bit gradients from the matrix kernels (without the accumulate flag: the slots without data come back as
    // zeros), widened into the caller's fp32 buffers or added to them
    Grads g = backward(c, narrowed(q), narrowed(k), narrowed(v), narrowed(kd), narrowed(vd), narrowed(o), lse, narrowed(d_o), stages,
                       nullptr, Tensor(), kOverwrite);
    for (int i = 0; i < 5; i++) {
      if (!out || !(*out)[i].defined()) {
        if (g[i].defined()) g[i] = g[i].to(at::kFloat);
      } else {
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
    if (out && (*out)[i].defined()) {
      g[i] = (*out)[i];
      CONTRACT(ins[i]->defined() && g[i].sizes() == ins[i]->sizes() && g[i].scalar_type() == ins[i]->scalar_type(),
               "reused gradient buffers must match their inputs in shape and dtype");
    } else if (ins[i]->defined()) {
      g[i] = at::empty(ins[i]->sizes(), ins[i]->options());
    }
  }
  Grads to = g;  // what the library sees: no depth gradients of an empty stream
  if (e.L == 0) kd = vd = to[3] = to[4] = Tensor();
  if (e.L > 0) d.flags = depth_grads;
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
  auto launch = [&] {
    return moda_hip_bwd_stages(&d, in_ptr(q), in_ptr(k), in_ptr(v), in_ptr(kd), in_ptr(vd), in_ptr(o), (const float*)in_ptr(lse),
                               in_ptr(d_o), out_ptr(to[0]), out_ptr(to[1]), out_ptr(to[2]), out_ptr(to[3]), out_ptr(to[4]),
                               out_ptr(ws), (size_t)ws.nbytes(), stages, stream_of(q));
  };
  if (own_slot) {
    d.flags |= MODA_HIP_FLAG_ADD_OWN_SLOT;
    const int rc = launch();
    if (rc != MODA_HIP_EUNSUPPORTED) {
      check_rc(rc, "moda_hip_bwd");
      *add_own_slot = true;
      return g;
    }
    d.flags &= ~MODA_HIP_FLAG_ADD_OWN_SLOT;
  }
  check_rc(launch(), "moda_hip_bwd");
  return g;
}

// What a backward node refuses.  The translator at the end of this file sees calls from Python only; the engine that runs
// the nodes hands a Python error on as it is and makes a RuntimeError of any other.
[[noreturn]] void throw_python(PyObject* type, const char* what) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(type, what);
  python_error error;
  error.persist();
  throw error;
}
template <typename F>
variable_list in_engine(F&& node) {
  try {
    return node();
  } catch (const ContractError& e) {
    throw_python(PyExc_AssertionError, e.what());
  } catch (const py::type_error& e) {
    throw_python(PyExc_TypeError, e.what());
  }
}

Tensor value(const OptTensor& x) { return x.has_value() ? *x : Tensor(); }
OptTensor optional(const Tensor& x) { return x.defined() ? OptTensor(x) : OptTensor(); }

// What a node keeps from its forward pass besides tensors, in the node's saved data: a tensor that owns it.  Compiled
// autograd, which replays nodes from a graph of its own, carries tensors through that graph; capsules it refuses.
template <typename State>
Tensor owning(const c10::intrusive_ptr<State>& state) {
  auto* kept = new c10::intrusive_ptr<State>(state);
  return at::from_blob(kept, {(int64_t)sizeof(*kept)}, [kept](void*) { delete kept; }, at::TensorOptions().dtype(at::kByte));
}
template <typename State>
c10::intrusive_ptr<State> owned(AutogradContext* ctx) {
  return *static_cast<const c10::intrusive_ptr<State>*>(ctx->saved_data["state"].toTensor().const_data_ptr());
}

// The autograd node of every operator (moda_v14.py:2649-2789, moda_v16.py:3456-3493, fda_v12.py:1207-1338,
// fla/ops/attn/parallel.py:632-675).  lse has no gradient and is no output of the node: it leaves by the pointer.
struct Attend : torch::autograd::Function<Attend> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd,
                               const OptTensor& vd, const c10::intrusive_ptr<Call>& call, Tensor* lse) {
    auto r = ::forward(*call, q, value(k), value(v), value(kd), value(vd));
    *lse = r.second;
    ctx->save_for_backward({q, value(k), value(v), value(kd), value(vd), r.first, r.second});
    ctx->saved_data["state"] = owning(call);
    ctx->set_materialize_grads(false);
    return {r.first};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return in_engine([&] { return gradients(ctx, grads); });
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const auto call = owned<Call>(ctx);
    if (!grads[0].defined()) return variable_list(7);
    Grads g = ::backward(*call, s[0], s[1], s[2], s[3], s[4], s[5], s[6], grads[0].to(s[5].scalar_type()), MODA_HIP_STAGE_ALL,
                         nullptr, Tensor(), kOverwrite);
    return {g[0], g[1], g[2], g[3], g[4], Tensor(), Tensor()};
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
  Tensor o, lse;
  {
    py::gil_scoped_release nogil;
    if (folded) check_folded_contract(mode, q, value(k), value(kd), value(vd), G);
    if (cu_seqlens.has_value()) packed = pack(*cu_seqlens, q, mode == MODA_HIP_PLAIN_GQA ? 1 : G);
    CONTRACT(group_rows == 0 || group_rows % G == 0,
             "To keep depth alignment consistent with backward, BT % moda_group_num must be 0");
    const bool has_depth = kd.has_value() && vd.has_value();  // one without the other counts as none
    const double sc = scale.has_value() ? *scale : 1.0 / std::sqrt((double)q.size(-1));
    o = Attend::apply(q, k, v, has_depth ? kd : OptTensor(), has_depth ? vd : OptTensor(),
                      make_call(mode, sc, G, chunk_tokens, depth_valid, std::move(packed)), &lse)[0];
  }
  return py::make_tuple(o, lse);
}

// ------------------------------------------------------------------------------------------------------------------
// depth stream of a training step (moda_amd/modules.py: DepthStream)
// ------------------------------------------------------------------------------------------------------------------

// Unit inner stride is all the slot kernels ask of a layer tensor.
Tensor layer_view(const Tensor& x) { return x.stride(3) == 1 || x.size(3) == 1 ? x : x.contiguous(); }

void check_layer(const Tensor& x, const Tensor& cache, int64_t L_total) {
  CONTRACT(x.dim() == 4, "a layer must be a [B, T, H, D] tensor");
  CONTRACT(cache.is_contiguous() && has_shape(cache, {x.size(0), x.size(1) * L_total, x.size(2), x.size(3)}),
           "cache must be a contiguous ", shape_text({x.size(0), x.size(1) * L_total, x.size(2), x.size(3)}), " tensor");
  CONTRACT(x.scalar_type() == cache.scalar_type() && x.device() == cache.device(), "layers and cache must share dtype and device");
}

// one layer's K and V into slot `slot` of the caches
void depth_push(const Tensor& k_in, const Tensor& v_in, const Tensor& cache_k, const Tensor& cache_v, int64_t slot, int64_t L_total) {
  check_layer(k_in, cache_k, L_total);
  check_layer(v_in, cache_v, L_total);
  CONTRACT(k_in.sizes() == v_in.sizes(), "a layer's k and v must agree in shape");
  CONTRACT(slot >= 0 && slot < L_total, "slots out of range");
  check_device(cache_k);
  const Tensor k = layer_view(k_in), v = layer_view(v_in);
  const moda_hip_strides sk = strides_of(k), sv = strides_of(v);
  c10::OptionalDeviceGuard guard(k.device());
  check_rc(moda_hip_depth_push(in_ptr(k), in_ptr(v), &sk, &sv, slot, L_total, k.size(0), k.size(1), k.size(2), k.size(3), dtype_code(k),
                               out_ptr(cache_k), out_ptr(cache_v), stream_of(k)),
           "moda_hip_depth_push");
}

// Cache and gradient buffers of one forward / backward pass, [B, T * L, H, D] each, allocated by the first push and never
// initialised: slots are read once written.  The nodes of a backward pass run from the last layer to the first; the first
// attention call among them overwrites the gradients of the slots it saw (`written`), the others, which saw fewer, add to
// theirs.  Another pass over a retained graph starts over, however much of the stream the one before it reached.
struct StreamBuffers : c10::intrusive_ptr_target {
  Tensor k, v, gk, gv;
  int64_t L = 0, written = 0;
  int pass = -1;  // the engine's number of the pass that `written` is about

  void enter_pass() {
    const int id = torch::autograd::get_current_graph_task_id();
    if (id != pass) written = 0;
    pass = id;
  }
};
// An attention call of the stream: what it saw, and the slot its own k, v were pushed to afterwards (-1: none).
struct StreamCall : c10::intrusive_ptr_target {
  Call call;
  c10::intrusive_ptr<StreamBuffers> buf;
  int64_t n = 0, slot = -1;
};

// A tensor that carries no data, only the order of the stream's operations (autograd runs them last to first).
Tensor order_token(const Tensor& like) { return at::empty({0}, like.options().dtype(at::kFloat)); }

// Attention over the sequence and the first n slots of the cache (which is not an autograd input: its gradient goes to
// the buffers).  Where the layer's k, v themselves went to a slot, their gradient is the call's own plus that slot's,
// complete by the time this node runs.
struct StreamAttend : torch::autograd::Function<StreamAttend> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& /*token*/,
                               const c10::intrusive_ptr<StreamCall>& call) {
    const bool depth = call->n > 0;
    auto r = ::forward(call->call, q, k, v, depth ? call->buf->k : Tensor(), depth ? call->buf->v : Tensor());
    ctx->save_for_backward({q, k, v, r.first, r.second});
    ctx->saved_data["state"] = owning(call);
    ctx->set_materialize_grads(false);
    return {r.first, order_token(q)};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return in_engine([&] { return gradients(ctx, grads); });
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const auto call = owned<StreamCall>(ctx);
    StreamBuffers& buf = *call->buf;
    buf.enter_pass();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &o = s[3], &lse = s[4];
    const Tensor d_o = grads[0].defined() ? grads[0].to(o.scalar_type()) : at::zeros_like(o);
    const int64_t n = call->n;
    Grads g;
    const bool join = call->slot >= 0 && call->slot < buf.written;  // later layers have seen this one's slot
    bool joined = join && call->slot == n;
    if (n > 0) {
      bool first = buf.written == 0;
      if (first && narrows(q)) {  // gradients computed in another type arrive as sums
        buf.gk.zero_();
        buf.gv.zero_();
        first = false;
      }
      const Grads into{Tensor(), Tensor(), Tensor(), buf.gk, buf.gv};
      g = ::backward(call->call, q, k, v, buf.k, buf.v, o, lse, d_o, MODA_HIP_STAGE_ALL, &into, Tensor(), first ? kKeepSlots : kAccumulate,
                     &joined);
      buf.written = std::max(buf.written, n);
    } else {
      g = ::backward(call->call, q, k, v, {}, {}, o, lse, d_o, MODA_HIP_STAGE_ALL, nullptr, Tensor(), kOverwrite);
      joined = false;
    }
    if (join && !joined) {
      const moda_hip_strides sk = strides_of(g[1]), sv = strides_of(g[2]);
      c10::OptionalDeviceGuard guard(k.device());
      check_rc(moda_hip_depth_slot_add(out_ptr(g[1]), out_ptr(g[2]), &sk, &sv, call->slot, buf.L, k.size(0), k.size(1), k.size(2), k.size(3),
                                       dtype_code(k), in_ptr(buf.gk), in_ptr(buf.gv), stream_of(k)),
               "moda_hip_depth_slot_add");
    }
    return {g[0], g[1], g[2], Tensor(), Tensor()};
  }
};

// K/V pushed without having been attended over by their own layer: their gradient is their slot's.
struct StreamPush : torch::autograd::Function<StreamPush> {
  static variable_list forward(AutogradContext* ctx, const Tensor& k, const Tensor& /*v*/, const Tensor& /*token*/,
                               const c10::intrusive_ptr<StreamCall>& call) {
    ctx->saved_data["state"] = owning(call);
    ctx->set_materialize_grads(false);
    return {order_token(k)};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list&) {
    const auto call = owned<StreamCall>(ctx);
    StreamBuffers& buf = *call->buf;
    buf.enter_pass();
    const int64_t B = buf.k.size(0), T = buf.k.size(1) / buf.L, H = buf.k.size(2), D = buf.k.size(3);
    auto slot = [&](const Tensor& g) {
      if (call->slot >= buf.written) return at::zeros({B, T, H, D}, g.options());
      return g.view({B, T, buf.L, H, D}).select(2, call->slot).contiguous();
    };
    return {slot(buf.gk), slot(buf.gv), Tensor(), Tensor()};
  }
};

class TrainStream {
 public:
  explicit TrainStream(int64_t max_layers) : buf_(c10::make_intrusive<StreamBuffers>()) { buf_->L = max_layers; }

  Tensor attend(const Tensor& q, const Tensor& k, const Tensor& v, double scale, int64_t G, int mode, int64_t chunk_tokens) {
    py::gil_scoped_release nogil;
    auto call = c10::make_intrusive<StreamCall>();
    call->call.mode = mode;
    call->call.scale = scale;
    call->call.G = G;
    call->call.chunk_tokens = chunk_tokens;
    if (n_ > 0) call->call.depth_valid = n_;
    call->buf = buf_;
    call->n = n_;
    const variable_list r = StreamAttend::apply(q, k, v, token_.defined() ? OptTensor(token_) : OptTensor(), call);
    token_ = r[1];
    last_ = r[0].requires_grad() ? call : c10::intrusive_ptr<StreamCall>();
    last_k_ = k;
    last_v_ = v;
    return r[0];
  }

  void push(const Tensor& k, const Tensor& v) {
    py::gil_scoped_release nogil;
    CONTRACT(k.dim() == 4, "k must be [B, T, H, D]");
    if (!buf_->k.defined()) {
      buf_->k = at::empty({k.size(0), k.size(1) * buf_->L, k.size(2), k.size(3)}, k.options());
      for (Tensor* x : {&buf_->v, &buf_->gk, &buf_->gv}) *x = at::empty_like(buf_->k);
    }
    depth_push(k, v, buf_->k, buf_->v, n_, buf_->L);
    if (at::GradMode::is_enabled()) {
      if (last_ && k.is_same(last_k_) && v.is_same(last_v_)) {
        last_->slot = n_;
      } else if (k.requires_grad() || v.requires_grad()) {
        auto call = c10::make_intrusive<StreamCall>();
        call->buf = buf_;
        call->slot = n_;
        token_ = StreamPush::apply(k, v, token_.defined() ? token_ : order_token(k), call)[0];
      }
    }
    last_.reset();
    last_k_ = last_v_ = Tensor();
    n_++;
  }

 private:
  c10::intrusive_ptr<StreamBuffers> buf_;
  c10::intrusive_ptr<StreamCall> last_;  // the latest attention call, until something is pushed
  Tensor token_, last_k_, last_v_;
  int64_t n_ = 0;
};

// ------------------------------------------------------------------------------------------------------------------
// a stack of blocks without gradients (moda_amd/modules.py: MoDAStack)
// ------------------------------------------------------------------------------------------------------------------

struct Block {
  Tensor norm1_w, norm1_b, q_w, q_b, kv_w, kv_b, proj_w, proj_b, norm2_w, norm2_b, fc1_w, fc1_b, fc2_w, fc2_b, kv_ffn_w, kv_ffn_b;
  double eps1, eps2;
};

// Whether the blocks run as native launches, by who is faster (four blocks, 64 .. 50 432 tokens, times of the modules over
// ours).  Up to width 512 we are: 1.2 - 3.9, replayed from a captured graph 1.13 - 1.6.  Above, the library's products are the
// faster kernels (width 1024, 12 608 tokens: 2246 against 1915 us; 2048: 7.6 against 5.6 ms; 4096, 197 tokens: 2294 against 908
// us), and what is left to gain is the modules' host time, some 170 us a block, where that is more than the launches take:
// width 1024 up to 3 152 tokens 1.1 - 2.1, 1280 up to 788 tokens 1.4 - 1.75 (3 152: 0.81), 1536 up to 197 tokens 1.16 - 1.5 (788:
// 0.97).  A captured graph has no host time: 1024 at 197 tokens replays at 0.89.
bool stack_runs_native(int64_t rows, int64_t width, void* stream) {
  if (width <= 512) return true;
  if (rows * width > (width <= 1024 ? 3 << 20 : width <= 1536 ? 1 << 20 : 0)) return false;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing((hipStream_t)stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
}

// Whether a block's dense part runs as one launch (moda_hip_block_tail): the kernel's range, and where it is the faster way.
bool tail_is_one_launch(bool fp16, int64_t rows, int64_t width, int64_t hidden, int64_t kv, int device) {
  if ((width != 128 && width != 256 && width != 384 && width != 512) || hidden % 128 != 0 || hidden >= 1 << 20 || kv % 16 != 0) return false;
  int compute_units = 0;
  return hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && compute_units > 0 &&
         moda::block_tail_pays(fp16, rows, width, hidden, kv, compute_units);
}

bool attention_joins(const Tensor& x, int64_t heads, int64_t kv_heads, int64_t slots, bool causal) {
  int compute_units = 0;
  return hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, x.get_device()) == hipSuccess && compute_units > 0 &&
         moda::attention_joins_tail(x.size(0), x.size(1), x.size(2), heads, kv_heads, slots, causal, compute_units);
}

// Forward pass of all blocks of one stack, launches only: the residual stream, one depth cache and four work tensors
// are all there is.  A layer's K and V are projected straight into their slot of the cache, where its own attention reads
// them as the sequence and later layers as a depth slot.  Returns nothing where a kernel's contract is not met (the
// caller then runs the modules one by one): 16-bit types, widths the linear kernel takes, 16-byte rows; or where the
// modules are faster.
std::optional<Tensor> stack_forward(const Tensor& x_in, const std::vector<Block>& blocks, int64_t heads, int64_t kv_heads, bool is_causal,
                                    int64_t chunk_tokens, bool post_norm) {
  const auto type = x_in.scalar_type();
  if (!x_in.is_cuda() || x_in.dim() != 3 || (type != at::kBFloat16 && type != at::kHalf) || x_in.numel() == 0) return {};
  const int64_t B = x_in.size(0), N = x_in.size(1), C = x_in.size(2), hd = C / heads, kv = kv_heads * hd, M = B * N;
  if (hd % 8 != 0 || hd > 256 || C % 64 != 0) return {};
  c10::OptionalDeviceGuard guard(x_in.device());
  void* stream = stream_of(x_in);
  if (!stack_runs_native(M, C, stream)) return {};
  const int64_t hidden = blocks[0].fc1_w.size(0);
  auto fits = [&](const Tensor& x, std::initializer_list<int64_t> shape) {
    return x.defined() && has_shape(x, shape) && x.scalar_type() == type && x.device() == x_in.device() && x.is_contiguous() &&
           (uintptr_t)x.const_data_ptr() % 16 == 0;
  };
  auto bias_fits = [&](const Tensor& x, int64_t n) { return !x.defined() || fits(x, {n}); };
  if (hidden % 64 != 0) return {};
  int64_t L = 0;
  for (const Block& b : blocks) {
    if (!(fits(b.norm1_w, {C}) && fits(b.norm1_b, {C}) && fits(b.norm2_w, {C}) && fits(b.norm2_b, {C}) && fits(b.q_w, {C, C}) &&
          fits(b.kv_w, {2 * kv, C}) && fits(b.proj_w, {C, C}) && fits(b.fc1_w, {hidden, C}) && fits(b.fc2_w, {C, hidden}) &&
          bias_fits(b.q_b, C) && bias_fits(b.kv_b, 2 * kv) && bias_fits(b.proj_b, C) && bias_fits(b.fc1_b, hidden) && bias_fits(b.fc2_b, C) &&
          bias_fits(b.kv_ffn_b, 2 * kv) && (!b.kv_ffn_w.defined() || fits(b.kv_ffn_w, {2 * kv, C}))))
      return {};
    L += b.kv_ffn_w.defined() ? 2 : 1;
  }
  const int dt = type == at::kHalf ? MODA_HIP_FP16 : MODA_HIP_BF16;
  const int64_t es = 2;
  const auto opt = x_in.options().requires_grad(false);
  const Tensor x0 = x_in.contiguous();
  if ((uintptr_t)x0.const_data_ptr() % 16 != 0) return {};
  const bool tails = tail_is_one_launch(type == at::kHalf, M, C, hidden, kv, x_in.get_device());
  // Attention and tail as one launch.  (Of chunks of more than 64 query rows the depth columns are summed from where a workgroup's own
  // begin: those keep the forward kernel's workgroups, and with them the bits.)
  const bool joined = tails && chunk_tokens * (heads / kv_heads) <= 64 && attention_joins(x_in, heads, kv_heads, L, is_causal || chunk_tokens > 0);
  Tensor x = at::empty({B, N, C}, opt), h = at::empty({M, C}, opt), q = at::empty({M, C}, opt), x1 = tails ? Tensor() : at::empty({M, C}, opt),
         hid = tails ? Tensor() : at::empty({M, hidden}, opt), ck = at::empty({B, N * L, kv}, opt), cv = at::empty({B, N * L, kv}, opt),
         lse = joined ? Tensor() : at::empty({M * heads}, opt.dtype(at::kFloat));
  auto part = [&](const Tensor& w, const Tensor& b, int64_t first, int64_t n, void* y, int64_t ldy) {
    return moda_hip_linear_part{(const char*)in_ptr(w) + first * w.size(1) * es, b.defined() ? (const char*)in_ptr(b) + first * es : nullptr, y,
                                ldy, n};
  };
  auto linear = [&](const void* in, int64_t K, std::initializer_list<moda_hip_linear_part> parts, const void* residual, bool gelu) {
    check_rc(moda_hip_linear(dt, M, K, in, K, parts.begin(), (int32_t)parts.size(), residual, C, gelu, stream), "moda_hip_linear");
  };
  auto norm = [&](const void* in, const Tensor& w, const Tensor& b, double eps, const Tensor& out) {
    check_rc(moda_hip_layer_norm(dt, M, C, in, in_ptr(w), in_ptr(b), (float)eps, out_ptr(out), stream), "moda_hip_layer_norm");
  };
  auto slot_of = [&](const Tensor& cache, int64_t slot) { return (char*)out_ptr(cache) + slot * kv * es; };

  moda_hip_desc d = {};
  d.struct_size = sizeof(d);
  d.dtype = dt;
  d.mode = chunk_tokens > 0 ? MODA_HIP_CHUNK_VISIBLE : is_causal ? MODA_HIP_CAUSAL : MODA_HIP_NONCAUSAL;
  d.B = B;
  d.T = N;
  d.H = kv_heads;
  d.G = heads / kv_heads;
  d.D = d.Dv = hd;
  d.chunk_tokens = chunk_tokens;
  d.scale = (float)(1.0 / std::sqrt((double)hd));
  d.q = d.o = {N * C, kv, hd};
  d.k = d.v = {N * L * kv, L * kv, hd};
  d.kd = d.vd = {N * L * kv, kv, hd};

  auto projections = [&](const Block& b, int64_t slot) {
    char *ks = slot_of(ck, slot), *vs = slot_of(cv, slot);
    return std::array<moda_hip_linear_part, 3>{part(b.q_w, b.q_b, 0, C, out_ptr(q), C), part(b.kv_w, b.kv_b, 0, kv, ks, L * kv),
                                               part(b.kv_w, b.kv_b, kv, kv, vs, L * kv)};
  };
  // packed copies of the weights, in the order proj, fc1, fc2, q, kv of each block (the first block's q, kv are not packed),
  // and the table behind them
  Tensor packed;
  const int64_t block_elems = C * C + 2 * hidden * C + C * C + 2 * kv * C;
  auto packed_at = [&](size_t i) { return (char*)out_ptr(packed) + (int64_t)i * block_elems * es; };
  if (tails) {
    packed = at::empty({(int64_t)blocks.size() * block_elems + MODA_HIP_GELU_TABLE_BYTES / es}, opt);
    std::vector<moda_hip_weight> weights;
    for (size_t i = 0; i < blocks.size(); i++) {
      const Block& b = blocks[i];
      char* to = packed_at(i);
      for (const Tensor* w : {&b.proj_w, &b.fc1_w, &b.fc2_w, &b.q_w, &b.kv_w}) {
        if (i > 0 || (w != &b.q_w && w != &b.kv_w)) weights.push_back({in_ptr(*w), to, w->size(0), w->size(1)});
        to += w->numel() * es;
      }
    }
    const Block& b = blocks[0];
    const moda_hip_norm_rows first = {in_ptr(x0), in_ptr(b.norm1_w), in_ptr(b.norm1_b), out_ptr(h), M, C, (float)b.eps1, dt};
    check_rc(post_norm ? moda_hip_pack_weights(weights.data(), (int32_t)weights.size(), packed_at(blocks.size()), stream)
                       : moda_hip_pack_weights_and_norm(weights.data(), (int32_t)weights.size(), packed_at(blocks.size()), &first, stream),
             "moda_hip_pack_weights");
  }

  const void* cur = in_ptr(x0);  // the residual stream
  int64_t n = 0;                 // filled slots
  bool projected = false;        // the block's q, k, v came with the previous block's last launch
  for (size_t i = 0; i < blocks.size(); i++) {
    const Block& b = blocks[i];
    if (!projected) {
      const void* in = cur;
      if (!post_norm) {
        if (!tails) norm(cur, b.norm1_w, b.norm1_b, b.eps1, h);  // (the first block's, else: with the weights)
        in = in_ptr(h);
      }
      const auto p = projections(b, n);
      linear(in, C, {p[0], p[1], p[2]}, nullptr, false);
    }
    d.L = n > 0 ? L : 0;
    d.L_valid = (int32_t)n;
    if (!joined)
      check_rc(moda_hip_fwd(&d, in_ptr(q), slot_of(ck, n), slot_of(cv, n), n > 0 ? in_ptr(ck) : nullptr, n > 0 ? in_ptr(cv) : nullptr,
                            out_ptr(h), (float*)out_ptr(lse), stream),
               "moda_hip_fwd");
    const int64_t slots = b.kv_ffn_w.defined() ? 2 : 1;
    if (tails) {
      moda_hip_block_tail_args t = {};
      t.struct_size = sizeof(t);
      t.dtype = dt;
      t.rows = M;
      t.width = C;
      t.hidden = hidden;
      t.gelu_table = packed_at(blocks.size());
      t.attention = in_ptr(h);
      t.residual = cur;
      t.x = out_ptr(x);
      t.proj_w = packed_at(i);
      t.proj_b = in_ptr(b.proj_b);
      t.fc1_w = packed_at(i) + C * C * es;
      t.fc1_b = in_ptr(b.fc1_b);
      t.fc2_w = packed_at(i) + (C + hidden) * C * es;
      t.fc2_b = in_ptr(b.fc2_b);
      const Block* next = i + 1 < blocks.size() ? &blocks[i + 1] : nullptr;
      t.post_norm = post_norm;
      t.mid_norm_w = in_ptr(post_norm ? b.norm1_w : b.norm2_w);
      t.mid_norm_b = in_ptr(post_norm ? b.norm1_b : b.norm2_b);
      t.mid_norm_eps = (float)(post_norm ? b.eps1 : b.eps2);
      if (post_norm || next) {
        t.end_norm_w = in_ptr(post_norm ? b.norm2_w : next->norm1_w);
        t.end_norm_b = in_ptr(post_norm ? b.norm2_b : next->norm1_b);
        t.end_norm_eps = (float)(post_norm ? b.eps2 : next->eps1);
      }
      if (next) {
        const auto p = projections(*next, n + slots);
        std::copy(p.begin(), p.end(), t.parts);
        const char* qkv = packed_at(i + 1) + (C + 2 * hidden) * C * es;
        t.parts[0].w = qkv;
        t.parts[1].w = qkv + C * C * es;
        t.parts[2].w = qkv + (C + kv) * C * es;
        t.n_parts = 3;
      }
      if (joined)
        check_rc(moda_hip_attend_block_tail(&d, in_ptr(q), slot_of(ck, n), slot_of(cv, n), n > 0 ? in_ptr(ck) : nullptr,
                                            n > 0 ? in_ptr(cv) : nullptr, &t, stream),
                 "moda_hip_attend_block_tail");
      else
        check_rc(moda_hip_block_tail(&t, stream), "moda_hip_block_tail");
      projected = true;
    } else {
      linear(in_ptr(h), C, {part(b.proj_w, b.proj_b, 0, C, out_ptr(x1), C)}, cur, false);
      if (post_norm) {
        norm(in_ptr(x1), b.norm1_w, b.norm1_b, b.eps1, x1);
        linear(in_ptr(x1), C, {part(b.fc1_w, b.fc1_b, 0, hidden, out_ptr(hid), hidden)}, nullptr, true);
        linear(in_ptr(hid), hidden, {part(b.fc2_w, b.fc2_b, 0, C, out_ptr(h), C)}, in_ptr(x1), false);
        norm(in_ptr(h), b.norm2_w, b.norm2_b, b.eps2, x);
      } else {
        norm(in_ptr(x1), b.norm2_w, b.norm2_b, b.eps2, h);
        linear(in_ptr(h), C, {part(b.fc1_w, b.fc1_b, 0, hidden, out_ptr(hid), hidden)}, nullptr, true);
        linear(in_ptr(hid), hidden, {part(b.fc2_w, b.fc2_b, 0, C, out_ptr(x), C)}, in_ptr(x1), false);
      }
    }
    cur = in_ptr(x);
    n++;
    if (b.kv_ffn_w.defined()) {
      linear(cur, C, {part(b.kv_ffn_w, b.kv_ffn_b, 0, kv, slot_of(ck, n), L * kv), part(b.kv_ffn_w, b.kv_ffn_b, kv, kv, slot_of(cv, n), L * kv)},
             nullptr, false);
      n++;
    }
  }
  return x;
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
  py::class_<TrainStream>(m, "TrainStream").def(py::init<int64_t>()).def("attend", &TrainStream::attend).def("push", &TrainStream::push);
  m.def("depth_push", &depth_push);
  m.def("stack_forward", [](const Tensor& x, const std::vector<std::vector<OptTensor>>& params, const std::vector<std::array<double, 2>>& eps,
                            int64_t heads, int64_t kv_heads, bool is_causal, int64_t chunk_tokens, bool post_norm) {
    std::vector<Block> blocks;
    for (size_t i = 0; i < params.size(); i++) {
      std::array<Tensor, 16> t;
      for (size_t j = 0; j < 16; j++) t[j] = value(params[i].at(j));
      blocks.push_back(Block{t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], t[13], t[14], t[15], eps[i][0], eps[i][1]});
    }
    py::gil_scoped_release nogil;
    std::optional<Tensor> y = stack_forward(x, blocks, heads, kv_heads, is_causal, chunk_tokens, post_norm);
    return y.has_value() ? OptTensor(*y) : OptTensor();
  });
  m.def("set_fp32_compute", [](int code) { fp32_compute.store(code); });
  m.def("pack", &pack);
  m.def("check_shapes", [](int mode, const Tensor& q, const OptTensor& k, const OptTensor& v, const OptTensor& kd, const OptTensor& vd,
                           int64_t G, const OptTensor& o, const OptTensor& d_o, const OptTensor& lse) {
    const Extent e = check_shapes(mode, q, value(k), value(v), value(kd), value(vd), G, value(o), value(d_o), value(lse));
    return py::make_tuple(e.T, e.L);
  });
  m.def("check_folded_contract", [](int mode, const Tensor& q, const OptTensor& k, const OptTensor& cached_k, const OptTensor& cached_v,
                                    int64_t G) { check_folded_contract(mode, q, value(k), value(cached_k), value(cached_v), G); });
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
                               value(kd), value(vd), o, lse, d_o, stages, out.has_value() ? &buffers : nullptr, value(ws),
                               accumulate ? kAccumulate : kOverwrite);
      for (int i = 0; i < 5; i++) r[i] = optional(g[i]);
    }
    return py::make_tuple(r[0], r[1], r[2], r[3], r[4]);
  });
}
