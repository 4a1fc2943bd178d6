// Host path between torch and libfta.so in C++: what attention() and TriangleAttention run for tensors that the
// kernels read in place.  A call checks its arguments, allocates outputs and launches, without going through
// the Python interpreter, and its backward runs in the autograd thread without taking the interpreter lock
// for more than one flag.  Anything it does not take -- wrong types or shapes, layouts that need a copy,
// another device than the current one, a thread whose operations something else watches -- it leaves to the
// Python path by returning None, which copies, records or raises as documented there.
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <atomic>
#include <unordered_set>

#include "fta.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Strided views with a unit last stride, rows on 16-byte boundaries.
bool readable(const Tensor& t) {
  const auto s = t.strides();
  const int64_t n = t.dim();
  if (s[n - 1] != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (s[i] % 8 != 0) return false;
  return true;
}
// t if the kernels read it in place, else a copy of its own (contiguous() would leave a dense tensor off the 16-byte
// boundary where it is: a gradient that the backward of a concatenation cut out, for instance).
Tensor readable_copy(const Tensor& t) { return readable(t) ? t : t.clone(at::MemoryFormat::Contiguous); }
Tensor packed_copy(const Tensor& t) {
  return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone(at::MemoryFormat::Contiguous);
}
// A tensor saved in the forward.  Hooks may have packed it and may return it with other strides, which the copies above
// take; another tensor than they were given (kept in fewer bits, left on the host) must not reach a kernel, which
// reads it by the sizes of the call.
const Tensor& saved(const Tensor& t, at::IntArrayRef sizes, at::ScalarType dtype, const at::Device& device) {
  TORCH_CHECK(t.defined() && t.layout() == at::kStrided && t.device() == device && t.scalar_type() == dtype && t.sizes() == sizes,
              "a hook for saved tensors returned a tensor of another type, device or size than it was given");
  return t;
}
// A plain tensor on the current GPU: no subclass or transform that has to see the operations, and no tangent (the
// operator has no forward-mode derivative: the Python function says so, here the output would come without one).
bool plain(const Tensor& t, int device) {
  return t.is_cuda() && t.device().index() == device && t.layout() == at::kStrided && !t._fw_grad(/*level=*/0).defined() &&
         !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchVmapMode,
                                                   c10::DispatchKey::Functionalize}));
}
// A torch.Tensor or Parameter itself.  A subclass, which may do without __torch_dispatch__, keeps its type through
// the Python path.
bool exact_tensor(py::handle h) { return THPVariable_CheckExact(h.ptr()); }
// Whether something watches or rewrites this thread's operations: jit tracing, a Python dispatch mode, a functorch
// transform (which need not show in this call's tensors).  The launches below are no operations, so a trace would hold
// the allocations of the outputs alone, and replay them.
bool watched() {
  return torch::jit::tracer::isTracing() ||
         c10::impl::tls_local_dispatch_key_set().included_.has_any(
             c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Functionalize}));
}
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

fta_tensor5 t5(const Tensor& t) {
  const auto s = t.strides();
  return fta_tensor5{t.data_ptr(), {s[0], s[1], s[2], s[3]}};
}
fta_tensor4 t4(const Tensor& t) {
  const auto s = t.strides();
  return fta_tensor4{t.data_ptr(), {s[0], s[1], s[2]}};
}
void check(int rc) {
  TORCH_CHECK(rc == FTA_OK, "libfta: ", fta_strerror(rc), " (status ", rc, ")");
}
// A forward call whose arguments the library refused (before any launch): left to the Python path, which raises its errors.
struct Refused {};
void check_forward(int rc) {
  if (rc < 0) throw Refused{};
  check(rc);
}

fta_options make_options(at::ScalarType dtype, double dropout_p, uint64_t seed, bool precise) {
  fta_options o{};
  o.dtype = dtype == at::kBFloat16 ? FTA_DTYPE_BF16 : FTA_DTYPE_F16;
  o.dropout_p = (float)dropout_p;
  o.seed = seed;
  o.precise = precise ? 1 : 0;
  return o;
}

// Whether rows of L2 keys run forward and backward with these options: asked once per length and kind.
bool length_supported(int64_t L2, int64_t D, const fta_options& o) {
  static std::atomic<uint8_t> known[2][2][2][FTA_MAX_L2 + 1];  // head dim, type, dropout: 0 unknown, 1 no, 2 yes
  if (L2 < 1 || L2 > FTA_MAX_L2 || (D != 32 && D != 64) || !(o.dropout_p < 1.f)) return false;  // (not what the table is about)
  auto& k = known[D == 64][o.dtype == FTA_DTYPE_BF16][o.dropout_p > 0.f][L2];
  uint8_t v = k.load(std::memory_order_relaxed);
  if (v == 0) {
    v = fta_seq_len_supported_ex((int)L2, (int)D, &o) ? 2 : 1;
    k.store(v, std::memory_order_relaxed);
  }
  return v == 2;
}

// The globals of the Python module a call came from, for its backward.  One reference per module is kept for good: the
// backward may run after the module itself is gone.  (Called under the interpreter lock.)
int64_t held(py::dict globals) {
  static std::unordered_set<PyObject*> kept;
  if (kept.insert(globals.ptr()).second) globals.inc_ref();
  return (int64_t) reinterpret_cast<intptr_t>(globals.ptr());
}
// The module switch PRECISE_BACKWARD of the Python module whose globals these are, at this moment.
bool precise_now(PyObject* globals) {
  py::gil_scoped_acquire gil;
  PyObject* v = PyDict_GetItemString(globals, "PRECISE_BACKWARD");
  return v != nullptr && PyObject_IsTrue(v) == 1;
}

// ---- attention -----------------------------------------------------------------------------------------
// Outputs of the forward, straight from the allocator: nothing watches this thread's operations here (see `watched`), every element is
// overwritten, and two trips through the dispatcher were a fifth of what a call costs the host.  A dense tensor's strides
// are kept, as at::empty_like keeps them; any other layout is left to that.
Tensor output_like(const Tensor& t) {
  if (!t.is_non_overlapping_and_dense()) return at::empty_like(t);
  return Tensor(at::detail::empty_strided_cuda(t.sizes(), t.strides(), t.scalar_type(), t.device()));
}
int attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, double scale, const fta_options& opt,
                      Tensor& o, Tensor& lse) {
  o = output_like(q);
  if (!readable(o)) o = at::empty(q.sizes(), q.options());
  const auto n = q.sizes();
  lse = Tensor(at::detail::empty_cuda({n[0], n[1], n[2], n[3]}, at::kFloat, q.device(), std::nullopt));
  const fta_tensor5 tq = t5(q), tk = t5(k), tv = t5(v), to = t5(o);
  const fta_tensor4 tb = t4(b);
  return fta_fwd_ex(&tq, &tk, &tv, &tb, &to, lse.data_ptr<float>(), (int)n[0], (int)n[1], (int)n[2], (int)n[3], (int)n[4],
                    (float)scale, &opt, current_stream(q));
}

struct Attention : public torch::autograd::Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, double scale,
                        double dropout_p, int64_t seed, int64_t globals) {
    Tensor o, lse;
    check_forward(attention_forward(q, k, v, b, scale, make_options(q.scalar_type(), dropout_p, (uint64_t)seed, false), o, lse));
    ctx->save_for_backward({q, k, v, o, b, lse});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["dropout_p"] = dropout_p;
    ctx->saved_data["seed"] = seed;
    ctx->saved_data["globals"] = globals;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::NoGradGuard no_grad;
    const variable_list s = ctx->get_saved_variables();
    const Tensor dout = readable_copy(grads[0]);  // (of the output's type, sizes and device: the engine sees to that)
    const at::Device dev = dout.device();
    const at::ScalarType dt = dout.scalar_type();
    c10::OptionalDeviceGuard guard(dev);
    const auto n = dout.sizes();
    const Tensor q = readable_copy(saved(s[0], n, dt, dev)), k = readable_copy(saved(s[1], n, dt, dev)),
                 v = readable_copy(saved(s[2], n, dt, dev)), o = readable_copy(saved(s[3], n, dt, dev)),
                 lse = packed_copy(saved(s[5], n.slice(0, 4), at::kFloat, dev));
    Tensor b = saved(s[4], {n[0], n[1], n[3], n[3]}, dt, dev);
    if (b.stride(3) != 1) b = b.contiguous();
    const fta_options opt = make_options(q.scalar_type(), ctx->saved_data["dropout_p"].toDouble(),
                                         (uint64_t)ctx->saved_data["seed"].toInt(),
                                         precise_now(reinterpret_cast<PyObject*>(ctx->saved_data["globals"].toInt())));
    const int B = (int)n[0], H = (int)n[1], L1 = (int)n[2], L2 = (int)n[3], D = (int)n[4];
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), db = at::empty_like(b);
    const size_t bytes = fta_bwd_workspace_bytes_ex(B, H, L1, L2, D, &opt);
    const Tensor ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    const fta_tensor5 tq = t5(q), tk = t5(k), tv = t5(v), to = t5(o), tdo = t5(dout), tdq = t5(dq), tdk = t5(dk), tdv = t5(dv);
    const fta_tensor4 tb = t4(b), tdb = t4(db);
    check(fta_bwd_ex(&tq, &tk, &tv, &tb, &to, lse.data_ptr<float>(), &tdo, &tdq, &tdk, &tdv, &tdb, ws.data_ptr(), bytes, B, H, L1, L2,
                     D, (float)ctx->saved_data["scale"].toDouble(), &opt, current_stream(q)));
    return {dq, dk, dv, db, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

py::object attention(py::handle qh, py::handle kh, py::handle vh, py::handle bh, double scale, double dropout_p, int64_t seed,
                     py::dict globals) {
  const py::object none = py::none();
  for (const py::handle h : {qh, kh, vh, bh})
    if (!exact_tensor(h)) return none;
  const Tensor &q = THPVariable_Unpack(qh.ptr()), &k = THPVariable_Unpack(kh.ptr()), &v = THPVariable_Unpack(vh.ptr()),
               &b = THPVariable_Unpack(bh.ptr());
  if (watched()) return none;
  const at::ScalarType dt = q.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16) || k.scalar_type() != dt || v.scalar_type() != dt || b.scalar_type() != dt) return none;
  if (q.dim() != 5 || b.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes() || !q.is_cuda()) return none;
  const auto n = q.sizes(), nb = b.sizes();
  if ((n[4] != 32 && n[4] != 64) || nb[0] != n[0] || nb[1] != n[1] || nb[2] != n[3] || nb[3] != n[3]) return none;
  if (!(dropout_p >= 0.0 && dropout_p < 1.0) || q.numel() == 0) return none;
  const int dev = (int)c10::hip::current_device();
  if (!plain(q, dev) || !plain(k, dev) || !plain(v, dev) || !plain(b, dev)) return none;
  if (!readable(q) || !readable(k) || !readable(v) || b.stride(3) != 1) return none;
  const fta_options opt = make_options(dt, dropout_p, (uint64_t)seed, false);
  if (!length_supported(n[3], n[4], opt)) return none;
  try {
    if (!wants_grad({&q, &k, &v, &b})) {
      Tensor o, lse;
      at::AutoDispatchBelowADInplaceOrView below;
      check_forward(attention_forward(q, k, v, b, scale, opt, o, lse));
      return py::cast(o);
    }
    return py::cast(Attention::apply(q, k, v, b, scale, dropout_p, seed, held(globals)));
  } catch (const Refused&) {
    return none;
  }
}

// ---- the block -----------------------------------------------------------------------------------------
struct BlockCall {
  int64_t C, H, D, seed, starting;
  double eps, dropout_p;
};

// The sizes of the weights: norm weight, norm bias, q, k, v, b, gate weight, gate bias, output weight, output bias.
struct WeightSizes {
  int64_t rows[10], cols[10];
  explicit WeightSizes(const BlockCall& c)
      : rows{c.C, c.C, c.H * c.D, c.H * c.D, c.H * c.D, c.H, c.H * c.D, c.H * c.D, c.C, c.C},
        cols{0, 0, c.C, c.C, c.C, c.C, c.C, 0, c.H * c.D, 0} {}
  c10::SmallVector<int64_t, 2> operator[](int n) const {
    return cols[n] ? c10::SmallVector<int64_t, 2>{rows[n], cols[n]} : c10::SmallVector<int64_t, 2>{rows[n]};
  }
};

// weights in that order
fta_block block_args(const Tensor& z, const Tensor& mask, const Tensor* w, const BlockCall& c, bool precise) {
  fta_block b{};
  b.B = (int)z.size(0); b.L = (int)z.size(1); b.C = (int)c.C; b.H = (int)c.H; b.D = (int)c.D;
  b.dtype = z.scalar_type() == at::kFloat ? FTA_DTYPE_F32 : z.scalar_type() == at::kBFloat16 ? FTA_DTYPE_BF16 : FTA_DTYPE_F16;
  b.eps = (float)c.eps;
  b.sm_scale = (float)(1.0 / std::sqrt((double)c.D));
  b.dropout_p = (float)c.dropout_p;
  b.seed = (uint64_t)c.seed;
  b.precise = precise ? 1 : 0;
  b.z = z.data_ptr();
  b.z_stride[0] = z.stride(0);
  b.z_stride[1] = z.stride(c.starting ? 1 : 2);
  b.z_stride[2] = z.stride(c.starting ? 2 : 1);
  b.mask = mask.defined() ? mask.data_ptr() : nullptr;
  const void** dst[10] = {&b.norm_weight, &b.norm_bias, &b.wq, &b.wk, &b.wv, &b.wb, &b.wg, &b.bg, &b.wo, &b.bo};
  for (int i = 0; i < 10; ++i) *dst[i] = w[i].defined() ? w[i].data_ptr() : nullptr;
  return b;
}
void node_strides(const Tensor& t, int64_t starting, int64_t (&s)[3]) {
  s[0] = t.stride(0);
  s[1] = t.stride(starting ? 1 : 2);
  s[2] = t.stride(starting ? 2 : 1);
}
int block_forward(const Tensor& z, const fta_block& b, int64_t starting, Tensor& out, Tensor& state) {
  out = at::empty(z.sizes(), z.options());
  state = at::empty({(int64_t)fta_block_state_bytes(&b)}, z.options().dtype(at::kByte));
  int64_t os[3];
  node_strides(out, starting, os);
  return fta_block_fwd(&b, out.data_ptr(), os, state.data_ptr(), current_stream(z));
}

// Gradients that are to be differentiated again, through a node that refuses it: the kernels' results have no graph, and a
// loss made of them would lose that part of its gradient without a word.
variable_list not_twice(variable_list grads) {
  at::AutoGradMode enabled(true);
  for (Tensor& t : grads)
    if (t.defined()) t = t.detach().set_requires_grad(true);
  const auto node = std::make_shared<torch::autograd::DelayedError>("TriangleAttention cannot be differentiated twice", (int64_t)grads.size());
  return (*node)(std::move(grads));
}

struct Block : public torch::autograd::Function<Block> {
  static Tensor forward(AutogradContext* ctx, const Tensor& z, const std::optional<Tensor>& mask, const Tensor& w0, const Tensor& w1,
                        const Tensor& w2, const Tensor& w3, const Tensor& w4, const Tensor& w5, const Tensor& w6,
                        const std::optional<Tensor>& w7, const Tensor& w8, const std::optional<Tensor>& w9, int64_t C, int64_t H,
                        int64_t D, int64_t seed, int64_t starting, double eps, double dropout_p, int64_t globals) {
    const Tensor w[10] = {w0, w1, w2, w3, w4, w5, w6, w7.value_or(Tensor()), w8, w9.value_or(Tensor())};
    const Tensor m = mask.value_or(Tensor());
    const BlockCall c{C, H, D, seed, starting, eps, dropout_p};
    Tensor out, state;
    check_forward(block_forward(z, block_args(z, m, w, c, false), starting, out, state));
    variable_list keep{z, m, state};
    for (const Tensor& t : w) keep.push_back(t);
    ctx->save_for_backward(keep);
    ctx->saved_data["i"] = c10::List<int64_t>({C, H, D, seed, starting, globals});
    ctx->saved_data["d"] = c10::List<double>({eps, dropout_p});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool create_graph = at::GradMode::is_enabled();
    at::NoGradGuard no_grad;
    const variable_list s = ctx->get_saved_variables();
    const auto i = ctx->saved_data["i"].toIntVector();
    const auto d = ctx->saved_data["d"].toDoubleVector();
    const BlockCall c{i[0], i[1], i[2], i[3], i[4], d[0], d[1]};
    const Tensor dout = readable_copy(grads[0]);
    const at::Device dev = dout.device();
    const at::ScalarType dt = dout.scalar_type();
    c10::OptionalDeviceGuard guard(dev);
    const Tensor z = readable_copy(saved(s[0], dout.sizes(), dt, dev));
    const Tensor mask = s[1].defined() ? packed_copy(saved(s[1], {z.size(0), z.size(1)}, dt, dev)) : Tensor();
    const WeightSizes sizes(c);
    Tensor w[10];
    for (int n = 0; n < 10; ++n)
      if (s[3 + n].defined()) w[n] = packed_copy(saved(s[3 + n], sizes[n], dt, dev));
    const fta_block b = block_args(z, mask, w, c, precise_now(reinterpret_cast<PyObject*>(i[5])));
    const Tensor state = packed_copy(saved(s[2], {(int64_t)fta_block_state_bytes(&b)}, at::kByte, dev));
    Tensor dz = at::empty_like(z), dw[10];
    if (!readable(dz)) dz = at::empty(z.sizes(), z.options());
    fta_block_grads g{};
    g.z = dz.data_ptr();
    node_strides(dz, c.starting, g.z_stride);
    void** dst[10] = {&g.norm_weight, &g.norm_bias, &g.wq, &g.wk, &g.wv, &g.wb, &g.wg, &g.bg, &g.wo, &g.bo};
    for (int n = 0; n < 10; ++n)
      if (w[n].defined()) {
        dw[n] = at::empty(w[n].sizes(), w[n].options());
        *dst[n] = dw[n].data_ptr();
      }
    const size_t bytes = fta_block_bwd_workspace_bytes(&b);
    const Tensor ws = at::empty({(int64_t)bytes}, z.options().dtype(at::kByte));
    int64_t ds[3];
    node_strides(dout, c.starting, ds);
    check(fta_block_bwd(&b, state.data_ptr(), dout.data_ptr(), ds, &g, ws.data_ptr(), bytes, current_stream(z)));
    variable_list out{dz, Tensor()};
    for (const Tensor& t : dw) out.push_back(t);
    if (create_graph) out = not_twice(std::move(out));
    out.resize(2 + 10 + 8);
    return out;
  }
};

py::object block(py::handle zh, py::handle key_mask, const std::vector<py::object>& weights, int64_t H, int64_t D,
                 bool starting, double eps, double dropout_p, std::optional<int64_t> given_seed, py::dict globals) {
  const py::object none = py::none();
  if (!exact_tensor(zh)) return none;
  const Tensor& z = THPVariable_Unpack(zh.ptr());
  if (watched()) return none;
  const at::ScalarType dt = z.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16 && dt != at::kFloat) || z.dim() != 4 || z.size(1) != z.size(2) || z.numel() == 0) return none;
  if (!z.is_cuda() || at::autocast::is_autocast_enabled(at::kCUDA) || weights.size() != 10) return none;
  const int dev = (int)c10::hip::current_device();
  BlockCall c{z.size(3), H, D, given_seed.value_or(0), starting ? 1 : 0, eps, dropout_p};
  if (!plain(z, dev) || !readable(z) || !(dropout_p >= 0.0 && dropout_p < 1.0)) return none;
  const WeightSizes sizes(c);
  Tensor w[10];
  for (int n = 0; n < 10; ++n) {
    if (weights[n].is_none()) {
      if (n != 7 && n != 9) return none;
      continue;
    }
    if (!exact_tensor(weights[n])) return none;
    w[n] = THPVariable_Unpack(weights[n].ptr());
    if (w[n].scalar_type() != dt || !plain(w[n], dev) || !w[n].is_contiguous() || reinterpret_cast<uintptr_t>(w[n].data_ptr()) % 16 != 0)
      return none;
    if (w[n].sizes() != at::IntArrayRef(sizes[n])) return none;
  }
  Tensor mask;
  if (!key_mask.is_none()) {
    if (!exact_tensor(key_mask)) return none;
    const Tensor& m = THPVariable_Unpack(key_mask.ptr());
    if (m.requires_grad() || !plain(m, dev) || m.dim() != 2 || m.size(0) != z.size(0) || m.size(1) != z.size(1)) return none;
    mask = m.to(dt).contiguous();
  }
  fta_block b = block_args(z, mask, w, c, false);
  if (!length_supported(b.L, D, make_options(dt, dropout_p, 0, false)) || fta_block_check(&b) != FTA_OK) return none;
  if (dropout_p > 0.0 && !given_seed) {  // (drawn only now that the call is taken: the Python path draws its own)
    c.seed = py::cast<int64_t>(globals["_draw_seed"]());
    b.seed = (uint64_t)c.seed;
  }
  auto opt_t = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  try {
    if (!wants_grad({&z, &w[0], &w[1], &w[2], &w[3], &w[4], &w[5], &w[6], &w[7], &w[8], &w[9]})) {
      Tensor out, state;
      at::AutoDispatchBelowADInplaceOrView below;
      check_forward(block_forward(z, b, c.starting, out, state));
      return py::cast(out);
    }
    return py::cast(Block::apply(z, opt_t(mask), w[0], w[1], w[2], w[3], w[4], w[5], w[6], opt_t(w[7]), w[8], opt_t(w[9]), c.C, H, D, c.seed,
                                 c.starting, eps, dropout_p, held(globals)));
  } catch (const Refused&) {
    return none;
  }
}

}  // namespace

PYBIND11_MODULE(fta_native, m) {
  m.doc() = "C++ host path of attention() and TriangleAttention; None = not taken, use the Python path";
  m.attr("built_for") = "fta_native built for torch " FTA_TORCH_VERSION;  // (read from the file before it is loaded, too)
  m.def("attention", &attention, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("b_pw"), py::arg("sm_scale"),
        py::arg("dropout_p") = 0.0, py::arg("seed") = 0, py::arg("globals"));
  m.def("block", &block);
}
