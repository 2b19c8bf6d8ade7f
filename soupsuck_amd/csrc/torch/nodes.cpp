// Autograd nodes of the per-layer entry points in native code, over the C ABI.
//
// A Python autograd.Function costs more host time than these layers' kernels run:
// forward and backward of one frozen projection took 165 us of host time against 89 us
// of kernels at T = 101 (7B down) and 124 us at T = 2048 (q / o), most of it interpreter
// work on two threads that take turns with the interpreter lock.  With these nodes the
// pairs take 80 and 115 us, and the row norms of 16384 x 1536 90 us instead of 144.  The nodes here do what
// the Python ones of the same layers do (kernels/nf4_gemm.py, kernels/rownorm.py,
// lora.py): same kernels, buffers, saved tensors, dtypes and error texts.  Arguments are
// checked by the callers in Python before they get here; the Python nodes stay for timing
// hooks and for the variants that need more (generic ranks, unaligned codes).
//
// Everything a node keeps is a tensor (no raw pointer outlives a call); the streams are
// torch's current ones at the call, which for a backward is its forward's.
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/extension.h>

#include "soupsuck_amd.h"

namespace {

using at::Tensor;
// An absent tensor argument of a node (apply() takes no undefined Tensor).
using OptionalTensor = std::optional<at::Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

void check(int rc, const char* name) {
  if (rc == SS_OK) return;
  const std::string text = ss_last_error();
  if (rc == SS_ERR_INVALID_ARGUMENT) TORCH_CHECK_VALUE(false, name, ": ", text);
  TORCH_CHECK(false, name, " failed (", rc, "): ", text);
}

template <class T>
T* ptr(const Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}
uint16_t* half_ptr(const Tensor& t) { return ptr<uint16_t>(t); }

int code_of(at::ScalarType t) {
  TORCH_CHECK_VALUE(t == at::kHalf || t == at::kFloat, "unsupported dtype ", t,
                    "; expected float16 or float32");
  return t == at::kHalf ? SS_F16 : SS_F32;
}
int code_of(const Tensor& t) { return t.defined() ? code_of(t.scalar_type()) : SS_F16; }

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dtype) {
  return at::empty(sizes, like.options().dtype(dtype));
}

Tensor workspace(size_t bytes, const Tensor& like) {
  return bytes ? empty({(int64_t)bytes}, like, at::kByte) : Tensor();
}

// Gradients of a node that cannot be differentiated again: as Python's
// once_differentiable, they fail when a graph through them is used.
variable_list once(const variable_list& incoming, variable_list grads) {
  bool track = at::GradMode::is_enabled();
  bool wanted = false;
  for (const Tensor& g : incoming) wanted |= g.defined() && g.requires_grad();
  if (!track || !wanted) return grads;
  for (Tensor& g : grads) {
    if (!g.defined()) continue;
    auto fail = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", 1);
    g = (*fail)({g.detach().requires_grad_(true)})[0];
  }
  return grads;
}

// One frozen NF4 weight: codes, block codes, second-level scales and table, offset.
struct Weight {
  Tensor packed, absmax, absmax2, code2, offset;
  int64_t n, k;
  std::vector<Tensor> tensors() const { return {packed, absmax, absmax2, code2, offset}; }
  static Weight from(const std::vector<Tensor>& t, int64_t n, int64_t k) {
    return Weight{t[0], t[1], t[2], t[3], t[4], n, k};
  }
};

#define WEIGHT_ARGS(w)                                                                   \
  ptr<uint8_t>((w).packed), ptr<uint8_t>((w).absmax), ptr<float>((w).absmax2),           \
      ptr<float>((w).code2), ptr<float>((w).offset), (w).n, (w).k

Tensor nf4_forward(const Tensor& x, const Weight& w, const Tensor& bias) {
  std::vector<int64_t> sizes = x.sizes().vec();
  sizes.back() = w.n;
  Tensor y = empty(sizes, x, at::kHalf);
  const int64_t t = x.numel() / w.k;
  if (t == 0) return y;
  const size_t bytes = ss_nf4_gemm_workspace_size(t, w.n, w.k);
  const Tensor ws = workspace(bytes, x);
  check(ss_nf4_gemm_fwd(half_ptr(x), w.k, t, WEIGHT_ARGS(w), half_ptr(bias), half_ptr(y), w.n,
                        ptr<void>(ws), bytes, stream_of(x)),
        "ss_nf4_gemm_fwd");
  return y;
}

// dx [.., K] of g [.., N].
Tensor nf4_dx(const Tensor& g, const Weight& w) {
  std::vector<int64_t> sizes = g.sizes().vec();
  sizes.back() = w.k;
  Tensor dx = empty(sizes, g, at::kHalf);
  const int64_t t = g.numel() / w.n;
  if (t == 0) return dx;
  const size_t bytes = ss_nf4_gemm_workspace_size(t, w.n, w.k);
  const Tensor ws = workspace(bytes, g);
  check(ss_nf4_gemm_dx(half_ptr(g), w.n, t, WEIGHT_ARGS(w), half_ptr(dx), w.k, 0,
                       ptr<void>(ws), bytes, stream_of(g)),
        "ss_nf4_gemm_dx");
  return dx;
}

// ------------------------------------------------------------ frozen projection

struct NF4Linear : public Function<NF4Linear> {
  static Tensor forward(AutogradContext* ctx, Tensor x, Tensor packed, const Weight& w,
                        const OptionalTensor& bias) {
    ctx->save_for_backward({packed});
    ctx->saved_data["w"] = w.tensors();
    ctx->saved_data["n"] = w.n;
    ctx->saved_data["k"] = w.k;
    return nf4_forward(x, w, bias.value_or(Tensor()));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();  // version check, hooks
    Weight w = Weight::from(ctx->saved_data["w"].toTensorVector(), ctx->saved_data["n"].toInt(),
                            ctx->saved_data["k"].toInt());
    w.packed = saved[0];
    Tensor dx;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(grads[0].device());
      dx = nf4_dx(grads[0].contiguous(), w);
    }
    return once(grads, {dx, Tensor(), Tensor(), Tensor()});
  }
};

// The node is needed: t has a gradient to come, or a forward-mode tangent (which it refuses).
bool tracked(const Tensor& t) {
  return t.defined() &&
         ((at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined());
}

Tensor nf4_linear(const Tensor& x, const Tensor& packed, const Tensor& absmax,
                  const Tensor& absmax2, const Tensor& code2, const Tensor& offset, int64_t n,
                  int64_t k, const OptionalTensor& bias) {
  c10::DeviceGuard guard(x.device());
  const Weight w{packed, absmax, absmax2, code2, offset, n, k};
  if (!tracked(x)) return nf4_forward(x, w, bias.value_or(Tensor()));
  return NF4Linear::apply(x, packed, w, bias);
}

// --------------------------------------------------- add-RMSNorm, RMSNorm (rownorm.py)

struct NormForward {
  Tensor s, y, rstd;
};

NormForward norm_forward(const Tensor& x, const Tensor& delta, const Tensor& weight, double eps,
                         at::ScalarType s_dtype, at::ScalarType y_dtype) {
  const int64_t h = x.size(-1);
  const int64_t rows = x.numel() / h;
  NormForward f;
  f.y = empty(x.sizes(), x, y_dtype);
  f.rstd = empty({rows}, x, at::kFloat);
  void* stream = stream_of(x);
  if (!delta.defined()) {
    f.s = x;
    if (rows) {
      const int64_t stride = x.dim() == 2 ? x.stride(0) : x.view({rows, h}).stride(0);
      check(ss_rmsnorm_fwd(ptr<void>(x), code_of(x), stride, ptr<void>(weight), code_of(weight),
                           weight.stride(0), ptr<void>(f.y), code_of(f.y), ptr<float>(f.rstd),
                           rows, h, (float)eps, stream),
            "ss_rmsnorm_fwd");
    }
    return f;
  }
  f.s = empty(x.sizes(), x, s_dtype);
  if (rows)
    check(ss_add_rmsnorm_fwd(ptr<void>(x), code_of(x), ptr<void>(delta), code_of(delta),
                             ptr<void>(weight), code_of(weight), weight.stride(0), ptr<void>(f.s),
                             code_of(f.s), ptr<void>(f.y), code_of(f.y), ptr<float>(f.rstd), rows,
                             h, (float)eps, stream),
          "ss_add_rmsnorm_fwd");
  return f;
}

struct RowNorm : public Function<RowNorm> {
  static variable_list forward(AutogradContext* ctx, Tensor x, const OptionalTensor& added,
                               Tensor weight, double eps, at::ScalarType s_dtype, at::ScalarType exact_dtype,
                               at::ScalarType y_dtype) {
    const Tensor delta = added.value_or(Tensor());
    const NormForward f = norm_forward(x, delta, weight, eps, s_dtype, y_dtype);
    ctx->saved_data["x"] = (int64_t)x.scalar_type();
    ctx->saved_data["d"] = delta.defined() ? (int64_t)delta.scalar_type() : -1;
    ctx->saved_data["half"] = exact_dtype == at::kHalf;
    ctx->save_for_backward({f.s, weight, f.rstd});
    ctx->set_materialize_grads(false);
    if (!delta.defined()) return {f.y};
    return {f.s, f.y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const int64_t d_code = ctx->saved_data["d"].toInt();
    const bool add = d_code >= 0;
    const Tensor g_s = add ? grads[0] : Tensor(), g_y = add ? grads[1] : grads[0];
    variable_list out(7);
    if (!g_s.defined() && !g_y.defined()) return out;
    const variable_list saved = ctx->get_saved_variables();
    const bool want_x = ctx->needs_input_grad(0), want_d = add && ctx->needs_input_grad(1);
    const bool want_w = ctx->needs_input_grad(add ? 2 : 1);  // counts tensors that are there
    {
      at::NoGradGuard no_grad;
      const Tensor &s = saved[0], &weight = saved[1], &rstd = saved[2];
      c10::DeviceGuard guard(s.device());
      const int64_t h = s.size(-1);
      const int64_t rows = s.numel() / h;
      Tensor dx, dd, dw;
      if (want_x) dx = empty(s.sizes(), s, (at::ScalarType)ctx->saved_data["x"].toInt());
      if (want_d) dd = empty(s.sizes(), s, (at::ScalarType)d_code);
      const Tensor s2 = rows ? s.reshape({rows, h}).contiguous() : s;
      const Tensor gs2 = g_s.defined() ? g_s.reshape({rows, h}) : Tensor();
      const Tensor gy2 = g_y.defined() ? g_y.reshape({rows, h}) : Tensor();
      const int64_t gs_row = gs2.defined() ? gs2.stride(0) : 0;
      const int64_t gs_col = gs2.defined() ? gs2.stride(1) : 0;
      const int64_t gy_row = gy2.defined() ? gy2.stride(0) : 0;
      const int64_t gy_col = gy2.defined() ? gy2.stride(1) : 0;
      void* stream = stream_of(s);
      if (want_w && rows && gy2.defined()) {
        dw = at::empty(weight.sizes(), weight.options());
        const Tensor partial = empty({ss_add_rmsnorm_dgamma_waves(rows), h}, s, at::kFloat);
        check(ss_add_rmsnorm_bwd_dgamma(
                  ptr<void>(s2), code_of(s2), ptr<void>(weight), code_of(weight),
                  weight.stride(0), ptr<float>(rstd), ptr<void>(gs2), code_of(gs2), gs_row,
                  gs_col, ptr<void>(gy2), code_of(gy2), gy_row, gy_col, ptr<void>(dx),
                  code_of(dx), ptr<void>(dd), code_of(dd), ctx->saved_data["half"].toBool(),
                  ptr<float>(partial), ptr<void>(dw), code_of(dw), rows, h, stream),
              "ss_add_rmsnorm_bwd_dgamma");
      } else {
        if (rows && (want_x || want_d))
          check(ss_add_rmsnorm_bwd(ptr<void>(s2), code_of(s2), ptr<void>(weight), code_of(weight),
                                   weight.stride(0), ptr<float>(rstd), ptr<void>(gs2),
                                   code_of(gs2), gs_row, gs_col, ptr<void>(gy2), code_of(gy2),
                                   gy_row, gy_col, ptr<void>(dx), code_of(dx), ptr<void>(dd),
                                   code_of(dd), rows, h, stream),
                "ss_add_rmsnorm_bwd");
        // No output gradient reaches the weight (or there are no rows): zero.
        if (want_w) dw = at::zeros(weight.sizes(), weight.options());
      }
      out[0] = dx;
      out[1] = dd;
      out[2] = dw;
    }
    return once(grads, out);
  }
};

std::vector<Tensor> row_norm(const Tensor& x, const OptionalTensor& delta,
                             const Tensor& weight, double eps, bool half_out) {
  c10::DeviceGuard guard(x.device());
  const Tensor d = delta.value_or(Tensor());
  const at::ScalarType s_dtype =
      d.defined() ? at::promote_types(x.scalar_type(), d.scalar_type()) : x.scalar_type();
  const at::ScalarType exact = at::promote_types(s_dtype, weight.scalar_type());
  const at::ScalarType y_dtype = half_out ? at::kHalf : exact;
  if (!tracked(x) && !tracked(d) && !tracked(weight)) {
    const NormForward f = norm_forward(x, d, weight, eps, s_dtype, y_dtype);
    if (!d.defined()) return {f.y};
    return {f.s, f.y};
  }
  return RowNorm::apply(x, delta, weight, eps, s_dtype, exact, y_dtype);
}

// -------------------------------------------------- fused QLoRA projection (lora.py)

Tensor as_half(const Tensor& w) { return w.to(at::kHalf).contiguous(); }

struct Dropout {
  bool on;
  uint64_t seed;
  double p;
};

struct QLoRA : public Function<QLoRA> {
  static Tensor forward(AutogradContext* ctx, Tensor x, Tensor lora_a, Tensor lora_b,
                        const Weight& w, const OptionalTensor& bias_arg, double scaling,
                        const Dropout& drop, const OptionalTensor& workspace,
                        const Tensor& rank_ws) {
    const Tensor bias = bias_arg.value_or(Tensor()), ws = workspace.value_or(Tensor());
    const int64_t t = x.numel() / w.k;
    const Tensor x2d = x.view({t, w.k});
    const Tensor a16 = as_half(lora_a), b16 = as_half(lora_b);
    const Tensor z = empty({t, 16}, x, at::kHalf);
    std::vector<int64_t> sizes = x.sizes().vec();
    sizes.back() = w.n;
    Tensor y = empty(sizes, x, at::kHalf);
    const size_t ws_bytes = ws.defined() ? ws.numel() : 0;
    void* stream = stream_of(x);
    if (!drop.on)
      check(ss_qlora_forward(half_ptr(x2d), w.k, t, WEIGHT_ARGS(w), half_ptr(bias),
                             half_ptr(a16), half_ptr(b16), (float)scaling, half_ptr(z),
                             half_ptr(y), w.n, ptr<void>(ws), ws_bytes, ptr<void>(rank_ws),
                             rank_ws.numel(), stream),
            "ss_qlora_forward");
    else
      check(ss_qlora_forward_dropout(half_ptr(x2d), w.k, t, WEIGHT_ARGS(w), half_ptr(bias),
                                     half_ptr(a16), half_ptr(b16), (float)scaling, drop.seed,
                                     (float)drop.p, half_ptr(z), half_ptr(y), w.n, ptr<void>(ws),
                                     ws_bytes, ptr<void>(rank_ws), rank_ws.numel(), stream),
            "ss_qlora_forward_dropout");
    ctx->save_for_backward({x2d, z, a16, b16});
    ctx->saved_data["w"] = w.tensors();
    ctx->saved_data["scratch"] =
        ws.defined() ? std::vector<Tensor>{rank_ws, ws} : std::vector<Tensor>{rank_ws};
    ctx->saved_data["ints"] = std::vector<int64_t>{
        w.n, w.k, (int64_t)lora_a.scalar_type(), (int64_t)lora_b.scalar_type(), drop.on,
        (int64_t)drop.seed};
    ctx->saved_data["reals"] = std::vector<double>{scaling, drop.p};
    ctx->saved_data["shape"] = x.sizes().vec();
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const std::vector<int64_t> ints = ctx->saved_data["ints"].toIntVector();
    const std::vector<double> reals = ctx->saved_data["reals"].toDoubleVector();
    const Weight w = Weight::from(ctx->saved_data["w"].toTensorVector(), ints[0], ints[1]);
    const std::vector<Tensor> scratch = ctx->saved_data["scratch"].toTensorVector();
    const Tensor rank_ws = scratch[0], ws = scratch.size() > 1 ? scratch[1] : Tensor();
    variable_list out(9);
    {
      at::NoGradGuard no_grad;
      const Tensor &x2d = saved[0], &z = saved[1], &a16 = saved[2], &b16 = saved[3];
      c10::DeviceGuard guard(x2d.device());
      const int64_t t = x2d.size(0), n = w.n, k = w.k;
      const Tensor g = grads[0].reshape({t, n}).to(at::kHalf).contiguous();
      // dZ (used inside the call), dB and dA in one allocation; dX apart
      const Tensor rank = empty({t * 16 + n * 16 + 16 * k}, g, at::kHalf);
      const Tensor dz = rank.narrow(0, 0, t * 16);
      const Tensor db = rank.narrow(0, t * 16, n * 16).view({n, 16});
      const Tensor da = rank.narrow(0, t * 16 + n * 16, 16 * k).view({16, k});
      const Tensor dx = empty(ctx->saved_data["shape"].toIntVector(), g, at::kHalf);
      const size_t ws_bytes = ws.defined() ? ws.numel() : 0;
      void* stream = stream_of(g);
      if (!ints[4])
        check(ss_qlora_backward(half_ptr(g), n, t, WEIGHT_ARGS(w), half_ptr(x2d), k, half_ptr(z),
                                half_ptr(a16), half_ptr(b16), (float)reals[0], half_ptr(dx), k,
                                half_ptr(dz), half_ptr(da), half_ptr(db), ptr<void>(ws), ws_bytes,
                                ptr<void>(rank_ws), rank_ws.numel(), stream),
              "ss_qlora_backward");
      else
        check(ss_qlora_backward_dropout(half_ptr(g), n, t, WEIGHT_ARGS(w), half_ptr(x2d), k,
                                        half_ptr(z), half_ptr(a16), half_ptr(b16),
                                        (float)reals[0], (uint64_t)ints[5], (float)reals[1],
                                        half_ptr(dx), k, half_ptr(dz), half_ptr(da),
                                        half_ptr(db), ptr<void>(ws), ws_bytes,
                                        ptr<void>(rank_ws), rank_ws.numel(), stream),
              "ss_qlora_backward_dropout");
      out[0] = dx;
      out[1] = da.to((at::ScalarType)ints[2]);
      out[2] = db.to((at::ScalarType)ints[3]);
    }
    return once(grads, out);
  }
};

Tensor qlora(const Tensor& x, const Tensor& lora_a, const Tensor& lora_b, const Tensor& packed,
             const Tensor& absmax, const Tensor& absmax2, const Tensor& code2,
             const Tensor& offset, int64_t n, int64_t k, const OptionalTensor& bias,
             double scaling, const std::optional<std::pair<int64_t, double>>& dropout,
             const OptionalTensor& ws, const Tensor& rank_ws) {
  const Weight w{packed, absmax, absmax2, code2, offset, n, k};
  Dropout drop{false, 0, 0.0};
  if (dropout) drop = Dropout{true, (uint64_t)dropout->first, dropout->second};
  return QLoRA::apply(x, lora_a, lora_b, w, bias, scaling, drop, ws, rank_ws);
}

// Python's view of the node, under the name that the Python node has there.
template <class Node>
void name_node(const char* name) {
  static PyTypeObject type;
  torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<Node>), &type);
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  name_node<NF4Linear>("NF4LinearBackward");
  name_node<RowNorm>("RowNormBackward");
  name_node<QLoRA>("_QLoRAFusedBackward");
  // Without the interpreter lock: a call may wait for room in the launch queue or for memory,
  // and other threads run meanwhile, as they do during a ctypes call.
  using Unlocked = pybind11::call_guard<pybind11::gil_scoped_release>;
  m.def("nf4_linear", &nf4_linear, Unlocked());
  m.def("row_norm", &row_norm, Unlocked());
  m.def("qlora", &qlora, Unlocked());
}
