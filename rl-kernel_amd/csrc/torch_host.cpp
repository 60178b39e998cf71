// The host side of the smallest calls in C++: checks, allocations and launches of an everyday inference projection, the packed
// FFN, the differentiable linear layer and the GRPO loss, on top of the C entry points of librlk_gfx950.so.
//
// Small calls are bound by their host time. In Python / here, us a call: a projection 13.9 / 5.2 (5 were the dispatch of the
// torch.library operator around it), the packed FFN 28.7 / 11.0, a linear layer with both gradients 40.6 / 27.0, the FFN with all
// its gradients 116 / 58, the GRPO loss with its gradient 59.7 / 33.5, beside kernels of 2 to 12 each; 87 / 50, 197 / 99 and 114 / 59
// in the stretches in which autograd's device thread has to be woken for every backward.
//
// Every function takes everyday arguments only and answers None to anything else - other types, layouts and devices, subclasses,
// batched and functorch tensors, tangents, dispatch and function modes (torch.set_default_device() is one), tracing, profilers -, for
// which the caller goes the way it went before. The autograd functions hand what is not everyday in a backward (an operand that wants
// no gradient, gradients or saved tensors that are more than their values) to the Python functions that bind() was given. Under
// create_graph the loss does so too, whose gradient is differentiable; those of the linear layer and the FFN have no graph either way.
// Nothing is kept from one call for the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <climits>

#include "../../include/rlk.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using c10::DispatchKeySet;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The library's entry points, from the library that Python has loaded, and the Python functions of the general ways.
decltype(&rlk_det_gemm_bf16) gemm_entry = nullptr;
decltype(&rlk_linear_bwd_bf16) linear_bwd_entry = nullptr;
decltype(&rlk_det_gemm_swiglu_workspace_bytes) swiglu_workspace_entry = nullptr;
decltype(&rlk_det_gemm_swiglu_bf16) swiglu_entry = nullptr;
decltype(&rlk_det_gemm_swiglu_training_bf16) swiglu_training_entry = nullptr;
decltype(&rlk_swiglu_bwd) swiglu_bwd_entry = nullptr;
decltype(&rlk_grpo_workspace_bytes) grpo_workspace_entry = nullptr;
decltype(&rlk_grpo_ratio_kl_loss) grpo_entry = nullptr;
decltype(&rlk_grpo_ratio_kl_loss_bwd) grpo_bwd_entry = nullptr;
decltype(&rlk_last_error) last_error_entry = nullptr;
PyObject* general_linear_gradients = nullptr;  // (a, weight, grad, need_a, need_weight) -> (da, dw)
PyObject* general_ffn_gradients = nullptr;     // (x, gate, up, activated, three weights, grad, need of x and the weights) -> four
PyObject* general_grpo_gradient = nullptr;     // (cur, old, ref, adv, mask, g_loss, g_policy, g_kl, clip_eps, beta) -> grad

// What _lib.check() raises.
void check_status(int status, const char* what) {
  if (status == RLK_OK) return;
  const char* message = last_error_entry();
  if (message == nullptr || message[0] == 0) message = what;
  TORCH_CHECK_VALUE(status != RLK_ERR_INVALID_ARGUMENT, message);
  throw std::runtime_error(message);
}

// Nothing on this thread takes over operations: no dispatch, function or tracing mode, no functorch level.
bool everyday_thread() {
  static const uint64_t usual = (DispatchKeySet(DispatchKey::BackendSelect) | DispatchKeySet(DispatchKey::ADInplaceOrView)).raw_repr();
  return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~usual) == 0 && !at::impl::torch_function_mode_enabled();
}
// ... and nothing looks at them: under a profiler the calls show as the operators that they are.
bool everyday_caller() { return everyday_thread() && !at::hasCallbacks(); }

// A tensor of values in GPU memory and nothing else.
bool everyday(const Tensor& t, at::ScalarType dtype) {
  static const uint64_t usual = (DispatchKeySet(DispatchKey::CUDA) | DispatchKeySet(DispatchKey::AutogradCUDA) |
                                 DispatchKeySet(DispatchKey::ADInplaceOrView) | DispatchKeySet(DispatchKey::AutocastCUDA)).raw_repr();
  return t.defined() && t.is_cuda() && (t.key_set().raw_repr() & ~usual) == 0 && t.scalar_type() == dtype && t.has_storage() &&
         !t._fw_grad(0).defined();
}
bool everyday(const Tensor& t, at::ScalarType dtype, const Tensor& beside) {
  return everyday(t, dtype) && t.get_device() == beside.get_device();
}

// A Python argument that is a Tensor or a Parameter, no subclass.
const Tensor* exact_tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

void* stream_of(const Tensor& t) {
  return reinterpret_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream());
}
Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const Tensor& like) {
  return at::empty(shape, like.options().dtype(dtype).requires_grad(false));
}

// A new reference, or the Python error that is set.
struct PyRef {
  explicit PyRef(PyObject* o) : object(o) {
    if (object == nullptr) throw python_error();
  }
  ~PyRef() { Py_DECREF(object); }
  PyRef(const PyRef&) = delete;
  PyRef& operator=(const PyRef&) = delete;
  PyObject* get() const { return object; }
  PyObject* const object;
};
Tensor tensor_or_none(PyObject* o) {
  if (o == nullptr) throw python_error();
  return o == Py_None ? Tensor() : THPVariable_Unpack(o);
}

constexpr auto kBf16 = at::kBFloat16;
bool everyday_matrix(const Tensor& t) { return t.dim() == 2 && t.is_contiguous() && t.numel() > 0; }

// a[M,K] @ weight[N,K].T
Tensor project(const Tensor& a, const Tensor& weight) {
  const int64_t m = a.size(0), k = a.size(1), n = weight.size(0);
  Tensor out = empty({m, n}, kBf16, a);
  check_status(gemm_entry(a.data_ptr(), k, 1, weight.data_ptr(), 1, k, out.data_ptr(), n, (int)m, (int)n, (int)k, 0, 0, stream_of(a)),
               "rlk_det_gemm_bf16 failed");
  return out;
}
bool projects(const Tensor& a, const Tensor& weight) {
  return everyday(a, kBf16) && everyday(weight, kBf16, a) && everyday_matrix(a) && everyday_matrix(weight) &&
         a.size(1) == weight.size(1) && a.size(0) <= INT_MAX && a.size(1) <= INT_MAX && weight.size(0) <= INT_MAX;
}

// ---------------------------------------------------------------------------
// Linear layer under autograd
// ---------------------------------------------------------------------------

// A row-major operand that the K-major loader takes as it is (_C._rows_of_chunks).
bool rows_of_chunks(const Tensor& t) {
  return t.size(1) % 8 == 0 && t.stride(1) == 1 && t.stride(0) % 8 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}

// Both gradients of a @ weight.T in one library call.
bool takes_both_gradients(const Tensor& a, const Tensor& weight, const Tensor& grad) {
  return everyday(grad, kBf16) && everyday_matrix(grad) && projects(a, weight) && everyday(a, kBf16, grad) &&
         grad.size(0) == a.size(0) && grad.size(1) == weight.size(0) && rows_of_chunks(a) && rows_of_chunks(weight) &&
         rows_of_chunks(grad);
}
variable_list both_gradients(const Tensor& a, const Tensor& weight, const Tensor& grad, int config) {
  const int64_t m = a.size(0), k = a.size(1), n = weight.size(0);
  Tensor da = empty({m, k}, kBf16, grad), dw = empty({n, k}, kBf16, grad);
  check_status(linear_bwd_entry(grad.data_ptr(), n, a.data_ptr(), k, weight.data_ptr(), k, da.data_ptr(), k, dw.data_ptr(), k, (int)m,
                                (int)k, (int)n, config, stream_of(grad)),
               "rlk_linear_bwd_bf16 failed");
  return {da, dw};
}

struct LinearFn : torch::autograd::Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& weight) {
    ctx->save_for_backward({a, weight});
    return project(a, weight);
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &a = saved[0], &weight = saved[1], &grad = grads[0];
    const bool need_a = ctx->needs_input_grad(0), need_weight = ctx->needs_input_grad(1);
    if (need_a && need_weight && everyday_thread() && takes_both_gradients(a, weight, grad)) {
      const c10::OptionalDeviceGuard guard(grad.device());
      return both_gradients(a, weight, grad, RLK_LINEAR_BWD_CFG_AUTO);
    }
    const pybind11::gil_scoped_acquire gil;
    const PyRef py_a(THPVariable_Wrap(a)), py_weight(THPVariable_Wrap(weight)), py_grad(THPVariable_Wrap(grad));
    const PyRef result(PyObject_CallFunctionObjArgs(general_linear_gradients, py_a.get(), py_weight.get(), py_grad.get(),
                                                    need_a ? Py_True : Py_False, need_weight ? Py_True : Py_False, nullptr));
    return {tensor_or_none(PyTuple_GetItem(result.get(), 0)), tensor_or_none(PyTuple_GetItem(result.get(), 1))};
  }
};


// ---------------------------------------------------------------------------
// Packed gated FFN (inference)
// ---------------------------------------------------------------------------

bool takes_ffn(const Tensor& x, const Tensor& gate_up, const Tensor& down) {
  return everyday(x, kBf16) && everyday(gate_up, kBf16, x) && everyday_matrix(gate_up) && x.dim() >= 1 && x.is_contiguous() &&
         x.numel() > 0 && everyday(down, kBf16, x) && everyday_matrix(down) && gate_up.size(0) % 2 == 0 &&
         gate_up.size(1) == x.size(-1) && down.size(1) == gate_up.size(0) / 2 && x.numel() / x.size(-1) <= INT_MAX &&
         x.size(-1) <= INT_MAX && gate_up.size(0) <= INT_MAX && down.size(0) <= INT_MAX;
}

Tensor packed_ffn(const Tensor& x, const Tensor& gate_up, const Tensor& down) {
  const int64_t k = x.size(-1), m = x.numel() / k, inter = gate_up.size(0) / 2, n = down.size(0);
  Tensor activated = empty({m, inter}, kBf16, x);
  const size_t bytes = swiglu_workspace_entry(x.data_ptr(), k, gate_up.data_ptr(), k, (int)m, (int)inter, (int)k);
  Tensor workspace;
  if (bytes > 0) workspace = empty({(int64_t)(bytes / 2)}, kBf16, x);
  void* const stream = stream_of(x);
  check_status(swiglu_entry(x.data_ptr(), k, gate_up.data_ptr(), k, activated.data_ptr(), inter,
                            bytes > 0 ? workspace.data_ptr() : nullptr, bytes, (int)m, (int)inter, (int)k, stream),
               "rlk_det_gemm_swiglu_bf16 failed");
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = n;
  Tensor out = empty(shape, kBf16, x);
  check_status(gemm_entry(activated.data_ptr(), inter, 1, down.data_ptr(), 1, inter, out.data_ptr(), n, (int)m, (int)n, (int)inter, 0,
                          0, stream),
               "rlk_det_gemm_bf16 failed");
  return out;
}

// ---------------------------------------------------------------------------
// Gated FFN under autograd (_DeterministicFFNFunction in backends/rocm/ffn/ffn.py, three weights)
// ---------------------------------------------------------------------------

bool takes_ffn_training(const Tensor& x, const Tensor& gate, const Tensor& up, const Tensor& down) {
  return everyday(x, kBf16) && x.dim() >= 1 && x.is_contiguous() && x.numel() > 0 && x.numel() / x.size(-1) <= INT_MAX &&
         x.size(-1) <= INT_MAX && everyday(gate, kBf16, x) && everyday_matrix(gate) && gate.size(1) == x.size(-1) &&
         everyday(up, kBf16, x) && up.is_contiguous() && up.sizes() == gate.sizes() && everyday(down, kBf16, x) &&
         everyday_matrix(down) && down.size(0) == gate.size(1) && down.size(1) == gate.size(0) && gate.size(0) <= INT_MAX;
}

struct FfnFn : torch::autograd::Function<FfnFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& input, const Tensor& gate_weight, const Tensor& up_weight,
                        const Tensor& down_weight) {
    const Tensor x = input.dim() == 2 ? input : input.view({-1, input.size(-1)});
    const int64_t m = x.size(0), k = x.size(1), inter = gate_weight.size(0);
    const Tensor gate = empty({m, inter}, kBf16, x), up = empty({m, inter}, kBf16, x), activated = empty({m, inter}, kBf16, x);
    check_status(swiglu_training_entry(x.data_ptr(), k, gate_weight.data_ptr(), up_weight.data_ptr(), k, gate.data_ptr(), up.data_ptr(),
                                       activated.data_ptr(), inter, (int)m, (int)inter, (int)k, stream_of(x)),
                 "rlk_det_gemm_swiglu_training_bf16 failed");
    ctx->save_for_backward({x, gate, up, activated, gate_weight, up_weight, down_weight});
    ctx->saved_data["shape"] = input.sizes().vec();
    const Tensor out = project(activated, down_weight);
    return input.dim() == 2 ? out : out.view(input.sizes());
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();  // x, gate, up, activated, weights of gate, up and down
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    bool need[4], all = true;
    for (int i = 0; i < 4; ++i) all &= need[i] = ctx->needs_input_grad(i);
    if (all && everyday_thread() && everyday(grads[0], kBf16) && grads[0].is_contiguous() && grads[0].sizes() == at::IntArrayRef(shape)) {
      const Tensor grad = shape.size() == 2 ? grads[0] : grads[0].view({-1, shape.back()});
      if (takes_both_gradients(s[3], s[6], grad) && everyday(s[1], kBf16, grad) && everyday_matrix(s[1]) && rows_of_chunks(s[1]) &&
          s[1].sizes() == s[3].sizes() && everyday(s[2], kBf16, grad) && everyday_matrix(s[2]) && s[2].sizes() == s[3].sizes() &&
          takes_both_gradients(s[0], s[4], s[1]) && takes_both_gradients(s[0], s[5], s[2])) {
        const c10::OptionalDeviceGuard guard(grad.device());
        // three weights that are together more than the memory-side cache holds (_MANY_WEIGHTS_BYTES)
        const int config = 3 * (int64_t)s[6].nbytes() >= ((int64_t)128 << 20) ? RLK_LINEAR_BWD_CFG_MANY_WEIGHTS : RLK_LINEAR_BWD_CFG_AUTO;
        const variable_list of_down = both_gradients(s[3], s[6], grad, config);
        const int64_t m = grad.size(0), inter = s[1].size(1);
        const Tensor d_gate = empty({m, inter}, kBf16, grad), d_up = empty({m, inter}, kBf16, grad);
        check_status(swiglu_bwd_entry(of_down[0].data_ptr(), inter, s[1].data_ptr(), inter, s[2].data_ptr(), inter, d_gate.data_ptr(),
                                      inter, d_up.data_ptr(), inter, (int)m, (int)inter, RLK_DTYPE_BF16, stream_of(grad)),
                     "rlk_swiglu_bwd failed");
        const variable_list of_gate = both_gradients(s[0], s[4], d_gate, config), of_up = both_gradients(s[0], s[5], d_up, config);
        Tensor dx = of_gate[0];
        dx.add_(of_up[0]);
        return {shape.size() == 2 ? dx : dx.view(shape), of_gate[1], of_up[1], of_down[1]};
      }
    }
    const pybind11::gil_scoped_acquire gil;
    const PyRef args(PyTuple_New(12));
    for (int i = 0; i < 7; ++i) PyTuple_SET_ITEM(args.get(), i, THPVariable_Wrap(s[i]));
    PyTuple_SET_ITEM(args.get(), 7, THPVariable_Wrap(grads[0]));
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(args.get(), 8 + i, PyBool_FromLong(need[i]));
    const PyRef result(PyObject_CallObject(general_ffn_gradients, args.get()));
    variable_list out;
    for (int i = 0; i < 4; ++i) out.push_back(tensor_or_none(PyTuple_GetItem(result.get(), i)));
    if (out[0].defined()) out[0] = out[0].reshape(shape);
    return out;
  }
};

// ---------------------------------------------------------------------------
// GRPO loss
// ---------------------------------------------------------------------------

// Log-probs [rollouts, tokens], one advantage per rollout, a mask of bools or none.
struct GrpoInputs {
  Tensor cur, old, ref, adv, mask;
  double clip_eps, beta;

  bool usual() const {
    constexpr auto kF32 = at::kFloat;
    return everyday(cur, kF32) && cur.dim() == 2 && cur.is_contiguous() && cur.numel() > 0 && cur.size(0) <= INT_MAX &&
           cur.size(1) <= INT_MAX && everyday(old, kF32, cur) && old.sizes() == cur.sizes() && old.is_contiguous() &&
           everyday(ref, kF32, cur) && ref.sizes() == cur.sizes() && ref.is_contiguous() && everyday(adv, kF32, cur) &&
           adv.numel() == cur.size(0) && adv.is_contiguous() &&
           (!mask.defined() || (everyday(mask, at::kBool, cur) && mask.sizes() == cur.sizes() && mask.is_contiguous()));
  }
  const uint8_t* mask_bytes() const { return mask.defined() ? static_cast<const uint8_t*>(mask.data_ptr()) : nullptr; }
};
struct GrpoOutputs {
  Tensor out3, ratio, k3, workspace;
};
const float* floats(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr; }

GrpoOutputs grpo(const GrpoInputs& in) {
  const int64_t rollouts = in.cur.size(0), tokens = in.cur.size(1);
  const size_t bytes = grpo_workspace_entry((int)rollouts);
  GrpoOutputs out{empty({3}, at::kFloat, in.cur), empty({rollouts, tokens}, at::kFloat, in.cur),
                  empty({rollouts, tokens}, at::kFloat, in.cur), empty({(int64_t)(bytes / 4)}, at::kFloat, in.cur)};
  check_status(grpo_entry(floats(in.cur), floats(in.old), floats(in.ref), floats(in.adv), in.mask_bytes(), (int)rollouts, (int)tokens,
                          (float)in.clip_eps, (float)in.beta, static_cast<float*>(out.ratio.data_ptr()),
                          static_cast<float*>(out.k3.data_ptr()), static_cast<float*>(out.out3.data_ptr()), out.workspace.data_ptr(),
                          bytes, stream_of(in.cur)),
               "rlk_grpo_ratio_kl_loss failed");
  return out;
}

// The three scalars with respect to the current log-probs (_GrpoLossAutograd in backends/rocm/loss/grpo.py, with the same
// conditions for the kernel in the backward). The workspace holds the kernel's own numbers: it is not for saved-tensor hooks.
struct GrpoFn : torch::autograd::Function<GrpoFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& cur, const GrpoInputs* in, GrpoOutputs* out) {
    *out = grpo(*in);
    variable_list saved = {cur, in->old, in->ref, in->adv};
    if (in->mask.defined()) saved.push_back(in->mask);
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["workspace"] = out->workspace;
    ctx->saved_data["clip_eps"] = in->clip_eps;
    ctx->saved_data["beta"] = in->beta;
    ctx->set_materialize_grads(false);  // an unused output costs no zero tensor
    return out->out3.unbind(0);
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    if (!grads[0].defined() && !grads[1].defined() && !grads[2].defined()) return {Tensor(), Tensor(), Tensor()};
    const variable_list saved = ctx->get_saved_variables();
    GrpoInputs in{saved[0], saved[1], saved[2], saved[3], saved.size() > 4 ? saved[4] : Tensor(),
                  ctx->saved_data["clip_eps"].toDouble(), ctx->saved_data["beta"].toDouble()};
    const Tensor workspace = ctx->saved_data["workspace"].toTensor();
    bool values = !at::GradMode::is_enabled() && everyday_thread() && in.usual() && in.cur.get_device() == workspace.get_device();
    for (const Tensor& g : grads) values = values && (!g.defined() || (everyday(g, at::kFloat, in.cur) && g.numel() == 1));
    if (values) {
      const c10::OptionalDeviceGuard guard(in.cur.device());
      Tensor grad = empty(in.cur.sizes(), at::kFloat, in.cur);
      check_status(grpo_bwd_entry(floats(in.cur), floats(in.old), floats(in.ref), floats(in.adv), in.mask_bytes(), workspace.data_ptr(),
                                  workspace.nbytes(), floats(grads[0]), floats(grads[1]), floats(grads[2]), (int)in.cur.size(0),
                                  (int)in.cur.size(1), (float)(1.0 - in.clip_eps), (float)(1.0 + in.clip_eps), (float)in.beta,
                                  static_cast<float*>(grad.data_ptr()), stream_of(in.cur)),
                   "rlk_grpo_ratio_kl_loss_bwd failed");
      return {grad, Tensor(), Tensor()};
    }
    const pybind11::gil_scoped_acquire gil;  // THPVariable_Wrap makes None of an undefined tensor
    const PyRef cur(THPVariable_Wrap(in.cur)), old(THPVariable_Wrap(in.old)), ref(THPVariable_Wrap(in.ref)), adv(THPVariable_Wrap(in.adv)),
        mask(THPVariable_Wrap(in.mask)), g_loss(THPVariable_Wrap(grads[0])), g_policy(THPVariable_Wrap(grads[1])),
        g_kl(THPVariable_Wrap(grads[2])), clip(PyFloat_FromDouble(in.clip_eps)), beta(PyFloat_FromDouble(in.beta));
    const PyRef grad(PyObject_CallFunctionObjArgs(general_grpo_gradient, cur.get(), old.get(), ref.get(), adv.get(), mask.get(),
                                                  g_loss.get(), g_policy.get(), g_kl.get(), clip.get(), beta.get(), nullptr));
    return {tensor_or_none(grad.get()), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// The Python module
// ---------------------------------------------------------------------------

PyObject* none() { Py_RETURN_NONE; }

// linear(a, weight) -> a @ weight.T, differentiable where an operand asks for it, or None
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 2 || gemm_entry == nullptr) return none();
  const Tensor *a = exact_tensor(args[0]), *weight = exact_tensor(args[1]);
  if (a == nullptr || weight == nullptr || !everyday_caller() || !projects(*a, *weight)) return none();
  const bool differentiable = at::GradMode::is_enabled() && (a->requires_grad() || weight->requires_grad());
  Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(a->device());
    out = differentiable ? LinearFn::apply(*a, *weight) : project(*a, *weight);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// packed_ffn(x, gate_up, down) -> down @ swiglu(gate_up @ x), or None
PyObject* py_packed_ffn(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 3 || gemm_entry == nullptr) return none();
  const Tensor *x = exact_tensor(args[0]), *gate_up = exact_tensor(args[1]), *down = exact_tensor(args[2]);
  if (x == nullptr || gate_up == nullptr || down == nullptr || !everyday_caller() || !takes_ffn(*x, *gate_up, *down)) return none();
  if (at::GradMode::is_enabled() && (x->requires_grad() || gate_up->requires_grad() || down->requires_grad())) return none();
  Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(x->device());
    out = packed_ffn(*x, *gate_up, *down);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ffn(x, gate, up, down) -> down @ (silu(gate @ x) * (up @ x)) with the gradients of all four, or None
PyObject* py_ffn(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 4 || gemm_entry == nullptr) return none();
  const Tensor* t[4];
  for (int i = 0; i < 4; ++i) {
    t[i] = exact_tensor(args[i]);
    if (t[i] == nullptr) return none();
  }
  if (!everyday_caller() || !takes_ffn_training(*t[0], *t[1], *t[2], *t[3])) return none();
  Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(t[0]->device());
    out = FfnFn::apply(*t[0], *t[1], *t[2], *t[3]);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// grpo(cur, old, ref, adv, mask or None, clip_eps, beta) -> (loss, policy, kl, ratio, k3), or None
PyObject* py_grpo(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 7 || gemm_entry == nullptr) return none();
  const Tensor* t[5] = {};
  for (int i = 0; i < 5; ++i) {
    if (i == 4 && args[i] == Py_None) break;
    t[i] = exact_tensor(args[i]);
    if (t[i] == nullptr) return none();
  }
  for (int i = 5; i < 7; ++i)
    if (!PyFloat_CheckExact(args[i]) && !PyLong_CheckExact(args[i])) return none();
  GrpoInputs in{*t[0], *t[1], *t[2], *t[3], t[4] != nullptr ? *t[4] : Tensor(), PyFloat_AsDouble(args[5]), PyFloat_AsDouble(args[6])};
  if (PyErr_Occurred()) throw python_error();
  if (!everyday_caller() || !in.usual()) return none();
  variable_list three;
  GrpoOutputs out;
  {
    const pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(in.cur.device());
    if (at::GradMode::is_enabled() && in.cur.requires_grad()) {
      for (Tensor* s : {&in.old, &in.ref, &in.adv})
        if (s->requires_grad()) *s = s->detach();
      three = GrpoFn::apply(in.cur, &in, &out);
    } else {
      out = grpo(in);
      three = out.out3.unbind(0);
    }
  }
  const PyRef loss(THPVariable_Wrap(three[0])), policy(THPVariable_Wrap(three[1])), kl(THPVariable_Wrap(three[2])),
      ratio(THPVariable_Wrap(out.ratio)), k3(THPVariable_Wrap(out.k3));
  return PyTuple_Pack(5, loss.get(), policy.get(), kl.get(), ratio.get(), k3.get());
  END_HANDLE_TH_ERRORS
}

// bind(addresses of the entry points by name, the general gradients of the linear layer, the FFN and the GRPO loss)
PyObject* py_bind(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *addresses, *linear, *ffn, *loss;
  if (!PyArg_ParseTuple(args, "O!OOO", &PyDict_Type, &addresses, &linear, &ffn, &loss)) return nullptr;
  auto entry = [&](const char* name, auto& to) {
    PyObject* const at = PyDict_GetItemString(addresses, name);
    void* const address = at != nullptr ? PyLong_AsVoidPtr(at) : nullptr;
    if (PyErr_Occurred()) throw python_error();
    TORCH_CHECK(address != nullptr, "no address for ", name);
    to = reinterpret_cast<std::remove_reference_t<decltype(to)>>(address);
  };
  entry("rlk_last_error", last_error_entry);
  entry("rlk_linear_bwd_bf16", linear_bwd_entry);
  entry("rlk_det_gemm_swiglu_workspace_bytes", swiglu_workspace_entry);
  entry("rlk_det_gemm_swiglu_bf16", swiglu_entry);
  entry("rlk_det_gemm_swiglu_training_bf16", swiglu_training_entry);
  entry("rlk_swiglu_bwd", swiglu_bwd_entry);
  entry("rlk_grpo_workspace_bytes", grpo_workspace_entry);
  entry("rlk_grpo_ratio_kl_loss", grpo_entry);
  entry("rlk_grpo_ratio_kl_loss_bwd", grpo_bwd_entry);
  Py_INCREF(linear);
  Py_XSETREF(general_linear_gradients, linear);
  Py_INCREF(ffn);
  Py_XSETREF(general_ffn_gradients, ffn);
  Py_INCREF(loss);
  Py_XSETREF(general_grpo_gradient, loss);
  entry("rlk_det_gemm_bf16", gemm_entry);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_linear)), METH_FASTCALL, nullptr},
    {"packed_ffn", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_packed_ffn)), METH_FASTCALL, nullptr},
    {"ffn", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_ffn)), METH_FASTCALL, nullptr},
    {"grpo", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_grpo)), METH_FASTCALL, nullptr},
    {"bind", py_bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_host() { return PyModule_Create(&module); }
