// The eager host path of the neuron layers in native code: a Python extension module (spikingjelly_amd/_sjhip_torch.so)
// between torch's C++ autograd and the C ABI of libsjhip.so.
//
// Why: a training pass through a small layer is host time.  Through torch.autograd.Function and ctypes the forward and
// backward of one layer of 8192 neurons cost 200 us of Python for two kernels of 5 us; here a call allocates its outputs,
// launches and records one autograd node, and the backward runs on the autograd engine's thread without entering Python.
//
// The functions take the tensors of the public functionals as they are ([T, ...], no flattening views) and return None
// where they do not serve (layouts, sizes, tracing and transforms that the general Python path handles); the caller then
// takes that path.  Nothing is kept between calls.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/autograd.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/dynamo/compiled_autograd.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/torch.h>

#include <mutex>
#include <string>
#include <vector>

#include "sjhip.h"

namespace py = pybind11;

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

void check(int rc, const char *what) {
  TORCH_CHECK(rc == SJHIP_OK, "libsjhip ", what, " failed (", rc, "): ", sjhip_last_error());
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int dtype_id(at::ScalarType t, bool bytes = false) {
  switch (t) {
    case at::kFloat: return SJHIP_F32;
    case at::kHalf: return SJHIP_F16;
    case at::kBFloat16: return SJHIP_BF16;
    case at::kByte: case at::kBool: return bytes ? SJHIP_U8 : -1;
    default: return -1;
  }
}

bool aligned16(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

// A plain dense device tensor outside every transform that would have to see the operation: no functorch level, no
// dispatch mode or tensor subclass, no forward-mode derivative.
bool plain(const Tensor &t) {
  return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has(c10::DispatchKey::Python) && !t.is_neg() &&
         !torch::autograd::isFwGradDefined(t);
}
bool transforms_active() {  // (torch.jit.trace among them: a node made here would enter the trace as a constant)
  return torch::jit::tracer::isTracing() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python);
}

// One element that stands for the state of every neuron: an expanded view (the stride of a dimension of one element
// means nothing).
bool is_broadcast(const Tensor &v) {
  if (v.numel() <= 1) return false;
  for (int64_t d = 0; d < v.dim(); ++d)
    if (v.size(d) != 1 && v.stride(d) != 0) return false;
  return true;
}

Tensor empty(at::IntArrayRef sizes, const Tensor &like) { return at::empty(sizes, like.options()); }

// dense and on 16 bytes
Tensor dense16(const Tensor &t) {
  const Tensor d = t.contiguous();
  return aligned16(d) ? d : d.clone();
}

// A gradient as the kernels take it: dense, in the storage dtype, on 16 bytes.
Tensor dense_grad(const Tensor &g, at::ScalarType dtype) {
  if (!g.defined()) return g;
  return dense16(g.to(dtype));
}

// A saved tensor as the kernels take it.  A saved-tensor hook may hand the values back in another layout or type; what is
// not on the device of the forward, or has another size, is refused before a kernel reads it.
Tensor saved_values(const Tensor &t, const char *name, c10::Device device, at::ScalarType dtype, int64_t numel) {
  TORCH_CHECK(t.device() == device, "backend='hip': the saved ", name, " is on ", t.device(), " and not on ", device);
  TORCH_CHECK(t.layout() == at::kStrided && t.numel() == numel, "the saved ", name, " has ", t.numel(), " elements instead of ", numel);
  return t.scalar_type() == dtype ? t : t.to(dtype);
}

const void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

struct NeuronBackward : public torch::autograd::Node {
  SavedVariable x_, v_, k_;
  bool with_k = false, single = false;  // single: one step without a time dimension
  sjhip_neuron_params params{};  // without SJHIP_FLAG_V_INIT_BROADCAST, which follows the state as it is unpacked
  at::ScalarType storage = at::kFloat;
  c10::Device device = at::kCUDA;
  int neuron = 0, dtype = 0;
  int64_t T = 0, N = 0;

  std::string name() const override { return "HipNeuronBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x_.reset_data();
    v_.reset_data();
    k_.reset_data();
  }

  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list out(3);
    if (!grads[0].defined() && !grads[1].defined() && !grads[2].defined()) return out;
    const Tensor saved_x = x_.unpack(), saved_v = v_.unpack(), saved_k = with_k ? k_.unpack() : Tensor();
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(device);
    // (the library asks for tensors that begin on 16 bytes; a step taken out of a sequence may not)
    const Tensor x = dense16(saved_values(saved_x, "x_seq", device, storage, T * N));
    Tensor v = saved_values(saved_v, "v_init", device, storage, N);
    const Tensor k = with_k ? saved_values(saved_k, "k", device, at::kFloat, 1) : Tensor();
    sjhip_neuron_params p = params;
    if (is_broadcast(v)) p.flags |= SJHIP_FLAG_V_INIT_BROADCAST;
    else v = dense16(v);
    const Tensor gs = dense_grad(grads[0], x.scalar_type()), glast = dense_grad(grads[1], x.scalar_type()),
                 gv = dense_grad(grads[2], x.scalar_type());
    const Tensor gx = at::empty_like(x);
    Tensor gv0, gk, workspace;
    if (task_should_compute_output(1)) gv0 = empty(v.sizes(), x);
    if (with_k) {
      const auto f32 = x.options().dtype(at::kFloat);
      if (p.flags & SJHIP_FLAG_ATOMIC_REDUCE) {
        gk = at::zeros(k.sizes(), f32);
      } else {
        gk = at::empty(k.sizes(), f32);
        workspace = at::empty({sjhip_plif_workspace_floats(dtype, N)}, f32);
      }
    }
    check(sjhip_neuron_backward_recompute(neuron, dtype, &p, T, N, ptr(x), ptr(v), static_cast<const float *>(ptr(k)), ptr(gs),
                                          ptr(gv), ptr(glast), gx.data_ptr(), gv0.defined() ? gv0.data_ptr() : nullptr,
                                          gk.defined() ? gk.data_ptr<float>() : nullptr,
                                          workspace.defined() ? workspace.data_ptr<float>() : nullptr, stream_of(x)),
          "neuron_backward_recompute");
    if (task_should_compute_output(0)) out[0] = gx;
    out[1] = gv0;
    if (with_k && task_should_compute_output(2)) out[2] = gk;
    return out;
  }

  // Compiled autograd records the backward graph instead of running it: what the node holds (scalars are constants of the
  // graph), and the same backward as a call of the traceable operators.
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs &args) const override {
    args.collect(x_, false);
    args.collect(v_, false);
    args.collect(with_k);
    if (with_k) args.collect(k_, false);
    args.collect(single);
    args.collect((int64_t)neuron);
    args.collect((int64_t)params.sg_id);
    args.collect((int64_t)params.flags);
    for (float f : {params.tau, params.v_threshold, params.v_reset, params.sg_alpha, params.v_rest, params.v_c, params.a0, params.level_max,
                    params.grad_min, params.grad_max})
      args.collect((double)f);
  }
  variable_list apply_with_saved(const variable_list &grads, torch::dynamo::autograd::SwapSavedVariables &saved) override {
    saved.before(x_);
    saved.before(v_);
    if (with_k) saved.before(k_);
    variable_list out(3);
    if (grads[0].defined() || grads[1].defined() || grads[2].defined()) {
      py::gil_scoped_acquire gil;
      auto arg = [](const Tensor &t) { return t.defined() ? py::cast(t) : py::object(py::none()); };
      const auto result = py::cast<std::tuple<Tensor, c10::optional<Tensor>, c10::optional<Tensor>>>(
          py::module_::import("spikingjelly_amd.activation_based.hip_kernel.neuron_kernel")
              .attr("backward_as_operator")(neuron, arg(grads[0]), arg(grads[2]), arg(grads[1]), x_.unpack(), v_.unpack(),
                                            arg(with_k ? k_.unpack() : Tensor()), single,
                                            py::make_tuple(params.tau, params.v_threshold, params.v_reset, params.sg_alpha, params.sg_id,
                                                           params.flags, params.v_rest, params.v_c, params.a0, params.level_max,
                                                           params.grad_min, params.grad_max),
                                            should_compute_output(1)));
      if (should_compute_output(0)) out[0] = std::get<0>(result);
      if (should_compute_output(1)) out[1] = *std::get<1>(result);
      if (with_k && should_compute_output(2)) out[2] = *std::get<2>(result);
    }
    saved.after(x_);
    saved.after(v_);
    if (with_k) saved.after(k_);
    return out;
  }
};

// (spikes, v after the last step, v after every step or None), or None when the general path has to serve.
// x_seq [T, *] (single: [*], one step), v: the state in front of the first step ([*], dense or one expanded element),
// k: one fp32 element on the device for PLIF.  replay_steps: the longest sequence whose backward replays the forward in
// one piece, 0 when a training call has to save h.  extra: v_rest, v_c, a0 and level_max, grad_min, grad_max.
py::object neuron_sequence(const Tensor &x_seq, const Tensor &v_init, const c10::optional<Tensor> &k_opt, bool single, int neuron,
                           double tau, double v_th, double v_reset, int64_t flags, int64_t sg_id, double sg_alpha, bool store_v_seq,
                           int64_t replay_steps, const std::array<double, 6> &extra) {
  const int dtype = dtype_id(x_seq.scalar_type());
  if (dtype < 0 || x_seq.dim() < (single ? 1 : 2) || !plain(x_seq) || !x_seq.is_contiguous() || x_seq.numel() == 0 || transforms_active())
    return py::none();
  const int64_t T = single ? 1 : x_seq.size(0), N = x_seq.numel() / T;
  const auto step = single ? x_seq.sizes() : x_seq.sizes().slice(1);
  if (v_init.scalar_type() != x_seq.scalar_type() || v_init.device() != x_seq.device() || v_init.sizes() != step) return py::none();
  const Tensor k = k_opt.has_value() ? *k_opt : Tensor();
  const bool grad = at::GradMode::is_enabled() && (x_seq.requires_grad() || v_init.requires_grad() || (k.defined() && k.requires_grad()));
  const bool broadcast = is_broadcast(v_init);
  if (torch::autograd::isFwGradDefined(v_init) || (k.defined() && torch::autograd::isFwGradDefined(k)) ||
      (!broadcast && !v_init.is_contiguous()))
    return py::none();
  if (k.defined() && (k.scalar_type() != at::kFloat || k.device() != x_seq.device() || k.numel() != 1)) return py::none();
  if (grad && (T > replay_steps || N < (dtype == SJHIP_F32 ? 4 : 8))) return py::none();

  Tensor spikes, v_last, v_seq;
  sjhip_neuron_params p{(float)tau, (float)v_th, (float)v_reset, (float)sg_alpha, (int32_t)sg_id,
                        (uint32_t)flags | (broadcast ? SJHIP_FLAG_V_INIT_BROADCAST : 0u),
                        (float)extra[0], (float)extra[1], (float)extra[2], (float)extra[3], (float)extra[4], (float)extra[5]};
  {
    py::gil_scoped_release no_gil;
    at::AutoDispatchBelowADInplaceOrView below;
    c10::DeviceGuard guard(x_seq.device());
    spikes = at::empty_like(x_seq);
    v_last = empty(step, x_seq);
    if (store_v_seq) v_seq = at::empty_like(x_seq);
    check(sjhip_neuron_forward(neuron, dtype, &p, T, N, ptr(x_seq), ptr(v_init), static_cast<const float *>(ptr(k)), spikes.data_ptr(),
                               store_v_seq ? v_seq.data_ptr() : nullptr, v_last.data_ptr(), nullptr, stream_of(x_seq)),
          "neuron_forward");
  }
  if (grad) {
    auto node = std::shared_ptr<NeuronBackward>(new NeuronBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(x_seq, v_init, k));
    node->x_ = SavedVariable(x_seq, false);
    node->v_ = SavedVariable(v_init, false);
    node->with_k = k.defined();
    node->single = single;
    if (k.defined()) node->k_ = SavedVariable(k, false);
    node->params = p;
    node->params.flags &= ~(uint32_t)SJHIP_FLAG_V_INIT_BROADCAST;
    node->storage = x_seq.scalar_type();
    node->device = x_seq.device();
    node->neuron = neuron; node->dtype = dtype; node->T = T; node->N = N;
    torch::autograd::set_history(spikes, node);
    torch::autograd::set_history(v_last, node);
    if (store_v_seq) torch::autograd::set_history(v_seq, node);
    else node->add_input_metadata(torch::autograd::Node::undefined_input());
  }
  return py::make_tuple(spikes, v_last, store_v_seq ? py::cast(v_seq) : py::object(py::none()));
}

// (spike bits, v after the last step, v after every step or None) of an inference call with bit-packed spikes; None where
// the general path has to serve (rows that do not start on a byte among them).
py::object neuron_sequence_packed(const Tensor &x_seq, const Tensor &v_init, const c10::optional<Tensor> &k_opt, int neuron, double tau,
                                  double v_th, double v_reset, int64_t flags, bool store_v_seq) {
  const int dtype = dtype_id(x_seq.scalar_type());
  if (dtype < 0 || x_seq.dim() < 2 || !plain(x_seq) || !x_seq.is_contiguous() || x_seq.numel() == 0 || transforms_active()) return py::none();
  const int64_t T = x_seq.size(0), N = x_seq.numel() / T;
  const auto step = x_seq.sizes().slice(1);
  const bool broadcast = is_broadcast(v_init);
  if (N % 8 != 0 || v_init.scalar_type() != x_seq.scalar_type() || v_init.device() != x_seq.device() || v_init.sizes() != step ||
      (!broadcast && !v_init.is_contiguous()))
    return py::none();
  const Tensor k = k_opt.has_value() ? *k_opt : Tensor();
  if (k.defined() && (k.scalar_type() != at::kFloat || k.device() != x_seq.device() || k.numel() != 1)) return py::none();
  sjhip_neuron_params p{};
  p.tau = (float)tau; p.v_threshold = (float)v_th; p.v_reset = (float)v_reset;
  p.flags = (uint32_t)flags | (broadcast ? SJHIP_FLAG_V_INIT_BROADCAST : 0u);
  Tensor bits, v_last, v_seq;
  {
    py::gil_scoped_release no_gil;
    at::NoGradGuard no_grad;
    c10::DeviceGuard guard(x_seq.device());
    bits = at::empty({T * N / 8}, x_seq.options().dtype(at::kByte));
    v_last = empty(step, x_seq);
    if (store_v_seq) v_seq = at::empty_like(x_seq);
    check(sjhip_neuron_forward_packed(neuron, dtype, &p, T, N, ptr(x_seq), ptr(v_init), static_cast<const float *>(ptr(k)),
                                      bits.data_ptr<uint8_t>(), store_v_seq ? v_seq.data_ptr() : nullptr, v_last.data_ptr(),
                                      stream_of(x_seq)),
          "neuron_forward_packed");
  }
  return py::make_tuple(bits, v_last, store_v_seq ? py::cast(v_seq) : py::object(py::none()));
}

Tensor bit_pack(const Tensor &spikes) {
  py::gil_scoped_release no_gil;
  at::NoGradGuard no_grad;
  const Tensor src = spikes.contiguous();
  const int dtype = dtype_id(src.scalar_type(), true);
  c10::DeviceGuard guard(src.device());
  const Tensor bits = at::empty({(src.numel() + 7) / 8}, src.options().dtype(at::kByte));
  if (src.numel() > 0) check(sjhip_bit_pack(dtype, src.numel(), src.data_ptr(), bits.data_ptr<uint8_t>(), stream_of(src)), "bit_pack");
  return bits;
}

Tensor bit_unpack(const Tensor &bits, at::IntArrayRef shape, at::ScalarType type) {
  py::gil_scoped_release no_gil;
  at::NoGradGuard no_grad;
  const Tensor src = bits.contiguous();
  c10::DeviceGuard guard(src.device());
  const Tensor out = at::empty(shape, src.options().dtype(type));
  if (out.numel() > 0)
    check(sjhip_bit_unpack(dtype_id(type, true), out.numel(), src.data_ptr<uint8_t>(), out.data_ptr(), stream_of(src)), "bit_unpack");
  return out;
}

}  // namespace

PYBIND11_MODULE(_sjhip_torch, m) {
  m.def("abi_version", [] { return sjhip_abi_version(); });
  m.def("neuron_sequence", &neuron_sequence);
  m.def("neuron_sequence_packed", &neuron_sequence_packed);
  m.def("bit_pack", &bit_pack);
  m.def("bit_unpack", [](const Tensor &bits, const std::vector<int64_t> &shape, at::ScalarType type) { return bit_unpack(bits, shape, type); });
}
