// The module's and the hidden-state operator's passes as native autograd nodes over the C ABI
// (include/gmlp.h): one Python call per forward, none per backward.
//
// What bounds a small pass is the host: at M = K = N = 512 the kernels of a training step take
// 50 us, while the same step through torch.autograd.Function and ctypes took 150 to 210 us of host
// time (a backward in Python has to take the interpreter lock on the autograd engine's thread while the
// main thread gives it up, and every operand goes through Python attribute and ctypes conversions).
// Here a forward is about 15 us and a backward enqueues without the interpreter.
//
// The library's entry points arrive as addresses from the Python loader (bind), so that there is one
// libgmlp.so in the process whatever path it was loaded from.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "gmlp.h"

namespace {

namespace ag = torch::autograd;
using at::Tensor;
typedef std::optional<Tensor> OptTensor;

#define GMLP_ENTRY_POINTS(X)                                                                     \
  X(gmlp_last_error) X(gmlp_workspace_bytes) X(gmlp_mlp_workspace_bytes) X(gmlp_mlp_fwd)         \
  X(gmlp_mlp_bwd) X(gmlp_gateup_fwd) X(gmlp_decode_fwd) X(gmlp_decode_stream_fwd) X(gmlp_hidden_bwd) \
  X(gmlp_grads_workspace_bytes)
struct Library {
#define GMLP_MEMBER(name) decltype(&::name) name = nullptr;
  GMLP_ENTRY_POINTS(GMLP_MEMBER)
#undef GMLP_MEMBER
};
Library lib;

void bind(const std::vector<std::pair<std::string, uintptr_t>>& entry_points) {
  for (const auto& e : entry_points) {
#define GMLP_BIND(name) \
  if (e.first == #name) lib.name = reinterpret_cast<decltype(lib.name)>(e.second);
    GMLP_ENTRY_POINTS(GMLP_BIND)
#undef GMLP_BIND
  }
#define GMLP_BOUND(name) TORCH_CHECK(lib.name != nullptr, "libgmlp.so entry point " #name " was not bound");
  GMLP_ENTRY_POINTS(GMLP_BOUND)
#undef GMLP_BOUND
}

void check(int status) {
  if (status == GMLP_OK) return;
  const std::string msg = lib.gmlp_last_error();
  if (status == GMLP_ESHAPE) C10_THROW_ERROR(NotImplementedError, msg);
  if (status == GMLP_EINVAL || status == GMLP_EALIGN) C10_THROW_ERROR(ValueError, msg);
  C10_THROW_ERROR(Error, msg);
}

const Tensor& or_undefined(const OptTensor& t) {
  static const Tensor undefined;
  return t.has_value() ? *t : undefined;
}
const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* out_ptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
Tensor contiguous(const Tensor& t) { return t.defined() ? t.contiguous() : t; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// All given tensors on one GPU, of one dtype the kernels take; returns the GMLP_* dtype code.
int require_gpu(std::initializer_list<std::reference_wrapper<const Tensor>> tensors) {
  const Tensor* first = nullptr;
  for (const Tensor& t : tensors) {
    if (!t.defined()) continue;
    TORCH_CHECK(t.is_cuda(), "fused gated-MLP operators run on an AMD GPU only (tensor is on ", t.device(),
                "); use EagerGatedMLP for CPU execution");
    if (first == nullptr) first = &t;
    TORCH_CHECK(t.device() == first->device(), "tensors on different devices: ", first->device(), " and ", t.device());
    TORCH_CHECK_TYPE(t.scalar_type() == first->scalar_type(), "tensors of different dtypes: ", first->scalar_type(), " and ",
                     t.scalar_type());
  }
  switch (first->scalar_type()) {
    case at::kHalf: return GMLP_F16;
    case at::kBFloat16: return GMLP_BF16;
    case at::kFloat: return GMLP_F32;
    default:
      C10_THROW_ERROR(TypeError, c10::str("fused gated-MLP kernels take float16, bfloat16 or float32 tensors, got ",
                                          first->scalar_type()));
  }
}

struct Problem {
  int64_t M = 0, K = 0, N = 0;
  int code = 0, act = 0;
  double p = 0.0;
  uint64_t seed = 0, offset = 0;
};

void check_gate_up(const Tensor& x, const Tensor& W_gate, const Tensor& b_gate, const Tensor& W_up, const Tensor& b_up) {
  TORCH_CHECK_VALUE(x.dim() >= 1 && W_up.dim() == 2 && W_up.size(1) == x.size(-1), "dimension mismatch in WT_up ", W_up.sizes(),
                    " or x ", x.sizes());
  TORCH_CHECK_VALUE(W_gate.sizes() == W_up.sizes(), "dimension mismatch in WT_up ", W_up.sizes(), " or WT_gp ", W_gate.sizes());
  TORCH_CHECK_VALUE(!b_up.defined() || (b_up.dim() == 1 && b_up.size(0) == W_up.size(0)), "dimension mismatch in b_up");
  TORCH_CHECK_VALUE(!b_gate.defined() || (b_gate.dim() == 1 && b_gate.size(0) == W_up.size(0)), "dimension mismatch in b_gp");
}
// x: [..., K], its leading dimensions are the M token rows
Problem problem_of(const Tensor& x, const Tensor& W_up, int code, int64_t act) {
  Problem q;
  q.K = x.size(-1);
  q.M = q.K > 0 ? x.numel() / q.K : 0;
  q.N = W_up.size(0);
  q.code = code;
  q.act = (int)act;
  return q;
}

// None of the operators has a forward-mode derivative: a dual input would come out without its tangent
// (also where reverse mode records nothing: torch.no_grad() leaves forward mode on).  Nor rules for
// functorch: refused as torch.autograd.Function does for an operator without rules of its own.
void refuse_transforms(const char* name, std::initializer_list<std::reference_wrapper<const Tensor>> tensors) {
  // (the key is included while a transform is active)
  TORCH_CHECK(!c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode), name,
              " does not support functorch transforms (vmap, grad, jvp, jacrev, ...)");
  if (ag::ForwardADLevel::try_get_by_idx(0) == nullptr) return;  // outside forward mode nothing is dual
  for (const Tensor& t : tensors)
    TORCH_CHECK_NOT_IMPLEMENTED(!t.defined() || !t._fw_grad(/*level=*/0).defined(),
                                "the fused gated-MLP operators have no forward-mode derivative");
}
// The incoming gradient, or zeros where what used the result has none for it (as torch.autograd.Function
// does by default): the gradients are zeros then, not None.
Tensor materialized(const Tensor& grad, at::IntArrayRef sizes, const at::TensorOptions& options) {
  return grad.defined() ? grad : at::zeros(sizes, options);
}
// A tensor that the kernels are about to read in a backward pass: saved-tensor hooks may hand back a tensor
// on another device, of another type or size than was saved.
Tensor readable(const Tensor& t, int64_t numel, const Tensor& grad) {
  TORCH_CHECK(t.defined() && t.device() == grad.device() && t.scalar_type() == grad.scalar_type() && t.numel() == numel,
              "a saved tensor came back as ", t.defined() ? c10::str(t.sizes(), " ", t.scalar_type(), " on ", t.device()) : "undefined",
              ", expected ", numel, " elements of ", grad.scalar_type(), " on ", grad.device());
  return t.contiguous();
}

// The backward passes have no derivative themselves.  Where autograd records one (create_graph), its results
// get a node in the place of the derivative that raises when it is differentiated through; results without
// a graph would silently be taken for constants.  The node leads on to what a derivative would reach (the
// operator's inputs and the incoming gradient), so that autograd comes by whichever of them is asked for.
void refuse_second_derivative(const ag::Node& backward, const Tensor& grad, ag::variable_list& out) {
  if (!at::GradMode::is_enabled()) return;
  ag::edge_list next = backward.next_edges();
  if (grad.requires_grad()) next.push_back(ag::impl::gradient_edge(grad));
  const auto node = std::shared_ptr<ag::Error>(
      new ag::Error("the fused gated-MLP operators have no second derivative", std::move(next)), ag::deleteNode);
  for (Tensor& t : out)
    if (t.defined()) ag::set_history(t, node);
}

Tensor scratch(size_t bytes, const Tensor& like) {
  return bytes > 0 ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// G, U, H planes of one [3, M, N] allocation, or H alone
struct Activations {
  Tensor all;
  char *g = nullptr, *u = nullptr, *h = nullptr;
  Activations(const Problem& q, const Tensor& t, bool saved) : all(t) {
    char* base = (char*)out_ptr(t);
    const int64_t plane = q.M * q.N * (int64_t)t.element_size();
    if (saved) {
      g = base;
      u = base + plane;
      h = base + 2 * plane;
    } else {
      h = base;
    }
  }
};

// ------------------------------------------------------------------ whole MLP
// Rule of ops.fwd.decode_preferred (its docstring has the measurements).
bool decode_preferred(int64_t M, int64_t K, int64_t N, int code, int64_t num_cu) {
  if (code == GMLP_F32 || M < 1 || M > 32 || K % 256 != 0 || N % 256 != 0 || N < 16 * num_cu) return false;
  if (M > 16 && !(K >= 768 && N >= 768 && K * N < ((int64_t)1 << 30))) return false;
  return K >= (M <= 16 ? 8 : 14) * num_cu;
}
// The widths that rule leaves out, on the same streaming kernels (two launches against the general path's
// four, no partial sums in memory).  One token tile always wins: K=1024, N=2048 11 to 13 us against 16,
// K=2200, N=4608 20 to 24 / 30, K=5168, N=20480 110 to 122 / 130 to 136.  With two, its operands' traffic
// grows with the rows per compute unit: up to 32 rows of W_gate they win (K=1024, N=8192 27 / 28, K=3592,
// N=8200 54 to 59 / 59 to 62), and beyond where the blocks are high enough for the share (rows of whole lines,
// K from 8 rows per unit up: K=2560, N=10240 44 / 47, K=3072, N=12288 55 / 60, K=2048, N=16384 M=24 52 / 56;
// K=3328, N=13312 M=20 64 / 62, M=24 60 / 62; K=1024, N=16384 41 / 39; K=4800, N=14400 89 / 89).
bool narrow_decode_preferred(int64_t M, int64_t K, int64_t N, int code, int64_t num_cu) {
  if (code == GMLP_F32 || M < 1 || M > 32 || K % 8 != 0 || N % 8 != 0) return false;
  if (K < 768 || N < 768 || K * N >= ((int64_t)1 << 30)) return false;
  if (M <= 16 || N <= 33 * num_cu) return true;
  return K % 256 == 0 && N % 64 == 0 && K >= 8 * num_cu && (M > 20 || N <= 48 * num_cu);
}
int64_t compute_units(int device) {
  static std::atomic<int> known[64];
  if (device < 0 || device >= 64) return 256;
  int n = known[device].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) n = 256;
    known[device].store(n, std::memory_order_relaxed);
  }
  return n;
}

Problem check_mlp(const Tensor& x, const Tensor& W_gate, const Tensor& b_gate, const Tensor& W_up, const Tensor& b_up,
                  const Tensor& W_down, const Tensor& b_down, int64_t act) {
  const int code = require_gpu({x, W_gate, b_gate, W_up, b_up, W_down, b_down});
  check_gate_up(x, W_gate, b_gate, W_up, b_up);
  const Problem q = problem_of(x, W_up, code, act);
  TORCH_CHECK_VALUE(W_down.dim() == 2 && W_down.size(0) == q.K && W_down.size(1) == q.N, "dimension mismatch in W_down ",
                    W_down.sizes());
  TORCH_CHECK_VALUE(!b_down.defined() || (b_down.dim() == 1 && b_down.size(0) == q.K), "dimension mismatch in b_down");
  return q;
}

Tensor mlp_infer(const Tensor& x_in, const Tensor& Wg_in, const OptTensor& bg_in, const Tensor& Wu_in, const OptTensor& bu_in,
                 const Tensor& Wd_in, const OptTensor& bd_in, int64_t act) {
  refuse_transforms("FusedGatedMLP", {x_in, Wg_in, or_undefined(bg_in), Wu_in, or_undefined(bu_in), Wd_in, or_undefined(bd_in)});
  const Problem q = check_mlp(x_in, Wg_in, or_undefined(bg_in), Wu_in, or_undefined(bu_in), Wd_in, or_undefined(bd_in), act);
  at::AutoDispatchBelowADInplaceOrView below;
  const c10::DeviceGuard guard(x_in.device());
  const Tensor x = x_in.contiguous(), Wg = Wg_in.contiguous(), Wu = Wu_in.contiguous(), Wd = Wd_in.contiguous();
  const Tensor bg = contiguous(or_undefined(bg_in)), bu = contiguous(or_undefined(bu_in)), bd = contiguous(or_undefined(bd_in));
  const Tensor y = at::empty(x.sizes(), x.options());
  if (q.M == 0) return y;
  void* const stream = stream_of(x);
  const int64_t cus = compute_units(x.device().index());
  const bool decode = decode_preferred(q.M, q.K, q.N, q.code, cus);
  if (decode || narrow_decode_preferred(q.M, q.K, q.N, q.code, cus)) {
    const Tensor h = at::empty({q.M <= 16 ? 16 : 32, q.N}, x.options());  // in the library's layout
    if (decode)
      check(lib.gmlp_decode_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(Wd), ptr(bg), ptr(bu), ptr(bd), out_ptr(h), out_ptr(y), nullptr, q.M,
                                q.K, q.N, q.code, q.act, stream));
    else
      check(lib.gmlp_decode_stream_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(Wd), ptr(bg), ptr(bu), ptr(bd), out_ptr(h), out_ptr(y), q.M,
                                       q.K, q.N, q.code, q.act, stream));
    return y;
  }
  const Tensor h = at::empty({q.M, q.N}, x.options());
  const size_t bytes = lib.gmlp_mlp_workspace_bytes(GMLP_PASS_FWD, q.M, q.K, q.N, q.code);
  const Tensor ws = scratch(bytes, x);
  check(lib.gmlp_mlp_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(Wd), ptr(bg), ptr(bu), ptr(bd), out_ptr(y), out_ptr(h), nullptr, nullptr,
                         q.M, q.K, q.N, q.code, q.act, 0.0f, 0, 0, out_ptr(ws), bytes, stream));
  return y;
}

// The outputs that are there, as gmlp_grads_workspace_bytes takes them.
int wanted_grads(const ag::variable_list& out, std::initializer_list<int> grads) {
  int wanted = 0, i = 0;
  for (int grad : grads) wanted |= out[i++].defined() ? grad : 0;
  return wanted;
}

// dY -> (dX, dW_gate, db_gate, dW_up, db_up, dW_down, db_down), in the order of the edges
struct MlpBackward : public ag::Node {
  Problem q;
  bool recompute = false;
  bool has_bias[3] = {false, false, false};  // gate, up, down
  std::vector<int64_t> x_sizes;
  at::TensorOptions options;  // of x
  ag::SavedVariable x_, Wg_, Wu_, Wd_;
  ag::SavedVariable acts_;      // G, U, H
  ag::SavedVariable bg_, bu_;   // recompute: G, U, H are computed again, from the inputs

  std::string name() const override { return "FusedGatedMLPBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (ag::SavedVariable* v : {&x_, &Wg_, &Wu_, &Wd_, &acts_, &bg_, &bu_}) v->reset_data();
  }
  ag::variable_list apply(ag::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    ag::variable_list out(7);
    const Tensor grad = materialized(grads[0], x_sizes, options);
    // first of all, while autograd still records: an unpack hook may run a whole forward (checkpointing)
    const Tensor x_saved = x_.unpack(), Wg_saved = Wg_.unpack(), Wu_saved = Wu_.unpack(), Wd_saved = Wd_.unpack();
    const Tensor acts_saved = acts_.unpack(), bg_saved = bg_.unpack(), bu_saved = bu_.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(grad.device());
    const Tensor dy = readable(grad, q.M * q.K, grad), x = readable(x_saved, q.M * q.K, dy);
    const Tensor Wg = readable(Wg_saved, q.N * q.K, dy), Wu = readable(Wu_saved, q.N * q.K, dy);
    const Tensor Wd = readable(Wd_saved, q.K * q.N, dy);
    const bool want[7] = {true, true, has_bias[0], true, has_bias[1], true, has_bias[2]};
    const int64_t shape[7][2] = {{0, 0}, {q.N, q.K}, {q.N, 0}, {q.N, q.K}, {q.N, 0}, {q.K, q.N}, {q.K, 0}};
    for (int i = 0; i < 7; ++i) {
      if (!want[i] || !task_should_compute_output(i)) continue;
      const at::IntArrayRef sizes = i == 0 ? at::IntArrayRef(x_sizes) : at::IntArrayRef(shape[i], i % 2 == 1 ? 2 : 1);
      out[i] = q.M == 0 ? at::zeros(sizes, dy.options()) : at::empty(sizes, dy.options());
    }
    if (q.M == 0) return out;
    void* const stream = stream_of(dy);
    Tensor kept;
    if (recompute) {
      const Tensor bg = has_bias[0] ? readable(bg_saved, q.N, dy) : Tensor();
      const Tensor bu = has_bias[1] ? readable(bu_saved, q.N, dy) : Tensor();
      kept = at::empty({3, q.M, q.N}, x.options());
      const Activations a(q, kept, true);
      const size_t bytes = lib.gmlp_workspace_bytes(GMLP_OP_GATEUP_FWD, q.M, q.K, q.N, q.code);
      const Tensor ws = scratch(bytes, x);
      check(lib.gmlp_gateup_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(bg), ptr(bu), a.h, a.g, a.u, nullptr, q.M, q.K, q.N, q.code, q.act,
                                (float)q.p, q.seed, q.offset, out_ptr(ws), bytes, stream));
    } else {
      kept = readable(acts_saved, 3 * q.M * q.N, dy);
    }
    const Activations a(q, kept, true);
    // dG, dU and the library's workspace share one scratch allocation that is dropped on return
    const size_t plane = ((size_t)(q.M * q.N) * dy.element_size() + 255) / 256 * 256;
    const int wanted = wanted_grads(out, {GMLP_GRAD_X, GMLP_GRAD_W_GATE, GMLP_GRAD_B_GATE, GMLP_GRAD_W_UP, GMLP_GRAD_B_UP,
                                          GMLP_GRAD_W_DOWN, GMLP_GRAD_B_DOWN});
    const size_t bytes = lib.gmlp_grads_workspace_bytes(GMLP_PASS_BWD, wanted, q.M, q.K, q.N, q.code);
    const Tensor arena = scratch(2 * plane + bytes, x);
    char* const base = (char*)out_ptr(arena);
    check(lib.gmlp_mlp_bwd(ptr(dy), ptr(x), ptr(Wg), ptr(Wu), ptr(Wd), a.g, a.u, a.h, base, base + plane, out_ptr(out[0]),
                           out_ptr(out[1]), out_ptr(out[3]), out_ptr(out[5]), out_ptr(out[2]), out_ptr(out[4]), out_ptr(out[6]),
                           q.M, q.K, q.N, q.code, q.act, (float)q.p, q.seed, q.offset, bytes > 0 ? base + 2 * plane : nullptr,
                           bytes, stream));
    refuse_second_derivative(*this, grad, out);
    return out;
  }
};

Tensor mlp_train(const Tensor& x_in, const Tensor& Wg_in, const OptTensor& bg_in, const Tensor& Wu_in, const OptTensor& bu_in,
                 const Tensor& Wd_in, const OptTensor& bd_in, double p, uint64_t seed, uint64_t offset, bool recompute,
                 int64_t act) {
  const Tensor &bg_o = or_undefined(bg_in), &bu_o = or_undefined(bu_in), &bd_o = or_undefined(bd_in);
  refuse_transforms("FusedGatedMLPFullFunction", {x_in, Wg_in, bg_o, Wu_in, bu_o, Wd_in, bd_o});
  Problem q = check_mlp(x_in, Wg_in, bg_o, Wu_in, bu_o, Wd_in, bd_o, act);
  q.p = p;
  q.seed = seed;
  q.offset = offset;
  const bool graph = ag::compute_requires_grad(x_in, Wg_in, bg_o, Wu_in, bu_o, Wd_in, bd_o), keep = graph && !recompute;
  Tensor y, kept;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    const Tensor x = x_in.contiguous(), Wg = Wg_in.contiguous(), Wu = Wu_in.contiguous(), Wd = Wd_in.contiguous();
    const Tensor bg = contiguous(bg_o), bu = contiguous(bu_o), bd = contiguous(bd_o);
    y = at::empty(x.sizes(), x.options());
    kept = keep ? at::empty({3, q.M, q.N}, x.options()) : at::empty({q.M, q.N}, x.options());
    if (q.M > 0) {
      const Activations a(q, kept, keep);
      const size_t bytes = lib.gmlp_mlp_workspace_bytes(GMLP_PASS_FWD, q.M, q.K, q.N, q.code);
      const Tensor ws = scratch(bytes, x);
      check(lib.gmlp_mlp_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(Wd), ptr(bg), ptr(bu), ptr(bd), out_ptr(y), a.h, a.g, a.u, q.M, q.K,
                             q.N, q.code, q.act, (float)p, seed, offset, out_ptr(ws), bytes, stream_of(x)));
    }
  }
  if (graph) {
    auto node = std::shared_ptr<MlpBackward>(new MlpBackward(), ag::deleteNode);
    node->set_next_edges(ag::collect_next_edges(x_in, Wg_in, bg_o, Wu_in, bu_o, Wd_in, bd_o));
    node->q = q;
    node->recompute = recompute;
    node->has_bias[0] = bg_o.defined();
    node->has_bias[1] = bu_o.defined();
    node->has_bias[2] = bd_o.defined();
    node->x_sizes = x_in.sizes().vec();
    node->options = y.options();
    node->x_ = ag::SavedVariable(x_in, false);
    node->Wg_ = ag::SavedVariable(Wg_in, false);
    node->Wu_ = ag::SavedVariable(Wu_in, false);
    node->Wd_ = ag::SavedVariable(Wd_in, false);
    if (recompute) {
      node->bg_ = ag::SavedVariable(bg_o, false);
      node->bu_ = ag::SavedVariable(bu_o, false);
    } else {
      node->acts_ = ag::SavedVariable(kept, false);
    }
    ag::set_history(y, node);
  }
  return y;
}

// ------------------------------------------------------------------ hidden states alone
// dH -> (dX, dW_up, db_up, dW_gp, db_gp), in the order of the edges
struct HiddenBackward : public ag::Node {
  Problem q;
  bool has_bias[2] = {false, false};  // up, gate
  at::TensorOptions options;          // of x
  ag::SavedVariable x_, Wu_, Wg_;
  ag::SavedVariable gate_up_;  // [2, M, N]

  std::string name() const override { return "FusedGatedMLPHiddenBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (ag::SavedVariable* v : {&x_, &Wu_, &Wg_, &gate_up_}) v->reset_data();
  }
  ag::variable_list apply(ag::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    ag::variable_list out(5);
    const Tensor grad = materialized(grads[0], {q.M, q.N}, options);
    const Tensor x_saved = x_.unpack(), Wu_saved = Wu_.unpack(), Wg_saved = Wg_.unpack(), gate_up_saved = gate_up_.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(grad.device());
    const Tensor dh = readable(grad, q.M * q.N, grad), x = readable(x_saved, q.M * q.K, dh);
    const Tensor Wu = readable(Wu_saved, q.N * q.K, dh), Wg = readable(Wg_saved, q.N * q.K, dh);
    const Tensor kept = readable(gate_up_saved, 2 * q.M * q.N, dh);
    const bool want[5] = {true, true, has_bias[0], true, has_bias[1]};
    const int64_t shape[5][2] = {{q.M, q.K}, {q.N, q.K}, {q.N, 0}, {q.N, q.K}, {q.N, 0}};
    for (int i = 0; i < 5; ++i) {
      if (!want[i] || !task_should_compute_output(i)) continue;
      const at::IntArrayRef sizes(shape[i], i == 2 || i == 4 ? 1 : 2);
      out[i] = q.M == 0 ? at::zeros(sizes, dh.options()) : at::empty(sizes, dh.options());
    }
    if (q.M == 0) return out;
    // dG, dU and the library's workspace share one scratch allocation
    const size_t plane = ((size_t)(q.M * q.N) * dh.element_size() + 255) / 256 * 256;
    const int wanted = wanted_grads(out, {GMLP_GRAD_X, GMLP_GRAD_W_UP, GMLP_GRAD_B_UP, GMLP_GRAD_W_GATE, GMLP_GRAD_B_GATE});
    const size_t bytes = lib.gmlp_grads_workspace_bytes(GMLP_PASS_HIDDEN_BWD, wanted, q.M, q.K, q.N, q.code);
    const Tensor arena = scratch(2 * plane + bytes, x);
    char *const dg = (char*)out_ptr(arena), *const du = dg + plane, *const ws = bytes > 0 ? du + plane : nullptr;
    const char* g = (const char*)ptr(kept);
    const char* u = g + q.M * q.N * (int64_t)kept.element_size();
    check(lib.gmlp_hidden_bwd(ptr(dh), ptr(x), ptr(Wg), ptr(Wu), g, u, dg, du, out_ptr(out[0]), out_ptr(out[3]), out_ptr(out[1]),
                              out_ptr(out[4]), out_ptr(out[2]), q.M, q.K, q.N, q.code, q.act, (float)q.p, q.seed, q.offset, ws,
                              bytes, stream_of(dh)));
    refuse_second_derivative(*this, grad, out);
    return out;
  }
};

Tensor hidden(const Tensor& x_in, const Tensor& Wu_in, const OptTensor& bu_in, const Tensor& Wg_in, const OptTensor& bg_in,
              double p, uint64_t seed, uint64_t offset, int64_t act) {
  const Tensor &bu_o = or_undefined(bu_in), &bg_o = or_undefined(bg_in);
  refuse_transforms("FusedGatedMLPFunction", {x_in, Wg_in, bg_o, Wu_in, bu_o});
  TORCH_CHECK_VALUE(x_in.dim() == 2, "input tensor must be 2-D [M, K], got ", x_in.dim(), " dims");
  check_gate_up(x_in, Wg_in, bg_o, Wu_in, bu_o);
  Problem q = problem_of(x_in, Wu_in, require_gpu({x_in, Wg_in, bg_o, Wu_in, bu_o}), act);
  q.p = p;
  q.seed = seed;
  q.offset = offset;
  const bool graph = ag::compute_requires_grad(x_in, Wu_in, bu_o, Wg_in, bg_o);
  Tensor h, kept;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    const Tensor x = x_in.contiguous(), Wu = Wu_in.contiguous(), Wg = Wg_in.contiguous();
    const Tensor bu = contiguous(bu_o), bg = contiguous(bg_o);
    h = at::empty({q.M, q.N}, x.options());
    if (graph) kept = at::empty({2, q.M, q.N}, x.options());
    if (q.M > 0) {
      char* const g = (char*)out_ptr(kept);
      char* const u = graph ? g + q.M * q.N * (int64_t)x.element_size() : nullptr;
      const size_t bytes = lib.gmlp_workspace_bytes(GMLP_OP_GATEUP_FWD, q.M, q.K, q.N, q.code);
      const Tensor ws = scratch(bytes, x);
      check(lib.gmlp_gateup_fwd(ptr(x), ptr(Wg), ptr(Wu), ptr(bg), ptr(bu), out_ptr(h), g, u, nullptr, q.M, q.K, q.N, q.code,
                                q.act, (float)p, seed, offset, out_ptr(ws), bytes, stream_of(x)));
    }
  }
  if (graph) {
    auto node = std::shared_ptr<HiddenBackward>(new HiddenBackward(), ag::deleteNode);
    node->set_next_edges(ag::collect_next_edges(x_in, Wu_in, bu_o, Wg_in, bg_o));
    node->q = q;
    node->has_bias[0] = bu_o.defined();
    node->has_bias[1] = bg_o.defined();
    node->options = h.options();
    node->x_ = ag::SavedVariable(x_in, false);
    node->Wu_ = ag::SavedVariable(Wu_in, false);
    node->Wg_ = ag::SavedVariable(Wg_in, false);
    node->gate_up_ = ag::SavedVariable(kept, false);
    ag::set_history(h, node);
  }
  return h;
}

// ------------------------------------------------------------------ torch.jit.trace
// While a trace is being recorded a call goes through torch's dispatcher, as an operator with a schema: the
// tracer then records the call itself.  Called directly it would record the only torch operation that it
// sees, the output's at::empty, and the traced graph would return memory that nothing fills.  Whether an
// autograd node is recorded is decided when the operator runs, as in the module.  Every other call goes
// straight to the functions above.
Tensor mlp_op(const Tensor& x, const Tensor& Wg, const OptTensor& bg, const Tensor& Wu, const OptTensor& bu, const Tensor& Wd,
              const OptTensor& bd, double p, int64_t seed, int64_t offset, bool recompute, int64_t act) {
  if (p == 0.0 && !ag::compute_requires_grad(x, Wg, or_undefined(bg), Wu, or_undefined(bu), Wd, or_undefined(bd)))
    return mlp_infer(x, Wg, bg, Wu, bu, Wd, bd, act);
  return mlp_train(x, Wg, bg, Wu, bu, Wd, bd, p, (uint64_t)seed, (uint64_t)offset, recompute, act);
}
Tensor hidden_op(const Tensor& x, const Tensor& Wu, const OptTensor& bu, const Tensor& Wg, const OptTensor& bg, double p,
                 int64_t seed, int64_t offset, int64_t act) {
  return hidden(x, Wu, bu, Wg, bg, p, (uint64_t)seed, (uint64_t)offset, act);
}

template <typename F>
c10::TypedOperatorHandle<F> recorded_operator(const char* name, F*) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}

// The entry points of the Python side (mlp_infer is not called while tracing).
Tensor call_mlp_train(const Tensor& x, const Tensor& Wg, const OptTensor& bg, const Tensor& Wu, const OptTensor& bu,
                      const Tensor& Wd, const OptTensor& bd, double p, uint64_t seed, uint64_t offset, bool recompute,
                      int64_t act) {
  if (torch::jit::tracer::isTracing()) {
    static const auto op = recorded_operator("triton_gated_mlp::mlp", mlp_op);
    return op.call(x, Wg, bg, Wu, bu, Wd, bd, p, (int64_t)seed, (int64_t)offset, recompute, act);
  }
  return mlp_train(x, Wg, bg, Wu, bu, Wd, bd, p, seed, offset, recompute, act);
}
Tensor call_hidden(const Tensor& x, const Tensor& Wu, const OptTensor& bu, const Tensor& Wg, const OptTensor& bg, double p,
                   uint64_t seed, uint64_t offset, int64_t act) {
  if (torch::jit::tracer::isTracing()) {
    static const auto op = recorded_operator("triton_gated_mlp::hidden", hidden_op);
    return op.call(x, Wu, bu, Wg, bg, p, (int64_t)seed, (int64_t)offset, act);
  }
  return hidden(x, Wu, bu, Wg, bg, p, seed, offset, act);
}

}  // namespace

TORCH_LIBRARY(triton_gated_mlp, m) {
  m.def("mlp(Tensor x, Tensor W_gate, Tensor? b_gate, Tensor W_up, Tensor? b_up, Tensor W_down, Tensor? b_down, "
        "float dropout_p, int seed, int offset, bool recompute, int act) -> Tensor", mlp_op);
  m.def("hidden(Tensor x, Tensor W_up, Tensor? b_up, Tensor W_gp, Tensor? b_gp, float dropout_p, int seed, int offset, "
        "int act) -> Tensor", hidden_op);
}

PYBIND11_MODULE(_gmlp_torch, m) {
  m.def("bind", torch::wrap_pybind_function(bind));
  m.def("decode_preferred", torch::wrap_pybind_function(decode_preferred));
  m.def("mlp_infer", torch::wrap_pybind_function_no_gil(mlp_infer));
  m.def("mlp_train", torch::wrap_pybind_function_no_gil(call_mlp_train));
  m.def("hidden", torch::wrap_pybind_function_no_gil(call_hidden));
}
