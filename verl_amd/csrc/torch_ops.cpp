// Native host side of the [B, L] entry points that an update calls many times a step: argument conversion, allocation,
// the library call and the autograd nodes, which in Python cost more than the kernels they launch (GRPO, policy loss,
// entropy aggregation and KL loss with their backward at 512 x 4096: 61 us of kernels in 340 us).  The Python functions
// in verl_amd/trainer/ppo keep names, arguments and checks of configuration; everything from the tensors on is here.
//
// The backward nodes run on autograd's device thread without the interpreter, the losses' results come back through
// host memory the GPU writes (fetch()), and the counter buffers of the single-launch reductions are kept here, one per
// (device, stream), for Python's ctypes calls as well.
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/anomaly_mode.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/extension.h>

#include <array>
#include <atomic>
#include <chrono>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/verl_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

[[noreturn]] void raise_assertion(const std::string& text) {
  PyErr_SetString(PyExc_AssertionError, text.c_str());
  throw py::error_already_set();
}

void check(int rc) {
  TORCH_CHECK(rc == 0, "libverl_amd error ", rc, ": ", vamd_last_error());
}

// Device the kernels run on: the tensors' GPU, or the current GPU for CPU inputs.
at::Device compute_device(std::initializer_list<const Tensor*> tensors) {
  for (const Tensor* t : tensors)
    if (t->defined() && t->is_cuda()) return t->device();
  if (!at::hasCUDA() || c10::hip::device_count() == 0)
    throw std::runtime_error("verl_amd needs a ROCm GPU: no device is visible and there is no CPU fallback");
  at::globalContext().lazyInitDevice(at::kCUDA);
  return at::Device(at::kCUDA, c10::hip::current_device());
}

void* stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// fp32, contiguous, on `dev`
Tensor as_f32(const Tensor& t, const at::Device& dev) {
  Tensor x = t;
  if (x.device() != dev || x.scalar_type() != at::kFloat) x = x.to(dev, at::kFloat);
  return x.is_contiguous() ? x : x.contiguous();
}

std::string shape_text(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

Tensor matrix(const Tensor& t, const at::Device& dev) {
  Tensor x = as_f32(t, dev);
  if (x.dim() == 1) x = x.view({1, -1});
  if (x.dim() != 2) raise_assertion("expected a (batch, length) tensor, got shape " + shape_text(t));
  return x;
}

// Contiguous mask on `dev` in one of the element types the kernels read, with its VAMD_MASK_* code.
struct Mask {
  Tensor t;
  int code;
};
Mask mask_of(const Tensor& mask, const at::Device& dev) {
  Mask m{mask.device() == dev ? mask : mask.to(dev), 0};
  switch (mask.scalar_type()) {
    case at::kFloat: m.code = VAMD_MASK_F32; break;
    case at::kLong: m.code = VAMD_MASK_I64; break;
    case at::kBool:
    case at::kByte: m.code = VAMD_MASK_U8; break;
    case at::kInt: m.code = VAMD_MASK_I32; break;
    default:  // fp16 / bf16 / fp64 / int8 / int16: exact in fp32 for 0/1 masks
      m.t = m.t.to(at::kFloat);
      m.code = VAMD_MASK_F32;
  }
  if (!m.t.is_contiguous()) m.t = m.t.contiguous();
  return m;
}
Mask mask_matrix(const Tensor& mask, const at::Device& dev, const Tensor& like) {
  Mask m = mask_of(mask, dev);
  if (m.t.dim() == 1) m.t = m.t.view({1, -1});
  if (m.t.sizes() != like.sizes())
    raise_assertion("mask shape " + shape_text(mask) + " does not match " + shape_text(like));
  return m;
}

const float* f32(const Tensor& t) { return t.defined() ? t.const_data_ptr<float>() : nullptr; }
float* f32_out(const Tensor& t) { return t.defined() ? t.mutable_data_ptr<float>() : nullptr; }

Tensor new_f32(at::IntArrayRef shape, const at::Device& dev) {
  return at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(dev));
}

// Parts of a call's one result allocation as tensors of their own, not views of it to autograd: a loss may be changed in place
// (`loss /= n`, `loss.detach().mul_(s)`), and the version of what a node has saved is not that of the loss beside it.
Tensor part(const Tensor& t, int64_t first, int64_t count) {
  at::AutoDispatchBelowADInplaceOrView no_view;
  return t.narrow(0, first, count);
}
Tensor scalar_part(const Tensor& t, int64_t i) {
  at::AutoDispatchBelowADInplaceOrView no_view;
  return t.select(0, i);
}

// Scratch of the single-launch reductions: its first VAMD_TICKET_BYTES are arrival counters that are zero on entry and
// zero again on completion, so one zeroed buffer per (device, stream) is kept; kernels on one stream run in order and
// never share it.  Never destroyed: at exit the runtime may be gone first.
Tensor ticket_workspace(size_t bytes, const at::Device& dev) {
  static std::mutex mu;
  static auto* buffers = new std::map<std::pair<int, void*>, Tensor>;
  const int64_t need = bytes < 4096 ? 4096 : (int64_t)bytes;
  const std::pair<int, void*> key{(int)dev.index(), stream_of(dev)};
  const auto kept = [&](const Tensor& fresh) {
    std::lock_guard<std::mutex> lock(mu);
    Tensor& buf = (*buffers)[key];
    if (fresh.defined() && (!buf.defined() || buf.numel() < need)) buf = fresh;
    return buf;
  };
  const Tensor buf = kept(Tensor());
  if (buf.defined() && buf.numel() >= need) return buf;
  // Without the lock: an allocation may run Python (a dispatch mode), which may let a thread run that comes here, holding the
  // interpreter.
  return kept(at::zeros({need < (1 << 20) ? (1 << 20) : need}, at::TensorOptions().dtype(at::kByte).device(dev)));
}

bool wants_gradient(const Tensor& t) { return at::GradMode::is_enabled() && t.requires_grad(); }

// The losses have no forward-mode derivative.  Asked before the choice between a node and a plain call: a dual tensor needs
// no requires_grad, and a loss without a tangent would read as a derivative of zero.
void refuse_tangents(const char* loss, std::initializer_list<const Tensor*> inputs) {
  for (const Tensor* t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(), loss,
                                " cannot be differentiated in forward mode");
}

struct Aggregation {
  int mode;
  double dp_size, batch_num_tokens, global_batch_size, loss_scale_factor;
};

// A loss node saves the gradient per unit upstream gradient, which the forward pass wrote, and the rows' coefficients;
// what else its backward needs to hand the gradient back in the input's form is kept only where that is not
// (batch, length) fp32 on the compute device.
void save_form(AutogradContext* ctx, const Tensor& input, const at::Device& dev) {
  if (input.dim() == 2 && input.scalar_type() == at::kFloat && input.device() == dev) return;
  ctx->saved_data["shape"] = input.sizes().vec();
  ctx->saved_data["device"] = input.device();
  ctx->saved_data["dtype"] = (int64_t)input.scalar_type();
}
bool in_kernel_form(AutogradContext* ctx) { return ctx->saved_data.find("shape") == ctx->saved_data.end(); }
Tensor in_saved_form(AutogradContext* ctx, Tensor g) {
  if (in_kernel_form(ctx)) return g;
  return g.view(ctx->saved_data["shape"].toIntVector())
      .to(ctx->saved_data["device"].toDevice(), (at::ScalarType)ctx->saved_data["dtype"].toInt());
}

Tensor upstream(const Tensor& d_loss, const at::Device& dev) { return as_f32(d_loss, dev).reshape({1}); }

// ---- sums of gradients ---------------------------------------------------------------------------------------
// Two nodes that differentiate the same tensor (entropy and log-probs of the logits, KL loss and policy loss of the
// log-probs) each hand autograd a gradient, which it adds up in a pass of its own: two tensors read and one written.
// Instead the node that runs first may leave its gradient with the other one and hand back none; the other one adds its own
// to it in the kernel that forms that, and hands back the sum.  What autograd has been given is not touched: its buffers
// belong to all its threads, and a node of another one (a copy of the same tensor to the host or to another GPU) may add to
// them at any time.  A gradient is left with a node only if
//   - it differentiates the same input of the same receiver, and the backward pass at hand includes it and needs it;
//   - it has not run in this pass.  Ids of passes grow, so a node whose newest run was in an older pass has not;
//   - it runs on the same device, so on this thread or one that takes over from it, and on the same stream;
//   - nothing was left with it by another pass that still runs or has failed;
//   - neither node has hooks, which would see the gradients apart, the pass records no graph of its own, and anomaly
//     detection, which looks at each gradient, is off.
// Otherwise each node hands back its own gradient, as ever.  What was left lies in the other node's saved data: if the pass
// fails in between it goes with the graph.  (Figures: scale_rows_add_kernel and row_softmax_backward_kernel.)
using torch::autograd::Edge;
using torch::autograd::Node;

// The newest nodes that can add to a gradient left with them, of all threads: where a running node looks for another one.
// All that counts is asked of the node itself; a node that is no longer among them is not found.  In vectors, because a
// backward pass finds them in another core's cache: where there is nothing to sum it reads four lines of them (asking 32 nodes
// one by one whether they belong to the pass cost 3 us of the 165 us of a call with two losses).
constexpr int kJoinable = 16;
struct Joinables {
  std::mutex mu;  // also guards kLeft and kLeftPass of every node's saved data
  int next = 0;
  std::array<Node*, kJoinable> key{}, receiver{};  // compared, never followed
  std::array<int, kJoinable> ran{};                // the newest pass in which the node has run
  std::array<std::weak_ptr<Node>, kJoinable> node;
  std::array<AutogradContext*, kJoinable> ctx{};  // lives in the node
};
Joinables& joinables() {
  static auto* j = new Joinables;  // never destroyed: at exit threads of autograd may still run
  return *j;
}
constexpr const char *kLeft = "left", *kLeftPass = "left_pass";

// The node of F that made `output` can add to a gradient left with it, unless its own takes another form or another's place.
template <class F>
void joinable(const Tensor& output) {
  const auto& node = output.grad_fn();
  auto* const made = dynamic_cast<torch::autograd::CppNode<F>*>(node.get());
  if (!made || made->num_outputs() == 0 || !made->next_edge(0).is_valid() || !in_kernel_form(&made->ctx_)) return;
  const auto in_place = made->ctx_.saved_data.find("in_place");
  if (in_place != made->ctx_.saved_data.end() && in_place->second.toBool()) return;
  Joinables& all = joinables();
  std::lock_guard<std::mutex> lock(all.mu);
  const int i = all.next;
  all.next = (i + 1) % kJoinable;
  all.key[i] = made;
  all.receiver[i] = made->next_edge(0).function.get();
  all.ran[i] = -1;
  all.node[i] = node;
  all.ctx[i] = &made->ctx_;
}

// One node's part in the sum, from the start of its backward function.
class Summing {
 public:
  explicit Summing(AutogradContext* ctx)
      : pass_(torch::autograd::get_current_graph_task_id()),
        seen_apart_(at::GradMode::is_enabled() || torch::autograd::AnomalyMode::is_enabled()) {
    if (pass_ < 0) return;
    me_ = torch::autograd::get_current_node();
    Joinables& all = joinables();
    std::lock_guard<std::mutex> lock(all.mu);
    for (int i = 0; i < kJoinable; ++i)
      if (all.key[i] == me_.get() && all.ran[i] < pass_) all.ran[i] = pass_;
    auto& data = ctx->saved_data;
    const auto left = data.find(kLeft);
    if (left == data.end() || data[kLeftPass].toInt() != pass_) return;
    left_ = left->second.toTensor();
    data.erase(left);
  }

  // Looks for the other node.  Where this node's gradient of the form given goes: a tensor to which it adds its own, or an
  // undefined tensor, and then it makes one.
  Tensor target(at::IntArrayRef shape, at::ScalarType type, const at::Device& dev) {
    find_other(dev);
    const Tensor& sum = left_.defined() ? left_ : left_there_;
    if (sum.defined() && sum.sizes() == shape && sum.scalar_type() == type && sum.device() == dev) return sum;
    return Tensor();
  }

  // What the node hands back for `grad`, which holds its gradient and what was in target().
  Tensor result(const Tensor& grad) {
    Tensor sum = grad;
    if (left_.defined() && !(sum.defined() && sum.is_same(left_))) sum = sum.defined() ? sum.add(left_) : left_;
    if (!other_ || !sum.defined()) return sum;
    if (left_there_.defined()) return sum.is_same(left_there_) ? Tensor() : sum;
    if (!sum.is_cuda() || !sum.is_contiguous()) return sum;
    Joinables& all = joinables();
    std::lock_guard<std::mutex> lock(all.mu);
    auto& data = all.ctx[slot_]->saved_data;
    if (all.key[slot_] != other_.get() || all.ran[slot_] >= pass_ || data.count(kLeft)) return sum;
    data[kLeftPass] = (int64_t)pass_;
    data[kLeft] = sum;
    return Tensor();
  }

 private:
  void find_other(const at::Device& dev) {
    if (pass_ < 0 || seen_apart_ || !me_ || me_->num_outputs() == 0 || !me_->post_hooks().empty()) return;
    const Edge& edge = me_->next_edge(0);
    if (!edge.is_valid()) return;
    std::array<std::shared_ptr<Node>, kJoinable> seen;  // (a node whose last owner this is goes after the lock)
    Joinables& all = joinables();
    std::lock_guard<std::mutex> lock(all.mu);
    for (int i = 0; i < kJoinable; ++i) {
      if (all.receiver[i] != edge.function.get() || all.key[i] == me_.get() || all.ran[i] >= pass_) continue;
      const auto& node = seen[i] = all.node[i].lock();
      if (!node || !runs_later(*node, edge, dev)) continue;
      const auto& data = all.ctx[i]->saved_data;
      const auto left = data.find(kLeft);
      if (left != data.end()) {
        if (data.at(kLeftPass).toInt() != pass_) continue;
        left_there_ = left->second.toTensor();
      }
      other_ = node;
      slot_ = i;
      return;
    }
  }

  // Whether the pass at hand runs `node`, which has not run in it, after this one, as the comment above asks.
  bool runs_later(Node& node, const Edge& edge, const at::Device& dev) const {
    const auto* const nodes = torch::autograd::get_current_graph_task_nodes_in_graph();
    if (!nodes || !nodes->count(&node) || node.num_outputs() == 0 || node.next_edge(0) != edge ||
        node.device() != me_->device() || !node.post_hooks().empty())
      return false;
    const auto stream = node.stream();
    const auto mine = c10::hip::getCurrentHIPStream(dev.index());
    if (!stream || stream->device_index() != mine.device_index() || stream->id() != mine.id()) return false;
    const auto* const needed = torch::autograd::get_current_graph_task_exec_info();
    if (!needed || needed->empty()) return true;
    const auto info = needed->find(&node);
    return info != needed->end() && info->second.needed_;
  }

  int pass_;
  bool seen_apart_;  // the pass records a graph of its gradients, or looks at each
  std::shared_ptr<Node> me_, other_;
  int slot_ = 0;     // the other node's place among the joinable ones
  Tensor left_, left_there_;  // what was left with this node, and with the other one
};

// The gradient of a loss whose forward pass left it per unit upstream gradient.
variable_list scaled_gradient(AutogradContext* ctx, const variable_list& grads, float extra_scale, size_t inputs) {
  Summing summing(ctx);
  at::AutoGradMode no_grad(false);
  variable_list result(inputs);
  const auto saved = ctx->get_saved_variables();
  TORCH_CHECK(saved.size() == 2, "the forward pass was not asked for a gradient of this input");
  if (!grads[0].defined()) {
    result[0] = summing.result(Tensor());
    return result;
  }
  const Tensor &g = saved[0], &coef = saved[1];
  const at::Device dev = g.device();
  const c10::DeviceGuard guard(dev);
  const Tensor d = upstream(grads[0], dev);
  const Tensor sum = in_kernel_form(ctx) ? summing.target(g.sizes(), at::kFloat, dev) : Tensor();
  const Tensor out = sum.defined() ? sum : at::empty_like(g);
  check((sum.defined() ? vamd_scale_rows_add : vamd_scale_rows)(f32(g), f32(coef), f32(d), extra_scale, g.size(0),
                                                                g.size(1), f32_out(out), stream_of(dev)));
  result[0] = summing.result(in_saved_form(ctx, out));
  return result;
}

// ---- log-probs and entropies of materialised logits ----------------------------------------------------------
// Nodes in C++ because two of them on the same logits sum their gradients, and because up to a few hundred rows the host is what
// a call waits for.
struct Rows {
  Tensor t;     // [rows, vocab], unit stride along the vocabulary
  int64_t ld;   // row pitch
  int type;     // VAMD_DT_*
  const void* data() const { return t.const_data_ptr(); }
  int64_t n() const { return t.size(0); }
  int64_t vocab() const { return t.size(1); }
};
int row_type(at::ScalarType type) {
  return type == at::kFloat ? VAMD_DT_F32 : type == at::kBFloat16 ? VAMD_DT_BF16 : type == at::kHalf ? VAMD_DT_F16 : -1;
}
Rows logit_rows(const Tensor& logits) {
  if (!logits.is_cuda()) raise_assertion("the logits must live on the GPU: there is no CPU fallback");
  const int type = row_type(logits.scalar_type());
  if (type < 0) raise_assertion(std::string("logits must be fp32, bf16 or fp16, got ") + c10::toString(logits.scalar_type()));
  if (logits.dim() < 1 || logits.numel() == 0) raise_assertion("");
  const int64_t vocab = logits.size(-1);
  Tensor rows = logits.reshape({-1, vocab});
  if (rows.stride(1) != 1 || (rows.size(0) > 1 && rows.stride(0) < vocab)) rows = rows.contiguous();
  return {rows, rows.size(0) > 1 ? rows.stride(0) : vocab, type};
}
// The logits that a node saved.  Hooks on saved tensors may hand them back in other strides (save_on_cpu keeps none), so the
// pitch is that of what comes back.
Rows saved_rows(const Tensor& rows, at::IntArrayRef shape) {
  const Rows r = logit_rows(rows);
  if (r.t.numel() != c10::multiply_integers(shape) || r.vocab() != shape.back())
    raise_assertion("saved logits came back as " + shape_text(rows));
  return r;
}
Tensor label_rows(const Tensor& labels, const Tensor& logits) {
  if (logits.dim() < 1 || labels.sizes() != logits.sizes().slice(0, logits.dim() - 1))
    raise_assertion("labels " + shape_text(labels) + " do not match logits " + shape_text(logits));
  return labels.reshape({-1}).to(logits.device(), at::kLong).contiguous();
}

struct RowStats {
  Tensor value, lse, mean_z;  // log-prob or entropy in `type`; what the backward pass needs, in fp32
};
// log-probs of `labels`, or without labels entropies
RowStats row_stats(const Tensor& logits, const Rows& r, const Tensor& labels, at::ScalarType type, bool need_grad) {
  const at::Device dev = logits.device();
  const c10::DeviceGuard guard(dev);
  const bool entropy = !labels.defined();
  const Tensor value = at::empty(logits.sizes().slice(0, logits.dim() - 1), at::TensorOptions().dtype(type).device(dev));
  const Tensor kept = need_grad ? new_f32({entropy ? 2 : 1, r.n()}, dev) : Tensor();
  const Tensor lse = need_grad ? kept.select(0, 0) : Tensor(), mean_z = need_grad && entropy ? kept.select(0, 1) : Tensor();
  void* const out = value.mutable_data_ptr();
  check(vamd_row_softmax_stats_as(r.data(), r.type, r.n(), r.vocab(), r.ld,
                                  entropy ? nullptr : labels.const_data_ptr<int64_t>(), entropy ? nullptr : out,
                                  entropy ? out : nullptr, row_type(type), f32_out(lse), f32_out(mean_z), stream_of(dev)));
  return {value, lse, mean_z};
}

// What a node hands back for the logits, in `shape`.
Tensor row_gradient(const Rows& r, const Tensor& labels, const Tensor& lse, const Tensor& mean_z, const Tensor& upstream,
                    at::IntArrayRef shape, bool in_place, Summing& summing) {
  const at::Device dev = r.t.device();
  const c10::DeviceGuard guard(dev);
  const at::ScalarType type = upstream.scalar_type() == r.t.scalar_type() ? upstream.scalar_type() : at::kFloat;
  const Tensor g = upstream.detach().reshape({-1}).to(dev, type).contiguous();
  const bool entropy = mean_z.defined();
  const Tensor sum = in_place ? Tensor() : summing.target(shape, r.t.scalar_type(), dev);
  const Tensor out = in_place ? r.t : sum.defined() ? sum : at::empty(shape, r.t.options());
  check((sum.defined() ? vamd_row_softmax_backward_add : vamd_row_softmax_backward_as)(
      r.data(), r.type, r.n(), r.vocab(), r.ld, entropy ? nullptr : labels.const_data_ptr<int64_t>(), f32(lse), f32(mean_z),
      entropy ? nullptr : g.const_data_ptr(), entropy ? g.const_data_ptr() : nullptr, row_type(type), out.mutable_data_ptr(),
      in_place ? r.ld : r.vocab(), stream_of(dev)));
  return summing.result(in_place ? out.view(shape) : out);
}

class RowLogprobs : public torch::autograd::Function<RowLogprobs> {
 public:
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& labels, bool inplace_backward) {
    const Tensor lab = label_rows(labels, logits);
    const Rows r = logit_rows(logits);
    const RowStats s = row_stats(logits, r, lab, logits.scalar_type(), true);
    ctx->save_for_backward({r.t, lab, s.lse});
    ctx->saved_data["logits_shape"] = logits.sizes().vec();
    // writing the gradient over the logits needs the rows to be the caller's storage, and never overwrites a parameter
    ctx->saved_data["in_place"] = inplace_backward && r.data() == logits.const_data_ptr() && logits.is_contiguous() &&
                                  !(logits.is_leaf() && logits.requires_grad());
    return s.value;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const bool records = at::GradMode::is_enabled();
    Summing summing(ctx);
    Tensor d;
    {
      at::AutoGradMode no_grad(false);
      const auto saved = ctx->get_saved_variables();
      const bool in_place = ctx->saved_data["in_place"].toBool();
      if (in_place) {
        // the logits are about to become their own gradient: a second pass over this node would read gradients where
        // it expects logits
        TORCH_CHECK(!ctx->saved_data.count("logits_overwritten"),
                    "logprobs_from_logits(inplace_backward=True) wrote the gradient over the logits in its first backward "
                    "pass and cannot run a second one; pass inplace_backward=False to keep the logits");
        ctx->saved_data["logits_overwritten"] = true;
      }
      const auto shape = ctx->saved_data["logits_shape"].toIntVector();
      d = row_gradient(saved_rows(saved[0], shape), saved[1], saved[2], Tensor(), grads[0], shape, in_place, summing);
    }
    if (records && grads[0].requires_grad())  // the gradient is no function of its own to differentiate
      d = torch::autograd::DelayedError("trying to differentiate twice a function that was marked with @once_differentiable",
                                        1)({d.detach().requires_grad_()})[0];
    return {d, Tensor(), Tensor()};
  }
};

class RowEntropy : public torch::autograd::Function<RowEntropy> {
 public:
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, bool fp32_output) {
    const Rows r = logit_rows(logits);
    const RowStats s = row_stats(logits, r, Tensor(), fp32_output ? at::kFloat : logits.scalar_type(), true);
    ctx->save_for_backward({r.t, s.lse, s.mean_z});
    ctx->saved_data["logits_shape"] = logits.sizes().vec();
    return s.value;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    Summing summing(ctx);
    at::AutoGradMode no_grad(false);
    const auto saved = ctx->get_saved_variables();
    const auto shape = ctx->saved_data["logits_shape"].toIntVector();
    return {row_gradient(saved_rows(saved[0], shape), Tensor(), saved[1], saved[2], grads[0], shape, false, summing),
            Tensor()};
  }
};

Tensor logprobs_from_logits(const Tensor& logits, const Tensor& labels, bool inplace_backward) {
  refuse_tangents("logprobs_from_logits", {&logits});
  // (labels of a floating type may require a gradient, and get none)
  if (wants_gradient(logits) || wants_gradient(labels)) {
    const Tensor logprobs = RowLogprobs::apply(logits, labels, inplace_backward);
    joinable<RowLogprobs>(logprobs);
    return logprobs;
  }
  at::AutoGradMode no_grad(false);
  const Tensor lab = label_rows(labels, logits);
  return row_stats(logits, logit_rows(logits), lab, logits.scalar_type(), false).value;
}

Tensor entropy_from_logits(const Tensor& logits, bool fp32_output) {
  refuse_tangents("entropy_from_logits", {&logits});
  if (wants_gradient(logits)) {
    const Tensor entropy = RowEntropy::apply(logits, fp32_output);
    joinable<RowEntropy>(entropy);
    return entropy;
  }
  at::AutoGradMode no_grad(false);
  return row_stats(logits, logit_rows(logits), Tensor(), fp32_output ? at::kFloat : logits.scalar_type(), false).value;
}

// ---- policy loss ---------------------------------------------------------------------------------------------
struct PolicyArgs {
  int variant;
  double clip_low, clip_high, clip_c, tau_pos, tau_neg;
  Aggregation agg;
};
struct LossResult {
  Tensor loss, out, grad, coef;
  at::Device dev;
};

LossResult policy_forward(const Tensor& log_prob, const Tensor& old_log_prob, const Tensor& advantages,
                          const Tensor& mask, const std::optional<Tensor>& is_weights, const PolicyArgs& a,
                          bool need_grad) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&log_prob, &old_log_prob, &advantages, &mask});
  const Tensor lp = matrix(log_prob, dev), old = matrix(old_log_prob, dev), adv = matrix(advantages, dev);
  if (lp.sizes() != old.sizes() || old.sizes() != adv.sizes()) raise_assertion("");
  const Mask m = mask_matrix(mask, dev, lp);
  const Tensor isw = is_weights ? matrix(*is_weights, dev) : Tensor();
  const int64_t rows = lp.size(0), cols = lp.size(1);
  const c10::DeviceGuard guard(dev);
  // one allocation for the four result floats and the per-row coefficients (16-byte aligned both)
  const Tensor buf = new_f32({4 + rows}, dev), out = part(buf, 0, 4), coef = part(buf, 4, rows);
  const Tensor g = need_grad ? at::empty_like(lp) : Tensor();
  const Tensor ws = ticket_workspace(vamd_policy_loss_variant_workspace_bytes(rows, cols), dev);
  check(vamd_policy_loss_variant_forward(a.variant, f32(old), f32(lp), f32(adv), m.t.const_data_ptr(), m.code, f32(isw),
                                         rows, cols, (float)a.clip_low, (float)a.clip_high, (float)a.clip_c,
                                         (float)a.tau_pos, (float)a.tau_neg, a.agg.mode, a.agg.dp_size,
                                         a.agg.batch_num_tokens, a.agg.global_batch_size, a.agg.loss_scale_factor,
                                         f32_out(out), f32_out(g), f32_out(coef), ws.mutable_data_ptr(), ws.numel(),
                                         stream_of(dev)));
  // the loss shares the floats the kernel wrote with the metrics
  const Tensor result = log_prob.device() == dev ? out : out.to(log_prob.device());
  return {scalar_part(result, 0), result, g, coef, dev};
}

class PolicyLoss : public torch::autograd::Function<PolicyLoss> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& log_prob, const Tensor& old_log_prob,
                               const Tensor& advantages, const Tensor& mask,
                               const std::optional<Tensor>& is_weights, const PolicyArgs& args) {
    const LossResult r = policy_forward(log_prob, old_log_prob, advantages, mask, is_weights, args, true);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({r.grad, r.coef});
    save_form(ctx, log_prob, r.dev);
    ctx->mark_non_differentiable({r.out});
    return {r.loss, r.out};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return scaled_gradient(ctx, grads, 1.f, 6);
  }
};

std::pair<Tensor, Tensor> policy_loss(const Tensor& log_prob, const Tensor& old_log_prob, const Tensor& advantages,
                                      const Tensor& mask, const std::optional<Tensor>& is_weights, double clip_low,
                                      double clip_high, double clip_c, int mode, double dp_size, double bnt, double gbs,
                                      double lsf, int variant, double tau_pos, double tau_neg) {
  const PolicyArgs a{variant, clip_low, clip_high, clip_c, tau_pos, tau_neg, {mode, dp_size, bnt, gbs, lsf}};
  const Tensor weights = is_weights ? *is_weights : Tensor();
  refuse_tangents("the policy loss", {&log_prob, &old_log_prob, &advantages, &mask, &weights});
  if (wants_gradient(log_prob)) {
    const auto r = PolicyLoss::apply(log_prob, old_log_prob, advantages, mask, is_weights, a);
    joinable<PolicyLoss>(r[0]);
    return {r[0], r[1]};
  }
  const LossResult r = policy_forward(log_prob, old_log_prob, advantages, mask, is_weights, a, false);
  return {r.loss, r.out};
}

// ---- value loss ----------------------------------------------------------------------------------------------
LossResult value_forward(const Tensor& vpreds, const Tensor& returns, const Tensor& values, const Tensor& mask,
                         double clip, int mode, bool need_grad) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&vpreds, &returns, &values, &mask});
  const Tensor vp = matrix(vpreds, dev), ret = matrix(returns, dev), val = matrix(values, dev);
  if (vp.sizes() != ret.sizes() || ret.sizes() != val.sizes()) raise_assertion("");
  const Mask m = mask_matrix(mask, dev, vp);
  const int64_t rows = vp.size(0), cols = vp.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor buf = new_f32({4 + rows}, dev), out = part(buf, 0, 2), coef = part(buf, 4, rows);
  const Tensor g = need_grad ? at::empty_like(vp) : Tensor();
  const Tensor ws = ticket_workspace(vamd_value_loss_workspace_bytes(rows, cols), dev);
  check(vamd_value_loss_forward(f32(vp), f32(ret), f32(val), m.t.const_data_ptr(), m.code, rows, cols, (float)clip, mode,
                                f32_out(out), f32_out(g), f32_out(coef), ws.mutable_data_ptr(), ws.numel(),
                                stream_of(dev)));
  const Tensor result = vpreds.device() == dev ? out : out.to(vpreds.device());
  return {scalar_part(result, 0), result, g, coef, dev};
}

class ValueLoss : public torch::autograd::Function<ValueLoss> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& vpreds, const Tensor& returns, const Tensor& values,
                               const Tensor& mask, double clip, int mode) {
    const LossResult r = value_forward(vpreds, returns, values, mask, clip, mode, true);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({r.grad, r.coef});
    save_form(ctx, vpreds, r.dev);
    ctx->mark_non_differentiable({r.out});
    return {r.loss, r.out};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return scaled_gradient(ctx, grads, 0.5f, 6);
  }
};

// (loss, clip fraction)
std::pair<Tensor, Tensor> value_loss(const Tensor& vpreds, const Tensor& returns, const Tensor& values,
                                     const Tensor& mask, double clip, int mode) {
  refuse_tangents("the value loss", {&vpreds, &returns, &values, &mask});
  if (wants_gradient(vpreds)) {
    const auto r = ValueLoss::apply(vpreds, returns, values, mask, clip, mode);
    joinable<ValueLoss>(r[0]);
    return {r[0], r[1].select(0, 1)};
  }
  const LossResult r = value_forward(vpreds, returns, values, mask, clip, mode, false);
  return {r.loss, r.out.select(0, 1)};
}

// ---- KL loss -------------------------------------------------------------------------------------------------
struct KlArgs {
  int kind, straight_through;
  Aggregation agg;
};
LossResult kl_forward(const Tensor& logprob, const Tensor& ref_logprob, const Tensor& mask, const KlArgs& a,
                      bool need_grad) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&logprob, &ref_logprob, &mask});
  const Tensor lp = matrix(logprob, dev), ref = matrix(ref_logprob, dev);
  if (lp.sizes() != ref.sizes()) raise_assertion("");
  const Mask m = mask_matrix(mask, dev, lp);
  const int64_t rows = lp.size(0), cols = lp.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor buf = new_f32({4 + rows}, dev), out = scalar_part(buf, 0), coef = part(buf, 4, rows);
  const Tensor g = need_grad ? at::empty_like(lp) : Tensor();
  const Tensor ws = ticket_workspace(vamd_kl_loss_workspace_bytes(rows, cols), dev);
  check(vamd_kl_loss_forward(f32(lp), f32(ref), m.t.const_data_ptr(), m.code, rows, cols, a.kind, a.straight_through,
                             a.agg.mode, a.agg.dp_size, a.agg.batch_num_tokens, a.agg.global_batch_size,
                             a.agg.loss_scale_factor, f32_out(out), f32_out(g), f32_out(coef), ws.mutable_data_ptr(),
                             ws.numel(), stream_of(dev)));
  return {logprob.device() == dev ? out : out.to(logprob.device()), Tensor(), g, coef, dev};
}

class KlLoss : public torch::autograd::Function<KlLoss> {
 public:
  static Tensor forward(AutogradContext* ctx, const Tensor& logprob, const Tensor& ref_logprob, const Tensor& mask,
                        const KlArgs& args) {
    const bool need_grad = logprob.requires_grad();
    const LossResult r = kl_forward(logprob, ref_logprob, mask, args, need_grad);
    ctx->set_materialize_grads(false);
    if (need_grad) ctx->save_for_backward({r.grad, r.coef});
    save_form(ctx, logprob, r.dev);
    return r.loss;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    return scaled_gradient(ctx, grads, 1.f, 4);
  }
};

Tensor kl_loss(const Tensor& logprob, const Tensor& ref_logprob, const Tensor& mask, int kind, bool straight_through,
               int mode, double dp_size, double bnt, double gbs, double lsf) {
  const KlArgs a{kind, straight_through, {mode, dp_size, bnt, gbs, lsf}};
  refuse_tangents("the KL loss", {&logprob, &ref_logprob, &mask});
  if (wants_gradient(logprob) || wants_gradient(ref_logprob)) {
    const Tensor loss = KlLoss::apply(logprob, ref_logprob, mask, a);
    joinable<KlLoss>(loss);
    return loss;
  }
  return kl_forward(logprob, ref_logprob, mask, a, false).loss;
}

// ---- agg_loss ------------------------------------------------------------------------------------------------
struct AggResult {
  Tensor loss, coef, mask;
  int code;
  at::Device dev;
};
AggResult agg_forward(const Tensor& loss_mat, const Tensor& mask, const Aggregation& a) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&loss_mat, &mask});
  const Tensor x = matrix(loss_mat, dev);
  const Mask m = mask_matrix(mask, dev, x);
  const int64_t rows = x.size(0), cols = x.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor buf = new_f32({4 + rows}, dev), out = scalar_part(buf, 0), coef = part(buf, 4, rows);
  const Tensor ws = ticket_workspace(vamd_agg_loss_workspace_bytes(rows, cols), dev);
  check(vamd_agg_loss_forward(f32(x), m.t.const_data_ptr(), m.code, rows, cols, a.mode, a.dp_size, a.batch_num_tokens,
                              a.global_batch_size, a.loss_scale_factor, f32_out(out), f32_out(coef),
                              ws.mutable_data_ptr(), ws.numel(), stream_of(dev)));
  return {loss_mat.device() == dev ? out : out.to(loss_mat.device()), coef, m.t, m.code, dev};
}

class AggLoss : public torch::autograd::Function<AggLoss> {
 public:
  static Tensor forward(AutogradContext* ctx, const Tensor& loss_mat, const Tensor& mask, const Aggregation& args) {
    const AggResult r = agg_forward(loss_mat, mask, args);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({r.coef, r.mask});
    ctx->saved_data["code"] = (int64_t)r.code;
    save_form(ctx, loss_mat, r.dev);
    return r.loss;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    at::AutoGradMode no_grad(false);
    variable_list result(3);
    const auto saved = ctx->get_saved_variables();
    if (!grads[0].defined()) return result;
    const Tensor &coef = saved[0], &mask = saved[1];
    const at::Device dev = coef.device();
    const c10::DeviceGuard guard(dev);
    const Tensor d = upstream(grads[0], dev), g = new_f32(mask.sizes(), dev);
    check(vamd_agg_loss_backward(f32(d), f32(coef), mask.const_data_ptr(), (int)ctx->saved_data["code"].toInt(),
                                 mask.size(0), mask.size(1), f32_out(g), stream_of(dev)));
    result[0] = in_saved_form(ctx, g);
    return result;
  }
};

Tensor agg_loss(const Tensor& loss_mat, const Tensor& mask, int mode, double dp_size, double bnt, double gbs,
                double lsf) {
  const Aggregation a{mode, dp_size, bnt, gbs, lsf};
  refuse_tangents("agg_loss", {&loss_mat, &mask});
  if (wants_gradient(loss_mat) || wants_gradient(mask)) return AggLoss::apply(loss_mat, mask, a);
  return agg_forward(loss_mat, mask, a).loss;
}

// ---- advantages and statistics -------------------------------------------------------------------------------
Tensor in_form_of(const Tensor& x, const Tensor& input) {
  const Tensor y = x.sizes() == input.sizes() ? x : x.view(input.sizes());
  return y.device() == input.device() ? y : y.to(input.device());
}

// (advantages, the counter buffer the call used)
std::pair<Tensor, Tensor> grpo_advantage(const Tensor& rewards, const Tensor& mask, const Tensor& ids, int64_t groups,
                                         double epsilon, bool norm_by_std, int std_mode) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&rewards, &mask});
  const Tensor r = matrix(rewards, dev);
  const Mask m = mask_matrix(mask, dev, r);
  const int64_t rows = r.size(0), cols = r.size(1);
  TORCH_CHECK_VALUE(ids.numel() == rows, "index has ", ids.numel(), " entries for a batch of ", rows);
  const c10::DeviceGuard guard(dev);
  const Tensor adv = at::empty_like(r);
  const Tensor ws = ticket_workspace(vamd_grpo_workspace_bytes(rows, cols, groups), dev);
  check(vamd_grpo_advantage(f32(r), m.t.const_data_ptr(), m.code, ids.const_data_ptr<int64_t>(), rows, cols, groups,
                            (float)epsilon, norm_by_std, std_mode, f32_out(adv), nullptr, ws.mutable_data_ptr(),
                            ws.numel(), stream_of(dev)));
  return {in_form_of(adv, rewards), ws};
}

// (advantages, returns, moments)
std::tuple<Tensor, Tensor, Tensor> gae(const Tensor& rewards, const Tensor& values, const Tensor& mask, double gamma,
                                       double lam, int whiten) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&rewards, &values, &mask});
  const Tensor r = matrix(rewards, dev), v = matrix(values, dev);
  if (r.sizes() != v.sizes()) raise_assertion("");
  const Mask m = mask_matrix(mask, dev, r);
  const int64_t rows = r.size(0), cols = r.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor adv = at::empty_like(r), ret = at::empty_like(r);
  const Tensor mom = at::empty({5}, at::TensorOptions().dtype(at::kDouble).device(dev));
  const Tensor ws = ticket_workspace(vamd_gae_workspace_bytes(rows, cols), dev);
  check(vamd_gae(f32(r), f32(v), m.t.const_data_ptr(), m.code, rows, cols, (float)gamma, (float)lam, whiten,
                 f32_out(adv), f32_out(ret), mom.mutable_data_ptr<double>(), ws.mutable_data_ptr(), ws.numel(),
                 stream_of(dev)));
  return {in_form_of(adv, rewards), in_form_of(ret, rewards), mom};
}

// (token-level rewards, mean KL [1])
std::pair<Tensor, Tensor> kl_rewards(const Tensor& scores, const Tensor& logprob, const Tensor& ref_logprob,
                                     const Tensor& mask, int kind, double beta) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&scores, &logprob, &ref_logprob, &mask});
  const Tensor sc = matrix(scores, dev), lp = matrix(logprob, dev), rf = matrix(ref_logprob, dev);
  if (sc.sizes() != lp.sizes() || lp.sizes() != rf.sizes()) raise_assertion("");
  const Mask m = mask_matrix(mask, dev, sc);
  const int64_t rows = sc.size(0), cols = sc.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty_like(sc), kl = new_f32({1}, dev);
  const Tensor ws = ticket_workspace(vamd_apply_kl_penalty_workspace_bytes(rows, cols), dev);
  check(vamd_apply_kl_penalty(f32(sc), f32(lp), f32(rf), m.t.const_data_ptr(), m.code, rows, cols, kind, (float)beta,
                              f32_out(out), f32_out(kl), ws.mutable_data_ptr(), ws.numel(), stream_of(dev)));
  return {in_form_of(out, scores), kl};
}

Tensor scratch(size_t bytes, const at::Device& dev) {
  return at::empty({bytes < 256 ? 256 : (int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(dev));
}

// (weights or None, metrics)
std::pair<std::optional<Tensor>, Tensor> rollout_correction(const Tensor& old_log_prob,
                                                            const std::optional<Tensor>& rollout_log_prob,
                                                            const Tensor& mask, int level, double threshold,
                                                            bool batch_normalize, int64_t slots) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&old_log_prob, &mask});
  Tensor old = as_f32(old_log_prob, dev);
  if (old.dim() == 1) old = old.view({1, -1});
  if (old.dim() != 2) raise_assertion("expected (batch, length) log-probabilities, got " + shape_text(old_log_prob));
  const Tensor roll = rollout_log_prob ? as_f32(*rollout_log_prob, dev).view(old.sizes()) : Tensor();
  Mask m = mask_of(mask, dev);
  m.t = m.t.view(old.sizes());
  const int64_t rows = old.size(0), cols = old.size(1);
  const c10::DeviceGuard guard(dev);
  const Tensor weights = level ? at::empty_like(old) : Tensor();
  const Tensor out = at::empty({slots}, at::TensorOptions().dtype(at::kDouble).device(dev));
  const Tensor ws = scratch(vamd_rollout_correction_workspace_bytes(rows, cols), dev);
  check(vamd_rollout_correction(f32(old), f32(roll), m.t.const_data_ptr(), m.code, rows, cols, level, (float)threshold,
                                batch_normalize, f32_out(weights), out.mutable_data_ptr<double>(),
                                ws.mutable_data_ptr(), ws.numel(), stream_of(dev)));
  if (!level) return {std::nullopt, out};
  return {in_form_of(weights, old_log_prob), out};
}

Tensor data_metrics(const Tensor& scores, const Tensor& rewards, const Tensor& advantages, const Tensor& returns,
                    const std::optional<Tensor>& values, const Tensor& response_mask, const Tensor& attention_mask,
                    int64_t width, int64_t slots) {
  at::AutoGradMode no_grad(false);
  const at::Device dev = compute_device({&scores, &response_mask, &attention_mask});
  const Tensor sc = as_f32(scores, dev);
  if (sc.dim() != 2 || sc.size(1) != width)
    raise_assertion("token_level_scores " + shape_text(sc) + " vs response width " + std::to_string(width));
  const Tensor rw = as_f32(rewards, dev), adv = as_f32(advantages, dev), ret = as_f32(returns, dev);
  const Tensor val = values ? as_f32(*values, dev) : Tensor();
  for (const Tensor* t : {&rw, &adv, &ret, &val})
    if (t->defined() && t->sizes() != sc.sizes()) raise_assertion("");
  const Mask m = mask_of(response_mask, dev), att = mask_of(attention_mask, dev);
  const int64_t rows = sc.size(0);
  if (m.t.sizes() != sc.sizes() || att.t.size(0) != rows || att.t.size(1) < width) raise_assertion("");
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty({slots}, at::TensorOptions().dtype(at::kDouble).device(dev));
  const Tensor ws = scratch(vamd_data_metrics_workspace_bytes(rows, width), dev);
  check(vamd_data_metrics(f32(sc), f32(rw), f32(adv), f32(ret), f32(val), m.t.const_data_ptr(), m.code,
                          att.t.const_data_ptr(), att.code, rows, att.t.size(1) - width, width,
                          out.mutable_data_ptr<double>(), ws.mutable_data_ptr(), ws.numel(), stream_of(dev)));
  return out;
}

// ---- a few numbers to the host -------------------------------------------------------------------------------
// What a copy and a synchronisation take 13 us for on an idle stream: a kernel of one wavefront writes the numbers and
// then a sequence number into host memory, which this thread reads until it sees it.  Slots are taken for the length of a
// call; a call that finds none left, or numbers that do not fit, goes through a copy.
constexpr int kSlots = 32, kSlotBytes = 512, kFlagBytes = 64;
struct Slots {
  std::mutex mu;
  char* base = nullptr;
  bool failed = false;
  uint32_t sequence = 0;
  std::vector<int> free;

  // index of a slot and the sequence number to wait for, or -1
  int take(uint32_t& number) {
    std::lock_guard<std::mutex> lock(mu);
    if (!base && !failed) {
      void* p = nullptr;
      failed = hipHostMalloc(&p, kSlots * kSlotBytes, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess;
      if (!failed) {
        base = static_cast<char*>(p);
        for (int i = 0; i < kSlots; ++i) {
          *reinterpret_cast<uint32_t*>(base + i * kSlotBytes) = 0;
          free.push_back(i);
        }
      } else {
        (void)hipGetLastError();
      }
    }
    if (free.empty()) return -1;
    const int slot = free.back();
    free.pop_back();
    number = ++sequence ? sequence : ++sequence;  // never 0
    return slot;
  }
  void give_back(int slot) {
    std::lock_guard<std::mutex> lock(mu);
    free.push_back(slot);
  }
};

// The values of a contiguous fp32 or fp64 vector as Python floats.
std::vector<double> fetch(const Tensor& t) {
  static auto* slots = new Slots;  // never destroyed: at exit the runtime may be gone first
  const bool f64 = t.scalar_type() == at::kDouble;
  const int64_t n = t.numel(), bytes = n * (f64 ? 8 : 4);
  std::vector<double> values(n);
  auto read = [&](const void* p) {
    for (int64_t i = 0; i < n; ++i)
      values[i] = f64 ? static_cast<const double*>(p)[i] : (double)static_cast<const float*>(p)[i];
  };
  py::gil_scoped_release no_gil;
  if (t.is_cuda() && t.is_contiguous() && bytes <= kSlotBytes - kFlagBytes) {
    const c10::DeviceGuard guard(t.device());
    const hipStream_t stream = (hipStream_t)stream_of(t.device());
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    uint32_t number = 0;
    int slot = -1;
    if (hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone)
      slot = slots->take(number);
    if (slot >= 0) {
      char* const at = slots->base + slot * kSlotBytes;
      const int rc = vamd_write_to_host(t.const_data_ptr(), bytes, at + kFlagBytes, at, number, stream);
      hipError_t err = hipSuccess;
      if (rc == 0) {
        // Reads for as long as a step's small kernels may take, then waits for the stream, which does not keep a core busy.
        const auto* flag = reinterpret_cast<const std::atomic<uint32_t>*>(at);
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        while (flag->load(std::memory_order_acquire) != number) {
          if (std::chrono::steady_clock::now() < until) continue;
          err = hipStreamSynchronize(stream);
          break;
        }
        if (err == hipSuccess && flag->load(std::memory_order_acquire) == number) read(at + kFlagBytes);
        else if (err == hipSuccess) err = hipErrorUnknown;
      }
      // after an error the kernel may still write the slot: it is not used again
      if (rc != 0 || err == hipSuccess) slots->give_back(slot);
      check(rc);
      TORCH_CHECK(err == hipSuccess, "libverl_amd: results could not be read: ", hipGetErrorString(err));
      return values;
    }
  }
  const Tensor host = t.detach().to(at::kCPU).contiguous();
  read(host.const_data_ptr());
  return values;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("abi_version", [] { return VAMD_ABI_VERSION; });
  m.def("library_abi_version", [] { return vamd_abi_version(); });
  m.def("ticket_workspace", [](int64_t bytes, at::Device dev) {
    if (!dev.has_index()) dev.set_index(c10::hip::current_device());
    return ticket_workspace((size_t)(bytes < 0 ? 0 : bytes), dev);
  });
  m.def("logprobs_from_logits", &logprobs_from_logits);
  m.def("entropy_from_logits", &entropy_from_logits);
  m.def("policy_loss", &policy_loss);
  m.def("value_loss", &value_loss);
  m.def("kl_loss", &kl_loss);
  m.def("agg_loss", &agg_loss);
  m.def("grpo_advantage", &grpo_advantage);
  m.def("gae", &gae);
  m.def("kl_rewards", &kl_rewards);
  m.def("rollout_correction", &rollout_correction);
  m.def("data_metrics", &data_metrics);
  m.def("fetch", &fetch);
}
