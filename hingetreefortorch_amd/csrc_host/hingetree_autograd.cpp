// The autograd functions of the operator module as native graph nodes: what HingeTree/_HingeTree.py:92-258,370-506 does
// in Python (forward, save, backward on the autograd thread) without entering the interpreter in the backward pass and
// with a few microseconds instead of tens on either side, which is most of a training step on a small table. One node
// class per operator; the Python classes' `apply` calls these where the native host is in use. A call that torch follows by
// other means than the graph is declined (NotImplemented), and the Python classes take it (see hth::watched).
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/core/grad_mode.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include "hingetree_host.hpp"

namespace hth {
namespace {

using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

int backward_mode() { return deterministic_mode() ? HT_BACKWARD_DETERMINISTIC : HT_BACKWARD_ATOMIC; }

// Whether a call has to be recorded, from its differentiable inputs. Forward-mode tangents would be dropped silently.
bool recorded(std::initializer_list<const Tensor *> inputs) {
  bool any = false;
  for (const Tensor *t : inputs) {
    TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(0).defined(), "the hinge operators have no forward-mode derivative");
    any = any || t->requires_grad();
  }
  return any && at::GradMode::is_enabled();
}

template <typename N>
std::shared_ptr<N> new_node(std::initializer_list<const Tensor *> inputs) {
  std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
  torch::autograd::edge_list edges;
  edges.reserve(inputs.size());
  for (const Tensor *t : inputs) edges.push_back(torch::autograd::impl::gradient_edge(*t));
  node->set_next_edges(std::move(edges));
  return node;
}

// A node that keeps tensors of the forward pass; `saved` is released after the backward pass unless the graph is retained.
struct SavingNode : Node {
  std::vector<SavedVariable> saved;
  std::string label;

  void save(std::initializer_list<const Tensor *> tensors) {
    saved.reserve(tensors.size());
    for (const Tensor *t : tensors) saved.emplace_back(*t, /*is_output=*/false);
  }
  std::vector<Tensor> unpack() {
    std::vector<Tensor> r;
    r.reserve(saved.size());
    for (const SavedVariable &s : saved) r.push_back(s.unpack(getptr()));
    return r;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable &s : saved) s.reset_data();
  }
  std::string name() const override { return label; }
  Needs needs() const { return {wants(0), wants(1), wants(3)}; }  // (data, thresholds, ordinals, weights)
  bool wants(size_t i) const { return task_should_compute_output(i); }
};

// ---- forest / fern ---------------------------------------------------------------------------------------------------
struct ForestNode : SavingNode {
  int kind = HT_TREE;
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list r(4);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    const Tensor g = grads[0].contiguous();
    const Gradients d = t[4].defined() ? forest_backward_records(kind, backward_mode(), needs(), t[4], t[0], t[1], t[2], t[3], g)
                                       : forest_backward(kind, backward_mode(), needs(), t[0], t[1], t[2], t[3], g);
    r[0] = d.dx;
    r[1] = d.dthr;
    r[3] = d.dw;
    return r;
  }
};

Tensor forest_apply(int kind, const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w) {
  if (!recorded({&x, &thr, &w})) return forest_forward(kind, x, thr, ord, w);
  auto node = new_node<ForestNode>({&x, &thr, &ord, &w});
  node->kind = kind;
  node->label = kind == HT_TREE ? "HingeTreeBackward" : "HingeFernBackward";
  Tensor out, records;
  {
    const at::AutoGradMode no_grad(false);
    // the walk records spare the backward pass a second walk
    std::tie(out, records) = forest_forward_records(kind, x, thr, ord, w);
  }
  node->save({&x, &thr, &ord, &w, &records});
  torch::autograd::set_history(out, node);
  return out;
}

// ---- convolution -------------------------------------------------------------------------------------------------
struct ConvNode : SavingNode {
  int kind = HT_TREE, nd = 0;
  Extents kernel, stride, padding, dilation;
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (deterministic_mode() && grads[0].defined() && !grads[0].device().is_cpu())
      runtime(std::string("No deterministic implementation of backpropagation for hinge ") +
              (kind == HT_TREE ? "tree" : "fern") + " convolution on GPUs.");
    variable_list r(4);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    const Gradients d = conv_backward(kind, nd, needs(), t[0], t[1], t[2], t[3], grads[0].contiguous(), kernel, stride,
                                      padding, dilation);
    r[0] = d.dx;
    r[1] = d.dthr;
    r[3] = d.dw;
    return r;
  }
};

Tensor conv_apply(int kind, int nd, const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,
                  const Extents &kernel, const Extents &stride, const Extents &padding, const Extents &dilation) {
  if (!recorded({&x, &thr, &w})) return conv_forward(kind, nd, x, thr, ord, w, kernel, stride, padding, dilation);
  auto node = new_node<ConvNode>({&x, &thr, &ord, &w});
  node->kind = kind;
  node->nd = nd;
  node->kernel = kernel;
  node->stride = stride;
  node->padding = padding;
  node->dilation = dilation;
  node->label = std::string(kind == HT_TREE ? "HingeTreeConv" : "HingeFernConv") + std::to_string(nd) + "dBackward";
  Tensor out;
  {
    const at::AutoGradMode no_grad(false);
    out = conv_forward(kind, nd, x, thr, ord, w, kernel, stride, padding, dilation);
  }
  node->save({&x, &thr, &ord, &w});
  torch::autograd::set_history(out, node);
  return out;
}

// ---- forest stored as an image -------------------------------------------------------------------------------------
struct ExpandedNode : SavingNode {
  int kind = HT_TREE;
  Extents padding;
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list r(4);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    const Gradients d = forest_backward_expanded(kind, backward_mode(), needs(), t[0], t[1], t[2], t[3],
                                                 grads[0].contiguous(), padding);
    r[0] = d.dx;
    r[1] = d.dthr;
    r[3] = d.dw;
    return r;
  }
};

Tensor expanded_apply(int kind, const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,
                      const Extents &padding) {
  if (!recorded({&x, &thr, &w})) return forest_forward_expanded(kind, x, thr, ord, w, padding);
  auto node = new_node<ExpandedNode>({&x, &thr, &ord, &w});
  node->kind = kind;
  node->padding = padding;
  node->label = kind == HT_TREE ? "HingeTreeExpandedBackward" : "HingeFernExpandedBackward";
  Tensor out;
  {
    const at::AutoGradMode no_grad(false);
    out = forest_forward_expanded(kind, x, thr, ord, w, padding);
  }
  node->save({&x, &thr, &ord, &w});
  torch::autograd::set_history(out, node);
  return out;
}

// ---- forest -> linear --------------------------------------------------------------------------------------------
struct FusedLinearNode : SavingNode {
  int kind = HT_TREE;
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list r(6);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    const MixGradients d = fused_linear_backward(kind, backward_mode(), needs(), wants(4), wants(5), t[0], t[1], t[2], t[3],
                                                 t[4], t[5], grads[0].contiguous(), t[6], t[7]);
    r[0] = d.dx;
    r[1] = d.dthr;
    r[3] = d.dw;
    r[4] = d.dlin;
    r[5] = d.dbias;
    return r;
  }
};

Tensor fused_linear_apply(int kind, const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,
                          const Tensor &lin, const Tensor &bias) {
  if (!recorded({&x, &thr, &w, &lin, &bias})) return fused_linear_forward(kind, x, thr, ord, w, lin, bias, false).out;
  auto node = new_node<FusedLinearNode>({&x, &thr, &ord, &w, &lin, &bias});
  node->kind = kind;
  node->label = kind == HT_TREE ? "HingeTreeFusedLinearBackward" : "HingeFernFusedLinearBackward";
  MixForward f;
  {
    const at::AutoGradMode no_grad(false);
    // the forest's output and walk records are kept: the backward pass needs both
    f = fused_linear_forward(kind, x, thr, ord, w, lin, bias, true);
  }
  node->save({&x, &thr, &ord, &w, &lin, &bias, &f.f, &f.records});
  torch::autograd::set_history(f.out, node);
  return f.out;
}

// ---- linear -> batch norm [-> forest] ------------------------------------------------------------------------------
struct LinearBatchNormNode : SavingNode {
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list r(2);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    // (with an input gradient the operator works in place on the upstream gradient, which is the caller's)
    const Tensor g = wants(0) ? grads[0].contiguous().clone() : grads[0].contiguous();
    std::tie(r[0], r[1]) = linear_bn_backward(t[0], wants(0), t[1], wants(1), t[2], t[3], g);
    return r;
  }
};

py::tuple linear_bn_apply(const Tensor &x, const Tensor &lin, double eps) {
  const bool record = recorded({&x, &lin});
  std::shared_ptr<LinearBatchNormNode> node;
  if (record) node = new_node<LinearBatchNormNode>({&x, &lin});
  BatchNormed b;
  {
    const at::AutoGradMode no_grad(false);
    b = linear_bn_forward(x, lin, eps);
  }
  if (record) {
    node->label = "LinearBatchNormBackward";
    torch::autograd::set_history(b.z, node);
    node->save({&x, &lin});
    node->saved.emplace_back(b.z, /*is_output=*/true);
    node->saved.emplace_back(b.rstd, /*is_output=*/false);
  }
  return py::make_tuple(b.z, b.mean, b.var);
}

// The forest reads the un-normalised product z and normalises it on the way. The backward pass takes the gradient of the
// linear weights straight from the forest's walk records where the library serves that, else the two separate backward
// passes over the dense gradient of the normalised product.
struct LinearForestNode : SavingNode {
  int kind = HT_TREE;
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list r(5);
    if (!grads[0].defined()) return r;
    const at::AutoGradMode no_grad(false);
    const std::vector<Tensor> t = unpack();
    const Tensor &x = t[0], &lin = t[1], &thr = t[2], &ord = t[3], &w = t[4], &z = t[5], &mean = t[6], &rstd = t[7],
                 &records = t[8];
    const Tensor up = grads[0].contiguous();
    const bool need_x = wants(0), need_lin = wants(1), need_thr = wants(2), need_w = wants(4);
    const int mode = backward_mode();
    if (records.defined() && !need_x && mode == HT_BACKWARD_ATOMIC) {
      const LinearForestGradients d =
          linear_bn_forest_backward(kind, records, x, lin, need_lin, z, rstd, thr, need_thr, ord, w, need_w, up, mean);
      if (d.served) {
        r[1] = d.dlin;
        r[2] = d.dthr;
        r[4] = d.dw;
        return r;
      }
    }
    const Tensor zhat = (z - mean) * rstd;
    const Needs need = {need_x || need_lin, need_thr, need_w};
    const Gradients d = records.defined() ? forest_backward_records(kind, mode, need, records, zhat, thr, ord, w, up)
                                          : forest_backward(kind, mode, need, zhat, thr, ord, w, up);
    if (d.dx.defined()) std::tie(r[0], r[1]) = linear_bn_backward(x, need_x, lin, need_lin, zhat, rstd, d.dx);
    r[2] = d.dthr;
    r[4] = d.dw;
    return r;
  }
};

py::tuple linear_forest_apply(int kind, const Tensor &x, const Tensor &lin, double eps, const Tensor &thr, const Tensor &ord,
                              const Tensor &w) {
  const bool record = recorded({&x, &lin, &thr, &w});
  std::shared_ptr<LinearForestNode> node;
  if (record) node = new_node<LinearForestNode>({&x, &lin, &thr, &ord, &w});
  LinearForest f;
  {
    const at::AutoGradMode no_grad(false);
    f = linear_bn_forest_forward(kind, x, lin, eps, thr, ord, w, record);
  }
  if (record) {
    node->kind = kind;
    node->label = "LinearBatchNormForestBackward";
    node->save({&x, &lin, &thr, &ord, &w, &f.bn.z, &f.bn.mean, &f.bn.rstd, &f.records});
    torch::autograd::set_history(f.out, node);
  }
  return py::make_tuple(f.out, f.bn.mean, f.bn.var);
}

}  // namespace

bool watched() {
  const c10::DispatchKeySet on = c10::impl::tls_local_dispatch_key_set().included_;
  return torch::jit::tracer::isTracing() || on.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         on.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}

void bind_autograd(py::module &m) {
  py::dict apply;
  const auto add = [&](const char *name, py::cpp_function fn) { apply[name] = fn; };
  // `call` unless the call is watched
  const auto unwatched = [](auto call) -> py::object {
    if (watched()) return py::reinterpret_borrow<py::object>(Py_NotImplemented);
    if constexpr (std::is_same_v<decltype(call()), py::tuple>)
      return call();
    else
      return py::cast(call());
  };
#define HT_APPLY(Name, KIND)                                                                                          \
  add(Name, py::cpp_function([=](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w) {            \
        return unwatched([&] { return forest_apply(KIND, x, thr, ord, w); });                                         \
      }));                                                                                                            \
  add(Name "Expanded", py::cpp_function([=](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,   \
                                            py::object padding) {                                                     \
        return unwatched([&] {                                                                                        \
          return expanded_apply(KIND, x, thr, ord, w,                                                                 \
                                py::isinstance<py::int_>(padding)                                                     \
                                    ? Extents(size_t(w.dim() > 2 ? w.dim() - 2 : 0), padding.cast<int64_t>())         \
                                    : padding.cast<Extents>());                                                       \
        });                                                                                                           \
      }, py::arg(), py::arg(), py::arg(), py::arg(), py::arg("padding") = 0));                                        \
  add(Name "FusedLinear", py::cpp_function([=](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w, \
                                               const Tensor &lin, const Tensor &bias) {                               \
        return unwatched([&] { return fused_linear_apply(KIND, x, thr, ord, w, lin, bias); });                        \
      }));
  HT_APPLY("HingeTree", HT_TREE)
  HT_APPLY("HingeFern", HT_FERN)
#undef HT_APPLY
#define HT_APPLY_CONV(Name, KIND, ND)                                                                                 \
  add(Name, py::cpp_function([=](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,              \
                                 const Extents &kernel, const Extents &stride, const Extents &padding,                \
                                 const Extents &dilation) {                                                           \
        return unwatched([&] { return conv_apply(KIND, ND, x, thr, ord, w, kernel, stride, padding, dilation); });    \
      }));
  HT_APPLY_CONV("HingeTreeConv1d", HT_TREE, 1)
  HT_APPLY_CONV("HingeTreeConv2d", HT_TREE, 2)
  HT_APPLY_CONV("HingeTreeConv3d", HT_TREE, 3)
  HT_APPLY_CONV("HingeFernConv1d", HT_FERN, 1)
  HT_APPLY_CONV("HingeFernConv2d", HT_FERN, 2)
  HT_APPLY_CONV("HingeFernConv3d", HT_FERN, 3)
#undef HT_APPLY_CONV
  add("LinearBatchNorm", py::cpp_function([=](const Tensor &x, const Tensor &lin, double eps) {
        return unwatched([&] { return linear_bn_apply(x, lin, eps); });
      }));
  add("LinearBatchNormForest",
      py::cpp_function([=](const Tensor &x, const Tensor &lin, double eps, const Tensor &thr, const Tensor &ord,
                           const Tensor &w, bool fern) {
        return unwatched([&] { return linear_forest_apply(fern ? HT_FERN : HT_TREE, x, lin, eps, thr, ord, w); });
      }));
  m.attr("apply") = apply;  // by the names of the autograd functions
}

}  // namespace hth
