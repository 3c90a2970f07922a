// What the translation units of the native host module share: the operators as plain ATen functions (validation,
// allocation, launch), used by the pybind11 bindings, by the operators built on top of them and by the autograd nodes.
#pragma once
#include <torch/extension.h>

#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/hingetree_hip.h"

namespace hth {

using torch::Tensor;

[[noreturn]] void invalid(const std::string &msg);  // -> Python ValueError
[[noreturn]] void runtime(const std::string &msg);  // -> Python RuntimeError
void check(int rc);

int64_t prod(c10::IntArrayRef v, size_t from);
void *ptr(const Tensor &t);
inline float *fptr(const Tensor &t) { return static_cast<float *>(ptr(t)); }
inline const int64_t *iptr(const Tensor &t) { return static_cast<const int64_t *>(ptr(t)); }
// The stream torch is using on the tensor's device.
void *current_stream(const Tensor &t);
// Device memory for results and scratch that the kernels overwrite completely. Taken from the caching allocator
// directly: torch.empty would fill the memory first under torch.use_deterministic_algorithms(True) (a guard for readers
// of uninitialised memory, of which there are none here), which for a forest's output costs as much as writing it.
Tensor fresh(c10::IntArrayRef sizes, at::ScalarType dtype, const Tensor &like);
inline Tensor fresh_like(const Tensor &t) { return fresh(t.sizes(), t.scalar_type(), t); }
Tensor workspace(size_t bytes, const Tensor &like);
std::string sizes_text(c10::IntArrayRef v);

bool deterministic_mode();

// hingetree.cpp:649-663: data types, devices, contiguity -- in that order
void common_checks(const std::vector<const Tensor *> &reals, const Tensor &ordinals, bool with_grad);
void require_gpu(const Tensor &t);
ht_forest_shape forest_shape(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                             const Tensor &inWeights, const Tensor *outDataGrad, std::vector<int64_t> *out_sizes);

struct Needs {
  bool dx, dthr, dw;
};
struct Gradients {
  Tensor dx, dthr, dw;
};

Tensor forest_forward(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                      const Tensor &inWeights);
// (out, walk records; the records undefined where the library offers none for the shape)
std::pair<Tensor, Tensor> forest_forward_records(int kind, const Tensor &inData, const Tensor &inThresholds,
                                                 const Tensor &inOrdinals, const Tensor &inWeights);
Gradients forest_backward(int kind, int mode, Needs need, const Tensor &inData, const Tensor &inThresholds,
                          const Tensor &inOrdinals, const Tensor &inWeights, const Tensor &outDataGrad);
Gradients forest_backward_records(int kind, int mode, Needs need, const Tensor &records, const Tensor &inData,
                                  const Tensor &inThresholds, const Tensor &inOrdinals, const Tensor &inWeights,
                                  const Tensor &outDataGrad);

using Extents = std::vector<int64_t>;
Tensor conv_forward(int kind, int nd, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                    const Tensor &inWeights, const Extents &kernelSize, const Extents &stride, const Extents &padding,
                    const Extents &dilation);
Gradients conv_backward(int kind, int nd, Needs need, const Tensor &inData, const Tensor &inThresholds,
                        const Tensor &inOrdinals, const Tensor &inWeights, const Tensor &outDataGrad,
                        const Extents &kernelSize, const Extents &stride, const Extents &padding,
                        const Extents &dilation);

// ---- hingetree_compose.cpp -----------------------------------------------------------------------------------
Tensor contract(const Tensor &inData, const Extents &window, const Extents &padding);
Tensor expand(const Tensor &inData, const Extents &padding);
Tensor forest_forward_expanded(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                               const Tensor &inWeights, const Extents &padding);
Gradients forest_backward_expanded(int kind, int mode, Needs need, const Tensor &inData, const Tensor &inThresholds,
                                   const Tensor &inOrdinals, const Tensor &inWeights, const Tensor &outImageGrad,
                                   const Extents &padding);

struct MixForward {
  Tensor out, f, records;  // f, records: only with keep (records where the library offers them)
};
MixForward fused_linear_forward(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                                const Tensor &inWeights, const Tensor &inLinearWeights, const Tensor &inLinearBias,
                                bool keep);
struct MixGradients {
  Tensor dx, dthr, dw, dlin, dbias;
};
MixGradients fused_linear_backward(int kind, int mode, Needs need, bool need_lin, bool need_bias, const Tensor &inData,
                                   const Tensor &inThresholds, const Tensor &inOrdinals, const Tensor &inWeights,
                                   const Tensor &inLinearWeights, const Tensor &inLinearBias, const Tensor &outDataGrad,
                                   const Tensor &f, const Tensor &records);

struct BatchNormed {
  Tensor z, mean, rstd, var;  // z: normalised (linear_bn_forward) or not (linear_bn_forest_forward)
};
BatchNormed linear_bn_forward(const Tensor &inData, const Tensor &inLinearWeights, double eps);
// (dx, dlin); with need_dx outDataGrad is overwritten
std::pair<Tensor, Tensor> linear_bn_backward(const Tensor &inData, bool need_dx, const Tensor &inLinearWeights,
                                             bool need_lin, const Tensor &zhat, const Tensor &rstd,
                                             const Tensor &outDataGrad);
struct LinearForest {
  Tensor out, records;
  BatchNormed bn;
};
LinearForest linear_bn_forest_forward(int kind, const Tensor &inData, const Tensor &inLinearWeights, double eps,
                                      const Tensor &inThresholds, const Tensor &inOrdinals, const Tensor &inWeights,
                                      bool want_records);
struct LinearForestGradients {
  bool served = false;
  Tensor dlin, dthr, dw;
};
LinearForestGradients linear_bn_forest_backward(int kind, const Tensor &records, const Tensor &inData,
                                                const Tensor &inLinearWeights, bool need_lin, const Tensor &zhat,
                                                const Tensor &rstd, const Tensor &inThresholds, bool need_thr,
                                                const Tensor &inOrdinals, const Tensor &inWeights, bool need_w,
                                                const Tensor &outDataGrad, const Tensor &mean);

void bind_compose(py::module &m);
// Whether torch follows the current call by other means than the autograd graph: torch.jit.trace, which sees an operator that
// is dispatched or a Python function but not what native code launches by itself, or a functorch transform.
bool watched();
void bind_autograd(py::module &m);

}  // namespace hth
