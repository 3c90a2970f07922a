// Operators of the native host built on the forest operators: tiles (contract / expand, the forest stored as an image),
// the linear mix behind a forest, and the projection + batch normalisation in front of one. Same checks, messages and
// results as the Python host's functions of the same names.
#include <c10/core/DeviceGuard.h>

#include <sstream>

#include "hingetree_host.hpp"

namespace hth {
namespace {

ht_tile_shape tile_geometry(int64_t planes, const Tensor &like, const Extents &size, const Extents &tiles,
                            const Extents &window, const Extents &padding) {
  ht_tile_shape g{};
  g.planes = planes;
  g.nd = int(window.size());
  g.elem_size = int(like.element_size());
  for (size_t i = 0; i < window.size(); ++i) {
    g.size[i] = size[i];
    g.tiles[i] = tiles[i];
    g.window[i] = window[i];
    g.padding[i] = padding[i];
  }
  return g;
}

bool tile_dtype(at::ScalarType t) {
  switch (t) {
    case torch::kUInt8: case torch::kInt8: case torch::kInt16: case torch::kInt32: case torch::kInt64:
    case torch::kFloat32: case torch::kFloat64: return true;
    default: return false;
  }
}

Extents tail(const Tensor &t, size_t from) { return Extents(t.sizes().begin() + from, t.sizes().end()); }

// expand.cpp:180-181,239-241
Extents image_size(const Extents &tiles, const Extents &window, const Extents &padding) {
  Extents size(tiles.size());
  for (size_t i = 0; i < tiles.size(); ++i) size[i] = tiles[i] * window[i] - ((2 * padding[i]) / window[i]) * window[i];
  return size;
}

bool any_negative(const Extents &v) {
  for (int64_t p : v)
    if (p < 0) return true;
  return false;
}
bool any_below_one(const Extents &v) {
  for (int64_t p : v)
    if (p < 1) return true;
  return false;
}

void need_float(const Tensor &t) {
  if (t.scalar_type() != torch::kFloat32) invalid("Error: the projection supports torch.float32 only.");
}
void need_contiguous(const Tensor &t) {
  if (!t.is_contiguous()) invalid("Error: All tensors are expected to be contiguous.");
}
void need_gpu(const Tensor &t) {
  if (!t.is_cuda()) runtime("Error: this build has no CPU back-end; tensors must be on a GPU.");
}
void need_same_device(const Tensor &a, const Tensor &b) {
  if (a.device() != b.device()) invalid("Error: All tensors are expected to be on the same device.");
}
void need_projection(const Tensor &inData, const Tensor &inLinearWeights) {
  if (inData.dim() != 2 || inLinearWeights.dim() != 2 || inData.size(1) != inLinearWeights.size(1))
    invalid("Error: inData must be [batch, in_features] and inLinearWeights [out_features, in_features].");
}

}  // namespace

// ---- contract / expand (expand.cpp:37-163,366-463 and :169-330,474-570) ------------------------------------------
Tensor contract(const Tensor &inData, const Extents &window, const Extents &padding) {
  if (window.empty() || window.size() != padding.size())
    invalid("Error: window and padding must be non-empty and the same size.");
  need_contiguous(inData);
  if (!tile_dtype(inData.scalar_type()))
    invalid("Error: Only torch.{uint8,int8,int16,int32,int64,float32,float64} are supported.");
  const int64_t nd = int64_t(window.size());
  if (nd != 2 && nd != 3) invalid("Error: Only 2D and 3D window sizes are supported.");
  if (inData.dim() != nd + 2 || any_negative(padding))
    invalid("Error: inData must have " + std::to_string(nd + 2) + " dimensions. Padding must be non-negative.");
  const Extents size = tail(inData, 2);
  Extents tiles(size.size());
  for (size_t i = 0; i < size.size(); ++i) {
    if (window[i] < 1 || window[i] > size[i] + 2 * padding[i])
      invalid("Error: Window dimensions must be at least 1 but no greater than the size of the padded image.");
    tiles[i] = (size[i] + 2 * padding[i] - window[i]) / window[i] + 1;
  }
  need_gpu(inData);
  std::vector<int64_t> out_sizes = {inData.size(0), inData.size(1)};
  out_sizes.insert(out_sizes.end(), tiles.begin(), tiles.end());
  out_sizes.insert(out_sizes.end(), window.begin(), window.end());
  const ht_tile_shape g = tile_geometry(inData.size(0) * inData.size(1), inData, size, tiles, window, padding);
  const c10::DeviceGuard guard(inData.device());
  Tensor out = fresh(out_sizes, inData.scalar_type(), inData);
  check(ht_contract(&g, ptr(inData), ptr(out), current_stream(inData)));
  return out;
}

Tensor expand(const Tensor &inData, const Extents &padding) {
  if (padding.empty()) invalid("Error: padding must be non-empty.");
  need_contiguous(inData);
  if (!tile_dtype(inData.scalar_type()))
    invalid("Error: Only torch.{uint8,int8,int16,int32,int64,float32,float64} are supported.");
  const int64_t nd = int64_t(padding.size());
  if (nd != 2 && nd != 3) invalid("Error: Only 2D and 3D padding sizes are supported.");
  if (inData.dim() != 2 * nd + 2 || any_negative(padding))
    invalid("Error: inData must have " + std::to_string(2 * nd + 2) + " dimensions. Padding must be non-negative.");
  const Extents tiles(inData.sizes().begin() + 2, inData.sizes().begin() + 2 + nd), window = tail(inData, size_t(2 + nd));
  if (any_below_one(window)) invalid("Error: The expanded size of the image must be non-empty.");
  const Extents size = image_size(tiles, window, padding);
  if (any_below_one(size)) invalid("Error: The expanded size of the image must be non-empty.");
  need_gpu(inData);
  std::vector<int64_t> out_sizes = {inData.size(0), inData.size(1)};
  out_sizes.insert(out_sizes.end(), size.begin(), size.end());
  const ht_tile_shape g = tile_geometry(inData.size(0) * inData.size(1), inData, size, tiles, window, padding);
  const c10::DeviceGuard guard(inData.device());
  Tensor out = fresh(out_sizes, inData.scalar_type(), inData);
  check(ht_expand(&g, ptr(inData), ptr(out), current_stream(inData)));
  return out;
}

// ---- the forest whose result is stored as the image that expand would make of it ---------------------------------
Tensor forest_forward_expanded(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                               const Tensor &inWeights, const Extents &padding) {
  common_checks({&inData, &inThresholds, &inWeights}, inOrdinals, false);
  std::vector<int64_t> out_sizes;
  const ht_forest_shape s = forest_shape(kind, inData, inThresholds, inOrdinals, inWeights, nullptr, &out_sizes);
  const size_t nd = padding.size();
  const Extents tiles = tail(inData, 2), window = tail(inWeights, 2);
  if (nd != 2 && nd != 3) invalid("Error: Only 2D and 3D padding sizes are supported.");
  if (tiles.size() != nd || window.size() != nd || any_negative(padding))
    invalid("Error: inData and inWeights must have " + std::to_string(nd + 2) +
            " dimensions. Padding must be non-negative.");
  if (any_below_one(window)) invalid("Error: The expanded size of the image must be non-empty.");
  const Extents size = image_size(tiles, window, padding);
  if (any_below_one(size)) invalid("Error: The expanded size of the image must be non-empty.");
  if (s.K == 1 || s.B == 0 || s.T == 0)
    return expand(forest_forward(kind, inData, inThresholds, inOrdinals, inWeights), padding);
  const ht_tile_shape g = tile_geometry(s.B * s.T, inData, size, tiles, window, padding);
  out_sizes.resize(2);
  out_sizes.insert(out_sizes.end(), size.begin(), size.end());
  const c10::DeviceGuard guard(inData.device());
  Tensor out = fresh(out_sizes, inData.scalar_type(), inData);
  const size_t bytes = ht_forest_forward_workspace(&s);
  const Tensor ws = workspace(bytes, inData);
  check(ht_forest_forward_image(&s, &g, ptr(inData), ptr(inThresholds), iptr(inOrdinals), ptr(inWeights), ptr(out),
                                ptr(ws), bytes, current_stream(inData)));
  return out;
}

Gradients forest_backward_expanded(int kind, int mode, Needs need, const Tensor &inData, const Tensor &inThresholds,
                                   const Tensor &inOrdinals, const Tensor &inWeights, const Tensor &outImageGrad,
                                   const Extents &padding) {
  const size_t nd = padding.size();
  const Extents window = tail(inWeights, 2), tiles = tail(inData, 2);
  bool fused = (nd == 2 || nd == 3) && window.size() == nd && tiles.size() == nd && !any_negative(padding) &&
               !any_below_one(window) && outImageGrad.is_contiguous() && outImageGrad.scalar_type() == torch::kFloat32 &&
               inData.scalar_type() == torch::kFloat32 && outImageGrad.device() == inData.device() &&
               inData.numel() > 0 && inWeights.numel() > 0;
  ht_forest_shape s{};
  ht_tile_shape g{};
  if (fused) {
    common_checks({&inData, &inThresholds, &inWeights}, inOrdinals, true);
    std::vector<int64_t> want;
    s = forest_shape(kind, inData, inThresholds, inOrdinals, inWeights, nullptr, &want);
    const Extents size = image_size(tiles, window, padding);
    want.resize(2);
    want.insert(want.end(), size.begin(), size.end());
    fused = outImageGrad.sizes() == c10::IntArrayRef(want);
    if (fused) {
      g = tile_geometry(s.B * s.T, inData, size, tiles, window, padding);
      fused = ht_forest_backward_image_supported(&s, &g, mode, need.dx, need.dthr, need.dw) == 1;
    }
  }
  if (!fused)
    return forest_backward(kind, mode, need, inData, inThresholds, inOrdinals, inWeights,
                           contract(outImageGrad.contiguous(), window, padding));
  const c10::DeviceGuard guard(inData.device());
  Gradients r;
  r.dx = need.dx ? fresh_like(inData) : Tensor();
  r.dthr = need.dthr ? fresh_like(inThresholds) : Tensor();
  r.dw = need.dw ? fresh_like(inWeights) : Tensor();
  const size_t bytes = ht_forest_backward_workspace(&s, mode, need.dx, need.dthr, need.dw);
  const Tensor ws = workspace(bytes, inData);
  check(ht_forest_backward_image(&s, &g, ptr(inData), ptr(inThresholds), iptr(inOrdinals), ptr(inWeights),
                                 ptr(outImageGrad), ptr(r.dx), ptr(r.dthr), ptr(r.dw), mode, ptr(ws), bytes,
                                 current_stream(inData)));
  return r;
}

// ---- forest -> linear (hingetree_fused_linear.cpp:75-412) ------------------------------------------------------------
static void fused_linear_checks(const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                                const Tensor &inWeights, const Tensor &inLinearWeights, const Tensor &inLinearBias,
                                const Tensor *outDataGrad) {
  std::vector<const Tensor *> reals = {&inData, &inThresholds, &inWeights, &inLinearWeights, &inLinearBias};
  if (outDataGrad) reals.push_back(outDataGrad);
  common_checks(reals, inOrdinals, outDataGrad != nullptr);
  if (inData.dim() < 2 || inThresholds.dim() != 2 || inOrdinals.dim() != 2 || inWeights.dim() < 2 ||
      inLinearWeights.dim() != 2 || inLinearBias.dim() != 1 || (outDataGrad && outDataGrad->dim() < 2))
    invalid("Error: inData, inWeights must have at least 2 dimensions. inThresholds, inOrdinals, inLinearWeights "
            "must have 2 dimensions. inLinearBias must have 1 dimension.");
  if (inThresholds.sizes() != inOrdinals.sizes() || inWeights.size(0) != inThresholds.size(0) ||
      inWeights.size(0) != inLinearWeights.size(1) || inLinearWeights.size(0) != inLinearBias.size(0))
    invalid("Error: inThresholds and inOrdinals must be the same shape. inWeights.shape[0] must be the same as "
            "inThresholds.shape[0]. inLinearWeightrs.shape[0] must be the same as inLinearBias.shape[0].");
}

struct MixSizes {
  int64_t B, T, O, R;
  std::vector<int64_t> out;
  // Whether the float32 mix moves its operands to planes first: with R values per (sample, tree) the product per
  // sample has results of O x R, a sliver of a matrix-core tile, while the R slices taken as samples make one product
  // of B * R rows.
  bool planes;
};

static MixSizes mix_sizes(const Tensor &inData, const Tensor &inWeights, const Tensor &inLinearWeights) {
  MixSizes m;
  m.B = inData.size(0);
  m.T = inWeights.size(0);
  m.O = inLinearWeights.size(0);
  m.R = prod(inData.sizes(), 2) * prod(inWeights.sizes(), 2);
  m.out = {m.B, m.O};
  m.out.insert(m.out.end(), inData.sizes().begin() + 2, inData.sizes().end());
  m.out.insert(m.out.end(), inWeights.sizes().begin() + 2, inWeights.sizes().end());
  m.planes = inData.scalar_type() == torch::kFloat32 && m.R > 1 && m.R < 128 && m.B > 1;
  return m;
}

MixForward fused_linear_forward(int kind, const Tensor &inData, const Tensor &inThresholds, const Tensor &inOrdinals,
                                const Tensor &inWeights, const Tensor &inLinearWeights, const Tensor &inLinearBias,
                                bool keep) {
  fused_linear_checks(inData, inThresholds, inOrdinals, inWeights, inLinearWeights, inLinearBias, nullptr);
  MixForward r;
  if (keep)
    std::tie(r.f, r.records) = forest_forward_records(kind, inData, inThresholds, inOrdinals, inWeights);
  else
    r.f = forest_forward(kind, inData, inThresholds, inOrdinals, inWeights);
  const MixSizes m = mix_sizes(inData, inWeights, inLinearWeights);
  const c10::DeviceGuard guard(inData.device());
  const at::ScalarType dt = inData.scalar_type();
  r.out = fresh(m.out, dt, inData);
  void *stream = current_stream(inData);
  if (m.planes) {
    const Tensor planes = fresh({m.R * m.B * m.T}, dt, inData), mixed = fresh({m.R * m.B * m.O}, dt, inData);
    check(ht_rows_to_planes(m.B * m.T, m.R, fptr(r.f), fptr(planes), stream));
    check(ht_tree_mix_forward(m.R * m.B, m.T, m.O, 1, fptr(planes), fptr(inLinearWeights), fptr(inLinearBias), fptr(mixed),
                              stream));
    check(ht_planes_to_rows(m.B * m.O, m.R, fptr(mixed), fptr(r.out), stream));
  } else if (dt == torch::kFloat32) {
    check(ht_tree_mix_forward(m.B, m.T, m.O, m.R, fptr(r.f), fptr(inLinearWeights), fptr(inLinearBias), fptr(r.out), stream));
  } else {
    check(ht_tree_mix_forward_f64(m.B, m.T, m.O, m.R, static_cast<const double *>(ptr(r.f)),
                                  static_cast<const double *>(ptr(inLinearWeights)),
                                  static_cast<const double *>(ptr(inLinearBias)), static_cast<double *>(ptr(r.out)), stream));
  }
  return r;
}

MixGradients fused_linear_backward(int kind, int mode, Needs need, bool need_lin, bool need_bias, const Tensor &inData,
                                   const Tensor &inThresholds, const Tensor &inOrdinals, const Tensor &inWeights,
                                   const Tensor &inLinearWeights, const Tensor &inLinearBias, const Tensor &outDataGrad,
                                   const Tensor &kept_f, const Tensor &records) {
  fused_linear_checks(inData, inThresholds, inOrdinals, inWeights, inLinearWeights, inLinearBias, &outDataGrad);
  const MixSizes m = mix_sizes(inData, inWeights, inLinearWeights);
  if (outDataGrad.sizes() != c10::IntArrayRef(m.out))
    invalid("Error: outDataGrad.shape does not match the expected shape (" + sizes_text(outDataGrad.sizes()) + " != " +
            sizes_text(m.out) + ").");
  MixGradients r;
  const bool need_forest = need.dx || need.dthr || need.dw;
  const at::ScalarType dt = inData.scalar_type();
  const c10::DeviceGuard guard(inData.device());
  void *stream = current_stream(inData);
  Tensor f = kept_f;
  if (!f.defined() && need_lin) f = forest_forward(kind, inData, inThresholds, inOrdinals, inWeights);
  Tensor h;
  if (need_forest) {
    std::vector<int64_t> sizes = m.out;
    sizes[1] = m.T;
    h = fresh(sizes, dt, inData);
  }
  if (need_lin) r.dlin = fresh_like(inLinearWeights);
  if (h.defined() || r.dlin.defined()) {
    const int det = mode == HT_BACKWARD_DETERMINISTIC;
    if (m.planes) {
      const Tensor g_planes = fresh({m.R * m.B * m.O}, dt, inData);
      check(ht_rows_to_planes(m.B * m.O, m.R, fptr(outDataGrad), fptr(g_planes), stream));
      Tensor f_planes, h_planes;
      if (r.dlin.defined()) {
        f_planes = fresh({m.R * m.B * m.T}, dt, inData);
        check(ht_rows_to_planes(m.B * m.T, m.R, fptr(f), fptr(f_planes), stream));
      }
      if (h.defined()) h_planes = fresh({m.R * m.B * m.T}, dt, inData);
      const size_t bytes = ht_tree_mix_backward_workspace(m.R * m.B, m.T, m.O, 1);
      const Tensor ws = workspace(bytes, inData);
      check(ht_tree_mix_backward_ws(m.R * m.B, m.T, m.O, 1, fptr(f_planes), fptr(inLinearWeights), fptr(g_planes),
                                    fptr(h_planes), fptr(r.dlin), det, ptr(ws), bytes, stream));
      if (h.defined()) check(ht_planes_to_rows(m.B * m.T, m.R, fptr(h_planes), fptr(h), stream));
    } else if (dt == torch::kFloat32) {
      const size_t bytes = ht_tree_mix_backward_workspace(m.B, m.T, m.O, m.R);
      const Tensor ws = workspace(bytes, inData);
      check(ht_tree_mix_backward_ws(m.B, m.T, m.O, m.R, fptr(f), fptr(inLinearWeights), fptr(outDataGrad), fptr(h),
                                    fptr(r.dlin), det, ptr(ws), bytes, stream));
    } else {  // float64: plain kernels with a fixed summation order in either mode
      check(ht_tree_mix_backward_f64(m.B, m.T, m.O, m.R, static_cast<const double *>(ptr(f)),
                                     static_cast<const double *>(ptr(inLinearWeights)),
                                     static_cast<const double *>(ptr(outDataGrad)), static_cast<double *>(ptr(h)),
                                     static_cast<double *>(ptr(r.dlin)), stream));
    }
  }
  if (need_forest) {
    const Gradients g = records.defined()
                            ? forest_backward_records(kind, mode, need, records, inData, inThresholds, inOrdinals, inWeights, h)
                            : forest_backward(kind, mode, need, inData, inThresholds, inOrdinals, inWeights, h);
    r.dx = g.dx;
    r.dthr = g.dthr;
    r.dw = g.dw;
  }
  if (need_bias) {  // a plain sum, like the reference's outDataGrad.sum(...) (hingetree_fused_linear.cpp:388)
    std::vector<int64_t> dims = {0};
    for (int64_t i = 2; i < outDataGrad.dim(); ++i) dims.push_back(i);
    r.dbias = outDataGrad.sum(dims);
  }
  return r;
}

// ---- projection + batch normalisation in front of a forest (README.md:117-129) -----------------------------------------
BatchNormed linear_bn_forward(const Tensor &inData, const Tensor &inLinearWeights, double eps) {
  need_float(inData);
  need_float(inLinearWeights);
  need_same_device(inData, inLinearWeights);
  need_gpu(inData);
  need_contiguous(inData);
  need_contiguous(inLinearWeights);
  need_projection(inData, inLinearWeights);
  const int64_t B = inData.size(0), K = inData.size(1), N = inLinearWeights.size(0);
  if (B == 0) invalid("Error: batch statistics need at least one sample.");  // torch.nn.BatchNorm1d refuses it too
  const c10::DeviceGuard guard(inData.device());
  BatchNormed r;
  r.z = fresh({B, N}, torch::kFloat32, inData);
  r.mean = fresh({N}, torch::kFloat32, inData);
  r.rstd = fresh({N}, torch::kFloat32, inData);
  r.var = fresh({N}, torch::kFloat32, inData);
  const size_t bytes = ht_projection_workspace(B, K, N);
  const Tensor ws = workspace(bytes, inData);
  check(ht_projection_forward(B, K, N, fptr(inData), fptr(inLinearWeights), eps, fptr(r.z), fptr(r.mean), fptr(r.rstd),
                              fptr(r.var), ptr(ws), bytes, current_stream(inData)));
  return r;
}

std::pair<Tensor, Tensor> linear_bn_backward(const Tensor &inData, bool need_dx, const Tensor &inLinearWeights,
                                             bool need_lin, const Tensor &zhat, const Tensor &rstd,
                                             const Tensor &outDataGrad) {
  for (const Tensor *t : {&inData, &inLinearWeights, &zhat, &rstd, &outDataGrad}) {
    need_float(*t);
    need_contiguous(*t);
    need_same_device(*t, inData);
  }
  need_gpu(inData);
  need_projection(inData, inLinearWeights);
  const int64_t B = inData.size(0), K = inData.size(1), N = inLinearWeights.size(0);
  const std::vector<int64_t> bn = {B, N}, n = {N};
  if (zhat.sizes() != c10::IntArrayRef(bn) || outDataGrad.sizes() != c10::IntArrayRef(bn) || rstd.sizes() != c10::IntArrayRef(n))
    invalid("Error: shapes of zhat / rstd / outDataGrad do not match the projection.");
  const c10::DeviceGuard guard(inData.device());
  Tensor dx, dlin;
  if (need_dx) dx = fresh_like(inData);
  if (need_lin) dlin = fresh_like(inLinearWeights);
  const size_t bytes = ht_projection_backward_workspace(B, K, N);
  const Tensor ws = workspace(bytes, inData);
  check(ht_projection_backward(B, K, N, fptr(inData), fptr(inLinearWeights), fptr(zhat), fptr(rstd), fptr(outDataGrad),
                               fptr(dlin), fptr(dx), ptr(ws), bytes, current_stream(inData)));
  return {dx, dlin};
}

LinearForest linear_bn_forest_forward(int kind, const Tensor &inData, const Tensor &inLinearWeights, double eps,
                                      const Tensor &inThresholds, const Tensor &inOrdinals, const Tensor &inWeights,
                                      bool want_records) {
  for (const Tensor *t : {&inData, &inLinearWeights, &inThresholds, &inWeights}) need_float(*t);
  need_contiguous(inData);
  need_contiguous(inLinearWeights);
  need_same_device(inData, inLinearWeights);
  need_gpu(inData);
  need_projection(inData, inLinearWeights);
  const int64_t B = inData.size(0), K = inData.size(1), N = inLinearWeights.size(0);
  if (B == 0) invalid("Error: batch statistics need at least one sample.");
  const c10::DeviceGuard guard(inData.device());
  LinearForest r;
  r.bn.z = fresh({B, N}, torch::kFloat32, inData);
  common_checks({&r.bn.z, &inThresholds, &inWeights}, inOrdinals, false);
  std::vector<int64_t> out_sizes;
  const ht_forest_shape s = forest_shape(kind, r.bn.z, inThresholds, inOrdinals, inWeights, nullptr, &out_sizes);
  r.bn.mean = fresh({N}, torch::kFloat32, inData);
  r.bn.rstd = fresh({N}, torch::kFloat32, inData);
  r.bn.var = fresh({N}, torch::kFloat32, inData);
  r.out = fresh(out_sizes, torch::kFloat32, inData);
  const size_t rec_bytes = want_records ? ht_forest_records_bytes(&s) : 0;
  r.records = workspace(rec_bytes, inData);
  const size_t bytes = ht_projection_forest_forward_workspace(&s, K);
  const Tensor ws = workspace(bytes, inData);
  check(ht_projection_forest_forward(&s, K, fptr(inData), fptr(inLinearWeights), eps, fptr(inThresholds), iptr(inOrdinals),
                                     fptr(inWeights), fptr(r.out), fptr(r.bn.z), fptr(r.bn.mean), fptr(r.bn.rstd),
                                     fptr(r.bn.var), ptr(r.records), rec_bytes, ptr(ws), bytes, current_stream(inData)));
  return r;
}

LinearForestGradients linear_bn_forest_backward(int kind, const Tensor &records, const Tensor &inData,
                                                const Tensor &inLinearWeights, bool need_lin, const Tensor &zhat,
                                                const Tensor &rstd, const Tensor &inThresholds, bool need_thr,
                                                const Tensor &inOrdinals, const Tensor &inWeights, bool need_w,
                                                const Tensor &outDataGrad, const Tensor &mean) {
  if (!records.defined() || records.scalar_type() != torch::kUInt8 || !records.is_contiguous())
    invalid("Error: records must be the contiguous uint8 tensor a *_forward_records call returned.");
  for (const Tensor *t : {&inData, &inLinearWeights, &zhat, &rstd, &inThresholds, &inWeights, &outDataGrad}) need_float(*t);
  for (const Tensor *t : {&inData, &inLinearWeights, &zhat, &rstd, &records, &mean}) {
    if (!t->defined()) continue;  // (mean may be left out)
    need_contiguous(*t);
    need_same_device(*t, inData);
  }
  if (mean.defined() && (mean.scalar_type() != torch::kFloat32 || mean.sizes() != rstd.sizes()))
    invalid("Error: shapes of zhat / rstd do not match the projection.");
  need_gpu(inData);
  common_checks({&zhat, &inThresholds, &inWeights, &outDataGrad}, inOrdinals, true);
  if (inData.dim() != 2 || inLinearWeights.dim() != 2 || zhat.dim() != 2)
    invalid("Error: inData must be [batch, in_features], inLinearWeights [out_features, in_features], zhat [batch, "
            "out_features].");
  const int64_t B = inData.size(0), K = inData.size(1), N = inLinearWeights.size(0);
  if (inLinearWeights.size(1) != K || zhat.size(0) != B || zhat.size(1) != N || rstd.dim() != 1 || rstd.size(0) != N)
    invalid("Error: shapes of zhat / rstd do not match the projection.");
  std::vector<int64_t> out_sizes;
  const ht_forest_shape s = forest_shape(kind, zhat, inThresholds, inOrdinals, inWeights, &outDataGrad, &out_sizes);
  if (size_t(records.numel()) != ht_forest_records_bytes(&s)) invalid("Error: records do not belong to a forest of this shape.");
  LinearForestGradients r;
  const size_t bytes = ht_projection_forest_backward_workspace(&s, K);
  if (bytes == 0) return r;
  const c10::DeviceGuard guard(inData.device());
  if (need_lin) r.dlin = fresh_like(inLinearWeights);
  if (need_thr) r.dthr = fresh_like(inThresholds);
  if (need_w) r.dw = fresh_like(inWeights);
  const Tensor ws = workspace(bytes, inData);
  check(ht_projection_forest_backward(&s, K, fptr(inData), fptr(inLinearWeights), fptr(zhat), fptr(mean), fptr(rstd),
                                      fptr(inWeights), fptr(outDataGrad), ptr(records), size_t(records.numel()),
                                      fptr(r.dthr), fptr(r.dw), fptr(r.dlin), ptr(ws), bytes, current_stream(inData)));
  r.served = true;
  return r;
}

// running <- (1 - momentum) running + momentum * batch for the mean and the unbiased variance, and the batch counter, in
// place; false where the tensors are not what the kernel takes or torch follows the call (the caller then does it with
// torch operations).
static bool update_running_stats(Tensor running_mean, Tensor running_var, Tensor batches, const Tensor &mean,
                                 const Tensor &var, double momentum, int64_t B) {
  if (watched()) return false;
  for (const Tensor *t : std::initializer_list<const Tensor *>{&running_mean, &running_var, &mean, &var})
    if (!t->is_cuda() || t->scalar_type() != torch::kFloat32 || !t->is_contiguous() || t->numel() != mean.numel() ||
        t->device() != mean.device())
      return false;
  if (!batches.is_cuda() || batches.scalar_type() != torch::kInt64 || batches.numel() != 1 || batches.device() != mean.device())
    return false;
  const c10::DeviceGuard guard(mean.device());
  check(ht_running_stats(mean.numel(), B, momentum, fptr(mean), fptr(var), fptr(running_mean), fptr(running_var),
                         static_cast<int64_t *>(ptr(batches)), current_stream(mean)));
  for (Tensor *t : {&running_mean, &running_var, &batches}) t->unsafeGetTensorImpl()->bump_version();
  return true;
}

// ---- bindings: the Python host's names and signatures -----------------------------------------------------------------
static py::object opt(const Tensor &t) { return t.defined() ? py::cast(t) : py::none(); }
static Tensor given(const std::optional<Tensor> &t) { return t ? *t : Tensor(); }

static void no_ordinal_gradient(bool wanted) {
  if (wanted) runtime("Error: Gradient on inOrdinals is requested, but inOrdinals never has a gradient.");
}

static int mode_of(bool deterministic) { return deterministic ? HT_BACKWARD_DETERMINISTIC : HT_BACKWARD_ATOMIC; }

static py::list py_mix_backward(int kind, int mode, const Tensor &x, bool bx, const Tensor &thr, bool bthr, const Tensor &ord,
                                bool bord, const Tensor &w, bool bw, const Tensor &lin, bool blin, const Tensor &bias,
                                bool bbias, const Tensor &g, const Tensor &f, const Tensor &records) {
  no_ordinal_gradient(bord);
  const MixGradients r = fused_linear_backward(kind, mode, {bx, bthr, bw}, blin, bbias, x, thr, ord, w, lin, bias, g, f, records);
  py::list out;
  out.append(opt(r.dx));
  out.append(opt(r.dthr));
  out.append(py::none());
  out.append(opt(r.dw));
  out.append(opt(r.dlin));
  out.append(opt(r.dbias));
  return out;
}

void bind_compose(py::module &m) {
  m.def("contract", &contract, py::arg("inData"), py::arg("window"), py::arg("padding"));
  m.def("expand", &expand, py::arg("inData"), py::arg("padding"));
  m.def("update_running_stats", &update_running_stats);
  m.def("linear_bn_forward", [](const Tensor &x, const Tensor &lin, double eps) {
    const BatchNormed r = linear_bn_forward(x, lin, eps);
    py::list out;
    for (const Tensor *t : {&r.z, &r.mean, &r.rstd, &r.var}) out.append(*t);
    return out;
  }, py::arg("inData"), py::arg("inLinearWeights"), py::arg("eps") = 1e-5);
  m.def("linear_bn_backward", [](const Tensor &x, bool bx, const Tensor &lin, bool blin, const Tensor &zhat,
                                 const Tensor &rstd, const Tensor &g) {
    const auto r = linear_bn_backward(x, bx, lin, blin, zhat, rstd, g);
    py::list out;
    out.append(opt(r.first));
    out.append(opt(r.second));
    return out;
  }, py::arg("inData"), py::arg("bInDataGrad"), py::arg("inLinearWeights"), py::arg("bInLinearWeightsGrad"), py::arg("zhat"),
     py::arg("rstd"), py::arg("outDataGrad"));

#define HT_COMPOSED_OPS(prefix, KIND)                                                                                 \
  m.def(prefix "_forward_expanded", [](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,        \
                                       const Extents &padding) {                                                      \
    return forest_forward_expanded(KIND, x, thr, ord, w, padding);                                                    \
  });                                                                                                                 \
  m.def(prefix "_backward_expanded", [](bool deterministic, const Extents &padding, const Tensor &x, bool bx,         \
                                        const Tensor &thr, bool bthr, const Tensor &ord, bool bord, const Tensor &w,  \
                                        bool bw, const Tensor &g) {                                                   \
    no_ordinal_gradient(bord);                                                                                        \
    const Gradients r = forest_backward_expanded(KIND, mode_of(deterministic), {bx, bthr, bw}, x, thr, ord, w, g,     \
                                                 padding);                                                            \
    py::list out;                                                                                                     \
    out.append(opt(r.dx));                                                                                            \
    out.append(opt(r.dthr));                                                                                          \
    out.append(py::none());                                                                                           \
    out.append(opt(r.dw));                                                                                            \
    return out;                                                                                                       \
  });                                                                                                                 \
  m.def(prefix "_fused_linear_forward", [](const Tensor &x, const Tensor &thr, const Tensor &ord, const Tensor &w,    \
                                           const Tensor &lin, const Tensor &bias) {                                   \
    return fused_linear_forward(KIND, x, thr, ord, w, lin, bias, false).out;                                          \
  });                                                                                                                 \
  m.def(prefix "_fused_linear_forward_records", [](const Tensor &x, const Tensor &thr, const Tensor &ord,             \
                                                   const Tensor &w, const Tensor &lin, const Tensor &bias) {          \
    const MixForward r = fused_linear_forward(KIND, x, thr, ord, w, lin, bias, true);                                 \
    return py::make_tuple(r.out, r.f, opt(r.records));                                                                \
  });                                                                                                                 \
  m.def(prefix "_fused_linear_backward", [](const Tensor &x, bool bx, const Tensor &thr, bool bthr, const Tensor &ord, \
                                            bool bord, const Tensor &w, bool bw, const Tensor &lin, bool blin,        \
                                            const Tensor &bias, bool bbias, const Tensor &g) {                        \
    return py_mix_backward(KIND, HT_BACKWARD_ATOMIC, x, bx, thr, bthr, ord, bord, w, bw, lin, blin, bias, bbias, g,   \
                           Tensor(), Tensor());                                                                       \
  });                                                                                                                 \
  m.def(prefix "_fused_linear_backward_deterministic", [](const Tensor &x, bool bx, const Tensor &thr, bool bthr,     \
                                                          const Tensor &ord, bool bord, const Tensor &w, bool bw,     \
                                                          const Tensor &lin, bool blin, const Tensor &bias,           \
                                                          bool bbias, const Tensor &g) {                              \
    return py_mix_backward(KIND, HT_BACKWARD_DETERMINISTIC, x, bx, thr, bthr, ord, bord, w, bw, lin, blin, bias,      \
                           bbias, g, Tensor(), Tensor());                                                             \
  });                                                                                                                 \
  m.def(prefix "_fused_linear_backward_records",                                                                      \
        [](const std::pair<Tensor, std::optional<Tensor>> &state, bool deterministic, const Tensor &x, bool bx,       \
           const Tensor &thr, bool bthr, const Tensor &ord, bool bord, const Tensor &w, bool bw, const Tensor &lin,   \
           bool blin, const Tensor &bias, bool bbias, const Tensor &g) {                                              \
          return py_mix_backward(KIND, mode_of(deterministic), x, bx, thr, bthr, ord, bord, w, bw, lin, blin, bias,   \
                                 bbias, g, state.first, given(state.second));                                         \
        });                                                                                                           \
  m.def(prefix "_linear_bn_forward_records",                                                                          \
        [](const Tensor &x, const Tensor &lin, double eps, const Tensor &thr, const Tensor &ord, const Tensor &w,     \
           bool want_records) {                                                                                       \
          const LinearForest r = linear_bn_forest_forward(KIND, x, lin, eps, thr, ord, w, want_records);              \
          py::list out;                                                                                               \
          out.append(r.out);                                                                                          \
          out.append(opt(r.records));                                                                                 \
          for (const Tensor *t : {&r.bn.z, &r.bn.mean, &r.bn.rstd, &r.bn.var}) out.append(*t);                        \
          return out;                                                                                                 \
        },                                                                                                            \
        py::arg("inData"), py::arg("inLinearWeights"), py::arg("eps"), py::arg("inThresholds"), py::arg("inOrdinals"), \
        py::arg("inWeights"), py::arg("want_records") = true);                                                        \
  m.def(prefix "_linear_bn_backward_records",                                                                         \
        [](const Tensor &records, const Tensor &x, const Tensor &lin, bool blin, const Tensor &zhat,                  \
           const Tensor &rstd, const Tensor &thr, bool bthr, const Tensor &ord, const Tensor &w, bool bw,             \
           const Tensor &g, const std::optional<Tensor> &mean) -> py::object {                                        \
          const LinearForestGradients r = linear_bn_forest_backward(KIND, records, x, lin, blin, zhat, rstd, thr,     \
                                                                    bthr, ord, w, bw, g, given(mean));                \
          if (!r.served) return py::none();                                                                           \
          py::list out;                                                                                               \
          for (const Tensor *t : {&r.dlin, &r.dthr, &r.dw}) out.append(opt(*t));                                      \
          return out;                                                                                                 \
        },                                                                                                            \
        py::arg("records"), py::arg("inData"), py::arg("inLinearWeights"), py::arg("bInLinearWeightsGrad"),           \
        py::arg("zhat"), py::arg("rstd"), py::arg("inThresholds"), py::arg("bInThresholdsGrad"),                      \
        py::arg("inOrdinals"), py::arg("inWeights"), py::arg("bInWeightsGrad"), py::arg("outDataGrad"),               \
        py::arg("mean") = py::none());
  HT_COMPOSED_OPS("tree", HT_TREE)
  HT_COMPOSED_OPS("fern", HT_FERN)
#undef HT_COMPOSED_OPS
}

}  // namespace hth
