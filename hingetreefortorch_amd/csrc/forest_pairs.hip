// Forest / fern kernels for problems of few (sample, tree) pairs, where a pass is a matter of latency: the number of
// launches, and the chain of dependent loads of one walk.
//
//   forward   one launch, no workspace: a lane per pair reads the threshold and ordinal arrays as they are (no packed
//             copy, no sample tile)
//   backward  from the walk records: a workgroup per tree (dW, dThr) and workgroups of a few samples (dX) in one grid,
//             every gradient accumulated in LDS and written once, so nothing has to be cleared first; where the samples of
//             a tree are shared out, a second launch adds the shares' tables, which the workspace holds
#include <type_traits>

#include "forest_tile.hpp"
#include "lds_accumulate.hpp"
#include "records.hpp"

namespace ht {
namespace {

// ---------------------------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------------------------
// Pairs are numbered like the output, ((b T) + t) K + k, so a wavefront's 64 pairs own 64 M consecutive outputs whatever
// T and K are. A level of a tree costs one round trip to L2, not two: both children of a vertex lie next to each
// other, and their thresholds and ordinals are requested together with the feature that decides between them.
// What it measures (16 rows of 16 features, 100 trees of depth 7, 26 outputs per leaf): 5.6 us against 13.5 us for the
// vertex-packing pre-pass and the tile kernel it replaces there, both bound by latency (1 MB of traffic).
constexpr int kPairThreads = 256;

template <typename Real, bool FERN, int VW, bool RECORD, bool COMPACT>
__global__ __launch_bounds__(kPairThreads) void forward_pairs_kernel(ForestDims d, const Real *__restrict__ x,
                                                                     const Real *__restrict__ thr,
                                                                     const int64_t *__restrict__ ord,
                                                                     const Real *__restrict__ w, Real *__restrict__ out,
                                                                     Records<Real, COMPACT> rec, uint32_t pairs,
                                                                     FastDiv div_m, ImageStore img,
                                                                     FeatureNorm<Real> norm) {
  typedef Real Vec __attribute__((ext_vector_type(VW)));
  const int lane = threadIdx.x & (kWave - 1);
  MarginBits margin_bound;
  const uint32_t stride = gridDim.x * kPairThreads;
  for (uint32_t p0 = blockIdx.x * kPairThreads + (threadIdx.x & ~uint32_t(kWave - 1)); p0 < pairs; p0 += stride) {
    const uint32_t p = min(p0 + uint32_t(lane), pairs - 1);  // surplus lanes repeat the last pair
    const uint32_t q = d.K == 1 ? p : p / uint32_t(d.K);
    const uint32_t k = d.K == 1 ? 0u : p - q * uint32_t(d.K);
    const uint32_t b = q / uint32_t(d.T), t = q - b * uint32_t(d.T);
    const Real *xs = x + (long long)b * d.FK + k;
    const Real *th = thr + (long long)t * d.V;
    const int64_t *od = ord + (long long)t * d.V;
    auto feature = [&](int f) -> Real {
      const Real v = xs[(long long)f * d.K];
      return norm.mean != nullptr ? (v - norm.mean[f]) * norm.rstd[f] : v;
    };
    uint32_t v = 0, key = 0, vertex = 0, sel = 0;
    Real best = Real(0), margin = Real(0);
    Real th_v = th[0];
    int64_t od_v = od[0];
    for (int lvl = 0; lvl < d.depth; ++lvl) {
      const int f = clamp_ordinal(od_v, d.F);
      const Real xv = feature(f);
      Real th_n[2] = {Real(0), Real(0)};
      int64_t od_n[2] = {0, 0};
      if (lvl + 1 < d.depth) {
        if (FERN) {
          th_n[0] = th[lvl + 1];
          od_n[0] = od[lvl + 1];
        } else {
          __builtin_memcpy(th_n, th + 2 * v + 1, sizeof(th_n));
          __builtin_memcpy(od_n, od + 2 * v + 1, sizeof(od_n));
        }
      }
      const Real m = xv - th_v;
      const uint32_t bit = (m > Real(0)) ? 1u : 0u;
      const Real a = ht_abs(m);
      if (lvl == 0 || a < best) {
        best = a;
        margin = m;
        vertex = FERN ? uint32_t(lvl) : v;
        sel = uint32_t(f);
      }
      key |= bit << lvl;
      v = 2u * v + 1u + bit;
      th_v = (!FERN && bit) ? th_n[1] : th_n[0];
      od_v = (!FERN && bit) ? od_n[1] : od_n[0];
    }
    if (RECORD) {
      if (p0 + lane < pairs) rec.put((long long)t * d.pitch + ((long long)b * d.K + k), key, vertex, sel, margin);
      margin_bound.take(margin);
    }
    // the wavefront's outputs, lanes along them
    const uint32_t row = t * uint32_t(d.L) + key;
    const int total = int(min(uint32_t(kWave), pairs - p0)) * d.M / VW;
    Real *obase = out + (long long)p0 * d.M;
    constexpr int kUnroll = 4;
    for (int u0 = 0; u0 < total; u0 += kWave * kUnroll) {
      Real a[kUnroll];
      Vec wv[kUnroll];
      long long at[kUnroll];
#pragma unroll
      for (int i = 0; i < kUnroll; ++i) {
        const int e = min(u0 + i * kWave + lane, total - 1) * VW;
        const int src = div_m.div(e), m = e - src * d.M;
        a[i] = ht_abs(__shfl(margin, src, kWave));
        const long long r = (long long)uint32_t(__shfl(int(row), src, kWave)) * d.M + m;
        wv[i] = *reinterpret_cast<const Vec *>(w + r);
        at[i] = e;
        if (img.nd) {
          // the pair's plane (b, t) and position k
          const long long plane = uint32_t(__shfl(int(q), src, kWave));
          const long long in_plane = img.offset(__shfl(int(k), src, kWave), m);
          at[i] = in_plane < 0 ? -1 : plane * img.plane + in_plane;
        }
      }
#pragma unroll
      for (int i = 0; i < kUnroll; ++i) {
        if (u0 + i * kWave + lane >= total || at[i] < 0) continue;
        Vec o;
#pragma unroll
        for (int j = 0; j < VW; ++j) o[j] = a[i] * wv[i][j];
        *reinterpret_cast<Vec *>((img.nd ? out : obase) + at[i]) = o;
      }
    }
  }
  if (RECORD) {
    // There is no pre-pass that cleared the bound's slots: every workgroup stores its own slot (there are no more
    // workgroups than slots), the first one also the surplus slots.
    __shared__ uint32_t part[kPairThreads / kWave];
    uint32_t bits = margin_bound.bits;
    for (int off = 32; off > 0; off >>= 1) bits = max(bits, uint32_t(__shfl_xor(int(bits), off, kWave)));
    if (lane == 0) part[threadIdx.x / kWave] = bits;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int i = 1; i < kPairThreads / kWave; ++i) bits = max(bits, part[i]);
      rec.bound[blockIdx.x] = (unsigned long long)__double_as_longlong(margin_bound_value<Real>(bits));
    }
    if (blockIdx.x == 0)
      for (int i = int(gridDim.x) + int(threadIdx.x); i < kBoundSlots; i += kPairThreads) rec.bound[i] = 0ull;
  }
}

template <typename Real, bool FERN, int VW, bool RECORD, bool COMPACT>
int launch_forward_pairs(const ForestDims &d, const Real *x, const Real *thr, const int64_t *ord, const Real *w,
                         Real *out, void *records, const ImageStore &img, const FeatureNorm<Real> &norm,
                         hipStream_t stream) {
  Records<Real, COMPACT> rec{};
  if (RECORD) rec = carve_records<Real, COMPACT>(d, records, nullptr);
  const uint32_t pairs = uint32_t(d.S * d.T);
  uint32_t blocks = (pairs + kPairThreads - 1) / kPairThreads;
  if (blocks > uint32_t(kBoundSlots)) blocks = kBoundSlots;
  hipLaunchKernelGGL((forward_pairs_kernel<Real, FERN, VW, RECORD, COMPACT>), dim3(blocks), dim3(kPairThreads), 0, stream,
                     d, x, thr, ord, w, out, rec, pairs, FastDiv(d.M), img, norm);
  HT_LAUNCH_CHECK("forest forward (pairs)");
  return HT_OK;
}

template <typename Real, bool FERN, int VW>
int forward_pairs_rec(const ForestDims &d, const Real *x, const Real *thr, const int64_t *ord, const Real *w, Real *out,
                      void *records, const ImageStore &img, const FeatureNorm<Real> &norm, hipStream_t stream) {
  if (!records) return launch_forward_pairs<Real, FERN, VW, false, true>(d, x, thr, ord, w, out, records, img, norm, stream);
  if (compact_ok(d)) return launch_forward_pairs<Real, FERN, VW, true, true>(d, x, thr, ord, w, out, records, img, norm, stream);
  return launch_forward_pairs<Real, FERN, VW, true, false>(d, x, thr, ord, w, out, records, img, norm, stream);
}

template <typename Real, bool FERN>
int forward_pairs_vw(const ForestDims &d, const Real *x, const Real *thr, const int64_t *ord, const Real *w, Real *out,
                     void *records, const ImageStore &img, const FeatureNorm<Real> &norm, hipStream_t stream) {
  const uintptr_t pw = reinterpret_cast<uintptr_t>(w), po = reinterpret_cast<uintptr_t>(out);
  auto fits = [&](int vw) {
    if (d.M % vw != 0 || pw % (vw * sizeof(Real)) != 0 || po % (vw * sizeof(Real)) != 0) return false;
    return img.nd == 0 || (img.win[2] % vw == 0 && img.pad[2] % vw == 0 && img.size[2] % vw == 0);
  };
  if (fits(4)) return forward_pairs_rec<Real, FERN, 4>(d, x, thr, ord, w, out, records, img, norm, stream);
  if (fits(2)) return forward_pairs_rec<Real, FERN, 2>(d, x, thr, ord, w, out, records, img, norm, stream);
  return forward_pairs_rec<Real, FERN, 1>(d, x, thr, ord, w, out, records, img, norm, stream);
}

// ---------------------------------------------------------------------------------------------------------------
// backward from records
// ---------------------------------------------------------------------------------------------------------------
// Workgroups [0, T * parts) own a tree each and pass over one of `parts` shares of the samples; the others own `per`
// consecutive samples and pass over all trees. Both form c = sign(margin) * sum_m w g of the pairs they meet (twice in all:
// the second read of a small problem's rows comes from L2), so neither waits for the other. What bounds such a pass is
// the chain record -> leaf row, so a lane takes kPairBatch pairs at a time and requests everything it needs of them
// before it uses any of it. P adjacent lanes serve a pair, lane li its elements li, li + P, ..., kPairElems of them per
// round. LDS cells are fp64 (see lds_accumulate.hpp). With parts > 1 every share stores its table as it is, and
// merge_shares_kernel adds them: one rounding to the result's type in all. (Met in float32 atomics, the 100 shares of 25600
// samples x 64 outputs of depth 7 left an error of dW against float64 of 1.8e-7 of its norm.)
__device__ __forceinline__ float fused_multiply_add(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fused_multiply_add(double a, double b, double c) { return __builtin_fma(a, b, c); }

constexpr int kPairBackThreads = 512;
constexpr int kPairBatch = 2;

template <typename Real, int P, int E, bool COMPACT>
__global__ __launch_bounds__(kPairBackThreads) void backward_pairs_kernel(ForestDims d, const Real *__restrict__ w,
                                                                          const Real *__restrict__ gout,
                                                                          Records<Real, COMPACT> rec, Real *dx,
                                                                          Real *dthr, Real *dw, double *shares,
                                                                          int tree_groups, int parts,
                                                                          long long part_size, int per) {
  constexpr int NT = kPairBackThreads, U = kPairBatch;
  constexpr int NP = NT / P;  // pairs of the workgroup per step
  extern __shared__ __align__(16) unsigned char smem[];
  double *acc = reinterpret_cast<double *>(smem);
  const int grp = threadIdx.x / P, li = threadIdx.x % P;
  // c of U pairs, one rounding per product as in the tree kernels; every term |margin| * g goes to add(u, m, term)
  auto pairs = [&](const long long (&goff)[U], const long long (&woff)[U], const Real (&mg)[U], const bool (&on)[U],
                   Real (&c)[U], auto add) {
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = Real(0);
    for (int m0 = 0; m0 < d.M; m0 += P * E) {
      Real gv[U][E], wv[U][E];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int m = min(m0 + e * P + li, d.M - 1);
          gv[u][e] = gout[goff[u] + m];
          wv[u][e] = w[woff[u] + m];
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int m = m0 + e * P + li;
          if (m >= d.M) break;
          c[u] = fused_multiply_add(wv[u][e], gv[u][e], c[u]);
          if (on[u]) add(u, m, ht_abs(mg[u]) * gv[u][e]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      for (int off = 1; off < P; off <<= 1) c[u] += __shfl_xor(c[u], off, kWave);
      c[u] *= ht_sign(mg[u]);
    }
  };
  if (int(blockIdx.x) < tree_groups) {
    const int t = int(blockIdx.x) / parts, part = int(blockIdx.x) - t * parts;
    const int n_w = dw ? d.L * d.M : 0, n_t = dthr ? d.V : 0;
    double *acc_t = acc + n_w;
    for (int i = threadIdx.x; i < n_w + n_t; i += NT) acc[i] = 0.0;
    __syncthreads();
    const long long s_begin = part * part_size, s_end = min(d.S, s_begin + part_size);
    for (long long s = s_begin + grp; s < s_end; s += NP * U) {
      uint32_t key[U], vertex[U];
      Real mg[U], c[U];
      bool on[U];
      long long goff[U], woff[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        on[u] = s + u * NP < s_end;
        const long long su = on[u] ? s + u * NP : s, at = (long long)t * d.pitch + su;
        key[u] = rec.key(at);
        vertex[u] = rec.vertex(at);
        mg[u] = rec.margin[at];
        goff[u] = out_offset(d, su, t, 0);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) woff[u] = ((long long)t * d.L + key[u]) * d.M;
      pairs(goff, woff, mg, on, c, [&](int u, int m, Real term) {
        if (dw) atomicAdd(acc + (key[u] * uint32_t(d.M) + uint32_t(m)), double(term));
      });
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (dthr && on[u] && li == 0) atomicAdd(acc_t + vertex[u], -double(c[u]));
    }
    __syncthreads();
    Real *dst_w = dw + (long long)t * n_w, *dst_t = dthr + (long long)t * n_t;
    if (parts > 1) {
      double *dst = shares + (long long)blockIdx.x * (n_w + n_t);
      for (int i = threadIdx.x; i < n_w + n_t; i += NT) dst[i] = acc[i];
    } else {
      for (int i = threadIdx.x; i < n_w; i += NT) dst_w[i] = Real(acc[i]);
      for (int i = threadIdx.x; i < n_t; i += NT) dst_t[i] = Real(acc_t[i]);
    }
    return;
  }
  const long long s0 = (long long)(int(blockIdx.x) - tree_groups) * per;
  const int ns = int(min<long long>(per, d.S - s0));
  for (int i = threadIdx.x; i < ns * d.F; i += NT) acc[i] = 0.0;
  __syncthreads();
  // pairs of the samples, tree running fastest (a sample's gradient row is contiguous along the trees for K == 1)
  const int total = ns * d.T;
  for (int i = grp; i < total; i += NP * U) {
    uint32_t cell[U];
    Real mg[U], c[U];
    bool on[U];
    long long goff[U], woff[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      on[u] = i + u * NP < total;
      const int iu = on[u] ? i + u * NP : i;
      const int j = iu / d.T, t = iu - j * d.T;
      const long long at = (long long)t * d.pitch + s0 + j;
      mg[u] = rec.margin[at];
      cell[u] = uint32_t(j) * uint32_t(d.F) + rec.ord(at);
      woff[u] = ((long long)t * d.L + rec.key(at)) * d.M;
      goff[u] = out_offset(d, s0 + j, t, 0);
    }
    pairs(goff, woff, mg, on, c, [](int, int, Real) {});
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (on[u] && li == 0) atomicAdd(acc + cell[u], double(c[u]));
  }
  __syncthreads();
  if (d.K == 1) {
    for (int i = threadIdx.x; i < ns * d.F; i += NT) dx[s0 * d.F + i] = Real(acc[i]);
  } else {
    for (int i = threadIdx.x; i < ns * d.F; i += NT) {
      const int f = i / ns, j = i - f * ns;
      const long long s = s0 + j;
      dx[(s / d.K) * d.FK + (long long)f * d.K + s % d.K] = Real(acc[j * d.F + f]);
    }
  }
}

// dW [T][n_w] and dThr [T][n_t] from the shares' tables [T][parts][n_w + n_t]: `lanes` threads per cell, each a run of the
// shares, eight requested together, whose sums meet in LDS; all in a fixed order. More than one lane where the cells are
// few: 100000 samples of a single tree of 64 leaves x 26 outputs, 500 shares, backward in all 26 us with a thread per cell,
// 17 with 16 (18 with shares that met in float32 atomics); 16384 samples x 8 trees x 512 leaves x 8 outputs 23 against 24.
constexpr int kMergeThreads = 256, kMergeLanes = 16;
template <typename Real>
__global__ __launch_bounds__(kMergeThreads) void merge_shares_kernel(const double *__restrict__ shares, int parts, int lanes,
                                                                     int n_w, int n_t, long long cells, Real *dw,
                                                                     Real *dthr) {
  __shared__ double sums[kMergeThreads];
  const int n = n_w + n_t, wide = kMergeThreads / lanes;  // cells of a step
  const int lane = int(threadIdx.x) / wide, run = (parts + lanes - 1) / lanes;
  const int p_begin = lane * run, p_end = min(parts, p_begin + run);
  for (long long i0 = (long long)blockIdx.x * wide; i0 < cells; i0 += (long long)gridDim.x * wide) {
    const long long i = i0 + int(threadIdx.x) % wide;
    const long long t = i / n;
    const int e = int(i - t * n);
    double sum = 0.0;
    if (i < cells) {
      const double *src = shares + t * parts * n + e;
      for (int p = p_begin; p < p_end; p += 8) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = src[(long long)min(p + k, p_end - 1) * n];
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (p + k < p_end) sum += v[k];
      }
    }
    sums[threadIdx.x] = sum;
    __syncthreads();
    if (lane == 0 && i < cells) {
      for (int l = 1; l < lanes; ++l) sum += sums[l * wide + int(threadIdx.x)];
      if (e < n_w)
        dw[t * n_w + e] = Real(sum);
      else
        dthr[t * n_t + e - n_w] = Real(sum);
    }
    __syncthreads();
  }
}

// Lanes per pair (four elements of a row each) ...
static int lanes_per_pair(int M) {
  int p = 1;
  while (4 * p < M && p < 16) p <<= 1;
  return p;
}

struct PairPlan {
  int parts, per;
  long long part_size;
};

// ... and the shares of the work: a tree's samples are split until a workgroup has about four steps left or the device
// is full; a dX workgroup takes as many samples as 64 KB of LDS and four steps hold, as long as every CU gets one.
static PairPlan plan_pairs(const ForestDims &d) {
  const long long step = kPairBackThreads / lanes_per_pair(d.M) * kPairBatch;  // pairs
  PairPlan p;
  long long parts = (d.S + 4 * step - 1) / (4 * step);
  const long long most = (2 * kNumCUs + d.T - 1) / d.T;
  if (parts > most) parts = most;
  p.part_size = (d.S + parts - 1) / parts;
  p.parts = int((d.S + p.part_size - 1) / p.part_size);
  const long long by_lds = (64 * 1024) / ((long long)d.F * 8), by_steps = 4 * step / d.T;
  long long per = by_lds < by_steps ? by_lds : by_steps;
  const long long spread = (d.S + kNumCUs - 1) / kNumCUs;
  if (per > spread) per = spread;
  p.per = int(per < 1 ? 1 : per);
  return p;
}

}  // namespace

// Measured against the vertex-packing pre-pass and the tile kernels (replayed graphs of either, T = 8 / 64 / 500 trees,
// 16 and 1000 features, depth 4 / 7 / 10, 1 / 10 / 26 outputs): a lane per pair is 1.2 to 2.7 x faster up to 2^16 pairs of
// any depth; beyond, its uncached vertex loads grow with pairs * depth, and it falls behind at 2^20 of these for trees
// (0.95 - 1.6 x there) and 2^21 for ferns, whose lanes read the same vertices. Walk records go out tree by tree from
// lanes that hold different trees: with them the lines cross at 2^16 pairs (1.4 - 2.6 x there, 0.7 x at 2^17).
template <typename Real>
bool forward_pairs_ok(const ForestDims &d, bool fern, bool records) {
  if (d.S <= 0 || d.T <= 0 || d.M < 1 || d.M > 4096 || d.V < 1 || (long long)d.T * d.L >= (1ll << 31)) return false;
  const long long pairs = d.S * d.T;
  if (pairs <= (1ll << 16)) return true;
  return !records && pairs <= (1ll << 19) && pairs * d.depth <= (fern ? 1ll << 21 : 1ll << 20);
}

template <typename Real>
int forward_pairs(const ForestDims &d, bool fern, const Real *x, const Real *thr, const int64_t *ord, const Real *w,
                  Real *out, void *records, const ImageStore &img, const FeatureNorm<Real> &norm, hipStream_t stream) {
  return fern ? forward_pairs_vw<Real, true>(d, x, thr, ord, w, out, records, img, norm, stream)
              : forward_pairs_vw<Real, false>(d, x, thr, ord, w, out, records, img, norm, stream);
}

// Time against the staged kernels (tree kernel, dThr, dX), replayed graphs of either, 4 to 500 trees, 32 and 1000 features, 16 to
// 10240 cells of dW per tree, three quarters of 2^17 to 2^20 pairs; float32, geometric mean, doubles below that:
//   up to 2^17   0.08 - 0.46 to 4096 cells, 0.41 - 0.84 to 8192. Beyond 8192 a CU holds one table: 0.52 at 4 trees, 0.85 at
//                60, 1.11 / 1.24 / 1.55 at 100 / 129 / 160, whose workgroups leave CUs idle, 0.82 at 200, 0.62 at 500
//   to 2^18      to 4096 cells 0.14 - 0.55; to 8192 0.48 - 0.90 up to 200 trees, at 300 and 500 1.01 (0.70 to 1.30) and 1.06
//                (0.63 to 1.81), doubles 0.75 and 0.68; beyond 0.64 - 1.79
//   to 2^20      to 4096 cells 0.17 - 0.56 up to 129 trees, 0.44 - 0.61 (1.03 the worst) at 160 and 200, 0.67 - 1.06 (1.54) at 300
//                and 500, where the staged kernels read gradient rows of adjacent trees together; to 8192 0.46 - 1.61
template <typename Real>
bool backward_pairs_ok(const ForestDims &d) {
  if (d.S <= 0 || d.T <= 0 || d.M < 1) return false;
  const long long pairs = d.S * d.T, cells = (long long)d.L * d.M;
  if ((cells + d.V) * 8 > kLdsBytes || (long long)d.F * 8 > kLdsBytes) return false;
  if (pairs <= (1ll << 17)) return cells <= 8192 || d.T <= 64 || d.T >= kNumCUs * 3 / 4;
  if (pairs <= (1ll << 18)) return cells <= (sizeof(Real) == 8 || d.T <= 200 ? 8192 : 4096);
  return pairs <= (1ll << 20) && d.T <= kNumCUs / 2 && cells <= 4096;
}

// The tables of the shares, where a tree's samples are shared out.
size_t backward_pairs_workspace(const ForestDims &d, bool need_dthr, bool need_dw) {
  const int parts = plan_pairs(d).parts;
  if (parts <= 1) return 0;
  return align_up(size_t(d.T) * parts * ((need_dw ? size_t(d.L) * d.M : 0) + (need_dthr ? size_t(d.V) : 0)) * 8, 256);
}

template <typename Real>
int backward_pairs(const ForestDims &d, const Real *w, const Real *gout, const void *records, Real *dx, Real *dthr,
                   Real *dw, void *ws, size_t ws_bytes, hipStream_t stream) {
  const PairPlan p = plan_pairs(d);
  const size_t need = backward_pairs_workspace(d, dthr != nullptr, dw != nullptr);
  if (need != 0 && (ws == nullptr || ws_bytes < need))
    return fail(HT_ERR_INVALID_ARGUMENT, "Error: workspace too small for the backward pass.");
  double *shares = static_cast<double *>(ws);
  const int tree_groups = (dthr || dw) ? d.T * p.parts : 0;
  const long long sample_groups = dx ? (d.S + p.per - 1) / p.per : 0;
  size_t lds = (size_t(dw ? (long long)d.L * d.M : 0) + size_t(dthr ? d.V : 0)) * 8;
  if (dx && size_t(p.per) * d.F * 8 > lds) lds = size_t(p.per) * d.F * 8;
  const unsigned grid = unsigned(tree_groups + sample_groups);
  if (grid == 0) return HT_OK;
  auto go = [&](auto p_tag, auto e_tag, auto compact_tag) -> int {
    constexpr bool COMPACT = decltype(compact_tag)::value;
    auto kernel = backward_pairs_kernel<Real, decltype(p_tag)::value, decltype(e_tag)::value, COMPACT>;
    HT_HIP_CHECK(grant_lds(reinterpret_cast<const void *>(kernel)));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kPairBackThreads), lds, stream, d, w, gout,
                       carve_records<Real, COMPACT>(d, const_cast<void *>(records), nullptr), dx, dthr, dw, shares,
                       tree_groups, p.parts, p.part_size, p.per);
    HT_LAUNCH_CHECK("forest backward (pairs)");
    if (need == 0) return HT_OK;
    const int n_w = dw ? d.L * d.M : 0, n_t = dthr ? d.V : 0;
    const long long cells = (long long)d.T * (n_w + n_t);
    int lanes = 1;
    while (2 * lanes <= p.parts && lanes < kMergeLanes && cells * lanes < kMergeThreads * kNumCUs) lanes *= 2;
    long long blocks = (cells * lanes + kMergeThreads - 1) / kMergeThreads;
    if (blocks > 8 * kNumCUs) blocks = 8 * kNumCUs;
    hipLaunchKernelGGL((merge_shares_kernel<Real>), dim3((unsigned)blocks), dim3(kMergeThreads), 0, stream, shares, p.parts,
                       lanes, n_w, n_t, cells, dw, dthr);
    HT_LAUNCH_CHECK("forest backward (sum of the shares)");
    return HT_OK;
  };
  auto by_lanes = [&](auto compact_tag) -> int {
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 4> four{};
    if (d.M == 1) return go(one, one, compact_tag);
    switch (lanes_per_pair(d.M)) {
      case 1: return go(one, four, compact_tag);
      case 2: return go(std::integral_constant<int, 2>{}, four, compact_tag);
      case 4: return go(four, four, compact_tag);
      case 8: return go(std::integral_constant<int, 8>{}, four, compact_tag);
      default: return go(std::integral_constant<int, 16>{}, four, compact_tag);
    }
  };
  return compact_ok(d) ? by_lanes(std::true_type{}) : by_lanes(std::false_type{});
}

#define HT_INSTANTIATE(Real)                                                                                          \
  template bool forward_pairs_ok<Real>(const ForestDims &, bool, bool);                                                           \
  template int forward_pairs<Real>(const ForestDims &, bool, const Real *, const Real *, const int64_t *, const Real *, \
                                   Real *, void *, const ImageStore &, const FeatureNorm<Real> &, hipStream_t);       \
  template bool backward_pairs_ok<Real>(const ForestDims &);                                                          \
  template int backward_pairs<Real>(const ForestDims &, const Real *, const Real *, const void *, Real *, Real *,     \
                                    Real *, void *, size_t, hipStream_t);
HT_INSTANTIATE(float)
HT_INSTANTIATE(double)
#undef HT_INSTANTIATE

}  // namespace ht
