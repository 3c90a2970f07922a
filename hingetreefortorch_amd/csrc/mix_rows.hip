// Linear mix over the tree axis behind a forest for few output channels (O <= kMixRowsMax), float32, f [B, T] rows:
//   forward : out[b, o] = bias[o] + sum_t lin[o, t] * f[b, t]
//   backward: h[b, t] = sum_o lin[o, t] * g[b, o],   dlin[o, t] = sum_b g[b, o] * f[b, t]
// With O this small nothing is left to reuse beyond one pass over f and h: the kernels are bound by streaming them, and a
// matrix-core tile of 128 x 128 results computes mostly padding and starts few workgroups. So a lane owns a row (forward)
// or a column (backward) with its O sums in registers, O known at compile time, and the small operand is broadcast.
// 30000 rows x 600 trees -> 10 channels, us: forward 52 -> 20 (72 MB, 3.6 TB/s), backward 107 in two products -> 39 (144 MB
// read and written, 3.7 TB/s); prediction of 2001 rows x 333 trees 51 -> 21 in all.
#include "common.hpp"

namespace ht {
namespace {

constexpr int kMixRows = 32;   // rows of a forward workgroup
constexpr int kMixChunk = 64;  // trees per step
constexpr int kMixThreads = 256;
constexpr int kMixParts = kMixThreads / kMixRows;    // shares of a chunk's trees
constexpr int kMixPer = kMixChunk / kMixParts;       // trees of a share
constexpr int kMixLoads = kMixRows * kMixChunk / kMixThreads;

// A chunk of f (32 rows x 64 trees) passes through LDS, whose rows the lanes then walk; thread = (row, share of the chunk's
// trees). The next chunk is on its way from memory meanwhile. The shares of a row's sum meet in a fixed order.
template <int O>
__global__ __launch_bounds__(kMixThreads) void mix_rows_forward_kernel(long long B, int T, const float *__restrict__ f,
                                                                       const float *__restrict__ lin,
                                                                       const float *__restrict__ bias,
                                                                       float *__restrict__ out) {
  constexpr int OP = (O + 3) / 4 * 4, LDF = kMixChunk + 1;
  __shared__ __align__(16) float fs[kMixRows * LDF];
  __shared__ __align__(16) float ls[kMixChunk * OP];
  __shared__ float sums[kMixParts * kMixRows * O];
  const long long b0 = (long long)blockIdx.x * kMixRows;
  const int tid = int(threadIdx.x), row = tid % kMixRows, part = tid / kMixRows;
  constexpr int kRowStep = kMixThreads / kMixChunk;  // rows between a thread's loads
  const int lt = tid % kMixChunk, lr = tid / kMixChunk;
  constexpr int kLinLoads = (kMixChunk * O + kMixThreads - 1) / kMixThreads;
  float fv[kMixLoads], lv[kLinLoads];
  auto load = [&](int t0) {
    const bool on = t0 + lt < T;
#pragma unroll
    for (int i = 0; i < kMixLoads; ++i) {
      const long long b = b0 + lr + i * kRowStep;
      fv[i] = (on && b < B) ? f[b * T + t0 + lt] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < kLinLoads; ++i) {
      const int e = tid + i * kMixThreads, o = e / kMixChunk, t = t0 + e % kMixChunk;
      lv[i] = (o < O && t < T) ? lin[(long long)o * T + t] : 0.f;
    }
  };
  if (OP != O)
    for (int i = tid; i < kMixChunk * OP; i += kMixThreads) ls[i] = 0.f;  // the pad stays zero
  float acc[OP];
#pragma unroll
  for (int o = 0; o < OP; ++o) acc[o] = 0.f;
  load(0);
  for (int t0 = 0; t0 < T; t0 += kMixChunk) {
    __syncthreads();  // the chunk before is no longer read
#pragma unroll
    for (int i = 0; i < kMixLoads; ++i) fs[(lr + i * kRowStep) * LDF + lt] = fv[i];
#pragma unroll
    for (int i = 0; i < kLinLoads; ++i) {
      const int e = tid + i * kMixThreads, o = e / kMixChunk;
      if (o < O) ls[(e % kMixChunk) * OP + o] = lv[i];
    }
    __syncthreads();
    if (t0 + kMixChunk < T) load(t0 + kMixChunk);
    const int n = min(kMixPer, T - t0 - part * kMixPer);  // (trees past the last are not multiplied: 0 * inf)
#pragma unroll
    for (int i = 0; i < kMixPer; ++i) {
      if (i >= n) break;
      const float x = fs[row * LDF + part * kMixPer + i];
      const float4 *l4 = reinterpret_cast<const float4 *>(ls + (part * kMixPer + i) * OP);
#pragma unroll
      for (int q = 0; q < OP / 4; ++q) {
        const float4 l = l4[q];
        acc[4 * q + 0] = __builtin_fmaf(x, l.x, acc[4 * q + 0]);
        if (4 * q + 1 < O) acc[4 * q + 1] = __builtin_fmaf(x, l.y, acc[4 * q + 1]);
        if (4 * q + 2 < O) acc[4 * q + 2] = __builtin_fmaf(x, l.z, acc[4 * q + 2]);
        if (4 * q + 3 < O) acc[4 * q + 3] = __builtin_fmaf(x, l.w, acc[4 * q + 3]);
      }
    }
  }
#pragma unroll
  for (int o = 0; o < O; ++o) sums[(part * kMixRows + row) * O + o] = acc[o];
  __syncthreads();
  for (int e = tid; e < kMixRows * O; e += kMixThreads) {
    float v = sums[e];
    for (int p = 1; p < kMixParts; ++p) v += sums[p * kMixRows * O + e];
    const int r = e / O, o = e - r * O;
    if (bias) v += bias[o];
    if (b0 + r < B) out[(b0 + r) * O + o] = v;
  }
}

constexpr int kMixBackThreads = 512;
constexpr int kMixBackWaves = kMixBackThreads / kWave;
constexpr int kMixBackRows = 4;  // rows in flight per wavefront

// Lane = tree, wavefronts of a workgroup on different rows (whose upstream gradients are scalar operands); h and dlin come
// from the same pass. dlin's shares meet in the workgroup's LDS, then by atomics on the cleared result.
template <int O>
__global__ __launch_bounds__(kMixBackThreads) void mix_rows_backward_kernel(long long B, int T, const float *__restrict__ f,
                                                                            const float *__restrict__ lin,
                                                                            const float *__restrict__ g,
                                                                            float *__restrict__ h, float *dlin,
                                                                            long long rows) {
  extern __shared__ __align__(16) unsigned char smem[];
  float *sums = reinterpret_cast<float *>(smem);  // [wavefront][O][64]
  const int lane = int(threadIdx.x) % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int t = int(blockIdx.x) * kWave + lane, tc = min(t, T - 1);
  const bool live = t < T;
  float l[O], acc[O];
#pragma unroll
  for (int o = 0; o < O; ++o) l[o] = lin[(long long)o * T + tc], acc[o] = 0.f;
  const long long end = min(B, ((long long)blockIdx.y + 1) * rows);
  float fv[kMixBackRows];
  auto load = [&](long long b) {
#pragma unroll
    for (int u = 0; u < kMixBackRows; ++u) fv[u] = f[min(b + u, end - 1) * T + tc];
  };
  long long b = (long long)blockIdx.y * rows + wave * kMixBackRows;
  if (dlin && b < end) load(b);
  for (; b < end; b += kMixBackWaves * kMixBackRows) {
    float cur[kMixBackRows];
#pragma unroll
    for (int u = 0; u < kMixBackRows; ++u) cur[u] = fv[u];
    if (dlin && b + kMixBackWaves * kMixBackRows < end) load(b + kMixBackWaves * kMixBackRows);
#pragma unroll
    for (int u = 0; u < kMixBackRows; ++u) {
      if (b + u >= end) break;
      const float *gr = g + (b + u) * O;
      float hv = 0.f;
#pragma unroll
      for (int o = 0; o < O; ++o) {
        const float gv = gr[o];
        hv = __builtin_fmaf(l[o], gv, hv);
        if (dlin) acc[o] = __builtin_fmaf(gv, cur[u], acc[o]);
      }
      if (h && live) h[(b + u) * T + t] = hv;
    }
  }
  if (!dlin) return;
#pragma unroll
  for (int o = 0; o < O; ++o) sums[(wave * O + o) * kWave + lane] = acc[o];
  __syncthreads();
  for (int e = int(threadIdx.x); e < O * kWave; e += kMixBackThreads) {
    float v = sums[e];
    for (int p = 1; p < kMixBackWaves; ++p) v += sums[p * O * kWave + e];
    const int o = e / kWave, te = int(blockIdx.x) * kWave + e % kWave;
    if (te < T) atomicAdd(dlin + (long long)o * T + te, v);
  }
}

template <int O>
int forward_as(long long B, int T, const float *f, const float *lin, const float *bias, float *out, hipStream_t stream) {
  hipLaunchKernelGGL(mix_rows_forward_kernel<O>, dim3((unsigned)((B + kMixRows - 1) / kMixRows)), dim3(kMixThreads), 0,
                     stream, B, T, f, lin, bias, out);
  HT_LAUNCH_CHECK("mix forward (rows)");
  return HT_OK;
}

template <int O>
int backward_as(long long B, int T, const float *f, const float *lin, const float *g, float *h, float *dlin,
                hipStream_t stream) {
  int rc;
  if (dlin && (rc = zero_fill(dlin, size_t(O) * size_t(T) * sizeof(float), stream)) != HT_OK) return rc;
  const long long chunks = (T + kWave - 1) / kWave;
  constexpr long long kStep = kMixBackWaves * kMixBackRows;
  // Four workgroups per CU, none with less than one step of rows; at most 128 shares, whose sums meet one by one in atomics
  // (626 of them at 20001 rows x 16 trees: error of dlin against float64 4.2e-7 of its norm, more than one long sum has).
  long long shares = chunks < 4 * kNumCUs ? 4 * kNumCUs / chunks : 1;
  if (shares > 128) shares = 128;
  long long rows = (B + shares - 1) / shares;
  rows = (rows + kStep - 1) / kStep * kStep;
  shares = (B + rows - 1) / rows;
  const size_t lds = dlin ? size_t(kMixBackWaves) * O * kWave * sizeof(float) : 0;
  HT_HIP_CHECK(grant_lds(reinterpret_cast<const void *>(mix_rows_backward_kernel<O>)));
  hipLaunchKernelGGL(mix_rows_backward_kernel<O>, dim3((unsigned)chunks, (unsigned)shares), dim3(kMixBackThreads), lds,
                     stream, B, T, f, lin, g, h, dlin, rows);
  HT_LAUNCH_CHECK("mix backward (rows)");
  return HT_OK;
}

}  // namespace

// (more rows or trees: the matrix-core product, whose grids are smaller)
constexpr long long kMixMost = 1ll << 28;
static_assert(kMixMost / kMixRows * kMixThreads < (1ll << 32) && kMixMost / kWave * kMixBackThreads < (1ll << 32),
              "a launch has less than 2^32 threads");
bool mix_rows_ok(long long B, long long T, long long O) {
  return O >= 1 && O <= kMixRowsMax && B >= 1 && T >= 1 && T <= kMixMost && B <= kMixMost;
}

#define HT_MIX_EACH(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) \
  X(19) X(20) X(21) X(22) X(23) X(24) X(25) X(26) X(27) X(28) X(29) X(30) X(31) X(32)

int mix_rows_forward(long long B, long long T, long long O, const float *f, const float *lin, const float *bias, float *out,
                     hipStream_t stream) {
  switch (O) {
#define HT_CASE(N) case N: return forward_as<N>(B, int(T), f, lin, bias, out, stream);
    HT_MIX_EACH(HT_CASE)
#undef HT_CASE
  }
  return fail(HT_ERR_RUNTIME, "Error: too many output channels for the row form of the mix.");
}

int mix_rows_backward(long long B, long long T, long long O, const float *f, const float *lin, const float *g, float *h,
                      float *dlin, hipStream_t stream) {
  switch (O) {
#define HT_CASE(N) case N: return backward_as<N>(B, int(T), f, lin, g, h, dlin, stream);
    HT_MIX_EACH(HT_CASE)
#undef HT_CASE
  }
  return fail(HT_ERR_RUNTIME, "Error: too many output channels for the row form of the mix.");
}

}  // namespace ht
