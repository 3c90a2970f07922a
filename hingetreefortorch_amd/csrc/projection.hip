// Dense projection in front of a forest: z = x * lin^T on the matrix cores, batch statistics of z in the same pass,
// normalisation in place, and the matching backward (batch-norm backward + dLin = dz^T * x, dX = dz * lin).
//
// This is the Linear -> BatchNorm1d(affine=False) -> RandomHingeForest composition of the reference's README
// (README.md:117-129, experiments/run_letter_seq.py:45-52) with the two dense stages written for gfx950: the only
// place of this library where MFMA applies. fp32 in, fp32 accumulate: large forward products and the two products behind the
// walk records' backward on split bf16 operands (split_gemm.hip), the others on v_mfma_f32_32x32x2_f32 here.
//
// GEMM tiling: a workgroup of 256 threads (4 wavefronts, 2 x 2) owns a 128 x 128 tile of the result; a wavefront
// owns 64 x 64 of it as 2 x 2 MFMA tiles (64 accumulator registers per lane). The reduction runs in steps of 16:
// both operand tiles are staged in LDS reduction-major (tile[r][i], pitch 132), so the MFMA operand of lane l
// (row l % 32, reduction index l / 32) is one conflict-free ds_read_b32, and the next step's global loads are in
// flight while the current step is multiplied (register double buffering).
#include <type_traits>

#include "common.hpp"
#include "records.hpp"
#include "split_gemm.hpp"

namespace ht {
namespace {

typedef float Acc16 __attribute__((ext_vector_type(16)));
typedef float Vec4 __attribute__((ext_vector_type(4)));

constexpr int kGemmThreads = 256;
constexpr int kTile = 128;  // result tile edge
constexpr int kRed = 16;    // reduction step
constexpr int kPitch = kTile + 4;

// Operand access patterns. An operand is a [rows x red] matrix that contributes tile[r][i] = op(i0 + i, r0 + r).
//   RED_CONTIG  : element (i, r) at p[i * ld + r]   (reduction index contiguous: x and lin in z = x * lin^T)
//   otherwise   : element (i, r) at p[r * ld + i]   (row index contiguous: dz and x in dLin = dz^T * x)
// Each thread moves 2 x float4 per operand and step.
struct Fetch {
  Vec4 v[2];
};

// `full` (uniform over the workgroup): the whole 128 x 16 tile lies inside the operand and may be read as float4s, so
// no thread needs a bounds check -- the common case, and the one whose instruction count matters.
template <bool RED_CONTIG>
__device__ __forceinline__ void fetch_tile(Fetch &f, const float *__restrict__ p, long long ld, int i0, int n_i,
                                           int r0, int n_r, bool vec_ok, bool full) {
  const int t = threadIdx.x;
  if (full) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float *src = RED_CONTIG ? p + (long long)(i0 + t / 4 + 64 * h) * ld + r0 + (t % 4) * 4
                                    : p + (long long)(r0 + t / 32 + 8 * h) * ld + i0 + (t % 32) * 4;
      f.v[h] = *reinterpret_cast<const Vec4 *>(src);
    }
    return;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    Vec4 v = {0.f, 0.f, 0.f, 0.f};
    if (RED_CONTIG) {
      // thread -> (row i = t / 4 + 64 h, reduction quad q = t % 4)
      const int i = i0 + t / 4 + 64 * h, r = r0 + (t % 4) * 4;
      if (i < n_i) {
        const float *src = p + (long long)i * ld + r;
        if (vec_ok && r + 3 < n_r) {
          v = *reinterpret_cast<const Vec4 *>(src);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (r + e < n_r) v[e] = src[e];
        }
      }
    } else {
      // thread -> (reduction index r = t / 32 + 8 h, row quad q = t % 32)
      const int r = r0 + t / 32 + 8 * h, i = i0 + (t % 32) * 4;
      if (r < n_r) {
        const float *src = p + (long long)r * ld + i;
        if (vec_ok && i + 3 < n_i) {
          v = *reinterpret_cast<const Vec4 *>(src);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (i + e < n_i) v[e] = src[e];
        }
      }
    }
    f.v[h] = v;
  }
}

template <bool RED_CONTIG>
__device__ __forceinline__ void stash_tile(float *tile, const Fetch &f) {
  const int t = threadIdx.x;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (RED_CONTIG) {
      const int i = t / 4 + 64 * h, r = (t % 4) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) tile[(r + e) * kPitch + i] = f.v[h][e];
    } else {
      const int r = t / 32 + 8 * h, i = (t % 32) * 4;
      *reinterpret_cast<Vec4 *>(tile + r * kPitch + i) = f.v[h];
    }
  }
}

// C[i, j] = sum_r A(i, r) * B(j, r) (+ bias_i[i] + bias_j[j]), i < n_i, j < n_j, r < n_r; C row-major with leading
// dimension ldc. A launch covers `batches` such problems whose operands lie stride_a / stride_b / stride_c elements
// apart: either one result per batch (blockIdx.z), or -- SUM_BATCHES -- one result summed over all of them (the
// batch index then simply extends the reduction).
// STATS: also accumulate per column j the sum and the sum of squares of C over i into stats[j], stats[n_j + j] (fp64
// atomics; the batch statistics of the projection).
struct GemmArgs {
  const float *A, *B;
  float *C;
  long long lda, ldb, ldc, stride_a, stride_b, stride_c;
  int n_i, n_j, n_r, batches;
  int tiles_i, tiles_j, rows_per_xcd;  // result tiles, and how many tile rows each of the 8 L2 domains takes
  int splits;                          // > 1: blockIdx.y takes a share of the reduction and adds into a zeroed C ...
  long long split_stride;              // ... or, if not 0, stores its share at C + blockIdx.y * split_stride
  bool vec_a, vec_b;
  double *stats;
  const float *bias_i, *bias_j;
  // A_BN: operand A is not read as it lies in memory but as the batch-norm backward of it, element (i, r) =
  // bn_rstd[i] * (A(i, r) - mean_1[i] - bn_zhat(i, r) * mean_2[i]) with mean_1[i] = bn_sums[i] / bn_count and
  // mean_2[i] = bn_sums[n_i + i] / bn_count (bn_zhat laid out like A)
  const float *bn_zhat, *bn_rstd;
  const double *bn_sums;
  double bn_count;
};

// The batch-norm backward of a fetched operand piece: rstd * (a - mean_1 - zh * mean_2) as two fused multiply-adds,
// a * rstd + (zh * (-rstd * mean_2) + (-rstd * mean_1)) -- a staging step of every reduction step, so its instruction
// count matters; bn_backward_apply_kernel rounds after each of its four operations instead, and the two forms differ
// in the last bits.
// rows: the tile's constants in LDS, [rstd | -rstd * mean_1 | -rstd * mean_2][kTile] (zeros for rows outside the
// operand, which makes their elements zero; in LDS because the kernel has no registers to spare for twelve more values
// per thread); row_ok: the piece's reduction index lies inside the operand (outside, the operand contributes zeros).
__device__ __forceinline__ void bn_backward_piece(Vec4 &a, const Vec4 &zh, const float *rows, bool row_ok) {
  const int i = (int(threadIdx.x) % 32) * 4;
  const Vec4 c0 = *reinterpret_cast<const Vec4 *>(rows + i), c1 = *reinterpret_cast<const Vec4 *>(rows + kTile + i),
             c2 = *reinterpret_cast<const Vec4 *>(rows + 2 * kTile + i);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float v = __builtin_fmaf(a[e], c0[e], __builtin_fmaf(zh[e], c2[e], c1[e]));
    a[e] = row_ok ? v : 0.f;
  }
}

template <bool A_RED_CONTIG, bool B_RED_CONTIG, bool STATS, bool SUM_BATCHES, bool A_BN = false>
__global__ __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(3, 4))) void gemm_kernel(GemmArgs g) {
  static_assert(!A_BN || (!A_RED_CONTIG && !SUM_BATCHES), "the fused batch-norm backward reads a row-contiguous operand");
  __shared__ float As[2][kRed * kPitch];
  __shared__ float Bs[2][kRed * kPitch];
  const int n_i = g.n_i, n_j = g.n_j, n_r = g.n_r;
  int tile_i, tile_j;
  // A launch slot runs on XCD slot % 8 whatever its share of a split reduction is (the grid's x extent is a multiple
  // of 8), and the tile map gives every XCD a band of tile rows: with few tile rows the shares would pile their work on
  // the same XCDs, so share y takes the band of the XCD y places further on.
  const int slot = int(blockIdx.x) - int(blockIdx.x) % kNumXCDs + (int(blockIdx.x) + int(blockIdx.y)) % kNumXCDs;
  if (!gemm_tile_of(slot, g.tiles_i, g.tiles_j, g.rows_per_xcd, &tile_i, &tile_j)) return;
  const int i0 = tile_i * kTile, j0 = tile_j * kTile;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * 64;  // this wavefront's 64 x 64 corner
  const int lr = lane & 31, lk = lane >> 5;
  const float *A = g.A, *B = g.B;
  float *C = g.C + (long long)blockIdx.y * g.split_stride;
  if (!SUM_BATCHES) {
    A += (long long)blockIdx.z * g.stride_a;
    B += (long long)blockIdx.z * g.stride_b;
    C += (long long)blockIdx.z * g.stride_c;
  }

  Acc16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  const int per_batch = (n_r + kRed - 1) / kRed;
  // this workgroup's share of the reduction steps (all of them unless the launch splits the reduction)
  const int all_steps = SUM_BATCHES ? per_batch * g.batches : per_batch;
  const int chunk = (all_steps + g.splits - 1) / g.splits;
  const int step0 = blockIdx.y * chunk;
  const int steps = max(0, min(chunk, all_steps - step0));
  if (g.splits > 1 && steps == 0) return;
  const bool rows_a_full = g.vec_a && i0 + kTile <= n_i, rows_b_full = g.vec_b && j0 + kTile <= n_j;
  __shared__ __align__(16) float bn[A_BN ? 3 * kTile : 4];
  if constexpr (A_BN) {
    if (threadIdx.x < kTile) {
      const int i = i0 + int(threadIdx.x);
      const bool in = i < n_i;
      const float rstd = in ? g.bn_rstd[i] : 0.f;
      bn[threadIdx.x] = rstd;
      bn[kTile + threadIdx.x] = in ? -rstd * float(g.bn_sums[i] / g.bn_count) : 0.f;
      bn[2 * kTile + threadIdx.x] = in ? -rstd * float(g.bn_sums[n_i + i] / g.bn_count) : 0.f;
    }
    __syncthreads();
  }
  // Pipeline: while step s is multiplied out of LDS buffer s & 1, the operands of step s + 1 (fetched during step
  // s - 1) are written to the other buffer in the middle of the multiply, and the global loads of step s + 2 are in
  // flight. A wavefront therefore issues its LDS writes and address arithmetic in the shadow of its own MFMAs, and one
  // barrier per step remains.
  // 32-wide blocks of this wavefront's corner that hold any result at all (wave uniform). In a tile on the ragged edge
  // of the result the others are skipped: a dLin of 784 columns ends in a tile column with 16 of them, where one
  // wavefront in two has nothing to multiply and the other one block column instead of two.
  const int na = __builtin_amdgcn_readfirstlane(max(0, min(2, (n_i - i0 - wi + 31) / 32)));
  const int nb = __builtin_amdgcn_readfirstlane(max(0, min(2, (n_j - j0 - wj + 31) / 32)));
  auto multiply = [&](const float *as, const float *bs, int kk_begin, int kk_end, auto edge_tag) {
    constexpr bool EDGE = decltype(edge_tag)::value;
#pragma unroll
    for (int kk = kk_begin; kk < kk_end; kk += 2) {
      const float a0 = as[(kk + lk) * kPitch + wi + lr], a1 = as[(kk + lk) * kPitch + wi + 32 + lr];
      const float b0 = bs[(kk + lk) * kPitch + wj + lr], b1 = bs[(kk + lk) * kPitch + wj + 32 + lr];
      if (!EDGE || (na > 0 && nb > 0)) acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
      if (!EDGE || (na > 0 && nb > 1)) acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
      if (!EDGE || (na > 1 && nb > 0)) acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
      if (!EDGE || (na > 1 && nb > 1)) acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
    }
  };
  // The loop exists twice: for workgroups whose operand tiles all lie inside the matrices (FULL: exactly four
  // unconditional float4 loads per fetch, so the wait in front of the LDS writes can leave the newest four in flight)
  // and for the edge tiles (bounds checks, a data-dependent number of loads, hence full waits).
  auto run = [&](auto full_tag) {
    constexpr bool FULL = decltype(full_tag)::value;
    // (A_BN: an operand piece of A travels with the matching piece of zhat, in the second half of the same structure)
    struct FetchA {
      Fetch a, zh;
    };
    auto fetch = [&](FetchA &fa, Fetch &fb, int s) {
      const int gs = s + step0;
      const int z = SUM_BATCHES ? gs / per_batch : 0;
      const int r0 = (gs - z * per_batch) * kRed;
      fetch_tile<A_RED_CONTIG>(fa.a, A + (long long)z * g.stride_a, g.lda, i0, n_i, r0, n_r, g.vec_a, FULL);
      if constexpr (A_BN) fetch_tile<false>(fa.zh, g.bn_zhat, g.lda, i0, n_i, r0, n_r, g.vec_a, FULL);
      fetch_tile<B_RED_CONTIG>(fb, B + (long long)z * g.stride_b, g.ldb, j0, n_j, r0, n_r, g.vec_b, FULL);
    };
    // operands of step s from registers into an LDS buffer
    auto stash = [&](int buffer, FetchA &fa, const Fetch &fb, int s) {
      if constexpr (A_BN) {
        const int r0 = (s + step0) * kRed;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          bn_backward_piece(fa.a.v[h], fa.zh.v[h], bn, FULL || r0 + int(threadIdx.x) / 32 + 8 * h < n_r);
      }
      stash_tile<A_RED_CONTIG>(As[buffer], fa.a);
      stash_tile<B_RED_CONTIG>(Bs[buffer], fb);
    };
    if constexpr (A_BN) {
      // One step of lookahead only: the operands of step s + 1 are requested when step s begins and written to LDS
      // when its products are done. With zhat travelling beside A, two steps in flight need more registers than three
      // wavefronts per SIMD leave, and the third wavefront hides more latency than the second step ahead did.
      FetchA fa;
      Fetch fb;
      if (steps > 0) {
        fetch(fa, fb, 0);
        stash(0, fa, fb, 0);
      }
      __syncthreads();
      for (int s = 0; s < steps; ++s) {
        const int cur = s & 1;
        const bool more = s + 1 < steps;
        if (more) fetch(fa, fb, s + 1);
        multiply(As[cur], Bs[cur], 0, kRed, std::integral_constant<bool, !FULL>{});
        if (more) stash(cur ^ 1, fa, fb, s + 1);
        __syncthreads();
      }
      return;
    }
    FetchA fa0, fa1;
    Fetch fb0, fb1;
    if (steps > 0) {
      fetch(fa0, fb0, 0);
      stash(0, fa0, fb0, 0);
      if (steps > 1) fetch(fa0, fb0, 1);
    }
    __syncthreads();
    // one step: `held` carries the operands of step s + 1, `next` receives those of step s + 2. PREFETCH is a
    // compile-time property of the call site: the steady-state loop always fetches (so the wait in front of the LDS
    // writes may leave exactly those newest loads in flight), the last two steps never do.
    auto step = [&](int s, FetchA &held_a, Fetch &held_b, FetchA &next_a, Fetch &next_b, auto prefetch_tag) {
      constexpr bool PREFETCH = decltype(prefetch_tag)::value;
      const int cur = s & 1;
      if (PREFETCH) fetch(next_a, next_b, s + 2);
      multiply(As[cur], Bs[cur], 0, kRed / 2, std::integral_constant<bool, !FULL>{});
      if (PREFETCH || s + 1 < steps) stash(cur ^ 1, held_a, held_b, s + 1);
      multiply(As[cur], Bs[cur], kRed / 2, kRed, std::integral_constant<bool, !FULL>{});
      __syncthreads();
    };
    int s = 0;
    for (; s + 3 < steps; s += 2) {  // both steps have a step s + 2 to fetch
      step(s, fa0, fb0, fa1, fb1, std::true_type{});
      step(s + 1, fa1, fb1, fa0, fb0, std::true_type{});
    }
    if (s + 2 < steps) {             // one more step that fetches; the operand registers swap roles once more
      step(s, fa0, fb0, fa1, fb1, std::true_type{});
      step(s + 1, fa1, fb1, fa0, fb0, std::false_type{});
      step(s + 2, fa0, fb0, fa1, fb1, std::false_type{});
    } else {
      if (s < steps) step(s, fa0, fb0, fa1, fb1, std::false_type{});
      if (s + 1 < steps) step(s + 1, fa1, fb1, fa0, fb0, std::false_type{});
    }
  };
  if (rows_a_full && rows_b_full && n_r % kRed == 0)
    run(std::true_type{});
  else
    run(std::false_type{});

  // accumulator element e of lane l is C(row 8 * (e / 4) + 4 * (l / 32) + e % 4, column l % 32) of its 32 x 32 tile
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int j = j0 + wj + 32 * b + lr;
    const bool first = blockIdx.y == 0;  // the biases belong to one share of a split reduction only
    const float bj = (g.bias_j && first && j < n_j) ? g.bias_j[j] : 0.f;
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int i = i0 + wi + 32 * a + 8 * (e / 4) + 4 * lk + (e % 4);
        if (i < n_i && j < n_j) {
          float v = acc[a][b][e];
          if (g.bias_i && first) v += g.bias_i[i];
          v += bj;
          if (g.splits > 1 && g.split_stride == 0) {
            atomicAdd(C + (long long)i * g.ldc + j, v);
          } else {
            C[(long long)i * g.ldc + j] = v;
          }
          if (STATS) {
            s1 += double(v);
            s2 += double(v) * double(v);
          }
        }
      }
    }
    if (STATS) {
      s1 += __shfl_xor(s1, 32, 64);
      s2 += __shfl_xor(s2, 32, 64);
      if (lk == 0 && j < n_j) {
        atomicAdd(g.stats + j, s1);
        atomicAdd(g.stats + n_j + j, s2);
      }
    }
  }
}

// mean, rstd (and the biased variance) of every column from the accumulated sums; a wavefront per column.
// x (optional): z [B x N] = x [B x K] * lin [N x K]^T came from split operands, where an infinity of x or lin leaves NaN
// instead of an infinity (split_gemm.hip). The NaN of a column, which its sum gives away, are then formed again as plain sums.
__global__ __launch_bounds__(256) void bn_finalize_kernel(const double *__restrict__ stats, long long N, long long B, double eps,
                                                          float *mean, float *rstd, float *var, const float *__restrict__ x,
                                                          const float *__restrict__ lin, long long K, float *z) {
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  for (long long j = (long long)blockIdx.x * (256 / kWave) + wave; j < N; j += (long long)gridDim.x * (256 / kWave)) {
    double s1 = stats[j], s2 = stats[N + j];
    if (x != nullptr && s1 != s1) {
      s1 = s2 = 0.0;
      for (long long b = lane; b < B; b += kWave) {
        float v = z[b * N + j];
        if (v != v) {
          v = 0.f;
          for (long long k = 0; k < K && v == v; ++k) v = __builtin_fmaf(x[b * K + k], lin[j * K + k], v);
          z[b * N + j] = v;
        }
        s1 += double(v);
        s2 += double(v) * double(v);
      }
      for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_xor(s1, off, kWave);
        s2 += __shfl_xor(s2, off, kWave);
      }
    }
    if (lane != 0) continue;
    const double m = s1 / double(B);
    double v = s2 / double(B) - m * m;
    if (v < 0.0) v = 0.0;
    mean[j] = float(m);
    rstd[j] = float(1.0 / sqrt(v + eps));
    if (var) var[j] = float(v);
  }
}

// The running statistics of BatchNorm1d after a training batch, as torch updates them: r <- (1 - m) r + m batch, with the
// unbiased variance, and the batch counter.
__global__ void running_stats_kernel(int N, float momentum, float unbias, const float *__restrict__ mean,
                                     const float *__restrict__ var, float *running_mean, float *running_var,
                                     long long *batches) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j == 0 && batches) *batches += 1;
  if (j >= N) return;
  running_mean[j] = running_mean[j] * (1.f - momentum) + momentum * mean[j];
  running_var[j] = running_var[j] * (1.f - momentum) + momentum * (var[j] * unbias);
}

// z <- (z - mean) * rstd, in place, row-major [B x N]. One thread per 4 consecutive columns of 8 rows.
__global__ __launch_bounds__(256) void bn_apply_kernel(float *z, long long B, int N, const float *__restrict__ mean,
                                                       const float *__restrict__ rstd) {
  const int j = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (j >= N) return;
  float m[4], r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    m[e] = j + e < N ? mean[j + e] : 0.f;
    r[e] = j + e < N ? rstd[j + e] : 0.f;
  }
  const bool vec = (N % 4 == 0) && (reinterpret_cast<uintptr_t>(z) % 16 == 0);
  for (long long i = blockIdx.y; i < B; i += gridDim.y) {
    float *p = z + i * N + j;
    if (vec) {
      Vec4 v = *reinterpret_cast<Vec4 *>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (v[e] - m[e]) * r[e];
      *reinterpret_cast<Vec4 *>(p) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j + e < N) p[e] = (p[e] - m[e]) * r[e];
    }
  }
}

// Column sums of g and of g * zhat over the rows (fp64 atomics into sums[j], sums[N + j]).
__global__ __launch_bounds__(256) void bn_backward_sums_kernel(const float *__restrict__ g,
                                                               const float *__restrict__ zhat, long long B, int N,
                                                               double *sums) {
  const int j = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (j >= N) return;
  double s1[4] = {0, 0, 0, 0}, s2[4] = {0, 0, 0, 0};
  const bool vec = (N % 4 == 0) && (reinterpret_cast<uintptr_t>(g) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(zhat) % 16 == 0);
  for (long long i = blockIdx.y; i < B; i += gridDim.y) {
    float gv[4], zv[4];
    if (vec) {
      const Vec4 a = *reinterpret_cast<const Vec4 *>(g + i * N + j), b = *reinterpret_cast<const Vec4 *>(zhat + i * N + j);
#pragma unroll
      for (int e = 0; e < 4; ++e) gv[e] = a[e], zv[e] = b[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        gv[e] = j + e < N ? g[i * N + j + e] : 0.f;
        zv[e] = j + e < N ? zhat[i * N + j + e] : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s1[e] += double(gv[e]);
      s2[e] += double(gv[e]) * double(zv[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (j + e < N) {
      atomicAdd(sums + j + e, s1[e]);
      atomicAdd(sums + N + j + e, s2[e]);
    }
}

// g <- rstd * (g - mean(g) - zhat * mean(g * zhat)), in place (batch-norm backward without affine parameters).
__global__ __launch_bounds__(256) void bn_backward_apply_kernel(float *g, const float *__restrict__ zhat, long long B,
                                                                int N, const float *__restrict__ rstd,
                                                                const double *__restrict__ sums) {
  const int j = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (j >= N) return;
  float r[4], m1[4], m2[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool in = j + e < N;
    r[e] = in ? rstd[j + e] : 0.f;
    m1[e] = in ? float(sums[j + e] / double(B)) : 0.f;
    m2[e] = in ? float(sums[N + j + e] / double(B)) : 0.f;
  }
  const bool vec = (N % 4 == 0) && (reinterpret_cast<uintptr_t>(g) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(zhat) % 16 == 0);
  for (long long i = blockIdx.y; i < B; i += gridDim.y) {
    float *p = g + i * N + j;
    const float *q = zhat + i * N + j;
    if (vec) {
      Vec4 a = *reinterpret_cast<Vec4 *>(p);
      const Vec4 b = *reinterpret_cast<const Vec4 *>(q);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = r[e] * (a[e] - m1[e] - b[e] * m2[e]);
      *reinterpret_cast<Vec4 *>(p) = a;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j + e < N) p[e] = r[e] * (p[e] - m1[e] - q[e] * m2[e]);
    }
  }
}

constexpr long long kMaxGridZ = 65535;  // limit of gridDim.z

// dst[i] = shares[0][i] + shares[1][i] + ... in that order (n elements per share).
__global__ __launch_bounds__(256) void sum_shares_kernel(const float *__restrict__ shares, int count, long long n,
                                                         float *dst, int mirror) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const int row = mirror ? int(i / mirror) : 0, col = mirror ? int(i - (long long)row * mirror) : 0;
    if (row / kSplitTile > col / kSplitTile) continue;
    // eight shares requested together, added in order
    float v = 0.f;
    for (int s = 0; s < count; s += 8) {
      float part[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) part[k] = shares[(long long)min(s + k, count - 1) * n + i];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (s + k < count) v = s + k == 0 ? part[k] : v + part[k];
    }
    dst[i] = v;
    if (row / kSplitTile != col / kSplitTile) dst[(long long)col * mirror + row] = v;
  }
}

bool aligned16(const void *p, long long ld, long long stride) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % 4 == 0 && stride % 4 == 0;
}

// The batch-norm backward that a product applies to its operand A while loading it (see GemmArgs).
struct BnOperand {
  const float *zhat, *rstd;
  const double *sums;
  double count;
};

template <bool A_RED_CONTIG, bool B_RED_CONTIG, bool STATS, bool SUM_BATCHES, bool A_BN = false>
int launch_gemm_batched(const float *A, long long lda, long long stride_a, const float *B, long long ldb,
                        long long stride_b, float *C, long long ldc, long long stride_c, long long n_i, long long n_j,
                        long long n_r, long long batches, double *stats, const float *bias_i, const float *bias_j,
                        hipStream_t stream, bool allow_split = false, float *partials = nullptr, int ordered_splits = 0,
                        const BnOperand *bn = nullptr) {
  if (n_i <= 0 || n_j <= 0 || batches <= 0) return HT_OK;
  if (!SUM_BATCHES && batches > kMaxGridZ) {
    // one result per batch rides on blockIdx.z: longer batch lists go out in several launches
    for (long long b0 = 0; b0 < batches; b0 += kMaxGridZ) {
      const long long nb = batches - b0 < kMaxGridZ ? batches - b0 : kMaxGridZ;
      int rc = launch_gemm_batched<A_RED_CONTIG, B_RED_CONTIG, STATS, SUM_BATCHES, false>(
          A + b0 * stride_a, lda, stride_a, B + b0 * stride_b, ldb, stride_b, C + b0 * stride_c, ldc, stride_c, n_i, n_j,
          n_r, nb, stats, bias_i, bias_j, stream, allow_split);
      if (rc != HT_OK) return rc;
    }
    return HT_OK;
  }
  const long long gi = (n_i + kTile - 1) / kTile, gj = (n_j + kTile - 1) / kTile;
  const long long per_batch = (n_r + kRed - 1) / kRed;
  if (gi > 0x7fffffffLL || gj > 0x7fffffffLL || n_r > 0x7fffffffLL || n_i > 0x7fffffffLL || n_j > 0x7fffffffLL ||
      batches > 0x7fffffffLL || per_batch * batches > 0x7fffffffLL)
    return fail(HT_ERR_RUNTIME, "Error: matrix product too large for this build.");
  GemmArgs g;
  g.A = A, g.B = B, g.C = C;
  g.lda = lda, g.ldb = ldb, g.ldc = ldc;
  g.stride_a = stride_a, g.stride_b = stride_b, g.stride_c = stride_c;
  g.n_i = int(n_i), g.n_j = int(n_j), g.n_r = int(n_r), g.batches = int(batches);
  g.tiles_i = int(gi), g.tiles_j = int(gj), g.rows_per_xcd = int((gi + kNumXCDs - 1) / kNumXCDs);
  const long long slots = (long long)g.rows_per_xcd * gj * kNumXCDs;
  if (slots > 0x7fffffffLL) return fail(HT_ERR_RUNTIME, "Error: matrix product too large for this build.");
  g.vec_a = aligned16(A, lda, stride_a), g.vec_b = aligned16(B, ldb, stride_b);
  g.stats = stats, g.bias_i = bias_i, g.bias_j = bias_j;
  g.bn_zhat = g.bn_rstd = nullptr, g.bn_sums = nullptr, g.bn_count = 1.0;
  if (A_BN) {
    if (!bn || batches != 1) return fail(HT_ERR_RUNTIME, "Error: fused batch-norm operand needs its statistics.");
    g.bn_zhat = bn->zhat, g.bn_rstd = bn->rstd, g.bn_sums = bn->sums, g.bn_count = bn->count;
    g.vec_a = g.vec_a && aligned16(bn->zhat, lda, 0);
  }
  // A product with few result tiles and a long reduction (dLin of a narrow linear head: 10 x 1000 from 65536 rows)
  // would leave most of the device idle: the reduction is then split over blockIdx.y and the shares are added into
  // the zeroed result with float atomics (a few thousand elements times the number of shares).
  g.splits = 1;
  g.split_stride = 0;
  const long long all_steps = SUM_BATCHES ? per_batch * batches : per_batch;
  if (ordered_splits > 1 && partials != nullptr && !STATS && ldc == n_j && batches == 1 && !bias_i && !bias_j) {
    // reproducible form of the split: every share stores its partial result, and the shares are added in a fixed order
    g.splits = ordered_splits;
    g.split_stride = n_i * n_j;
    g.C = partials;
    hipLaunchKernelGGL((gemm_kernel<A_RED_CONTIG, B_RED_CONTIG, STATS, SUM_BATCHES, A_BN>),
                       dim3((unsigned)slots, (unsigned)g.splits, 1u), dim3(kGemmThreads), 0, stream, g);
    HT_LAUNCH_CHECK("matrix product (matrix cores, split reduction)");
    const long long chunk = (all_steps + g.splits - 1) / g.splits;
    const int filled = int((all_steps + chunk - 1) / chunk);  // shares that had steps to do (the others wrote nothing)
    const long long n = n_i * n_j;
    return sum_shares(partials, filled, n, C, stream);
  }
  if (allow_split && !STATS && ldc == n_j && (SUM_BATCHES || batches == 1) && gi * gj < kNumCUs && all_steps >= 64) {
    long long want = (2 * kNumCUs + gi * gj - 1) / (gi * gj);
    if (want > all_steps / 16) want = all_steps / 16;
    if (want > 65535) want = 65535;
    if (want > 1) {
      g.splits = int(want);
      int rc = zero_fill(C, size_t(n_i) * size_t(n_j) * sizeof(float), stream);
      if (rc != HT_OK) return rc;
    }
  }
  hipLaunchKernelGGL((gemm_kernel<A_RED_CONTIG, B_RED_CONTIG, STATS, SUM_BATCHES, A_BN>),
                     dim3((unsigned)slots, (unsigned)g.splits, (unsigned)(SUM_BATCHES ? 1 : batches)), dim3(kGemmThreads),
                     0, stream, g);
  HT_LAUNCH_CHECK("matrix product (matrix cores)");
  return HT_OK;
}

template <bool A_RED_CONTIG, bool B_RED_CONTIG, bool STATS>
int launch_gemm(const float *A, long long lda, const float *B, long long ldb, float *C, long long ldc, long long n_i,
                long long n_j, long long n_r, double *stats, hipStream_t stream) {
  return launch_gemm_batched<A_RED_CONTIG, B_RED_CONTIG, STATS, false>(A, lda, 0, B, ldb, 0, C, ldc, 0, n_i, n_j, n_r, 1,
                                                                        stats, nullptr, nullptr, stream);
}

long long rows_grid(long long B) { return B < 64 ? (B < 1 ? 1 : B) : 64; }

}  // namespace

int sum_shares(const float *shares, int count, long long n, float *dst, hipStream_t stream, int mirror) {
  hipLaunchKernelGGL(sum_shares_kernel, dim3((unsigned)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192)), dim3(256), 0,
                     stream, shares, count, n, dst, mirror);
  HT_LAUNCH_CHECK("matrix product (sum of the shares)");
  return HT_OK;
}

int running_stats(long long N, long long B, double momentum, const float *mean, const float *var, float *running_mean,
                  float *running_var, int64_t *batches, hipStream_t stream) {
  if (N <= 0) return HT_OK;
  const double unbias = double(B) / double(B > 1 ? B - 1 : 1);
  hipLaunchKernelGGL(running_stats_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream, int(N), float(momentum),
                     float(unbias), mean, var, running_mean, running_var, reinterpret_cast<long long *>(batches));
  HT_LAUNCH_CHECK("running statistics");
  return HT_OK;
}

int gemm_tile_map(int tiles_i, int tiles_j, int *tile_i, int *tile_j) {
  const int rows_per_xcd = (tiles_i + kNumXCDs - 1) / kNumXCDs;
  const long long slots = (long long)rows_per_xcd * tiles_j * kNumXCDs;
  for (long long b = 0; b < slots; ++b)
    if (!gemm_tile_of(int(b), tiles_i, tiles_j, rows_per_xcd, &tile_i[b], &tile_j[b])) tile_i[b] = tile_j[b] = -1;
  return int(slots);
}

static size_t projection_workspace(long long N) { return align_up(size_t(2) * size_t(N) * sizeof(double), 256); }

// The split operands pay for their packing passes and their coarser tiles from about 10^9 multiply-adds on (measured:
// 2226 x 28 x 9144, 0.57e9, 91 against 88 us; 2679 x 88 x 5355, 1.26e9, 115 against 118; 8607 x 530 x 1380 151 against
// 306; 16384 x 784 x 12700 2.05 against 2.96 ms, normalisation pass included).
static bool split_pays(long long n_i, long long n_j, long long n_r) {
  return double(n_i) * double(n_j) * double(n_r) >= double(1ll << 30);
}

// z [B x N] = x [B x K] * lin [N x K]^T with the column sums of z and of its squares added to stats; ws: projection_product_workspace
static size_t projection_product_workspace(long long B, long long K, long long N) {
  return split_pays(B, N, K) ? align_up(split_pack_bytes(B, K), 256) + align_up(split_pack_bytes(N, K), 256) : 0;
}
size_t projection_forward_workspace(long long B, long long K, long long N) {
  return projection_workspace(N) + projection_product_workspace(B, K, N);
}
static int projection_product(long long B, long long K, long long N, const float *x, const float *lin, float *z, double *stats,
                              void *ws, hipStream_t stream) {
  if (!split_pays(B, N, K)) return launch_gemm<true, true, true>(x, K, lin, K, z, N, B, N, K, stats, stream);
  unsigned char *px = static_cast<unsigned char *>(ws), *pl = px + align_up(split_pack_bytes(B, K), 256);
  int rc;
  if ((rc = split_pack(x, K, B, K, true, px, stream, nullptr, 1.0, true)) != HT_OK) return rc;
  if ((rc = split_pack(lin, K, N, K, true, pl, stream)) != HT_OK) return rc;
  return split_gemm(px, pl, z, N, B, N, K, stats, stream);
}

// ... and the batch statistics of what it left
static int projection_statistics(long long B, long long K, long long N, const float *x, const float *lin, double eps, float *z,
                                 const double *stats, float *mean, float *rstd, float *var, hipStream_t stream) {
  const bool split = split_pays(B, N, K);
  const long long blocks = (N + 3) / 4 < 64 * kNumCUs ? (N + 3) / 4 : 64 * kNumCUs;
  hipLaunchKernelGGL(bn_finalize_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, stats, N, B, eps, mean, rstd, var,
                     split ? x : nullptr, lin, K, z);
  HT_LAUNCH_CHECK("batch statistics");
  return HT_OK;
}

// Shares of the reduction of a product with rows x cols results over `red` terms (1: no split): long reductions whose
// result tiles do not fill the device evenly by themselves.
int reduction_shares(long long rows, long long cols, long long red) {
  const long long tiles = ((rows + kTile - 1) / kTile) * ((cols + kTile - 1) / kTile), steps = (red + kRed - 1) / kRed;
  if (tiles <= 0 || steps < 64) return 1;
  long long want;
  if (tiles < kNumCUs / 2) {
    // a handful of tiles: enough shares to put four workgroups on every CU (a workgroup alone on a CU waits out every
    // operand latency by itself: a 784 x 784 product over 16 384 rows, 49 tiles, took 0.32 ms with 11 shares, 0.23 with 21)
    want = (4 * kNumCUs + tiles - 1) / tiles;
    if (want > steps / 16) want = steps / 16;
  } else {
    // A few tiles per CU: tiles are equal pieces of work, so 700 of them leave some CUs with three and some with two
    // while the product takes as long as three. About twenty pieces per CU level that out (the README model's dLin,
    // 100 x 7 tiles over 16 384 rows: backward pass 4.22 ms with one share, 3.90 with six, 3.79 with eight, 3.86 with
    // sixteen, the sum of the shares included), each still a reduction of 64 steps or more and all of them together
    // within a GiB of partial results.
    want = (20 * kNumCUs + tiles - 1) / tiles;
    if (want > steps / 64) want = steps / 64;
    const long long bytes = rows * cols * (long long)sizeof(float);
    if (bytes > 0 && want > (1LL << 30) / bytes) want = (1LL << 30) / bytes;
  }
  return want > 1 ? int(want) : 1;
}
// dLin [N x K] reduces over the batch, dX [B x K] over the N columns; the two products run one after the other and
// share the area for their partial results.
size_t shares_bytes(long long B, long long K, long long N) {
  const int s_lin = reduction_shares(N, K, B), s_x = reduction_shares(B, K, N);
  const size_t lin = s_lin > 1 ? size_t(s_lin) * size_t(N) * size_t(K) * sizeof(float) : 0;
  const size_t dx = s_x > 1 ? size_t(s_x) * size_t(B) * size_t(K) * sizeof(float) : 0;
  return lin > dx ? lin : dx;
}

size_t projection_backward_workspace(long long B, long long K, long long N) {
  return projection_workspace(N) + shares_bytes(B, K, N);
}

// zhat [B x N] = normalised (x [B x K] * lin [N x K]^T); mean, rstd, var [N] out; ws: projection_forward_workspace.
int projection_forward(long long B, long long K, long long N, const float *x, const float *lin, double eps,
                       float *zhat, float *mean, float *rstd, float *var, void *ws, hipStream_t stream) {
  int rc;
  double *stats = static_cast<double *>(ws);
  if ((rc = zero_fill(stats, size_t(2) * N * sizeof(double), stream)) != HT_OK) return rc;
  if (B == 0 || N == 0) return HT_OK;
  if ((rc = projection_product(B, K, N, x, lin, zhat, stats, static_cast<unsigned char *>(ws) + projection_workspace(N),
                               stream)) != HT_OK)
    return rc;
  if ((rc = projection_statistics(B, K, N, x, lin, eps, zhat, stats, mean, rstd, var, stream)) != HT_OK) return rc;
  hipLaunchKernelGGL(bn_apply_kernel, dim3((unsigned)((N + 1023) / 1024), (unsigned)rows_grid(B)), dim3(256), 0, stream,
                     zhat, B, int(N), mean, rstd);
  HT_LAUNCH_CHECK("normalisation");
  return HT_OK;
}

// g [B x N] holds dL/dzhat on entry; where dx is wanted it holds dL/dz on return, otherwise it is left as it came.
// dlin [N x K] and / or dx [B x K] out (either may be null).
int projection_backward(long long B, long long K, long long N, const float *x, const float *lin, const float *zhat,
                        const float *rstd, float *g, float *dlin, float *dx, void *ws, hipStream_t stream) {
  int rc;
  double *sums = static_cast<double *>(ws);
  if ((rc = zero_fill(sums, size_t(2) * N * sizeof(double), stream)) != HT_OK) return rc;
  if (B == 0 || N == 0) {
    if (dlin && (rc = zero_fill(dlin, size_t(N) * K * sizeof(float), stream)) != HT_OK) return rc;
    if (dx && (rc = zero_fill(dx, size_t(B) * K * sizeof(float), stream)) != HT_OK) return rc;
    return HT_OK;
  }
  const dim3 grid((unsigned)((N + 1023) / 1024), (unsigned)rows_grid(B));
  hipLaunchKernelGGL(bn_backward_sums_kernel, grid, dim3(256), 0, stream, g, zhat, B, int(N), sums);
  HT_LAUNCH_CHECK("batch-norm backward (sums)");
  float *partials = reinterpret_cast<float *>(static_cast<unsigned char *>(ws) + projection_workspace(N));
  if (dlin && !dx) {
    // dLin alone, the training case of a first layer: dL/dz is not written out and read back, the product's loader
    // turns dL/dzhat into it on the way into LDS (same arithmetic, same dLin bit for bit); g stays as it came
    const BnOperand bn = {zhat, rstd, sums, double(B)};
    return launch_gemm_batched<false, false, false, false, true>(g, N, 0, x, K, 0, dlin, K, 0, N, K, B, 1, nullptr, nullptr,
                                                                  nullptr, stream, false, partials,
                                                                  reduction_shares(N, K, B), &bn);
  }
  hipLaunchKernelGGL(bn_backward_apply_kernel, grid, dim3(256), 0, stream, g, zhat, B, int(N), rstd, sums);
  HT_LAUNCH_CHECK("batch-norm backward");
  // dlin[n, k] = sum_b g[b, n] * x[b, k]: both operands row contiguous, reduction over the batch. A small layer under a
  // large batch has a handful of result tiles and a long reduction: it is then split over workgroups whose shares are
  // summed in a fixed order (reproducible, unlike a split that meets in atomics).
  if (dlin && (rc = launch_gemm_batched<false, false, false, false>(g, N, 0, x, K, 0, dlin, K, 0, N, K, B, 1, nullptr,
                                                                     nullptr, nullptr, stream, false, partials,
                                                                     reduction_shares(N, K, B))) != HT_OK)
    return rc;
  // dx[b, k] = sum_n g[b, n] * lin[n, k]: g has the reduction index n contiguous, lin the row index k (split the same
  // way where a small batch meets a wide layer)
  if (dx && (rc = launch_gemm_batched<true, false, false, false>(g, N, 0, lin, K, 0, dx, K, 0, B, K, N, 1, nullptr,
                                                                  nullptr, nullptr, stream, false, partials,
                                                                  reduction_shares(B, K, N))) != HT_OK)
    return rc;
  return HT_OK;
}

namespace {

// ---- dLin of Linear -> BatchNorm(affine = False) -> forest, from the forest's walk records ------------------------
//
// The upstream gradient of the normalisation, g = dL/dzhat [B x N], is the forest's dX: one non-zero per (sample, tree)
// pair -- c at the feature the selected vertex looks at -- so B * T entries out of B * N (1.6 M of 208 M for the README
// model). Instead of writing that matrix densely, summing its columns, normalising it and multiplying it by x as a dense
// 2 * B * N * K product, the gradient is taken apart:
//   dz = rstd * (g - m1 - zhat * m2),  m1 = mean_b g,  m2 = mean_b (g * zhat)            (batch-norm backward)
//   dLin[n, k] = sum_b dz[b, n] * x[b, k]
//              = rstd[n] * (sum_b g[b, n] * xc[b, k]  -  m2[n] * sum_b zhat[b, n] * xc[b, k])
// with xc = x - mean_b x: the m1 term vanishes against the centring (sum_b xc = 0), and centring costs nothing on the
// zhat term because sum_b zhat = 0. The second sum is rstd[n] * (lin * Gc)[n, k] with Gc = xc^T xc [K x K], since
// zhat = (x lin^T - mean) * rstd: two small dense products (2 B K^2 + 2 N K^2 operations instead of 2 B N K).
// The first sum is sparse: per (tree, vertex) the rows of xc of the samples that selected it, weighted by c. No term is
// a difference of large numbers. m2 is sparse as well: c * zhat at the selected feature.
//
// Steps: column means of x and xc; per tree the samples bucketed by selected vertex (counting sort in LDS); one
// wavefront per (tree, vertex) segment sums c * xc rows in registers (lanes along K) and c * zhat; the two products on
// the matrix cores; an elementwise combination. The order of a segment's samples depends on scheduling (bucket cursors
// are LDS atomics), so like every atomic-mode gradient the last bits can differ between runs.

constexpr int kBucketThreads = 512;
constexpr int kMaxBucketVertices = 16384;  // LDS counters of the bucketing kernel
// Its vertices with a float64 sum in LDS: all of them, or as many as fit beside the counters of a depth-14 tree, the upper
// levels first (few samples of a block select a vertex of the last).
constexpr int bucket_sums(int V) {
  const int fit = (kLdsBytes - 64 - V * int(sizeof(uint32_t))) / int(sizeof(double));
  return V < fit ? V : fit;
}
constexpr size_t bucket_lds(int V) { return size_t(bucket_sums(V)) * sizeof(double) + size_t(V) * sizeof(uint32_t); }
static_assert(bucket_lds(kMaxBucketVertices) + 64 <= size_t(kLdsBytes) && bucket_sums(kMaxBucketVertices) > 8191,
              "counters and sums of the largest tree's upper levels");
constexpr int kChunk = 64;                 // columns of xc that are laid out (and summed) together
constexpr int kSampleBlock = 8192;         // samples that are ordered (and summed) together

// sums[k] += sum_b x[b, k] (fp64 atomics). A workgroup takes 64 columns x a share of the rows, its four wavefronts
// alternate rows, eight in flight, and meet in LDS: one atomic per column and workgroup.
__global__ __launch_bounds__(256) void col_sums_kernel(const float *__restrict__ x, long long B, int K, double *sums) {
  __shared__ double part[3][kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int k = blockIdx.x * kWave + lane;
  double s = 0.0;
  if (k < K) {
    constexpr int kRows = 8;
    const long long stride = (long long)gridDim.y * 4;
    for (long long b = (long long)blockIdx.y * 4 + wave; b < B; b += stride * kRows) {
      float v[kRows];
#pragma unroll
      for (int r = 0; r < kRows; ++r) v[r] = b + r * stride < B ? x[(b + r * stride) * K + k] : 0.f;
#pragma unroll
      for (int r = 0; r < kRows; ++r) s += double(v[r]);
    }
  }
  if (wave > 0) part[wave - 1][lane] = s;
  __syncthreads();
  if (wave == 0 && k < K) atomicAdd(sums + k, s + part[0][lane] + part[1][lane] + part[2][lane]);
}

// xc[chunk][b][k % 64] = x[b, k] - float(sums[k] / B), zeros beyond column K: 256-byte rows of 64 columns.
__global__ __launch_bounds__(256) void center_kernel(const float *__restrict__ x, long long B, int K,
                                                     const double *__restrict__ sums, float *__restrict__ xc) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int k = blockIdx.x * kChunk + lane;
  const float m = k < K ? float(sums[k] / double(B)) : 0.f;
  float *dst = xc + (long long)blockIdx.x * B * kChunk + lane;
  for (long long b = (long long)blockIdx.y * 4 + wave; b < B; b += (long long)gridDim.y * 4)
    dst[b * kChunk] = k < K ? x[b * K + k] - m : 0.f;
}

// What a pair contributes, in the order of its block of samples by selected vertex.
struct PairEntry {
  uint32_t sample;
  float c;
};

// One workgroup per (tree, block of kSampleBlock samples): the block's pairs ordered by the vertex they selected
// (counting sort in LDS), entries[t][.] and the features they look at, features[t][.]. On the way m2sum[n] += sum c * zhat
// over the pairs that look at feature n.
template <bool COMPACT>
__global__ __launch_bounds__(kBucketThreads) void bucket_kernel(ForestDims d, Records<float, COMPACT> rec,
                                                                const float *__restrict__ c,
                                                                const float *__restrict__ zhat,
                                                                const float *__restrict__ z_mean,
                                                                const float *__restrict__ z_rstd,
                                                                PairEntry *__restrict__ entries,
                                                                uint32_t *__restrict__ features, double *m2sum, int sums) {
  extern __shared__ __align__(16) unsigned char smem[];
  // sums of c * zhat by vertex first (fp64: a third of the samples may select the root, whose sum in global atomics took
  // ten times as long as the rest of the kernel; those past `sums` go there), then the counters
  double *m2 = reinterpret_cast<double *>(smem);
  uint32_t *count = reinterpret_cast<uint32_t *>(m2 + sums);  // [V], then the segments' cursors
  __shared__ uint32_t wave_total[kBucketThreads / kWave];
  const int t = blockIdx.x;
  const long long first = (long long)t * d.pitch;
  const long long s_begin = (long long)blockIdx.y * kSampleBlock, s_end = min(d.S, s_begin + kSampleBlock);
  for (int v = threadIdx.x; v < d.V; v += kBucketThreads) count[v] = 0u;
  for (int v = threadIdx.x; v < sums; v += kBucketThreads) m2[v] = 0.0;
  __syncthreads();
  for (long long s = s_begin + threadIdx.x; s < s_end; s += kBucketThreads)
    atomicAdd(&count[min(rec.vertex(first + s), uint32_t(d.V - 1))], 1u);
  __syncthreads();
  // exclusive scan over the V counters: a thread owns a run of `per` consecutive ones
  const int per = (d.V + kBucketThreads - 1) / kBucketThreads;
  const int v0 = min(int(threadIdx.x) * per, d.V), v1 = min(v0 + per, d.V);
  uint32_t mine = 0u;
  for (int v = v0; v < v1; ++v) mine += count[v];
  uint32_t scan = mine;  // inclusive over the wavefront
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t o = __shfl_up(scan, off, kWave);
    if (lane >= off) scan += o;
  }
  if (lane == kWave - 1) wave_total[wave] = scan;
  __syncthreads();
  uint32_t before = scan - mine;
  for (int wv = 0; wv < wave; ++wv) before += wave_total[wv];
  __syncthreads();
  for (int v = v0; v < v1; ++v) {
    const uint32_t n = count[v];
    count[v] = before;
    before += n;
  }
  __syncthreads();
  constexpr int kBatch = 4;  // the chain of loads behind a pair (record, c, zhat) is paid once per batch
  for (long long s0 = s_begin + threadIdx.x; s0 < s_end; s0 += kBucketThreads * kBatch) {
    uint32_t n[kBatch], v[kBatch];
    float cs[kBatch], zh[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const long long at = first + min(s0 + i * kBucketThreads, s_end - 1);
      n[i] = min(rec.ord(at), uint32_t(d.F - 1));
      v[i] = min(rec.vertex(at), uint32_t(d.V - 1));
      cs[i] = c[at];
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) zh[i] = zhat[min(s0 + i * kBucketThreads, s_end - 1) * d.F + n[i]];
    // (z_mean given: `zhat` holds the product before its normalisation, which is applied here as the forward applied it)
    if (z_mean != nullptr) {
#pragma unroll
      for (int i = 0; i < kBatch; ++i) zh[i] = (zh[i] - z_mean[n[i]]) * z_rstd[n[i]];
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const long long s = s0 + i * kBucketThreads;
      if (s >= s_end) break;
      if (cs[i] != 0.f) {
        const double term = double(cs[i]) * double(zh[i]);
        if (v[i] < uint32_t(sums))
          atomicAdd(m2 + v[i], term);
        else
          atomicAdd(m2sum + n[i], term);
      }
      const uint32_t at = atomicAdd(&count[v[i]], 1u);
      entries[first + s_begin + at] = PairEntry{uint32_t(s), cs[i]};
      features[first + s_begin + at] = n[i];
    }
  }
  __syncthreads();
  // (the cursors now stand at the segments' ends: a vertex that was selected by anything has its feature in front of it)
  for (int v = threadIdx.x; v < sums; v += kBucketThreads)
    if (m2[v] != 0.0) atomicAdd(m2sum + features[first + s_begin + count[v] - 1], m2[v]);
}

// Value of lane LANE of each row of 16 lanes, to all lanes of the row.
template <int LANE>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x150 + LANE /* row_newbcast */, 0xF, 0xF, false));
}

constexpr int kSegmentThreads = 256;
constexpr int kSegmentRun = 512;  // entries a row of 16 lanes works off, one after the other
constexpr int kSegmentSpan = kSegmentThreads / 16 * kSegmentRun;  // ... and a workgroup
constexpr long long kSegmentUnits = 1ll << 20;  // units of work of one launch
static_assert((kSegmentUnits + kNumXCDs) * kSegmentThreads < (1ll << 32), "a launch has less than 2^32 threads");

// acc[n, columns of the chunk] += sum of c * xc[sample, columns] over the entries of feature n. A unit of work is (chunk
// of 64 columns, block of 8192 samples, tree, span of entries), numbered in that order, and every XCD takes one
// contiguous eighth of the units: at a time it reads the 2 MB that one chunk of one block of samples is, out of its L2 --
// the rows of a tree's samples come in no useful order, and read from the memory-side cache, 3 KB each, they are what the
// pass costs (16384 samples x 784 columns x 100 trees of depth 7: 0.84 ms that way, 0.36 ms this way; 0.41 ms with blocks
// of 16384 samples, 4 MB, 0.38 ms with 4096). A row of 16 lanes takes kSegmentRun consecutive entries, one 16-byte piece of
// a sample's 256 bytes per lane, four samples in flight; the entries are ordered by feature, so the sum stays in
// registers until the feature changes and then goes out as atomics -- a third of the pass with runs of 128 entries
// (0.48 ms), whose ends are additional changes.
__global__ __launch_bounds__(kSegmentThreads) void segment_sums_kernel(ForestDims d, const PairEntry *__restrict__ entries,
                                                                       const uint32_t *__restrict__ features,
                                                                       const float *__restrict__ xc, int chunks,
                                                                       float *acc_out, long long unit0,
                                                                       long long units_per_xcd, long long units) {
  const int blocks = int((d.S + kSampleBlock - 1) / kSampleBlock), spans = (kSampleBlock + kSegmentSpan - 1) / kSegmentSpan;
  // (units [unit0, unit0 + units) of all)
  const long long nth = (long long)(blockIdx.x % kNumXCDs) * units_per_xcd + blockIdx.x / kNumXCDs, unit = unit0 + nth;
  if (blockIdx.x / kNumXCDs >= units_per_xcd || nth >= units) return;
  const int span = int(unit % spans);
  long long rest = unit / spans;
  const int t = int(rest % d.T);
  rest /= d.T;
  const int block = int(rest % blocks), chunk = int(rest / blocks);
  const long long first = (long long)t * d.pitch;
  const long long block_end = min(d.S, (long long)(block + 1) * kSampleBlock);
  const int row = threadIdx.x / 16, li = threadIdx.x % 16;
  const long long begin = (long long)block * kSampleBlock + (long long)span * kSegmentSpan + row * kSegmentRun;
  const long long end = min(block_end, begin + kSegmentRun);
  const float *base = xc + (long long)chunk * d.S * kChunk + li * 4;
  float *out = acc_out + (long long)chunk * kChunk + li * 4;
  const long long pitch = (long long)chunks * kChunk;
  Vec4 sum = {0.f, 0.f, 0.f, 0.f}, acc = {0.f, 0.f, 0.f, 0.f};  // of the feature's entries so far; of the sixteen at hand
  uint32_t cur = 0xffffffffu;
  auto flush = [&]() {
    if (cur == 0xffffffffu) return;
    float *dst = out + cur * pitch;
    sum += acc;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (sum[e] != 0.f) atomicAdd(dst + e, sum[e]);
  };
  for (long long i0 = begin; i0 < end; i0 += 16) {
    // (lanes past the end repeat the last entry with weight 0)
    const long long i = min(i0 + li, end - 1);
    const PairEntry en = entries[first + i];
    const uint32_t cb = i0 + li < end ? __float_as_uint(en.c) : 0u;
    const uint32_t nf = features[first + i];
    auto four = [&](auto k_tag) {
      constexpr int k = decltype(k_tag)::value;
      const uint32_t s[4] = {row_bcast<k>(en.sample), row_bcast<k + 1>(en.sample), row_bcast<k + 2>(en.sample),
                             row_bcast<k + 3>(en.sample)};
      const uint32_t n[4] = {row_bcast<k>(nf), row_bcast<k + 1>(nf), row_bcast<k + 2>(nf), row_bcast<k + 3>(nf)};
      const uint32_t w[4] = {row_bcast<k>(cb), row_bcast<k + 1>(cb), row_bcast<k + 2>(cb), row_bcast<k + 3>(cb)};
      Vec4 v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const Vec4 *>(base + (long long)s[r] * kChunk);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n[r] != cur) {
          flush();
          cur = n[r];
          sum = acc = Vec4{0.f, 0.f, 0.f, 0.f};
        }
        const float cr = __uint_as_float(w[r]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(cr, v[r][e], acc[e]);
      }
    };
    four(std::integral_constant<int, 0>{});
    four(std::integral_constant<int, 4>{});
    four(std::integral_constant<int, 8>{});
    four(std::integral_constant<int, 12>{});
    sum += acc;
    acc = Vec4{0.f, 0.f, 0.f, 0.f};
  }
  flush();
}

// dlin[n, k] = rstd[n] * (sparse[n, k] - (m2sum[n] / B) * rstd[n] * dense[n, k]); sparse rows are `pitch` apart
__global__ __launch_bounds__(256) void combine_dlin_kernel(long long N, int K, double B, const float *__restrict__ sparse,
                                                           long long pitch, const float *__restrict__ dense,
                                                           const float *__restrict__ rstd,
                                                           const double *__restrict__ m2sum, float *__restrict__ dlin) {
  for (long long n = blockIdx.x; n < N; n += gridDim.x) {
    const float r = rstd[n], f = float(m2sum[n] / B) * r;
    for (int k = threadIdx.x; k < K; k += 256) dlin[n * K + k] = r * (sparse[n * pitch + k] - f * dense[n * K + k]);
  }
}

struct ProjectionForestLayout {
  size_t forest, colsum, m2sum, sparse, xc, packed_x, packed_lin, packed_gram, gram, partials, dense, entries, features, total;
  int chunks, shares;
};

ProjectionForestLayout projection_forest_layout(const ForestDims &d, long long K) {
  ProjectionForestLayout l;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += align_up(bytes, 256);
    return here;
  };
  l.chunks = int((K + kChunk - 1) / kChunk);
  l.shares = split_gemm_shares(K, K, d.S, true);
  l.forest = take(forest_backward_keep_c_workspace<float>(d));
  l.colsum = take(size_t(K) * sizeof(double));
  l.m2sum = take(size_t(d.F) * sizeof(double));
  l.sparse = take(size_t(d.F) * l.chunks * kChunk * sizeof(float));
  l.xc = take(size_t(d.S) * l.chunks * kChunk * sizeof(float));
  l.packed_x = take(split_pack_bytes(K, d.S));
  l.packed_lin = take(split_pack_bytes(d.F, K));
  l.packed_gram = take(split_pack_bytes(K, K));
  l.gram = take(size_t(K) * K * sizeof(float));
  l.partials = take(l.shares > 1 ? size_t(l.shares) * K * K * sizeof(float) : 0);
  l.dense = take(size_t(d.F) * K * sizeof(float));
  l.entries = take(size_t(d.T) * d.pitch * sizeof(PairEntry));
  l.features = take(size_t(d.T) * d.pitch * sizeof(uint32_t));
  l.total = at;
  return l;
}

template <bool COMPACT>
int projection_forest_sparse(const ForestDims &d, const ProjectionForestLayout &l, const void *records, const float *c,
                             const float *zhat, const float *z_mean, const float *z_rstd, unsigned char *base,
                             hipStream_t stream) {
  // (the records are only read here; c comes from the forest pass)
  const Records<float, COMPACT> rec = carve_records<float, COMPACT>(d, const_cast<void *>(records), nullptr);
  PairEntry *entries = reinterpret_cast<PairEntry *>(base + l.entries);
  uint32_t *features = reinterpret_cast<uint32_t *>(base + l.features);
  const long long blocks = (d.S + kSampleBlock - 1) / kSampleBlock;
  HT_HIP_CHECK(grant_lds(reinterpret_cast<const void *>(bucket_kernel<COMPACT>)));
  hipLaunchKernelGGL(bucket_kernel<COMPACT>, dim3((unsigned)d.T, (unsigned)blocks), dim3(kBucketThreads),
                     bucket_lds(d.V), stream, d, rec, c, zhat, z_mean, z_rstd, entries, features,
                     reinterpret_cast<double *>(base + l.m2sum), bucket_sums(d.V));
  HT_LAUNCH_CHECK("projection + forest backward (samples by vertex)");
  const long long spans = (kSampleBlock + kSegmentSpan - 1) / kSegmentSpan;
  const long long all = spans * d.T * blocks * l.chunks;
  for (long long unit0 = 0; unit0 < all; unit0 += kSegmentUnits) {
    const long long units = all - unit0 < kSegmentUnits ? all - unit0 : kSegmentUnits;
    const long long per_xcd = (units + kNumXCDs - 1) / kNumXCDs;
    hipLaunchKernelGGL(segment_sums_kernel, dim3((unsigned)(per_xcd * kNumXCDs)), dim3(kSegmentThreads), 0, stream, d, entries,
                       features, reinterpret_cast<const float *>(base + l.xc), l.chunks,
                       reinterpret_cast<float *>(base + l.sparse), unit0, per_xcd, units);
    HT_LAUNCH_CHECK("projection + forest backward (segment sums)");
  }
  return HT_OK;
}

}  // namespace

size_t projection_forest_forward_workspace(const ForestDims &d, long long K) {
  return align_up(projection_workspace(d.F), 256) + align_up(forest_forward_workspace<float>(d), 256) +
         projection_product_workspace(d.S, K, d.F);
}

// The forward pass of the whole front: z [B x N] = x [B x K] * lin [N x K]^T with its batch statistics (mean, rstd, var
// [N] out), then the forest over the normalised product -- which is never written: the forest's kernels normalise z as
// they read it ((z - mean) * rstd, the arithmetic of bn_apply_kernel), one pass over [B x N] less than
// projection_forward + forest_forward. records (optional) as for forest_forward.
int projection_forest_forward(const ForestDims &d, bool fern, long long K, const float *x, const float *lin, double eps,
                              const float *thr, const int64_t *ord, const float *w, float *out, float *z, float *mean,
                              float *rstd, float *var, void *records, void *ws, size_t ws_bytes, hipStream_t stream) {
  int rc;
  if (d.K != 1) return fail(HT_ERR_INVALID_ARGUMENT, "Error: the projection's forest has no inner data dimensions.");
  if (ws == nullptr || ws_bytes < projection_forest_forward_workspace(d, K))
    return fail(HT_ERR_INVALID_ARGUMENT, "Error: workspace too small for the forward pass.");
  const long long B = d.S, N = d.F;
  double *stats = static_cast<double *>(ws);
  if ((rc = zero_fill(stats, size_t(2) * N * sizeof(double), stream)) != HT_OK) return rc;
  if (B == 0 || N == 0) return HT_OK;
  unsigned char *product_ws = static_cast<unsigned char *>(ws) + align_up(projection_workspace(N), 256) +
                              align_up(forest_forward_workspace<float>(d), 256);
  if ((rc = projection_product(B, K, N, x, lin, z, stats, product_ws, stream)) != HT_OK) return rc;
  if ((rc = projection_statistics(B, K, N, x, lin, eps, z, stats, mean, rstd, var, stream)) != HT_OK) return rc;
  FeatureNorm<float> norm;
  norm.mean = mean, norm.rstd = rstd;
  unsigned char *forest_ws = static_cast<unsigned char *>(ws) + align_up(projection_workspace(N), 256);
  return forest_forward<float>(d, fern, z, thr, ord, w, out, records, forest_ws,
                               ws_bytes - align_up(projection_workspace(N), 256), stream, nullptr, &norm);
}

// Whether projection_forest_backward serves a forest [B x N features, K = 1] behind a projection from K_in inputs.
bool projection_forest_backward_ok(const ForestDims &d, long long K) {
  if (is_empty(d) || d.K != 1 || K <= 0 || K > (1 << 20) || d.V > kMaxBucketVertices) return false;
  // (a ragged K was never served where the dense product is small: 2^20 multiply-adds take less than the launches here)
  if (K % 4 != 0 && double(d.S) * double(d.F) * double(K) < double(1 << 20)) return false;
  if ((long long)d.T * d.V > 0x7fffffffLL * 4 || d.S > 0x7fffffffLL || d.S * d.T > 0x7fffffffLL * 16) return false;
  return forest_backward_keeps_c<float>(d);
}

size_t projection_forest_backward_workspace(const ForestDims &d, long long K) {
  return projection_forest_backward_ok(d, K) ? projection_forest_layout(d, K).total : 0;
}

// dThr, dW of the forest and dLin of the projection in front of it, from the forest's walk records and upstream
// gradient gout; no dense dL/dzhat is formed. x [B x K], lin [N x K], zhat [B x N], rstd [N] as projection_forward left
// them -- or, with mean [N] given, `zhat` is the product before its normalisation as projection_forest_forward left it;
// dthr / dw / dlin may be null.
int projection_forest_backward(const ForestDims &d, bool fern, long long K, const float *x, const float *lin,
                               const float *zhat, const float *mean, const float *rstd, const float *w, const float *gout,
                               const void *records, float *dthr, float *dw, float *dlin, void *ws, size_t ws_bytes,
                               hipStream_t stream) {
  int rc;
  if (!projection_forest_backward_ok(d, K))
    return fail(HT_ERR_RUNTIME, "Error: this shape is not served by the records form of the projection backward.");
  const ProjectionForestLayout l = projection_forest_layout(d, K);
  if (ws == nullptr || ws_bytes < l.total)
    return fail(HT_ERR_INVALID_ARGUMENT, "Error: workspace too small for the backward pass.");
  if (reinterpret_cast<uintptr_t>(ws) % 16 != 0)
    return fail(HT_ERR_INVALID_ARGUMENT, "Error: the workspace must be 16-byte aligned.");
  unsigned char *base = static_cast<unsigned char *>(ws);
  const float *c = nullptr;
  const size_t forest_bytes = l.colsum - l.forest;
  if ((rc = forest_backward_records_keep_c<float>(d, fern, w, gout, records, dthr, dw, base + l.forest, forest_bytes,
                                                  stream, &c)) != HT_OK)
    return rc;
  if (!dlin) return HT_OK;
  const long long B = d.S, N = d.F;
  double *colsum = reinterpret_cast<double *>(base + l.colsum), *m2sum = reinterpret_cast<double *>(base + l.m2sum);
  float *xc = reinterpret_cast<float *>(base + l.xc), *gram = reinterpret_cast<float *>(base + l.gram);
  float *dense = reinterpret_cast<float *>(base + l.dense), *sparse = reinterpret_cast<float *>(base + l.sparse);
  // colsum, m2sum and sparse are neighbours: one clear
  if ((rc = zero_fill(colsum, l.xc - l.colsum, stream)) != HT_OK) return rc;
  // (x is small beside the matrices of the forward pass: shares of 16 rows or more, enough of them to fill the device)
  const dim3 grid((unsigned)l.chunks, (unsigned)(B < 64 ? 1 : (B / 64 < 256 ? B / 64 : 256)));
  hipLaunchKernelGGL(col_sums_kernel, grid, dim3(256), 0, stream, x, B, int(K), colsum);
  HT_LAUNCH_CHECK("projection + forest backward (column means)");
  hipLaunchKernelGGL(center_kernel, grid, dim3(256), 0, stream, x, B, int(K), colsum, xc);
  HT_LAUNCH_CHECK("projection + forest backward (centring)");
  // Gc = xc^T xc (reduction over the batch, shares summed in a fixed order), dense = lin * Gc (Gc is symmetric: its
  // rows serve as the columns the product wants, reduction index contiguous)
  if ((rc = split_pack(x, K, K, B, false, base + l.packed_x, stream, colsum, double(B))) != HT_OK) return rc;
  if ((rc = split_gemm(base + l.packed_x, base + l.packed_x, gram, K, K, K, B, nullptr, stream, l.shares,
                       reinterpret_cast<float *>(base + l.partials), true)) != HT_OK)
    return rc;
  if ((rc = split_pack(gram, K, K, K, true, base + l.packed_gram, stream)) != HT_OK) return rc;
  if ((rc = split_pack(lin, K, N, K, true, base + l.packed_lin, stream)) != HT_OK) return rc;
  if ((rc = split_gemm(base + l.packed_lin, base + l.packed_gram, dense, K, N, K, K, nullptr, stream)) != HT_OK) return rc;
  rc = compact_ok(d) ? projection_forest_sparse<true>(d, l, records, c, zhat, mean, rstd, base, stream)
                     : projection_forest_sparse<false>(d, l, records, c, zhat, mean, rstd, base, stream);
  if (rc != HT_OK) return rc;
  hipLaunchKernelGGL(combine_dlin_kernel, dim3((unsigned)(N < 16384 ? N : 16384)), dim3(256), 0, stream, N, int(K), double(B),
                     sparse, (long long)l.chunks * kChunk, dense, rstd, m2sum, dlin);
  HT_LAUNCH_CHECK("projection + forest backward (dLin)");
  return HT_OK;
}

// Linear mix over the tree axis behind a forest (the reference's "fused linear" operators,
// hingetree_fused_linear.cpp:75-412): f [B, T, R] are forest outputs (R = inner data positions x outputs per leaf).
//   forward : out[b, o, r] = bias[o] + sum_t lin[o, t] * f[b, t, r]
//   backward: h[b, t, r] = sum_o lin[o, t] * g[b, o, r]   (the upstream gradient of the forest)
//             dlin[o, t] = sum_{b, r} g[b, o, r] * f[b, t, r]
// rows [n][R] (the R values of a row contiguous) -> planes [R][n], and back. A thread takes a row: its R values are
// read (written) one after the other -- neighbouring threads' rows are neighbours in memory, so the lines are used
// whole -- and each plane is written (read) with consecutive threads on consecutive addresses.
__global__ __launch_bounds__(256) void rows_to_planes_kernel(long long n, int R, const float *__restrict__ rows,
                                                             float *__restrict__ planes) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    for (int r = 0; r < R; ++r) planes[(long long)r * n + i] = rows[i * R + r];
}
__global__ __launch_bounds__(256) void planes_to_rows_kernel(long long n, int R, const float *__restrict__ planes,
                                                             float *__restrict__ rows) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    for (int r = 0; r < R; ++r) rows[i * R + r] = planes[(long long)r * n + i];
}

int rows_to_planes(long long n, long long R, const float *rows, float *planes, bool back, hipStream_t stream) {
  if (n <= 0 || R <= 0) return HT_OK;
  if (R > 0x7fffffffLL) return fail(HT_ERR_RUNTIME, "Error: rows too long for this build.");
  long long blocks = (n + 255) / 256;
  if (blocks > 32 * kNumCUs) blocks = 32 * kNumCUs;
  if (back)
    hipLaunchKernelGGL(planes_to_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, n, int(R), rows, planes);
  else
    hipLaunchKernelGGL(rows_to_planes_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, n, int(R), rows, planes);
  HT_LAUNCH_CHECK("rows <-> planes");
  return HT_OK;
}

int mix_forward(long long B, long long T, long long O, long long R, const float *f, const float *lin,
                const float *bias, float *out, hipStream_t stream) {
  // (from 17 channels on the matrix-core tile below wins where its 128 rows leave enough workgroups: 30000 rows x 600 trees ->
  // 32 152 us against 178, 65536 x 1000 -> 26 408 against 424, but 4000 x 1000 -> 32 110 against 78)
  if (R == 1 && mix_rows_ok(B, T, O) && (O <= 16 || B <= 16384)) return mix_rows_forward(B, T, O, f, lin, bias, out, stream);
  if (R == 1)  // out [B x O] = f [B x T] * lin [O x T]^T, bias per column
    return launch_gemm_batched<true, true, false, false>(f, T, 0, lin, T, 0, out, O, 0, B, O, T, 1, nullptr, nullptr, bias,
                                                         stream);
  // per sample: out_b [O x R] = lin [O x T] * f_b [T x R], bias per row
  return launch_gemm_batched<true, false, false, false>(lin, T, 0, f, R, T * R, out, R, O * R, O, R, T, B, nullptr, bias,
                                                        nullptr, stream);
}

// Area for the shares of the reproducible split of dLin's reduction (R == 1: one product reducing over the samples).
size_t mix_backward_workspace(long long B, long long T, long long O, long long R) {
  if (R != 1) return 0;
  const int shares = reduction_shares(O, T, B);
  return shares > 1 ? size_t(shares) * size_t(O) * size_t(T) * sizeof(float) : 0;
}

// The row form's backward against the matrix-core products (500 to 65536 samples, 17 to 1000 trees, 1 to 32 channels, us, rows
// first). Both gradients in its one pass: 0.08 to 0.99 x the time up to 24 channels; beyond, 277 against 260 and 293 against 256
// at 65536 x 1000 -> 28 and 32, the worst, and 0.88 x at 65536 x 600 -> 32. dLin alone 203 against 152 at 65536 x 1000 -> 32, 60
// against 146 at one channel. The rows keep these few as well: the error of dLin against float64 is 2.6e-7 of its norm at 65536
// x 1000 -> 16, 6.0e-7 from the product. h alone is one product of few terms per result, which rounds alike either way: 165
// against 64 at 65536 x 600 -> 32, 24 against 10 at 65536 x 17 -> 16, 25 against 19 at 16384 x 600 -> 12, but 11 against 16 at
// 16384 x 100 -> 24 and 50 against 81 at 65536 x 1000 -> 1.
static bool mix_rows_backward_pays(long long B, long long T, long long O, bool h, bool dlin) {
  if (!mix_rows_ok(B, T, O) || (!h && !dlin)) return false;
  return dlin || O < 8 || (B * O < (1ll << 19) && double(B) * double(T) * double(O) < 1e8);
}

int mix_backward(long long B, long long T, long long O, long long R, const float *f, const float *lin, const float *g,
                 float *h, float *dlin, bool deterministic, hipStream_t stream, void *ws, size_t ws_bytes) {
  int rc;
  if (R == 1 && mix_rows_backward_pays(B, T, O, h != nullptr, dlin != nullptr && !deterministic)) {
    // one pass for both; the reproducible dLin comes from the product below, whose shares are summed in a fixed order
    if ((rc = mix_rows_backward(B, T, O, f, lin, g, h, deterministic ? nullptr : dlin, stream)) != HT_OK) return rc;
    if (!deterministic || !dlin) return HT_OK;
    h = nullptr;
  }
  if (h) {
    if (R == 1)  // h [B x T] = g [B x O] * lin [O x T]
      rc = launch_gemm_batched<true, false, false, false>(g, O, 0, lin, T, 0, h, T, 0, B, T, O, 1, nullptr, nullptr,
                                                          nullptr, stream);
    else  // per sample: h_b [T x R] = lin^T [T x O] * g_b [O x R]
      rc = launch_gemm_batched<false, false, false, false>(lin, T, 0, g, R, O * R, h, R, T * R, T, R, O, B, nullptr,
                                                           nullptr, nullptr, stream);
    if (rc != HT_OK) return rc;
  }
  if (dlin && (B == 0 || R == 0)) return zero_fill(dlin, size_t(O) * size_t(T) * sizeof(float), stream);
  if (dlin) {
    if (R == 1) {  // dlin [O x T] = g^T [O x B] * f [B x T]
      // deterministic mode with a workspace: shares of the reduction summed in a fixed order instead of one long pass
      const bool ordered = deterministic && ws != nullptr && ws_bytes >= mix_backward_workspace(B, T, O, R);
      rc = launch_gemm_batched<false, false, false, false>(g, O, 0, f, T, 0, dlin, T, 0, O, T, B, 1, nullptr, nullptr,
                                                           nullptr, stream, !deterministic,
                                                           ordered ? static_cast<float *>(ws) : nullptr,
                                                           ordered ? reduction_shares(O, T, B) : 0);
    }
    else  // dlin [O x T] = sum_b g_b [O x R] * f_b [T x R]^T
      rc = launch_gemm_batched<true, true, false, true>(g, R, O * R, f, R, T * R, dlin, T, 0, O, T, R, B, nullptr,
                                                        nullptr, nullptr, stream, !deterministic);
    if (rc != HT_OK) return rc;
  }
  return HT_OK;
}

}  // namespace ht
