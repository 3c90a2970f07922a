// Matrix products of float32 operands on the bf16 matrix cores, at float32 precision.
//
// A float32 number is the sum of three bfloat16 numbers, x = x1 + x2 + x3: x1 = bf16(x), x2 = bf16(x - x1), x3 =
// bf16(x - x1 - x2), every difference exact, each term rounded to nearest, so |x2| <= 2^-9 |x| and |x3| <= 2^-18 |x| and
// nothing is left over (3 x 8 significant bits) as long as bf16 can hold the last of them: its smallest number is 2^-133, so an
// operand below 2^-109 loses up to 2^-134 (at 2^-126, the smallest normal number, 2^-8 of itself). A product is then the sum of nine products of bf16 numbers, each exact
// in float32, of which the three smallest -- x2 y3, x3 y2 and x3 y3, together below 2^-26 |x y|, a quarter of the
// rounding of one float32 operation -- are left out. The other six accumulate in the float32 accumulators of
// v_mfma_f32_32x32x16_bf16. (The splitting is that of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", ARITH 2019.) Six products at 16 times the rate of
// v_mfma_f32_32x32x2_f32 leave a factor of 2.7 at the peaks. An infinity or NaN has no second and third part (zeros): it
// makes every result it enters infinite or NaN. Against the parts of a finite number, whose signs differ, an infinity sums to
// NaN: a caller to whom the difference matters forms such results again (bn_finalize_kernel).
//
// The matrix instructions round their sums towards minus infinity: over 16384 x 784 inputs the results lie 3.9e-8 of their rms
// too low on average, a tenth of their own error (4.2e-7, 5.0e-7 from v_mfma_f32_32x32x2_f32), but ten times the error of
// their column means. A product whose column sums are wanted therefore takes its first operand with the odd rows negated
// and negates those rows' results, which moves them up by as much.
//
// The operands are split once by a packing pass, which also lays them out as the product reads them: blocks of 128 rows x
// 16 reduction indices, [plane][half of the reduction step][row] in 16-byte pieces of eight bf16 numbers -- the operand
// of one lane of one matrix instruction. A block is 12 KB of consecutive memory and lands in LDS as it is; rows and
// reduction are padded with zeros, so the product's loop has no edges.
//
// The product: a workgroup of 8 wavefronts owns 256 x 256 results, a wavefront 64 x 128 of them as 2 x 4 MFMA tiles (128
// accumulator registers); per reduction step of 16 it reads 18 16-byte operands per lane from LDS for 48 matrix
// instructions (1536 cycles of its SIMD), and the workgroup fetches 48 KB, half the bytes per result of a 128 x 128 tile.
// LDS is a ring of three steps (144 KB); operands go from memory to LDS directly (global_load_lds_dwordx4).
#include "common.hpp"
#include "split_gemm.hpp"

namespace ht {
namespace {

typedef float Acc16 __attribute__((ext_vector_type(16)));
typedef __bf16 Bf8 __attribute__((ext_vector_type(8)));
typedef unsigned short U16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplitThreads = 512;
constexpr int kPackRows = 128, kPackRed = 16;     // a packed block
constexpr int kBlockUnits = 3 * 2 * kPackRows;    // ... in 16-byte units
constexpr int kStepUnits = 4 * kBlockUnits;       // both operands of a workgroup's step
constexpr size_t kSplitLds = 3 * size_t(kStepUnits) * 16;

__device__ __forceinline__ uint32_t bf16_nearest(float v) {
  const uint32_t b = __float_as_uint(v);
  if ((b & 0x7f800000u) == 0x7f800000u) return (b >> 16) | ((b & 0xffffu) ? 0x40u : 0u);  // inf, NaN (kept a NaN)
  const uint32_t r = (b + 0x7fffu + ((b >> 16) & 1u)) >> 16;
  return (r & 0x7fffu) == 0x7f80u ? b >> 16 : r;  // the largest numbers are cut instead of rounded to infinity
}

__device__ __forceinline__ void split3(float v, uint32_t (&p)[3]) {
  p[0] = bf16_nearest(v);
  const bool finite = (p[0] & 0x7f80u) != 0x7f80u;
  const float r1 = finite ? v - __uint_as_float(p[0] << 16) : 0.f;
  p[1] = bf16_nearest(r1);
  p[2] = bf16_nearest(r1 - __uint_as_float(p[1] << 16));
}

// Element (row, red) of the operand; outside the operand 0.
struct PackSource {
  const float *p;
  long long ld;
  int rows, red;
  const double *row_sums;  // optional: the operand is the element minus float(row_sums[row] / count)
  double count;
  bool negate_odd;
};

// One thread per (row, reduction octet): eight consecutive reduction indices of a row, split and stored as one 16-byte
// piece per plane. RED_CONTIG: element at p[row * ld + red], lanes along the octets of two rows' neighbourhood; otherwise
// p[red * ld + row], lanes along the rows.
template <bool RED_CONTIG>
__global__ __launch_bounds__(256) void split_pack_kernel(PackSource s, U32x4 *__restrict__ dst, int steps,
                                                         int octs, long long octets) {
  // octs: octets of a row; for RED_CONTIG rounded up to a multiple of eight, the surplus skipped
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < octets; i += (long long)gridDim.x * 256) {
    // i numbers the octets of a row block: block, then (step, half) and row, in the order that makes the source's reads
    // and the destination's writes run along lanes as far as both can
    const long long block = i / ((long long)octs * kPackRows);
    const int in = int(i - block * ((long long)octs * kPackRows));
    int r, oct;
    if (RED_CONTIG) {
      // 8 rows x 8 octets per wavefront: 8 runs of 128 bytes are written per plane, 256-byte runs are read
      const int tile = in / 64, l = in % 64;
      const int rt = tile % (kPackRows / 8), ot = tile / (kPackRows / 8);
      r = rt * 8 + l % 8;
      oct = ot * 8 + l / 8;
    } else {
      r = in % kPackRows;
      oct = in / kPackRows;
    }
    if (oct >= steps * 2) continue;
    const long long row = block * kPackRows + r;
    const int red0 = oct * 8;
    float v[8];
    if (row < s.rows) {
      const float shift = s.row_sums ? float(s.row_sums[row] / s.count) : 0.f;
      if (RED_CONTIG) {
        const float *src = s.p + row * s.ld + red0;
        if (red0 + 8 <= s.red) {
          __builtin_memcpy(v, src, sizeof(v));
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = red0 + e < s.red ? src[e] : 0.f;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = red0 + e < s.red ? s.p[(long long)(red0 + e) * s.ld + row] : 0.f;
      }
      if (s.row_sums) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = red0 + e < s.red ? v[e] - shift : 0.f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
    }
    if (s.negate_odd && (row & 1)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = -v[e];
    }
    uint32_t part[3][4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint32_t q[3];
      split3(v[e], q);
#pragma unroll
      for (int k = 0; k < 3; ++k) part[k][e / 2] = e % 2 ? part[k][e / 2] | (q[k] << 16) : q[k];
    }
    U32x4 *out = dst + (block * steps + oct / 2) * kBlockUnits + (oct % 2) * kPackRows + r;
#pragma unroll
    for (int k = 0; k < 3; ++k) out[k * 2 * kPackRows] = U32x4{part[k][0], part[k][1], part[k][2], part[k][3]};
  }
}

struct SplitArgs {
  const U32x4 *A, *B;
  float *C;
  long long ldc;
  int n_i, n_j, steps;
  int tiles_i, tiles_j, rows_per_xcd;
  int splits, tiles;  // shares of the reduction; the tiles of one
  long long split_stride;
  bool symmetric;
  double *stats;
};

template <bool STATS>
__global__ __launch_bounds__(kSplitThreads, 2) void split_gemm_kernel(SplitArgs g) {
  extern __shared__ __align__(16) U32x4 lds[];
  int tile_i, tile_j, share = 0;
  if (g.splits > 1) {
    // few tiles, shared out: tile running fastest, the diagonal and what is above it only for a symmetric product; the
    // hardware deals consecutive workgroups to the XCDs in turn, which spreads every share over all of them
    int tile = int(blockIdx.x) % g.tiles;
    share = int(blockIdx.x) / g.tiles;
    if (g.symmetric) {
      tile_i = 0;
      while (tile >= g.tiles_j - tile_i) tile -= g.tiles_j - tile_i, ++tile_i;
      tile_j = tile_i + tile;
    } else {
      tile_i = tile / g.tiles_j;
      tile_j = tile - tile_i * g.tiles_j;
    }
  } else {
    if (!gemm_tile_of(int(blockIdx.x), g.tiles_i, g.tiles_j, g.rows_per_xcd, &tile_i, &tile_j)) return;
    if (g.symmetric && tile_j < tile_i) return;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * 128;
  const int lr = lane & 31, lk = lane >> 5;
  const int chunk = (g.steps + g.splits - 1) / g.splits;
  const int step0 = share * chunk, steps = min(chunk, g.steps - step0);
  if (steps <= 0) return;

  // what this wavefront fetches: 6 of the step's 48 pieces of 64 units, each inside one packed block
  const U32x4 *src[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const int c = wave + 8 * i, part = c / 12;
    const int rb = part < 2 ? 2 * tile_i + part : 2 * tile_j + part - 2;
    src[i] = (part < 2 ? g.A : g.B) + ((long long)rb * g.steps + step0) * kBlockUnits + (c % 12) * 64 + lane;
  }
  // Written as assembly because the compiler, which knows the builtin form for a write to LDS, would make every later LDS
  // read wait for it; here the waits are `landed` below. m0 cannot be named among what the assembly overwrites (it is reserved,
  // and the compiler sets it in front of each of its own uses); nothing else in this kernel uses it: LDS instructions of this
  // part need no m0.
  const uint32_t lds_base = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) U32x4 *)lds));
  auto fetch = [&](int buffer, int s) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const uint32_t to = __builtin_amdgcn_readfirstlane(lds_base + uint32_t(buffer * kStepUnits + (wave + 8 * i) * 64) * 16u);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                   :
                   : "s"(to), "v"(src[i] + (long long)s * kBlockUnits)
                   : "memory");
    }
  };

  Acc16 acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  // this lane's operand units inside a step: row r of a block of the operand, its half of the reduction step
  int ua[2], ub[4];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = wi + 32 * a + lr;
    ua[a] = (r / kPackRows) * kBlockUnits + lk * kPackRows + r % kPackRows;
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int r = wj + 32 * b + lr;
    ub[b] = (2 + r / kPackRows) * kBlockUnits + lk * kPackRows + r % kPackRows;
  }

  // Everything this wavefront requested has landed, and so has what the others did. Nothing may be moved across: hoisted
  // above the matrix instructions the wait would expose the transfer it is meant to hide. LDS reads are not waited for.
  auto landed = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  Bf8 a0[2], a1[2], a2[2], b0[4], b1[4], b2[4], na0[2], nb2[4];
  auto read_a = [&](Bf8 (&to)[2], const U32x4 *buf, int plane) {
#pragma unroll
    for (int a = 0; a < 2; ++a) to[a] = __builtin_bit_cast(Bf8, buf[ua[a] + plane * 2 * kPackRows]);
  };
  auto read_b = [&](Bf8 (&to)[4], const U32x4 *buf, int plane) {
#pragma unroll
    for (int b = 0; b < 4; ++b) to[b] = __builtin_bit_cast(Bf8, buf[ub[b] + plane * 2 * kPackRows]);
  };
  auto multiply = [&](const Bf8 (&x)[2], const Bf8 (&y)[4]) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[a], y[b], acc[a][b], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Step s multiplies out of LDS buffer s % 3. Its middle is the one barrier of a step: by then the operands of step s + 1,
  // requested a step ago, are in LDS, and every wavefront is done with buffer (s - 1) % 3, so the operands of step s + 2 are
  // requested into that one and the first operands of step s + 1 are read in the shadow of the step's second half.
  fetch(0, 0);
  landed();
  if (steps > 1) fetch(1, 1);
  // a wavefront of a tile on the edge that holds no results only moves operands
  const bool idle = tile_i * kSplitTile + wi >= g.n_i || tile_j * kSplitTile + wj >= g.n_j;
  if (idle) {
    for (int s = 0, cur = 0; s < steps; ++s) {
      const int nxt = cur == 2 ? 0 : cur + 1, after = nxt == 2 ? 0 : nxt + 1;
      landed();
      if (s + 2 < steps) fetch(after, s + 2);
      cur = nxt;
    }
  } else {
    read_a(a0, lds, 0);
    read_b(b2, lds, 2);
    int cur = 0;
    for (int s = 0; s < steps; ++s) {
      const int nxt = cur == 2 ? 0 : cur + 1, after = nxt == 2 ? 0 : nxt + 1;
      const U32x4 *buf = lds + cur * kStepUnits;
      read_a(a1, buf, 1);
      read_b(b1, buf, 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(a0, b2);
      read_a(a2, buf, 2);
      read_b(b0, buf, 0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(a1, b1);
      multiply(a0, b1);
      landed();
      if (s + 2 < steps) fetch(after, s + 2);
      if (s + 1 < steps) {
        read_a(na0, lds + nxt * kStepUnits, 0);
        read_b(nb2, lds + nxt * kStepUnits, 2);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(a2, b0);
      multiply(a1, b0);
      multiply(a0, b0);
#pragma unroll
      for (int a = 0; a < 2; ++a) a0[a] = na0[a];
#pragma unroll
      for (int b = 0; b < 4; ++b) b2[b] = nb2[b];
      cur = nxt;
    }
  }
  __syncthreads();

  // accumulator element e of lane l is C(row 8 * (e / 4) + 4 * (l / 32) + e % 4, column l % 32) of its 32 x 32 tile
  const int i0 = tile_i * kSplitTile + wi, j0 = tile_j * kSplitTile + wj;
  float *C = g.C + (long long)share * g.split_stride;
  double *part = reinterpret_cast<double *>(lds);  // STATS: [row wavefront][sum, sum of squares][column of the tile]
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int j = j0 + 32 * b + lr;
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int i = i0 + 32 * a + 8 * (e / 4) + 4 * lk + (e % 4);
        const float v = STATS && e % 2 ? 0.f - acc[a][b][e] : acc[a][b][e];  // (i is odd where e is)
        if (i < g.n_i && j < g.n_j) {
          C[(long long)i * g.ldc + j] = v;
          if (g.symmetric && tile_i != tile_j && g.splits == 1) C[(long long)j * g.ldc + i] = v;
        }
        if (STATS) {  // (rows beyond the matrix are zeros)
          s1 += double(v);
          s2 += double(v) * double(v);
        }
      }
    if (STATS) {
      s1 += __shfl_xor(s1, 32, kWave);
      s2 += __shfl_xor(s2, 32, kWave);
      if (lk == 0) {
        part[((wave >> 1) * 2 + 0) * kSplitTile + wj + 32 * b + lr] = s1;
        part[((wave >> 1) * 2 + 1) * kSplitTile + wj + 32 * b + lr] = s2;
      }
    }
  }
  if (STATS) {
    __syncthreads();
    const int col = threadIdx.x % kSplitTile, which = threadIdx.x / kSplitTile;  // 512 threads: column x (sum | squares)
    const int j = tile_j * kSplitTile + col;
    if (j < g.n_j) {
      double v = 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) v += part[(r * 2 + which) * kSplitTile + col];
      atomicAdd(g.stats + (long long)which * g.n_j + j, v);
    }
  }
}

}  // namespace

size_t split_pack_bytes(long long rows, long long red) {
  const long long blocks = (rows + kSplitTile - 1) / kSplitTile * (kSplitTile / kPackRows);
  const long long steps = (red + kPackRed - 1) / kPackRed;
  return size_t(blocks) * size_t(steps) * kBlockUnits * 16;
}

int split_pack(const float *src, long long ld, long long rows, long long red, bool red_contig, void *dst,
               hipStream_t stream, const double *row_sums, double count, bool negate_odd) {
  if (rows <= 0 || red <= 0) return HT_OK;
  if (rows > 0x7fffff00LL || red > 0x7fffff00LL) return fail(HT_ERR_RUNTIME, "Error: matrix product too large for this build.");
  PackSource s{src, ld, int(rows), int(red), row_sums, count, negate_odd};
  const long long blocks = (rows + kSplitTile - 1) / kSplitTile * (kSplitTile / kPackRows);
  const long long steps = (red + kPackRed - 1) / kPackRed;
  const long long octs = red_contig ? (steps * 2 + 7) / 8 * 8 : steps * 2;
  const long long total = blocks * octs * kPackRows;
  long long grid = (total + 255) / 256;
  if (grid > 64 * kNumCUs) grid = 64 * kNumCUs;
  if (red_contig)
    hipLaunchKernelGGL(split_pack_kernel<true>, dim3((unsigned)grid), dim3(256), 0, stream, s, static_cast<U32x4 *>(dst),
                       int(steps), int(octs), total);
  else
    hipLaunchKernelGGL(split_pack_kernel<false>, dim3((unsigned)grid), dim3(256), 0, stream, s, static_cast<U32x4 *>(dst),
                       int(steps), int(octs), total);
  HT_LAUNCH_CHECK("matrix product (packing)");
  return HT_OK;
}

// One workgroup occupies a CU, so a product of few tiles is shared out until every CU has one, as long as a share keeps
// 8 steps (10 us). Tiles of which only a sliver holds results finish early and are not counted.
int split_gemm_shares(long long n_i, long long n_j, long long n_r, bool symmetric) {
  auto tiles_of = [](long long n) { const long long t = (n + kSplitTile / 2) / kSplitTile; return t < 1 ? 1ll : t; };
  const long long ti = tiles_of(n_i), tj = tiles_of(n_j);
  const long long tiles = symmetric ? ti * (ti + 1) / 2 : ti * tj, steps = (n_r + kPackRed - 1) / kPackRed;
  long long want = kNumCUs / tiles;
  if (want > steps / 8) want = steps / 8;
  return want > 1 ? int(want) : 1;
}

int split_gemm(const void *A, const void *B, float *C, long long ldc, long long n_i, long long n_j, long long n_r,
               double *stats, hipStream_t stream, int splits, float *partials, bool symmetric) {
  if (n_i <= 0 || n_j <= 0 || n_r <= 0) return HT_OK;
  SplitArgs g;
  g.A = static_cast<const U32x4 *>(A);
  g.B = static_cast<const U32x4 *>(B);
  g.C = C;
  g.ldc = ldc;
  g.n_i = int(n_i), g.n_j = int(n_j), g.steps = int((n_r + kPackRed - 1) / kPackRed);
  g.tiles_i = int((n_i + kSplitTile - 1) / kSplitTile), g.tiles_j = int((n_j + kSplitTile - 1) / kSplitTile);
  g.rows_per_xcd = (g.tiles_i + kNumXCDs - 1) / kNumXCDs;
  g.splits = 1, g.split_stride = 0, g.symmetric = symmetric, g.stats = stats;
  long long slots = (long long)g.rows_per_xcd * g.tiles_j * kNumXCDs;
  g.tiles = g.tiles_i * g.tiles_j;
  if (splits > 1 && partials != nullptr) {
    g.splits = splits;
    g.split_stride = n_i * n_j;
    g.C = partials;
    g.ldc = n_j;
    if (symmetric) g.tiles = g.tiles_i * (g.tiles_i + 1) / 2;
    slots = (long long)g.tiles * splits;
  }
  if (slots > 0x7fffffffLL) return fail(HT_ERR_RUNTIME, "Error: matrix product too large for this build.");
  auto kernel = stats ? split_gemm_kernel<true> : split_gemm_kernel<false>;
  HT_HIP_CHECK(grant_lds(reinterpret_cast<const void *>(kernel)));
  hipLaunchKernelGGL(kernel, dim3((unsigned)slots), dim3(kSplitThreads), kSplitLds, stream, g);
  HT_LAUNCH_CHECK("matrix product (split operands)");
  if (g.splits > 1) {
    const int per = (g.steps + g.splits - 1) / g.splits;
    return sum_shares(partials, (g.steps + per - 1) / per, n_i * n_j, C, stream, symmetric ? int(n_j) : 0);
  }
  return HT_OK;
}

}  // namespace ht
