// Matrix products of float32 operands on the bf16 matrix cores (split_gemm.hip), and what the two product kernels share.
#pragma once
#include "common.hpp"

namespace ht {

// Workgroup -> result tile. Workgroups are dealt to the 8 XCDs (each with its own L2) round robin by index, so
// index % 8 names the L2 a workgroup will use. Every XCD takes a contiguous band of tile rows and walks it in panels
// of 8 tile columns, row by row inside a panel: the ~100 workgroups an XCD runs at a time then cover about 12 x 8
// tiles and share their 12 + 8 operand tiles through that L2, instead of each fetching its own pair.
// Returns false for a launch slot that has no tile (bands are padded to the same number of slots).
__host__ __device__ inline bool gemm_tile_of(int block, int tiles_i, int tiles_j, int rows_per_xcd, int *tile_i,
                                             int *tile_j) {
  const int xcd = block % kNumXCDs, slot = block / kNumXCDs;
  const int row0 = xcd * rows_per_xcd;
  const int rows = rows_per_xcd < tiles_i - row0 ? rows_per_xcd : tiles_i - row0;
  if (rows <= 0 || slot >= rows * tiles_j) return false;
  constexpr int kPanel = 8;
  const int full = tiles_j / kPanel;  // panels of the full width
  int panel = slot / (rows * kPanel), rem = slot - panel * (rows * kPanel), width = kPanel;
  if (panel >= full) {
    panel = full;
    rem = slot - full * (rows * kPanel);
    width = tiles_j - full * kPanel;
  }
  const int r = rem / width;
  *tile_i = row0 + r;
  *tile_j = panel * kPanel + (rem - r * width);
  return true;
}

// An operand [rows x red] split and laid out for split_gemm (16-byte aligned, split_pack_bytes): element (i, r) at
// src[i * ld + r] (red_contig) or src[r * ld + i], minus float(row_sums[i] / count) where row_sums is given; the elements of odd
// rows negated with negate_odd.
size_t split_pack_bytes(long long rows, long long red);
int split_pack(const float *src, long long ld, long long rows, long long red, bool red_contig, void *dst,
               hipStream_t stream, const double *row_sums = nullptr, double count = 1.0, bool negate_odd = false);
// Shares of the reduction with which a product of this size fills the device (1: its tiles do).
int split_gemm_shares(long long n_i, long long n_j, long long n_r, bool symmetric);

// C[i, j] = sum_r A(i, r) B(j, r), i < n_i, j < n_j, from packed operands with the same n_r. stats (optional): [2 n_j]
// doubles that receive the column sums of C and of its squares (added to what is there); A then comes packed with its odd
// rows negated. splits > 1 with partials (splits x n_i x n_j floats): the reduction is shared out, and the shares are summed
// in a fixed order.
// symmetric: A and B are the same operand; tiles below the diagonal are mirrored from above.
int split_gemm(const void *A, const void *B, float *C, long long ldc, long long n_i, long long n_j, long long n_r,
               double *stats, hipStream_t stream, int splits = 1, float *partials = nullptr, bool symmetric = false);

// dst[i] = shares[0][i] + shares[1][i] + ... in that order (n elements per share). mirror > 0: a share is a mirror x mirror
// matrix whose tiles (of split_gemm) below the diagonal were not computed; they are taken from above it.
int sum_shares(const float *shares, int count, long long n, float *dst, hipStream_t stream, int mirror = 0);
constexpr int kSplitTile = 256;  // result tile edge of split_gemm

}  // namespace ht
