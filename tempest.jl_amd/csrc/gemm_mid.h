// The product's middle tiles (gemm_mid.hip): the arguments and the kernel for
// a tile, layouts and factor type, shared with the builder (gemm.hip).
#pragma once

#include <cstdint>

namespace thg {

struct MidArgs {
  const uint16_t* a;
  const uint16_t* b;
  void* c;               // result (parts: written by the fold)
  const void* d;         // C = D + A B where non-null, laid out at d_ld / d_batch
  const uint16_t* bias;  // bf16, per row of C, or null
  const uint16_t* aux;   // TH_EPI_GELU_BACKWARD: Z at aux_ld
  uint16_t* aux_out;     // TH_EPI_GELU: H, laid out as C
  float* parts;          // the fp32 sums of each part of K, or null: one part, finished in place
  float* row_parts;      // row sums per column block, [column block][m]
  float* loss_parts;     // loss per workgroup
  int64_t a_m, a_k, a_batch;
  int64_t b_k, b_n, b_batch;
  int64_t c_ld, c_batch;
  int64_t d_ld, d_batch;
  int64_t aux_ld;
  int64_t part_ld, part_split, part_batch;  // multiples of 4
  int32_t m, n, k;
  int32_t ksplit;   // K per part
  int32_t splits;   // parts
  int32_t tiles_m, tiles_n;
  int32_t result;   // TH_F32, TH_BF16 or TH_F16
  int32_t epilogue; // TH_EPI_*
  int32_t direct;   // the operands' whole steps may be loaded straight into LDS
};

constexpr int kFoldColumns = 32;  // columns a workgroup of the fold takes (128 rows)

// The kernel for tile (TH_TILE_128X128 .. TH_TILE_64X64) over fp16 or bf16
// factors, A k-contiguous (a_k == 1) or m-contiguous, B k-contiguous (b_k ==
// 1) or n-contiguous; nullptr for any other tile.  Rows and columns of the
// tile (bm, bn) and its LDS bytes go to *bm, *bn, *lds.
const void* mid_kernel(int tile, bool f16, bool a_kc, bool b_kc, int* bm, int* bn, int* lds);

// The fold of a product's parts of K: a workgroup per 128 rows x kFoldColumns
// columns (grid x, rows fastest) and product of the batch (grid z).
const void* mid_fold_kernel();

}  // namespace thg
