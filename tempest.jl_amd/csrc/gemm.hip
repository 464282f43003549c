// th_build_gemm: a product's launch on the kernel its tile names (the
// 256 x 256 kernel in gemm_kernel.h, the middle tiles in gemm_mid.hip, the
// general kernel in gemm_general.hip), the parts of K summed, and the folds
// the epilogues leave: bias gradients and the loss.  th_gemm_tune measures
// the choices.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>

#include "gemm_kernel.h"
#include "gemm_mid.h"
#include "th_core.h"

namespace thg {
namespace {

struct SumArgs {
  const float* rows;       // parts x m
  uint16_t* out;           // m, bf16
  const float* loss_parts; // count, or null
  float* loss;
  int32_t m, parts, count;
};

// The folds an epilogue leaves: out[i] = sum over parts of rows[p, i], in
// part order, 256 rows a workgroup; and, in the last workgroup, the loss.
__global__ __launch_bounds__(256) void sum_epilogue(SumArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (blockIdx.x < (a.m + 255) / 256) {
    if (i < a.m) a.out[i] = bf16_bits(thd::sum_in_order(a.rows + i, a.m, a.parts));
    return;
  }
  __shared__ double lds[4];
  double s = 0.0;
  for (int j = threadIdx.x; j < a.count; j += 256) s += (double)a.loss_parts[j];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (threadIdx.x % 64 == 0) lds[threadIdx.x / 64] = s;
  __syncthreads();
  if (threadIdx.x == 0) a.loss[0] = (float)(lds[0] + lds[1] + lds[2] + lds[3]);
}

// The launch of sum_epilogue after an epilogue with row sums (`parts` x m at
// at_rows of the workspace) and, for the square loss, `count` loss partials.
void add_sums(th::Builder& b, const th_gemm_desc* d, uint64_t at_rows, int parts, uint64_t at_loss, int count) {
  const bool loss = d->epilogue == TH_EPI_SQUARE_LOSS;
  SumArgs s{nullptr, static_cast<uint16_t*>(d->row_sums), nullptr, d->loss, d->m, parts, count};
  const int k = b.kernel((const void*)sum_epilogue, loss ? "sum_rows_and_loss" : "sum_rows",
                         dim3((d->m + 255) / 256 + (loss ? 1 : 0)), dim3(256), 0, s);
  b.ref(6, k, TH_OFFSET(SumArgs, out));
  b.ws_ref(k, TH_OFFSET(SumArgs, rows), at_rows);
  if (loss) {
    b.ref(7, k, TH_OFFSET(SumArgs, loss));
    b.ws_ref(k, TH_OFFSET(SumArgs, loss_parts), at_loss);
  }
}

// The launch that folds parts of K (mid_fold): `g` as the parts were written,
// with what the result takes from `d` filled in here.
int add_fold(th::Builder& b, const th_gemm_desc* d, MidArgs g, uint64_t at_parts) {
  const bool accumulate = (d->flags & TH_GEMM_ACCUMULATE) != 0;
  g.c = d->c, g.c_ld = d->c_ld, g.c_batch = d->c_batch, g.result = d->c_dtype;
  g.d = accumulate ? d->d : nullptr;
  g.d_ld = d->d_ld ? d->d_ld : d->c_ld;
  g.d_batch = d->d_ld ? d->d_batch : d->c_batch;
  g.bias = static_cast<const uint16_t*>(d->bias);
  g.aux = static_cast<const uint16_t*>(d->aux), g.aux_ld = d->aux_ld;
  g.aux_out = static_cast<uint16_t*>(d->aux_out);
  g.m = d->m, g.n = d->n, g.epilogue = d->epilogue;
  const unsigned blocks = (unsigned)(((d->m + 127) / 128) * (int64_t)((d->n + kFoldColumns - 1) / kFoldColumns));
  const int k = b.kernel(mid_fold_kernel(), "sum_splits", dim3(blocks, 1, std::max(1, d->batch)), dim3(256), 0, g);
  b.ws_ref(k, TH_OFFSET(MidArgs, parts), at_parts);
  b.ref(2, k, TH_OFFSET(MidArgs, c));
  b.ref(3, k, TH_OFFSET(MidArgs, bias));
  b.ref(4, k, TH_OFFSET(MidArgs, aux));
  b.ref(5, k, TH_OFFSET(MidArgs, aux_out));
  b.ref(8, k, TH_OFFSET(MidArgs, d));
  return k;
}

bool aligned(const void* p, int bytes) { return (reinterpret_cast<uintptr_t>(p) % bytes) == 0; }

// An fp32 factor as three bf16 copies along K, for the bf16x3 products:
// x = hi + lo + (below lo), hi = bf16(x), lo = bf16(x - hi); A's copies are
// (hi, hi, lo) and B's (hi, lo, hi), so that the product of the two tripled
// operands is A_hi B_hi + A_hi B_lo + A_lo B_hi.  Each copy is k8 deep (k
// rounded up to 8, zeros past k); rows past `rows` (up to the destination's
// padded count) are zeros.
struct SplitArgs {
  const float* src;
  uint16_t* dst;
  int64_t s_r, s_k, s_batch;  // source strides along the rows (m or n), along k, between products
  int64_t d_r, d_k, d_batch;  // destination strides
  int64_t total;              // destination elements of one copy of one product: rows_pad x k8
  int32_t rows, rows_pad, k, k8;
  int32_t order;   // 0: (hi, hi, lo), 1: (hi, lo, hi)
  int32_t k_fast;  // 1: k is the destination's contiguous axis
};

__global__ __launch_bounds__(256) void split_bf16x3(SplitArgs a) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= a.total) return;
  const int64_t z = blockIdx.y;
  int64_t r, l;
  if (a.k_fast) r = e / a.k8, l = e % a.k8;
  else r = e % a.rows_pad, l = e / a.rows_pad;
  const float x = (r < a.rows && l < a.k) ? a.src[z * a.s_batch + r * a.s_r + l * a.s_k] : 0.0f;
  const uint16_t hi = bf16_bits(x);
  const uint16_t lo = bf16_bits(x - bf16_float(hi));
  uint16_t* d = a.dst + z * a.d_batch + r * a.d_r + l * a.d_k;
  const int64_t step = (int64_t)a.k8 * a.d_k;
  d[0] = hi;
  d[step] = a.order == 0 ? hi : lo;
  d[2 * step] = a.order == 0 ? lo : hi;
}

}  // namespace
}  // namespace thg

using namespace thg;

// Whether the bf16 tile kernel takes the descriptor: bf16 factors, a unit
// stride on each operand, sizes and strides multiples of 8, 16-byte operands.
bool tile_kernel_takes(const th_gemm_desc* d) {
  if (d->flags & (TH_GEMM_F32_FACTORS | TH_GEMM_F16_FACTORS)) return false;
  if (d->c_dtype != TH_BF16 && d->c_dtype != TH_F32) return false;
  if (d->m % 8 || d->n % 8 || d->k % 8) return false;
  const bool ua = d->a_k == 1 || d->a_m == 1, ub = d->b_k == 1 || d->b_n == 1;
  if (!ua || !ub) return false;
  const int64_t sa = d->a_k == 1 ? d->a_m : d->a_k, sb = d->b_k == 1 ? d->b_n : d->b_k;
  if (sa % 8 || sb % 8 || d->c_ld % 8 || d->c_ld < d->m) return false;
  if (d->batch > 1 && (d->a_batch % 8 || d->b_batch % 8 || d->c_batch % 8)) return false;
  return aligned(d->a, 16) && aligned(d->b, 16) && aligned(d->c, 16);
}

// Whether the middle tiles take the descriptor: half factors, a unit stride
// on each operand, the other strides multiples of 8, 16-byte operands, a
// plain product with a result of the factors' type or fp32.
static bool mid_takes(const th_gemm_desc* d) {
  if (d->flags & TH_GEMM_F32_FACTORS) return false;
  if (d->epilogue != TH_EPI_STORE) return false;
  const int factor = (d->flags & TH_GEMM_F16_FACTORS) ? TH_F16 : TH_BF16;
  if (d->c_dtype != factor && d->c_dtype != TH_F32) return false;
  if (!(d->a_k == 1 || d->a_m == 1) || !(d->b_k == 1 || d->b_n == 1)) return false;
  const int64_t sa = d->a_k == 1 ? d->a_m : d->a_k, sb = d->b_k == 1 ? d->b_n : d->b_k;
  if (sa % 8 || sb % 8 || d->c_ld < d->m) return false;
  if (d->batch > 1 && (d->a_batch % 8 || d->b_batch % 8)) return false;
  return aligned(d->a, 16) && aligned(d->b, 16);
}

constexpr int kMidStep = 64;  // parts of K on the middle tiles are multiples of it

static int mid_rows(int tile) { return tile == TH_TILE_64X128 || tile == TH_TILE_64X64 ? 64 : 128; }
static int mid_cols(int tile) { return tile == TH_TILE_128X64 || tile == TH_TILE_64X64 ? 64 : 128; }

static int64_t tiles_of(const th_gemm_desc* d, int bm, int bn) {
  return (int64_t)((d->m + bm - 1) / bm) * ((d->n + bn - 1) / bn) * std::max(1, d->batch);
}

// The parts of K a tile takes when the caller leaves them to the builder:
// enough for about 256 workgroups where the tiles alone give fewer than 128,
// each part at least `least` deep (1024 on the 256 x 256 kernel, 512 on the
// middle tiles).
static int auto_splits(const th_gemm_desc* d, int tile) {
  if (d->epilogue != TH_EPI_STORE) return 1;
  const bool big = tile == TH_TILE_256;
  const int64_t tiles = big ? tiles_of(d, kTile, kTile) : tiles_of(d, mid_rows(tile), mid_cols(tile));
  const int least = big ? 1024 : 512;
  if (tiles >= 128 || d->k < 2 * least) return 1;
  return (int)std::max<int64_t>(1, std::min<int64_t>((256 + tiles - 1) / tiles, d->k / least));
}

// Whether the 256 x 256 kernel runs its direct sweep: whole tiles of C, whole
// steps of K, 32-bit byte offsets.
static bool interior_256(const th_gemm_desc* d) {
  const int64_t a_bytes = 2 * (d->a_k == 1 ? (int64_t)(d->m - 1) * d->a_m + d->k : (int64_t)(d->k - 1) * d->a_k + d->m);
  const int64_t b_bytes = 2 * (d->b_k == 1 ? (int64_t)(d->n - 1) * d->b_n + d->k : (int64_t)(d->k - 1) * d->b_k + d->n);
  return d->m % kTile == 0 && d->n % kTile == 0 && d->k % kDepth == 0 && a_bytes <= 0x7fffffff && b_bytes <= 0x7fffffff;
}

// Microseconds a product takes on a tile with K in `splits` parts, fitted to
// what the kernels measure on this device (2.4 GHz, 256 CUs): a step of 64 of
// K takes `alone` us with one workgroup on a CU and `pair` with two (the 256 x
// 256 kernel has room for one), the end of a tile `end`; a launch 3; the fold
// of parts 3 and their bytes at 8 TB/s.  Steps measured at 768 x 1024 x 3072,
// 4096 x 512 x 4096, 2048^3, 4096^3, 4096 x 2048 x 16384: 64 x 64 0.27 / 0.43 to 0.55,
// 128 x 64 0.44 / 0.75, 128 x 128 0.75 / 1.0 to 1.05, 256 x 256 1.55 to 1.8
// (over twice that where its tiles are ragged: 2000 x 8000 x 520 58.6 us
// against 33.8 on 128 x 128 tiles).  The estimate only has to order them.
static double estimate(const th_gemm_desc* d, int tile, int splits) {
  struct Cost { double alone, pair, end; };
  const Cost c = tile == TH_TILE_256       ? (interior_256(d) ? Cost{1.7, 1.7, 5.0} : Cost{4.0, 4.0, 8.0})
                 : tile == TH_TILE_128X128 ? Cost{0.75, 1.05, 2.0}
                 : tile == TH_TILE_64X64   ? Cost{0.27, 0.5, 0.5}
                                           : Cost{0.44, 0.75, 1.0};
  const bool big = tile == TH_TILE_256;
  const int64_t work = (big ? tiles_of(d, kTile, kTile) : tiles_of(d, mid_rows(tile), mid_cols(tile))) * splits;
  const int64_t room = big ? 256 : 512;  // workgroups the device holds
  const double steps = ((d->k + splits - 1) / splits + 63) / 64;
  const int64_t rounds = work / room, rest = work % room;
  double t = 3.0 + rounds * (steps * c.pair + c.end);
  if (rest > 0) t += steps * (rest <= 256 ? c.alone : c.pair) + c.end;
  if (splits > 1 || (big && (d->flags & TH_GEMM_ACCUMULATE)))
    t += 3.0 + 8.0 * splits * std::max(1, d->batch) * (double)d->m * d->n / 8e6;
  return t;
}

// Where the library chooses the tile: the kernel, and unless the caller
// names them the parts of K (at least 256 deep), with the least estimate
// among the 256 x 256 kernel (parts as it splits by itself) and the middle
// tiles, where they take the product; else the general kernel.  The middle
// tiles take what the 256 x 256 kernel takes, fused epilogues included, which
// then run in the fold of the parts.
static int choose_tile(const th_gemm_desc* d, int* splits) {
  const bool big = tile_kernel_takes(d), mid = d->epilogue == TH_EPI_STORE ? mid_takes(d) : big;
  *splits = d->splits > 0 ? d->splits : 1;
  if (!big && !mid) return TH_TILE_GENERAL;
  int best = TH_TILE_GENERAL;
  double least = INFINITY;
  auto consider = [&](int tile, int s) {
    const double t = estimate(d, tile, s);
    if (t < least) least = t, best = tile, *splits = s;
  };
  const int asked = d->splits;
  if (big) {
    const int s = asked > 0 ? asked : auto_splits(d, TH_TILE_256);
    // An fp32 result with a bias stays refused where the 256 x 256 tiles fill the device.
    if (d->c_dtype == TH_F32 && d->bias && tiles_of(d, kTile, kTile) * s >= 128) return *splits = s, TH_TILE_256;
    consider(TH_TILE_256, s);
  }
  if (mid)
    for (int t : {TH_TILE_128X128, TH_TILE_64X128, TH_TILE_128X64, TH_TILE_64X64})
      for (int s = 1; s <= 16 && (s == 1 || (asked == 0 && d->k / s >= 256)); ++s) consider(t, asked > 0 ? asked : s);
  return best;
}

static int build_tile256(const th_gemm_desc* d, th_launch** out);
static int build_mid(const th_gemm_desc* d, int tile, int splits, th_launch** out);

// What a fused epilogue needs, on whichever kernel.
static int check_epilogue(const th_gemm_desc* d) {
  const int epi = d->epilogue;
  if (epi == TH_EPI_STORE) return TH_OK;
  TH_REQUIRE(d->c_dtype == TH_BF16, "th_build_gemm: fused epilogues write bf16");
  TH_REQUIRE(!d->bias || aligned(d->bias, 8), "th_build_gemm: bias must be 8-byte aligned");
  TH_REQUIRE(d->splits <= 1, "th_build_gemm: only a plain product splits K");
  if (epi == TH_EPI_GELU)
    TH_REQUIRE(d->aux_out && d->bias && aligned(d->aux_out, 8), "th_build_gemm: GELU needs bias and aux_out");
  if (epi == TH_EPI_SQUARE_LOSS)
    TH_REQUIRE(d->bias && d->loss && d->row_sums, "th_build_gemm: the square loss needs bias, loss, row_sums");
  if (epi == TH_EPI_GELU_BACKWARD)
    TH_REQUIRE(d->aux && d->row_sums && d->aux_ld >= d->m && d->aux_ld % 4 == 0 && aligned(d->aux, 8),
               "th_build_gemm: the GELU backward needs aux (8-byte aligned, ld >= m, ld % 4 == 0) and row_sums");
  return TH_OK;
}

static int build_bf16x3(const th_gemm_desc* d, th_launch** out);

extern "C" int th_build_gemm(const th_gemm_desc* d, th_launch** out) {
  if (int r = th::require_ready()) return r;
  *out = nullptr;
  TH_REQUIRE(d != nullptr, "th_build_gemm: null descriptor");
  TH_REQUIRE(d->m >= 1 && d->n >= 1 && d->k >= 1, "th_build_gemm: m, n, k must be positive");
  TH_REQUIRE(d->a && d->b && d->c, "th_build_gemm: null operand");
  TH_REQUIRE((d->flags & ~(TH_GEMM_F32_FACTORS | TH_GEMM_F16_FACTORS | TH_GEMM_ACCUMULATE | TH_GEMM_BF16X3)) == 0 &&
                 (d->flags & (TH_GEMM_F32_FACTORS | TH_GEMM_F16_FACTORS)) != (TH_GEMM_F32_FACTORS | TH_GEMM_F16_FACTORS),
             "th_build_gemm: unknown flags");
  const bool accumulate = (d->flags & TH_GEMM_ACCUMULATE) != 0;
  TH_REQUIRE(!accumulate || d->d, "th_build_gemm: accumulating needs d");
  const int epi = d->epilogue;
  TH_REQUIRE(epi >= TH_EPI_STORE && epi <= TH_EPI_GELU_BACKWARD, "th_build_gemm: unknown epilogue");
  TH_REQUIRE(epi == TH_EPI_STORE || ((d->batch <= 1) && !accumulate),
             "th_build_gemm: fused epilogues take one product and nothing to add");
  TH_REQUIRE(d->tile >= TH_TILE_AUTO && d->tile <= TH_TILE_GENERAL, "th_build_gemm: unknown tile");
  TH_REQUIRE(d->splits >= 0, "th_build_gemm: splits must be >= 0");
  if (d->flags & TH_GEMM_BF16X3) return build_bf16x3(d, out);
  int splits = 0;
  const int tile = d->tile == TH_TILE_AUTO ? choose_tile(d, &splits) : d->tile;
  if (tile == TH_TILE_GENERAL) return th::build_gemm_general(d, out);
  if (tile == TH_TILE_256) {
    TH_REQUIRE(tile_kernel_takes(d),
               "th_build_gemm: the 256 x 256 kernel takes bf16 factors with a unit stride on each operand, m, n, k "
               "and the other strides multiples of 8 and 16-byte aligned operands");
    return build_tile256(d, out);
  }
  if (d->tile == TH_TILE_AUTO) {
    if (int r = check_epilogue(d)) return r;
    return build_mid(d, tile, splits, out);
  }
  TH_REQUIRE(mid_takes(d),
             "th_build_gemm: the middle tiles take bf16 or fp16 factors with a unit stride on each operand, the other "
             "strides multiples of 8, 16-byte aligned operands, TH_EPI_STORE and a result of the factors' type or fp32");
  return build_mid(d, tile, d->splits > 0 ? d->splits : auto_splits(d, tile), out);
}

static int build_tile256(const th_gemm_desc* d, th_launch** out) {
  const int M = d->m, N = d->n, K = d->k;
  const int batch = d->batch > 0 ? d->batch : 1;
  const bool accumulate = (d->flags & TH_GEMM_ACCUMULATE) != 0;
  const int epi = d->epilogue;
  const int la = d->a_k == 1 ? kK : kMN;
  const int lb = d->b_k == 1 ? kK : kMN;
  if (int r = check_epilogue(d)) return r;
  TH_REQUIRE(!d->bias || aligned(d->bias, 8), "th_build_gemm: bias must be 8-byte aligned");
  TH_REQUIRE(!(d->c_dtype == TH_F32 && d->bias), "th_build_gemm: an fp32 result takes no bias");
  const int tiles_m = (M + kTile - 1) / kTile, tiles_n = (N + kTile - 1) / kTile;
  // K split over parts (each a multiple of 64 deep) where asked, or where the
  // tiles alone would leave most CUs idle.
  int splits = d->splits > 0 ? d->splits : auto_splits(d, TH_TILE_256);
  TH_REQUIRE(splits == 1 || epi == TH_EPI_STORE, "th_build_gemm: only a plain product splits K");
  int ksplit = K;
  if (splits > 1) {
    ksplit = ((K + splits - 1) / splits + kDepth - 1) / kDepth * kDepth;
    splits = (K + ksplit - 1) / ksplit;
  }
  TH_REQUIRE(splits <= 65535 && batch <= 65535, "th_build_gemm: grid too large");
  // Parts and what is added go through an fp32 workspace and a second launch.
  const bool staged = splits > 1 || accumulate;
  // Ragged tiles and operands past 2 GiB take the bounds-checked kernel,
  // which addresses with 64-bit pointers.
  const bool check = !interior_256(d) || ksplit % kDepth;
  const void* fn = nullptr;
  const char* name = "";
  switch (epi) {
    case TH_EPI_STORE:
      fn = (staged || d->c_dtype == TH_F32) ? gemm_store_f32(la, lb, check) : gemm_store(la, lb, check);
      name = staged ? "gemm_bf16_parts_f32" : d->c_dtype == TH_F32 ? "gemm_bf16_store_f32" : "gemm_bf16_store";
      break;
    case TH_EPI_GELU: fn = gemm_gelu(la, lb, check), name = "gemm_bf16_gelu"; break;
    case TH_EPI_SQUARE_LOSS: fn = gemm_square_loss(la, lb, check), name = "gemm_bf16_square_loss"; break;
    default: fn = gemm_gelu_backward(la, lb, check), name = "gemm_bf16_gelu_backward"; break;
  }
  const size_t lds_bytes = check ? kLds : kLdsDirect;
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));

  th::Builder b("gemm_bf16", 9);
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(d->a);
  g.b = static_cast<const uint16_t*>(d->b);
  g.c = d->c;
  g.bias = staged ? nullptr : static_cast<const uint16_t*>(d->bias);
  g.aux = static_cast<const uint16_t*>(d->aux);
  g.aux_out = static_cast<uint16_t*>(d->aux_out);
  g.a_o = la == kK ? d->a_m : 1;
  g.a_k = la == kK ? 1 : d->a_k;
  g.b_o = lb == kK ? d->b_n : 1;
  g.b_k = lb == kK ? 1 : d->b_k;
  g.ldc = d->c_ld;
  g.aux_ld = d->aux_ld;
  g.m = M;
  g.n = N;
  g.k = K;
  g.tiles_m = tiles_m;
  g.tiles_n = tiles_n;
  g.a_batch = d->a_batch;
  g.b_batch = d->b_batch;
  g.c_batch = d->c_batch;
  g.c_split = 0;
  g.ksplit = ksplit;
  const int64_t mn = (int64_t)M * N;
  // Workspace: the fp32 sums of each part of K (staged products), then the
  // epilogue's per-tile row sums and loss partials.
  uint64_t at_parts = 0, at_sums = 0;
  if (staged) {
    at_parts = b.workspace((uint64_t)batch * splits * mn * sizeof(float));
    g.c = nullptr;
    g.ldc = M;
    g.c_batch = (int64_t)splits * mn;
    g.c_split = mn;
  }
  const bool sums = epi == TH_EPI_SQUARE_LOSS || epi == TH_EPI_GELU_BACKWARD;
  const int blocks = tiles_m * tiles_n;
  if (sums) at_sums = b.workspace(((uint64_t)2 * tiles_n * M + (uint64_t)4 * blocks) * sizeof(float));
  int k = b.kernel(fn, name, dim3(blocks, splits, batch), dim3(kThreads), (uint32_t)lds_bytes, g);
  if (staged) b.ws_ref(k, TH_OFFSET(GemmArgs, c), at_parts);
  if (sums) b.ws_ref(k, TH_OFFSET(GemmArgs, partial), at_sums);
  b.ref(0, k, TH_OFFSET(GemmArgs, a));
  b.ref(1, k, TH_OFFSET(GemmArgs, b));
  if (!staged) b.ref(2, k, TH_OFFSET(GemmArgs, c));
  if (!staged) b.ref(3, k, TH_OFFSET(GemmArgs, bias));
  b.ref(4, k, TH_OFFSET(GemmArgs, aux));
  b.ref(5, k, TH_OFFSET(GemmArgs, aux_out));
  for (int v : {0, 1, 2}) b.align(v, 16);
  for (int v : {3, 4, 5}) b.align(v, 8);
  if (staged) {
    MidArgs f{};
    f.part_ld = M, f.part_split = mn, f.part_batch = (int64_t)splits * mn, f.splits = splits;
    add_fold(b, d, f, at_parts);
  }
  if (sums) add_sums(b, d, at_sums, 2 * tiles_n, at_sums + (uint64_t)2 * tiles_n * M * sizeof(float), 4 * blocks);
  const double mm = M, nn = N, kk = K, bb = batch;
  const double cbytes = d->c_dtype == TH_F32 ? 4 : 2;
  double bytes = bb * (2.0 * (mm * kk + kk * nn) + cbytes * mm * nn * (accumulate ? 2 : 1));
  if (epi == TH_EPI_GELU || epi == TH_EPI_GELU_BACKWARD) bytes += 2.0 * mm * nn;
  b.work(bytes, 2.0 * bb * mm * nn * kk, (int64_t)blocks * splits * batch);
  *out = b.release();
  return TH_OK;
}

// The middle tiles: one launch of the tile kernel, for parts of K a second
// that folds them, and for an epilogue with folds a last one that ends them.
static int build_mid(const th_gemm_desc* d, int tile, int splits, th_launch** out) {
  const int M = d->m, N = d->n, K = d->k;
  const int batch = d->batch > 0 ? d->batch : 1;
  const bool accumulate = (d->flags & TH_GEMM_ACCUMULATE) != 0;
  const bool f16 = (d->flags & TH_GEMM_F16_FACTORS) != 0;
  int bm = 0, bn = 0, lds = 0;
  const bool a_kc = d->a_k == 1, b_kc = d->b_k == 1;
  const void* fn = mid_kernel(tile, f16, a_kc, b_kc, &bm, &bn, &lds);
  TH_REQUIRE(fn != nullptr, "th_build_gemm: unknown tile");
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  const int64_t tiles_m = (M + bm - 1) / bm, tiles_n = (N + bn - 1) / bn;
  TH_REQUIRE(tiles_m * tiles_n <= 0x7fffffff, "th_build_gemm: grid too large");
  int ksplit = K;
  if (splits > 1) {
    ksplit = ((K + splits - 1) / splits + kMidStep - 1) / kMidStep * kMidStep;
    splits = (K + ksplit - 1) / ksplit;
  }
  TH_REQUIRE(splits <= 65535 && batch <= 65535, "th_build_gemm: grid too large");
  const bool staged = splits > 1;
  const bool sums = d->epilogue >= TH_EPI_SQUARE_LOSS;
  th::Builder b("gemm_mid", 9);
  MidArgs g{};
  g.a = static_cast<const uint16_t*>(d->a);
  g.b = static_cast<const uint16_t*>(d->b);
  g.a_m = d->a_m, g.a_k = d->a_k, g.a_batch = d->a_batch;
  g.b_k = d->b_k, g.b_n = d->b_n, g.b_batch = d->b_batch;
  g.m = M, g.n = N, g.k = K, g.ksplit = ksplit, g.splits = splits;
  g.tiles_m = (int32_t)tiles_m, g.tiles_n = (int32_t)tiles_n, g.epilogue = d->epilogue;
  // Direct loads take 16-byte chunks that lie inside a row or outside all of
  // them, at 32-bit byte offsets.
  const int64_t a_bytes = 2 * (a_kc ? (int64_t)(M - 1) * d->a_m + K : (int64_t)(K - 1) * d->a_k + M);
  const int64_t b_bytes = 2 * (b_kc ? (int64_t)(N - 1) * d->b_n + K : (int64_t)(K - 1) * d->b_k + N);
  g.direct = (a_kc || M % 8 == 0) && (b_kc || N % 8 == 0) && a_bytes <= 0x7fffffff && b_bytes <= 0x7fffffff &&
             d->a_m >= 0 && d->a_k >= 0 && d->b_n >= 0 && d->b_k >= 0;
  uint64_t at_parts = 0, at_rows = 0, at_loss = 0;
  if (staged) {
    // Each part's fp32 sums, [batch][part][n][m], m padded to 8.
    g.part_ld = (M + 7) / 8 * 8, g.part_split = g.part_ld * N, g.part_batch = g.part_split * splits;
    at_parts = b.workspace((uint64_t)batch * g.part_batch * sizeof(float));
  } else {
    g.c = d->c, g.c_ld = d->c_ld, g.c_batch = d->c_batch, g.result = d->c_dtype;
    g.d = accumulate ? d->d : nullptr;
    g.d_ld = d->d_ld ? d->d_ld : d->c_ld;
    g.d_batch = d->d_ld ? d->d_batch : d->c_batch;
    g.bias = static_cast<const uint16_t*>(d->bias);
    g.aux = static_cast<const uint16_t*>(d->aux), g.aux_ld = d->aux_ld;
    g.aux_out = static_cast<uint16_t*>(d->aux_out);
  }
  // Column blocks of row sums and workgroups of loss partials, as the kernel that finishes has them.
  const int nb = staged ? (N + kFoldColumns - 1) / kFoldColumns : (int)tiles_n;
  const int64_t blocks = staged ? (int64_t)((M + 127) / 128) * nb : tiles_m * tiles_n;
  if (sums) {
    at_rows = b.workspace((uint64_t)nb * M * sizeof(float));
    at_loss = b.workspace((uint64_t)blocks * sizeof(float));
  }
  const char* name = staged ? "gemm_mid_parts_f32"
                     : d->epilogue == TH_EPI_STORE       ? "gemm_mid"
                     : d->epilogue == TH_EPI_GELU        ? "gemm_mid_gelu"
                     : d->epilogue == TH_EPI_SQUARE_LOSS ? "gemm_mid_square_loss"
                                                         : "gemm_mid_gelu_backward";
  const int k = b.kernel(fn, name, dim3((unsigned)(tiles_m * tiles_n), splits, batch), dim3(256), (uint32_t)lds, g);
  b.ref(0, k, TH_OFFSET(MidArgs, a));
  b.ref(1, k, TH_OFFSET(MidArgs, b));
  b.align(0, 16);
  b.align(1, 16);
  int last = k;
  if (staged) {
    b.ws_ref(k, TH_OFFSET(MidArgs, parts), at_parts);
    last = add_fold(b, d, g, at_parts);
  } else {
    b.ref(2, k, TH_OFFSET(MidArgs, c));
    b.ref(3, k, TH_OFFSET(MidArgs, bias));
    b.ref(4, k, TH_OFFSET(MidArgs, aux));
    b.ref(5, k, TH_OFFSET(MidArgs, aux_out));
    b.ref(8, k, TH_OFFSET(MidArgs, d));
  }
  if (sums) {
    b.ws_ref(last, TH_OFFSET(MidArgs, row_parts), at_rows);
    b.ws_ref(last, TH_OFFSET(MidArgs, loss_parts), at_loss);
    add_sums(b, d, at_rows, nb, at_loss, (int)blocks);
  }
  if (d->epilogue != TH_EPI_STORE) {  // as the 256 x 256 kernel asks of a fused product
    b.align(2, 16);
    for (int v : {3, 4, 5}) b.align(v, 8);
  }
  const double mm = M, nn = N, kk = K, bb = batch;
  const double cbytes = d->c_dtype == TH_F32 ? 4 : 2;
  double bytes = bb * (2.0 * (mm * kk + kk * nn) + cbytes * mm * nn * (accumulate ? 2 : 1));
  if (d->epilogue == TH_EPI_GELU || d->epilogue == TH_EPI_GELU_BACKWARD) bytes += 2.0 * mm * nn;
  b.work(bytes, 2.0 * bb * mm * nn * kk, tiles_m * tiles_n * splits * batch);
  *out = b.release();
  return TH_OK;
}

// fp32 factors as split bf16 on the bf16 tile kernels (TH_GEMM_BF16X3): each
// factor becomes three bf16 copies along K (split_bf16x3) in the launch's
// workspace, and one product over 3 k8 sums A_hi B_hi + A_hi B_lo + A_lo B_hi
// in fp32 — the MI355X counterpart of the reference's :tf32x3
// (src/Compiler/runtime/target.jl:42-44, ext/cuBLASExt.jl:61-65).  The
// launch is the two split kernels followed by the inner product's kernels;
// the inner product's operands point into the workspace.
static int build_bf16x3(const th_gemm_desc* d, th_launch** out) {
  TH_REQUIRE(d->flags & TH_GEMM_F32_FACTORS, "th_build_gemm: TH_GEMM_BF16X3 splits fp32 factors");
  TH_REQUIRE(d->epilogue == TH_EPI_STORE && !d->bias && d->c_dtype == TH_F32,
             "th_build_gemm: a bf16x3 product stores an fp32 result, with no epilogue or bias");
  TH_REQUIRE(d->tile == TH_TILE_AUTO || (d->tile >= TH_TILE_256 && d->tile <= TH_TILE_64X64),
             "th_build_gemm: a bf16x3 product runs on the bf16 tile kernels");
  const int batch = d->batch > 0 ? d->batch : 1;
  const int M = d->m, N = d->n, K = d->k;
  const int k8 = (K + 7) / 8 * 8, m8 = (M + 7) / 8 * 8, n8 = (N + 7) / 8 * 8;
  TH_REQUIRE((int64_t)3 * k8 <= 0x7fffffff, "th_build_gemm: K too large");
  // The tripled operands, dense, with the fp32 operand's unit-stride axis kept.
  th_gemm_desc in = *d;
  in.flags = d->flags & TH_GEMM_ACCUMULATE;
  in.k = 3 * k8;
  const bool a_kfast = d->a_k == 1 && d->a_m != 1;
  const bool b_kfast = d->b_k == 1 && d->b_n != 1;
  SplitArgs sa{}, sb{};
  sa.rows = M, sa.k = K, sa.k8 = k8, sa.order = 0, sa.k_fast = a_kfast;
  sa.s_r = d->a_m, sa.s_k = d->a_k, sa.s_batch = d->a_batch;
  if (a_kfast) sa.rows_pad = M, sa.d_r = 3 * k8, sa.d_k = 1, in.a_m = 3 * k8, in.a_k = 1;
  else sa.rows_pad = m8, sa.d_r = 1, sa.d_k = m8, in.a_m = 1, in.a_k = m8;
  sa.total = (int64_t)sa.rows_pad * k8;
  sa.d_batch = 3 * sa.total;
  sb.rows = N, sb.k = K, sb.k8 = k8, sb.order = 1, sb.k_fast = b_kfast;
  sb.s_r = d->b_n, sb.s_k = d->b_k, sb.s_batch = d->b_batch;
  if (b_kfast) sb.rows_pad = N, sb.d_r = 3 * k8, sb.d_k = 1, in.b_n = 3 * k8, in.b_k = 1;
  else sb.rows_pad = n8, sb.d_r = 1, sb.d_k = n8, in.b_n = 1, in.b_k = n8;
  sb.total = (int64_t)sb.rows_pad * k8;
  sb.d_batch = 3 * sb.total;
  in.a_batch = sa.d_batch, in.b_batch = sb.d_batch;
  // Stand-ins the inner build checks for alignment; the workspace replaces them.
  in.a = reinterpret_cast<const void*>(uintptr_t(256));
  in.b = reinterpret_cast<const void*>(uintptr_t(256));
  th_launch* inner = nullptr;
  if (int r = th_build_gemm(&in, &inner)) return r;
  const uint64_t a_bytes = (uint64_t)batch * sa.d_batch * 2, b_bytes = (uint64_t)batch * sb.d_batch * 2;
  th::Builder bl("gemm_bf16x3", 9);
  const uint64_t at_a = bl.workspace(a_bytes), at_b = bl.workspace(b_bytes);
  const uint64_t at_inner = bl.workspace(inner->ws_bytes);
  sa.src = static_cast<const float*>(d->a), sb.src = static_cast<const float*>(d->b);
  const int ka = bl.kernel((const void*)split_bf16x3, "split_bf16x3_a", dim3((unsigned)((sa.total + 255) / 256), batch),
                           dim3(256), 0, sa);
  const int kb = bl.kernel((const void*)split_bf16x3, "split_bf16x3_b", dim3((unsigned)((sb.total + 255) / 256), batch),
                           dim3(256), 0, sb);
  bl.ref(0, ka, TH_OFFSET(SplitArgs, src));
  bl.ref(1, kb, TH_OFFSET(SplitArgs, src));
  bl.ws_ref(ka, TH_OFFSET(SplitArgs, dst), at_a);
  bl.ws_ref(kb, TH_OFFSET(SplitArgs, dst), at_b);
  th_launch* l = bl.release();
  // The inner product's kernels after the splits: its operands a and b
  // become the tripled copies in the workspace, its other values ours.
  const int base = (int)l->kernels.size();
  for (const th::Kernel& k : inner->kernels) l->kernels.push_back(k);
  for (int v = 0; v < (int)inner->values.size() && v < (int)l->values.size(); ++v)
    for (const th::Ref& r : inner->values[v]) {
      if (v == 0) l->ws_refs.push_back(th::WsRef{base + r.kernel, r.offset, at_a});
      else if (v == 1) l->ws_refs.push_back(th::WsRef{base + r.kernel, r.offset, at_b});
      else l->values[v].push_back(th::Ref{base + r.kernel, r.offset});
    }
  for (const th::WsRef& w : inner->ws_refs) l->ws_refs.push_back(th::WsRef{base + w.kernel, w.offset, at_inner + w.at});
  for (int v = 2; v < (int)inner->align.size() && v < (int)l->align.size(); ++v) l->align[v] = inner->align[v];
  l->work.kernels = (int32_t)l->kernels.size();
  l->work.flops = 2.0 * batch * (double)M * N * K;
  l->work.bytes = batch * (4.0 * ((double)M * K + (double)K * N) + 4.0 * (double)M * N *
                          ((d->flags & TH_GEMM_ACCUMULATE) ? 2 : 1));
  l->work.blocks = inner->work.blocks;
  l->name = "gemm_bf16x3 (fp32 factors as hi + lo bf16, K tripled): " + inner->name;
  inner->kernels.clear();
  th_launch_destroy(inner);
  *out = l;
  return TH_OK;
}

// ---- measuring the choices -------------------------------------------------------

namespace {

struct Tuned {
  int32_t tile, splits;
  double seconds;
};

std::mutex g_tune_mutex;
std::map<std::string, Tuned> g_tuned;

std::string tune_key(const th_gemm_desc* d) {
  char buf[512];
  snprintf(buf, sizeof buf, "%d %d %d %d|%lld %lld %lld %lld %lld|%lld %lld %lld %lld %lld|%d %d %d %d %d|%d %d %d",
           d->m, d->n, d->k, std::max(1, d->batch), (long long)d->a_m, (long long)d->a_k, (long long)d->b_k,
           (long long)d->b_n, (long long)d->c_ld, (long long)d->a_batch, (long long)d->b_batch, (long long)d->c_batch,
           (long long)d->d_ld, (long long)d->d_batch, d->flags, d->c_dtype, d->epilogue, d->bias != nullptr,
           d->d != nullptr, (int)(reinterpret_cast<uintptr_t>(d->a) % 16 == 0),
           (int)(reinterpret_cast<uintptr_t>(d->b) % 16 == 0), (int)(reinterpret_cast<uintptr_t>(d->c) % 16 == 0));
  return buf;
}

// The parts of K with which a build for `tile` is what one left to the
// builder (splits 0) is: named, but for fp32 factors, whose builders choose among
// kernels by them too (0 stays 0).
int splits_of(const th_gemm_desc* d, int tile) {
  if (d->flags & TH_GEMM_F32_FACTORS) return 0;
  return tile == TH_TILE_GENERAL ? 1 : auto_splits(d, tile);
}

int measure(const th_gemm_desc* base, int tile, int splits, double* seconds) {
  th_gemm_desc d = *base;
  d.tile = tile;
  d.splits = splits;
  th_launch* l = nullptr;
  if (int r = th_build_gemm(&d, &l)) return r;
  const int r = th_time_launch(l, 0, seconds);
  th_launch_destroy(l);
  return r;
}

}  // namespace

extern "C" int th_gemm_tune(const th_gemm_desc* desc, int32_t* tile_out, int32_t* splits_out, double* seconds_out) {
  if (int r = th::require_ready()) return r;
  TH_REQUIRE(desc != nullptr && tile_out && splits_out && seconds_out, "th_gemm_tune: null argument");
  TH_REQUIRE(!((desc->flags & TH_GEMM_ACCUMULATE) && desc->d == desc->c),
             "th_gemm_tune: D + A B in place would add the product again at every measurement");
  const std::string key = tune_key(desc);
  std::lock_guard<std::mutex> lock(g_tune_mutex);
  auto hit = g_tuned.find(key);
  if (hit == g_tuned.end()) {
    th_gemm_desc d = *desc;
    d.tile = TH_TILE_AUTO;
    d.splits = 0;
    // Every choice is kept as it is measured (tile, splits), so that the launch
    // built from the answer is the one measured.
    std::vector<Tuned> choices;
    const bool x3 = (d.flags & TH_GEMM_BF16X3) != 0;
    auto add = [&](int tile) { choices.push_back(Tuned{tile, splits_of(&d, tile), 0.0}); };
    if (x3) {
      // The bf16 tiles the tripled product may run on: those that build.
      for (int t : {TH_TILE_256, TH_TILE_128X128, TH_TILE_128X64, TH_TILE_64X128, TH_TILE_64X64}) add(t);
    } else {
      if (tile_kernel_takes(&d)) add(TH_TILE_256);
      if (mid_takes(&d))
        for (int t : {TH_TILE_128X128, TH_TILE_128X64, TH_TILE_64X128, TH_TILE_64X64}) add(t);
      if (d.epilogue == TH_EPI_STORE && !d.bias) add(TH_TILE_GENERAL);
      // The library's own choice where it is none of these: parts of K it takes
      // by its estimate, or a fused product on a middle tile (which no caller names).
      int s = 0;
      const int t = choose_tile(&d, &s);
      if (d.epilogue != TH_EPI_STORE && t != TH_TILE_256 && !choices.empty()) choices.push_back(Tuned{TH_TILE_AUTO, 0, 0.0});
      else if (t != TH_TILE_256 && t != TH_TILE_GENERAL && s != splits_of(&d, t)) choices.push_back(Tuned{t, s, 0.0});
    }
    TH_REQUIRE(!choices.empty(), "th_gemm_tune: no kernel takes the product");
    // Stage one: every tile at the split the builder would choose.
    Tuned best{-1, 0, 0.0};
    auto consider = [&](Tuned c) -> int {
      if (int r = measure(&d, c.tile, c.splits, &c.seconds)) return r;
      if (best.tile < 0 || c.seconds < best.seconds) best = c;
      return TH_OK;
    };
    for (const Tuned& c : choices)
      if (int r = consider(c))
        if (!x3) return r;  // (x3: a tile the tripled product does not fit)
    TH_REQUIRE(best.tile >= 0, "th_gemm_tune: no kernel takes the product");
    // Stage two: the other splits of the best (plain products on the tile
    // kernels, and fp32 ones on the general kernel), each part at least 256 deep.
    const bool general_splits = d.flags & TH_GEMM_F32_FACTORS && d.c_dtype == TH_F32 && !d.bias;
    if ((best.tile != TH_TILE_GENERAL || general_splits) && d.epilogue == TH_EPI_STORE) {
      const Tuned first = best;
      for (int sp : {1, 2, 4, 8, 16}) {
        if (sp > 1 && d.k / sp < 256) break;
        if (sp == first.splits) continue;
        if (int r = consider(Tuned{first.tile, sp, 0.0})) return r;
      }
    }
    hit = g_tuned.emplace(key, best).first;
  }
  *tile_out = hit->second.tile;
  *splits_out = hit->second.splits;
  *seconds_out = hit->second.seconds;
  return TH_OK;
}

extern "C" int th_build_gemm_grouped(const th_gemm_desc* descs, int count, th_launch** out) {
  if (int r = th::require_ready()) return r;
  *out = nullptr;
  TH_REQUIRE(descs != nullptr && count >= 1, "th_build_gemm_grouped: no products");
  std::vector<th_launch*> parts;
  auto drop = [&]() {
    for (th_launch* l : parts) th_launch_destroy(l);
  };
  for (int i = 0; i < count; ++i) {
    th_launch* l = nullptr;
    if (int r = th_build_gemm(&descs[i], &l)) {
      drop();
      return r;
    }
    parts.push_back(l);
  }
  // One launch: every product's kernels in order, its values after the
  // previous products', its workspaces owned by the whole.
  th_launch* g = new th_launch();
  g->name = "gemm_grouped";
  for (th_launch* l : parts) {
    const int k0 = (int)g->kernels.size();
    g->kernels.insert(g->kernels.end(), l->kernels.begin(), l->kernels.end());
    for (size_t v = 0; v < l->values.size(); ++v) {
      std::vector<th::Ref> refs = l->values[v];
      for (th::Ref& r : refs) r.kernel += k0;
      g->values.push_back(refs);
      g->align.push_back(l->align[v]);
    }
    g->owned.insert(g->owned.end(), l->owned.begin(), l->owned.end());
    l->owned.clear();
    // Its workspace follows the previous products' in the whole's.
    for (th::WsRef r : l->ws_refs) {
      r.kernel += k0;
      r.at += g->ws_bytes;
      g->ws_refs.push_back(r);
    }
    g->ws_bytes += l->ws_bytes;
    g->work.bytes += l->work.bytes;
    g->work.flops += l->work.flops;
    g->work.blocks += l->work.blocks;
  }
  g->work.kernels = (int32_t)g->kernels.size();
  g->work.values = (int32_t)g->values.size();
  drop();
  *out = g;
  return TH_OK;
}
