// Op class (b), the product's middle tiles: C tiles of 128 x 128, 128 x 64,
// 64 x 128 and 64 x 64 on the half-precision matrix cores
// (v_mfma_f32_32x32x16_bf16 / _f16), the output tiles the reference's
// product sketch searches for half factors (ext/cuTileExt/contract.jl:36-39),
// for products whose 256 x 256 tiles would leave most of the device idle or
// whose sizes those tiles do not divide.  Factors bf16 or fp16, each operand
// with a unit stride along k or along its rows, any m, n, k, the other strides
// multiples of 8 and operands 16-byte aligned; K may be split over parts that
// a second launch folds (mid_fold), which then runs the epilogue.
//
// A workgroup of four waves takes one tile, each wave a quarter as 32 x 32
// blocks.  K advances 64 at a time through 2 to 4 LDS stages: whole steps are
// loaded straight into LDS (lds_dma.h), one to three steps ahead, one barrier
// a step; rows past the operand's end read its last rows again (their
// products are not stored).  What is left of K, and operands the direct loads
// do not take (an mn-contiguous one whose rows are not a multiple of 8, or
// over 2 GiB), go through registers with every element checked.
// A k-contiguous operand sits in LDS as rows of 64 k, 16-byte chunk c of row r
// at c ^ (r / 2 % 8) (16 rows' reads of one chunk fall on 16 distinct bank
// quads); an mn-contiguous one as rows of one k, chunk c of row k moved by 64
// bytes so that the four rows of a transposed read (ds_read_b64_tr_b16) fall
// on distinct banks.
// These tiles are bound by latency and by the L2's rate, not by the matrix
// cores: two workgroups a CU, each with its loads a step or more ahead.
// Measured (launch to launch, warm): 4096^3 on 128 x 128 tiles 203 us through
// registers 32 of K at a time, 138 here (992 TFLOP/s; the 256 x 256 kernel
// 108); 3072 x 1024 x 768 33.2 -> 11.5; 2000 x 8000 x 520 58.6 on ragged 256 x
// 256 tiles, 33.8 here.  An MLP's gradient at batch 1024, 768 x 3072 x 768, with
// its fused products here instead of on 12 or 48 tiles of 256 x 256: 266 -> 125.
#include <hip/hip_runtime.h>

#include "gemm_kernel.h"
#include "gemm_mid.h"
#include "th_core.h"

namespace thg {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));

constexpr int kKd = 64;  // K per step

// The n < 8 leading elements at p, the rest zero.
__device__ __forceinline__ u32x4 partial(const uint16_t* p, int n) {
  uint32_t e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = i < n ? p[i] : 0u;
  return u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
}

// One operand of R rows (m of A, n of B): element (row, k) at
// base[row * s + k] (KC) or base[row + k * s].
template <int R, bool KC>
struct Op {
  static constexpr int kElems = R * kKd;   // one stage
  static constexpr int kLoads = R / 32;    // 1 KB loads a wave issues a step; 16-byte chunks a thread moves
  __amdgpu_buffer_rsrc_t rsrc;
  int32_t off[kLoads];
  int32_t step;

  // Chunk c of LDS row l (KC: a row of the operand; else one k).
  __device__ __forceinline__ static int chunk(int l, int c) {
    if constexpr (KC) return l * kKd + 8 * (c ^ (l / 2 % 8));
    return l * R + 8 * (c ^ (R == 128 ? 4 * (l % 4) : 4 * (l / 2 % 2)));
  }

  __device__ __forceinline__ void init(const uint16_t* base, int64_t s, int row0, int rows, int kbeg) {
    rsrc = th_dev::buffer_of(base);
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    constexpr int per = KC ? 8 : R / 8;  // chunks an LDS row
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = 64 * (w * kLoads + i) + l, line = q / per;
      const int c = (q % per) ^ (chunk(line, 0) % (8 * per) / 8);  // the logical chunk that lies there
      off[i] = KC ? (int32_t)(((int64_t)min(row0 + line, rows - 1) * s + kbeg + 8 * c) * 2)
                  : (int32_t)((min(row0 + 8 * c, rows - 8) + (int64_t)(kbeg + line) * s) * 2);
    }
    step = (int32_t)((KC ? 1 : s) * kKd * 2);
  }
  // Whole step t into the stage at LDS byte `at`.
  __device__ __forceinline__ void direct(int t, uint32_t at) const {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) th_dev::dma16(rsrc, off[i], t * step, at + 1024 * (w * kLoads + i));
  }

  // Through registers: chunk i of this thread is q = threadIdx.x + 256 i.
  __device__ static void load(const uint16_t* base, int64_t s, int row0, int rows, int k0, int kend,
                              u32x4 (&r)[kLoads]) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = (int)threadIdx.x + 256 * i;
      u32x4 v = {0u, 0u, 0u, 0u};
      if constexpr (KC) {
        const int row = row0 + q / 8, k = k0 + 8 * (q % 8);
        if (row < rows && k < kend) {
          const uint16_t* at = base + (int64_t)row * s + k;
          v = k + 8 <= kend ? *reinterpret_cast<const u32x4*>(at) : partial(at, kend - k);
        }
      } else {
        const int k = k0 + q / (R / 8), row = row0 + 8 * (q % (R / 8));
        if (k < kend && row < rows) {
          const uint16_t* at = base + row + (int64_t)k * s;
          v = row + 8 <= rows ? *reinterpret_cast<const u32x4*>(at) : partial(at, rows - row);
        }
      }
      r[i] = v;
    }
  }
  __device__ static void store(uint16_t* lds, const u32x4 (&r)[kLoads]) {
    constexpr int per = KC ? 8 : R / 8;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = (int)threadIdx.x + 256 * i;
      *reinterpret_cast<u32x4*>(lds + chunk(q / per, q % per)) = r[i];
    }
  }

  // The fragment of rows r0 + lane % 32, k = 16 ks + 8 (lane / 32) + (0..7).
  __device__ static bf16x8 frag(const uint16_t* lds, int r0, int ks) {
    const int lane = threadIdx.x % 64;
    if constexpr (KC) {
      return *reinterpret_cast<const bf16x8*>(lds + chunk(r0 + lane % 32, 2 * ks + lane / 32));
    } else {
      // ds_read_b64_tr_b16 hands lane i of each 16 element i % 4 of the
      // 8-byte pieces addressed by lanes 4 q + i / 4 (q = 0..3).  Lane j
      // addresses k row 16 ks + 8 (lane / 32) + j / 4 (+ 4 for the upper
      // half, four rows on: the same permutation), rows r0 + 16 ((lane / 16)
      // % 2) + 4 (j % 4) + (0..3), so lane i receives k rows base + (0..3) of
      // row r0 + 16 ((lane / 16) % 2) + i.
      const int j = lane % 16;
      const int k = 16 * ks + 8 * (lane / 32) + j / 4;
      const int row = r0 + 16 * ((lane / 16) % 2) + 4 * (j % 4);
      const uint16_t* at = lds + chunk(k, row / 8) + row % 8;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * R));
      const s16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8, w);
    }
  }
};

template <bool F16>
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float widen(const void* p, int64_t i, int type) {
  if (type == TH_F32) return static_cast<const float*>(p)[i];
  const uint16_t h = static_cast<const uint16_t*>(p)[i];
  if (type == TH_BF16) return bf16_float(h);
  return (float)__builtin_bit_cast(_Float16, h);
}
__device__ __forceinline__ uint16_t narrow(float x, int type) {
  return type == TH_BF16 ? bf16_bits(x) : __builtin_bit_cast(uint16_t, (_Float16)x);
}

__device__ __forceinline__ u32x4 pack8(const uint16_t (&h)[8]) {
  return u32x4{h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16, h[4] | (uint32_t)h[5] << 16,
               h[6] | (uint32_t)h[7] << 16};
}

// The epilogue of eight sums v of column n, rows m.. (`live` of them inside
// C): bias, D, what the epilogue computes, one rounding, the store; rs and
// loss take this thread's share of the row sums and the loss.
__device__ __forceinline__ void finish8(const MidArgs& p, int64_t z, int m, int n, int live, float (&v)[8],
                                        float (&rs)[8], float& loss) {
  if (p.bias) {
    if (live == 8) {
      const u32x4 b = *reinterpret_cast<const u32x4_any*>(p.bias + m);
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] += half_of(b[r / 2], r % 2);
    } else {
      for (int r = 0; r < live; ++r) v[r] += bf16_float(p.bias[m + r]);
    }
  }
  const int64_t at = z * p.c_batch + m + (int64_t)n * p.c_ld;
  uint16_t* c = static_cast<uint16_t*>(p.c);
  uint16_t out[8];
  switch (p.epilogue) {
    case TH_EPI_GELU: {
      uint16_t h[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        out[r] = bf16_bits(v[r]);
        h[r] = bf16_bits(gelu(bf16_float(out[r])));
      }
      *reinterpret_cast<u32x4_any*>(p.aux_out + at) = pack8(h);
      break;
    }
    case TH_EPI_SQUARE_LOSS:
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float y = bf16_float(bf16_bits(v[r]));
        out[r] = bf16_bits(2.0f * y);
        loss = fmaf(y, y, loss);
        rs[r] += bf16_float(out[r]);
      }
      break;
    case TH_EPI_GELU_BACKWARD: {
      const u32x4 zz = *reinterpret_cast<const u32x4_any*>(p.aux + m + (int64_t)n * p.aux_ld);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        out[r] = bf16_bits(bf16_float(bf16_bits(v[r])) * gelu_grad(half_of(zz[r / 2], r % 2)));
        rs[r] += bf16_float(out[r]);
      }
      break;
    }
    default: {
      if (p.d) {
        const int64_t at_d = z * p.d_batch + m + (int64_t)n * p.d_ld;
#pragma unroll
        for (int r = 0; r < 8; ++r)
          if (r < live) v[r] += widen(p.d, at_d + r, p.result);
      }
      if (p.result == TH_F32) {
        float* f = static_cast<float*>(p.c) + at;
        typedef f32x4 f32x4_any __attribute__((aligned(4)));
        if (live == 8) {
          *reinterpret_cast<f32x4_any*>(f) = f32x4{v[0], v[1], v[2], v[3]};
          *reinterpret_cast<f32x4_any*>(f + 4) = f32x4{v[4], v[5], v[6], v[7]};
        } else {
#pragma unroll
          for (int r = 0; r < 8; ++r)
            if (r < live) f[r] = v[r];
        }
        return;
      }
#pragma unroll
      for (int r = 0; r < 8; ++r) out[r] = narrow(v[r], p.result);
    }
  }
  if (live == 8) {
    *reinterpret_cast<u32x4_any*>(c + at) = pack8(out);
  } else {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (r < live) c[at + r] = out[r];
  }
}

// A workgroup's row sums (rs: rows m0 + 8 (thread % G) + (0..7) over the
// thread's columns) and loss into the partials of column block nb and block
// `block`, the 256 / G threads of a row added in order.
template <int G>
__device__ __forceinline__ void finish_sums(const MidArgs& p, float* lds, int m0, int nb, int block,
                                            const float (&rs)[8], float loss) {
  __syncthreads();
  float* mine = lds + (threadIdx.x / G) * (8 * G + 4) + 8 * (threadIdx.x % G);
#pragma unroll
  for (int r = 0; r < 8; ++r) mine[r] = rs[r];
  float* per_wave = lds + (256 / G) * (8 * G + 4);
  loss = thd::wave_sum(loss);
  if (threadIdx.x % 64 == 0) per_wave[threadIdx.x / 64] = loss;
  __syncthreads();
  const int m = m0 + threadIdx.x;
  if (threadIdx.x < 8 * G && m < p.m) {
    float s = 0.0f;
    for (int i = 0; i < 256 / G; ++i) s += lds[i * (8 * G + 4) + threadIdx.x];
    p.row_parts[(int64_t)nb * p.m + m] = s;
  }
  if (threadIdx.x == 0) p.loss_parts[block] = per_wave[0] + per_wave[1] + per_wave[2] + per_wave[3];
}

template <int BM, int BN>
constexpr int kStages = BM + BN == 256 ? 2 : BM + BN == 192 ? 3 : 4;

template <int BM, int BN>
constexpr int lds_bytes() {
  const int sweep = kStages<BM, BN> * (BM + BN) * kKd * 2, tile = BN * (BM + 4) * 4;
  return sweep > tile ? sweep : tile;
}

template <int BM, int BN, bool F16, bool AKC, bool BKC>
__global__ __launch_bounds__(256, 2) void gemm_mid(MidArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  using OA = Op<BM, AKC>;
  using OB = Op<BN, BKC>;
  constexpr int BI = BM / 64, BJ = BN / 64;  // 32 x 32 blocks a wave
  constexpr int ST = kStages<BM, BN>, kStage = OA::kElems + OB::kElems;
  auto As = [&](int s) { return lds + s * kStage; };
  auto Bs = [&](int s) { return lds + s * kStage + OA::kElems; };
  const uint32_t ring = (uint32_t)(uintptr_t)lds;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int64_t z = blockIdx.z, part = blockIdx.y;
  const int kbeg = (int)part * p.ksplit, kend = min(p.k, kbeg + p.ksplit);
  const uint16_t* a = p.a + z * p.a_batch;
  const uint16_t* b = p.b + z * p.b_batch;
  const int64_t sa = AKC ? p.a_m : p.a_k, sb = BKC ? p.b_n : p.b_k;
  const int m0 = tm * BM, n0 = tn * BN;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int wm = wave / 2, wn = wave % 2;
  f32x16 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = f32x16{};
  auto multiply = [&](int s) {
#pragma unroll
    for (int ks = 0; ks < kKd / 16; ++ks) {
      bf16x8 fa[BI], fb[BJ];
#pragma unroll
      for (int i = 0; i < BI; ++i) fa[i] = OA::frag(As(s), wm * (BM / 2) + 32 * i, ks);
#pragma unroll
      for (int j = 0; j < BJ; ++j) fb[j] = OB::frag(Bs(s), wn * (BN / 2) + 32 * j, ks);
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) acc[i][j] = mfma<F16>(fa[i], fb[j], acc[i][j]);
    }
  };
  const int whole = p.direct ? (kend - kbeg) / kKd : 0, steps = (kend - kbeg + kKd - 1) / kKd;
  if (whole > 0) {
    OA A;
    OB B;
    A.init(a, sa, m0, p.m, kbeg);
    B.init(b, sb, n0, p.n, kbeg);
    constexpr int L = OA::kLoads + OB::kLoads;
    auto issue = [&](int t, int s) {
      A.direct(t, ring + s * kStage * 2);
      B.direct(t, ring + (s * kStage + OA::kElems) * 2);
    };
#pragma unroll
    for (int t = 0; t < ST - 1; ++t)
      if (t < whole) issue(t, t);
    int s = 0;
    for (int t = 0; t < whole; ++t) {
      // Step t has landed: the loads of at most ST - 2 later steps stay in
      // flight.  Past the barrier every wave is done with step t - 1, whose
      // stage step t + ST - 1 takes.
      const int later = min(ST - 2, whole - 1 - t);
      if (ST == 4 && later == 2) th_dev::wait_and_meet<2 * L>();
      else if (ST >= 3 && later == 1) th_dev::wait_and_meet<L>();
      else th_dev::wait_and_meet<0>();
      if (t + ST - 1 < whole) issue(t + ST - 1, s == 0 ? ST - 1 : s - 1);
      multiply(s);
      s = s + 1 == ST ? 0 : s + 1;
    }
  }
  if (whole < steps) {
    u32x4 ra[OA::kLoads], rb[OB::kLoads];
    auto load = [&](int t) {
      OA::load(a, sa, m0, p.m, kbeg + t * kKd, kend, ra);
      OB::load(b, sb, n0, p.n, kbeg + t * kKd, kend, rb);
    };
    auto store = [&](int s) {
      OA::store(As(s), ra);
      OB::store(Bs(s), rb);
    };
    load(whole);
    __syncthreads();  // every wave is done with the whole steps' stages
    store(0);
    __syncthreads();
    for (int t = whole; t < steps; ++t) {
      const int cur = (t - whole) & 1;
      if (t + 1 < steps) load(t + 1);
      multiply(cur);
      if (t + 1 < steps) store(cur ^ 1);
      __syncthreads();
    }
  }
  // The tile through LDS, column-major at BM + 4 floats, so that each thread
  // ends with eight consecutive rows of a column: lane holds C(m, n) for n =
  // the block's first column + lane % 32 and m = its first row + 8 g + 4
  // (lane / 32) + (0..3), register 4 g + (0..3).
  __syncthreads();
  float* T = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(T + (wn * (BN / 2) + 32 * j + lane % 32) * (BM + 4) + wm * (BM / 2) + 32 * i + 8 * g +
                                  4 * (lane / 32)) =
            f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
  __syncthreads();
  constexpr int G = BM / 8;  // threads a column
  const int m = m0 + 8 * (threadIdx.x % G), live = min(8, p.m - m);
  float rs[8] = {}, loss = 0.0f;
  for (int i = threadIdx.x / G; i < BN; i += 256 / G) {
    const int n = n0 + i;
    if (live <= 0 || n >= p.n) break;
    const f32x4 lo = *reinterpret_cast<const f32x4*>(T + i * (BM + 4) + (m - m0));
    const f32x4 hi = *reinterpret_cast<const f32x4*>(T + i * (BM + 4) + (m - m0) + 4);
    if (p.parts) {  // this part's sums, rows padded to 8
      float* to = p.parts + z * p.part_batch + part * p.part_split + m + (int64_t)n * p.part_ld;
      *reinterpret_cast<f32x4*>(to) = lo;
      *reinterpret_cast<f32x4*>(to + 4) = hi;
    } else {
      float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      finish8(p, z, m, n, live, v, rs, loss);
    }
  }
  if (!p.parts && p.epilogue >= TH_EPI_SQUARE_LOSS) finish_sums<G>(p, T, m0, tn, blockIdx.x, rs, loss);
}

// The parts of K summed, in part order, and the epilogue of the sums.  A
// workgroup takes 128 rows of kFoldColumns columns, a thread eight rows of a
// column at a time, the parts' loads issued four at a time.
__global__ __launch_bounds__(256) void mid_fold(MidArgs p) {
  __shared__ float lds[16 * 132 + 4];
  const int tiles_m = (p.m + 127) / 128;
  const int tm = blockIdx.x % tiles_m, tn = blockIdx.x / tiles_m;
  const int64_t z = blockIdx.z;
  const int m = tm * 128 + 8 * (threadIdx.x % 16), live = min(8, p.m - m);
  float rs[8] = {}, loss = 0.0f;
#pragma unroll
  for (int i = 0; i < kFoldColumns / 16; ++i) {
    const int n = tn * kFoldColumns + 16 * i + threadIdx.x / 16;
    if (live > 0 && n < p.n) {
      const f32x4* x = reinterpret_cast<const f32x4*>(p.parts + z * p.part_batch + m + (int64_t)n * p.part_ld);
      const int64_t step = p.part_split / 4;
      f32x4 lo = {}, hi = {};
      int s = 0;
      for (; s + 4 <= p.splits; s += 4) {
        f32x4 l[4], h[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) l[u] = x[(s + u) * step], h[u] = x[(s + u) * step + 1];
#pragma unroll
        for (int u = 0; u < 4; ++u) lo += l[u], hi += h[u];
      }
      for (; s < p.splits; ++s) lo += x[s * step], hi += x[s * step + 1];
      float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      finish8(p, z, m, n, live, v, rs, loss);
    }
  }
  if (p.epilogue >= TH_EPI_SQUARE_LOSS) finish_sums<16>(p, lds, tm * 128, tn, blockIdx.x, rs, loss);
}

template <int BM, int BN>
const void* for_tile(bool f16, bool a_kc, bool b_kc) {
#define TH_MID(F, A, B) (const void*)gemm_mid<BM, BN, F, A, B>
  if (f16) {
    if (a_kc) return b_kc ? TH_MID(true, true, true) : TH_MID(true, true, false);
    return b_kc ? TH_MID(true, false, true) : TH_MID(true, false, false);
  }
  if (a_kc) return b_kc ? TH_MID(false, true, true) : TH_MID(false, true, false);
  return b_kc ? TH_MID(false, false, true) : TH_MID(false, false, false);
#undef TH_MID
}

}  // namespace

const void* mid_fold_kernel() { return (const void*)mid_fold; }

const void* mid_kernel(int tile, bool f16, bool a_kc, bool b_kc, int* bm, int* bn, int* lds) {
  switch (tile) {
    case TH_TILE_128X128:
      *bm = 128, *bn = 128, *lds = lds_bytes<128, 128>();
      return for_tile<128, 128>(f16, a_kc, b_kc);
    case TH_TILE_128X64:
      *bm = 128, *bn = 64, *lds = lds_bytes<128, 64>();
      return for_tile<128, 64>(f16, a_kc, b_kc);
    case TH_TILE_64X128:
      *bm = 64, *bn = 128, *lds = lds_bytes<64, 128>();
      return for_tile<64, 128>(f16, a_kc, b_kc);
    case TH_TILE_64X64:
      *bm = 64, *bn = 64, *lds = lds_bytes<64, 64>();
      return for_tile<64, 64>(f16, a_kc, b_kc);
    default:
      return nullptr;
  }
}

}  // namespace thg
