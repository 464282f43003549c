// Op class (c) for fp32 arrays on the matrix cores at head dims 64 and 128, any
// lengths, grouped heads, causal or not.  fp32 attention with device-held masks,
// and other head dims, stay on attention_generic.hip.  The reference's cuTile
// sweep takes fp32 arrays (its TF32 mode rounds the factors to 10 bits,
// ext/cuTileExt/build.jl:326-532; TRIALS.md:2187); here all of fp32's 24 bits
// take part, as its default precision asks (src/Compiler/runtime/target.jl:42-44).
//
// The sweeps (*_parts) are the bf16 kernels' of attention_mfma.hip on operands
// split into three bf16 parts, tiles on their way into LDS, P and dS in
// registers: six products of parts (v_mfma_f32_32x32x16_bf16) for each product,
// what they leave out at most 2^-25 of each a b.  The fp32 matrix cores take
// 2.7 times as long for the same product.  Error against float64 over thirty
// drawn shapes: 0.89 of the fp32 products' on average, at most 6.7e-7 where
// theirs was 8.1e-7.  B2 H8 S1024 d64 causal, forward + backward: 168 us with
// fp32 products, 124 so; S2048 469 and 305; B6 H16 KV8 S640 d128 568 and 437.  One
// stage of LDS (the parts take 1.5 times fp32's bytes), the next tile in
// registers, two barriers a step; bound by the vector work of the splits and
// the wait at the barriers, the matrix cores busy 18 to 24 % of the time.
//
// Q, K, V and dO are scaled by 2^24 as they are split (kUp; dS with them, and the
// results back), so that a part of the least fp32 number is one of bf16's; a weight
// under 2^-109 keeps what bits of it lie above 2^-134.  A block whose results are not finite
// (also those of factors past 2^103) is computed again with fp32 products
// (v_mfma_f32_32x32x2_f32; *_block), forms of depth 2 instead of 16:
//   - products over d (S' = K Q', S = Q K', dP = dO V'): lane half h takes d
//     in [h D/2, (h + 1) D/2), step s the d h D/2 + s, so a lane's operand
//     of four steps is one 16-byte read of a tile row (rows of D + 4 floats:
//     16 lanes reading 16 rows start on 16 distinct bank quads), the other
//     operand (a position's row) in registers;
//   - products over positions (O' += V' P', dV' += dO' P, dK' += Q' dS,
//     dQ' += K' dS'): the score accumulator's register i is the B operand
//     of step i as it stands (lanes 0..31 holding position 8 (i / 4) + i % 4
//     of the block, lanes 32..63 the position 4 further), and the output's
//     row m of block b holds d = NB m + b (NB = D / 32 blocks), so that a
//     lane's A operands of the NB blocks are NB adjacent floats of one tile
//     row, one 8- or 16-byte read.
// Everything else as there: tiles of 64 positions staged through registers a
// step ahead (zeros past the sequence), the online softmax in exp2 units
// (folds.jl:186-222), P in fp32, lse = m + log(l); the backward FA2's,
// deterministic: delta = rowsum(dO .* O); dK, dV per 128 keys sweeping the query
// tiles of each query head of the group; dQ per 128 queries sweeping the key
// tiles.  Keys past the keys' length and, causal, keys after the query weigh 0;
// queries past the sequence are computed on zeros and not stored.
#include <hip/hip_runtime.h>

#include <cmath>

#include "attention_tiles.h"
#include "th_core.h"

namespace {

struct FArgs {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  float* lse;  // natural log, [b][s][h]
  const float* dout;
  float* delta;  // backward workspace: rowsum(dO .* O), [b][s][h]
  float* dq;
  float* dk;
  float* dv;
  int64_t q_sh, q_ss, q_sb;  // strides (elements) of q, o, dout, dq
  int64_t k_sh, k_ss, k_sb;  // strides of k, v, dk, dv
  int32_t seq, kv_seq, heads, kv_heads, batch, causal;
  float scale;
  // A sweep split into parts (small grids): nsplit parts of `span`
  // positions (a multiple of 64), partial results in `part`
  // ([part][b][position][head][d]) and the forward's (m, l) in `part_ml`.
  int32_t nsplit, span;
  float* part;
  float* part_ml;
  // The backward's dQ sweep, beside the dK/dV one above.
  int32_t q_nsplit, q_span;
  float* q_part;
};

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int D>
constexpr int kLd = D + 4;  // LDS row of a tile (floats)
template <int D>
constexpr int kTileF = 64 * kLd<D>;

// A position's row as the B operand of a product over d: f[s] = row[h D/2 + s].
template <int D>
__device__ __forceinline__ void row_half(const float* row, bool live, float (&f)[D / 2]) {
  const int h = (threadIdx.x % 64) / 32;
#pragma unroll
  for (int u = 0; u < D / 8; ++u) {
    const f32x4 x = live ? *reinterpret_cast<const f32x4*>(row + h * (D / 2) + 4 * u) : f32x4{};
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * u + e] = x[e];
  }
}

// acc += T[rows r0 + lane % 32] x f over d (D / 2 steps, four a read).
template <int D>
__device__ __forceinline__ void over_d(const float* t, int r0, const float (&f)[D / 2], f32x16& acc) {
  const int lane = threadIdx.x % 64;
  const float* row = t + (r0 + lane % 32) * kLd<D> + (lane / 32) * (D / 2);
#pragma unroll
  for (int u = 0; u < D / 8; ++u) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(row + 4 * u);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma2(a[e], f[4 * u + e], acc);
  }
}

// The NB adjacent floats of tile row `r` this lane gives the NB output
// blocks of a product over positions: columns NB (lane % 32) + (0..NB-1).
template <int D>
struct Cols {
  float x[D / 32];
};
template <int D>
__device__ __forceinline__ Cols<D> cols_of(const float* t, int r) {
  constexpr int NB = D / 32;
  const float* at = t + r * kLd<D> + NB * (threadIdx.x % 32);
  Cols<D> c;
  if constexpr (NB == 2) {
    const f32x2 x = *reinterpret_cast<const f32x2*>(at);
    c.x[0] = x[0], c.x[1] = x[1];
  } else {
    const f32x4 x = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
    for (int e = 0; e < NB; ++e) c.x[e] = x[e];
  }
  return c;
}

// out[db] += T'(d, positions of block pb) P over the block's 32 positions:
// step i pairs position 8 (i / 4) + i % 4 (lanes 0..31) with the one 4
// further (lanes 32..63), as register i of the score accumulator holds them.
template <int D>
__device__ __forceinline__ void over_positions(const float* t, int p0, const f32x16& pw, f32x16 (&out)[D / 32]) {
  const int lh = (threadIdx.x % 64) / 32;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const Cols<D> c = cols_of<D>(t, p0 + 8 * (i / 4) + 4 * lh + i % 4);
#pragma unroll
    for (int db = 0; db < D / 32; ++db) out[db] = mfma2(c.x[db], pw[i], out[db]);
  }
}

// Store an output block set: block db's register i holds d = NB (8 (i / 4) +
// 4 lh + i % 4) + db, for the lane's position; scaled by sc.
template <int D>
__device__ __forceinline__ void store_rows(float* row, const f32x16 (&x)[D / 32], float sc) {
  constexpr int NB = D / 32;
  const int lh = (threadIdx.x % 64) / 32;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    // d = NB (8 q + 4 lh) + (0 .. 4 NB - 1): register 4 q + e of block db at NB e + db.
    float* at = row + NB * (8 * q + 4 * lh);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (NB == 2) {
        *reinterpret_cast<f32x2*>(at + 2 * e) = f32x2{x[0][4 * q + e] * sc, x[1][4 * q + e] * sc};
      } else {
        *reinterpret_cast<f32x4*>(at + 4 * e) =
            f32x4{x[0][4 * q + e] * sc, x[1][4 * q + e] * sc, x[2][4 * q + e] * sc, x[3][4 * q + e] * sc};
      }
    }
  }
}

// A 64-position tile staged through registers: thread t holds the 16-byte
// chunks t + 256 i; rows past `limit` read as zeros.
template <int D>
struct StageF {
  static constexpr int kChunks = D / 4;
  static constexpr int kPer = 64 * kChunks / 256;
  f32x4 r[kPer];
  __device__ void load(const float* base, int64_t ss, int row0, int limit) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = threadIdx.x + 256 * i, row = c / kChunks, col = c % kChunks;
      r[i] = row0 + row < limit ? *reinterpret_cast<const f32x4*>(base + (int64_t)(row0 + row) * ss + 4 * col)
                                : f32x4{};
    }
  }
  __device__ void store(float* t) const {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = threadIdx.x + 256 * i, row = c / kChunks, col = c % kChunks;
      *reinterpret_cast<f32x4*>(t + row * kLd<D> + 4 * col) = r[i];
    }
  }
};

// The grid is (heads, batch, blocks): blocks slowest, the longest causal
// sweeps first, the short ones filling in behind them.

// ---- forward ---------------------------------------------------------------------

// Keys [k_lo, k_hi) of query block qb: all (split < 0) or part `split`,
// which leaves its unnormalised O' and (m, l) for the combining kernel.
template <int D>
__device__ __forceinline__ void fwd_block(const FArgs& p, const int qb, const int b, const int split) {
  constexpr int NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  const int h = blockIdx.x;
  const int hk = h / (p.heads / p.kv_heads);
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lr = lane % 32, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lr;
  const float* qbase = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const float* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const float* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  float qf[D / 2];
  row_half<D>(qbase + (int64_t)query * p.q_ss, query < p.seq, qf);
  f32x16 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) o[i] = f32x16{};
  float m = -INFINITY, l = 0.0f;
  const float c = p.scale * kLog2e;
  const int qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(p.kv_seq, qlast + 1) : p.kv_seq;
  const int k_lo = split < 0 ? 0 : split * p.span, k_hi = split < 0 ? kend : min(kend, k_lo + p.span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  StageF<D> sk, sv;
  auto K = [&](int s) { return flds + 2 * s * kTileF<D>; };
  auto V = [&](int s) { return flds + (2 * s + 1) * kTileF<D>; };
  if (nsteps > 0) {
    sk.load(kbase, p.k_ss, k_lo, p.kv_seq);
    sv.load(vbase, p.k_ss, k_lo, p.kv_seq);
    sk.store(K(0));
    sv.store(V(0));
  }
  __syncthreads();
  for (int j = 0; j < nsteps; ++j) {
    const int cur = j & 1, k0 = k_lo + 64 * j;
    if (j + 1 < nsteps) {
      sk.load(kbase, p.k_ss, k0 + 64, p.kv_seq);
      sv.load(vbase, p.k_ss, k0 + 64, p.kv_seq);
    }
    // S' (64 keys x 32 queries): key 32 kb + 8 (i / 4) + 4 lh + i % 4 in register i.
    f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) over_d<D>(K(cur), 32 * kb, qf, s[kb]);
    if (k0 + 64 > p.kv_seq || (p.causal && k0 + 63 > q0)) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
          if (key >= p.kv_seq || (p.causal && key > query)) s[kb][i] = -INFINITY;
        }
    }
    float mb = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mb = fmaxf(mb, s[kb][i]);
    mb = fmaxf(mb, other_half(mb)) * c;
    const float mn = fmaxf(m, mb);
    const float shift = isfinite(mn) ? mn : 0.0f;  // lse_shift (folds.jl:194)
    const float alpha = __builtin_amdgcn_exp2f(m - shift);
    l *= alpha;
#pragma unroll
    for (int i = 0; i < NB; ++i) o[i] *= alpha;
    m = mn;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float w = __builtin_amdgcn_exp2f(fmaf(s[kb][i], c, -shift));
        l += w;
        s[kb][i] = w;
      }
    // O' (D x 32 queries) += V' P'.
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) over_positions<D>(V(cur), 32 * kb, s[kb], o);
    if (j + 1 < nsteps) {
      // The other stage was last read in step j - 1, before the barrier that ended it.
      sk.store(K(cur ^ 1));
      sv.store(V(cur ^ 1));
    }
    __syncthreads();
  }
  l += other_half(l);
  if (query >= p.seq) return;
  if (split >= 0) {
    // This part's unnormalised O' and (m, l) (m = -inf, l = 0 where it saw no key).
    const int64_t row = (((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h;
    store_rows<D>(p.part + row * D, o, 1.0f);
    if (lh == 0) reinterpret_cast<f32x2*>(p.part_ml)[row] = f32x2{m, l};
    return;
  }
  store_rows<D>(p.o + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss, o, 1.0f / l);
  if (lh == 0 && p.lse) p.lse[((int64_t)b * p.seq + query) * p.heads + h] = (m + log2f(l)) * kLn2;
}

// The parts of a split forward combined: per (b, query, head) row, M = max
// m_s, L = sum l_s 2^(m_s - M), O = sum O_s 2^(m_s - M) / L in part order;
// lse = (M + log2 L) ln 2.  A thread per four features of a row.
struct FCombineArgs {
  FArgs p;  // first: its members sit at FArgs' offsets
  int32_t d;
};

__global__ __launch_bounds__(256) void f32_attn_combine(FCombineArgs a) {
  const FArgs& p = a.p;
  const int quads = a.d / 4;
  const int64_t rows = (int64_t)p.batch * p.seq * p.heads;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= rows * quads) return;
  const int64_t row = t / quads;
  const int c = 4 * (int)(t % quads);
  const f32x2* ml = reinterpret_cast<const f32x2*>(p.part_ml);
  float mx = -INFINITY;
  for (int s = 0; s < p.nsplit; ++s) mx = fmaxf(mx, ml[s * rows + row][0]);
  const float shift = isfinite(mx) ? mx : 0.0f;
  float l = 0.0f;
  f32x4 acc = {};
  for (int s = 0; s < p.nsplit; ++s) {
    const f32x2 x = ml[s * rows + row];
    const float w = __builtin_amdgcn_exp2f(x[0] - shift);
    l += w * x[1];
    acc += w * *reinterpret_cast<const f32x4*>(p.part + (s * rows + row) * a.d + c);
  }
  const int h = (int)(row % p.heads);
  const int64_t pos = (row / p.heads) % p.seq, b = row / ((int64_t)p.heads * p.seq);
  *reinterpret_cast<f32x4*>(p.o + b * p.q_sb + h * p.q_sh + pos * p.q_ss + c) = acc * (1.0f / l);
  if (c == 0 && p.lse) p.lse[row] = (mx + log2f(l)) * kLn2;
}

// dK, dV and dQ from split sweeps' parts, one launch: out = scale * sum_s
// part_s in part order; rows [b][position][head] of `d` features.
struct FSumArgsOne {
  const float* part;
  float* out;
  int64_t sh, ss, sb;
  int32_t positions, heads, nsplit;
  float scale;
  uint32_t blocks;  // workgroups, 256 quads of features each
};
struct FSumArgs {
  FSumArgsOne of[3];
  int32_t n, batch, d;
};

__global__ __launch_bounds__(256) void f32_attn_sum(FSumArgs all) {
  uint32_t block = blockIdx.x;
  int which = 0;
  while (which + 1 < all.n && block >= all.of[which].blocks) block -= all.of[which++].blocks;
  const FSumArgsOne& a = all.of[which];
  const int d = all.d, quads = d / 4;
  const int64_t rows = (int64_t)all.batch * a.positions * a.heads;
  const int64_t t = (int64_t)block * 256 + threadIdx.x;
  if (t >= rows * quads) return;
  const int64_t row = t / quads;
  const int c = 4 * (int)(t % quads);
  // Part s of this quad at a.part + (s rows + row) d + c: a stride of rows d / 4 quads.
  f32x4 acc = thd::sum_in_order(reinterpret_cast<const f32x4*>(a.part + row * d + c), rows * d / 4, a.nsplit);
  acc *= a.scale;
  const int h = (int)(row % a.heads);
  const int64_t pos = (row / a.heads) % a.positions, b = row / ((int64_t)a.heads * a.positions);
  *reinterpret_cast<f32x4*>(a.out + b * a.sb + h * a.sh + pos * a.ss + c) = acc;
}

// ---- backward: delta = rowsum(dO .* O) ---------------------------------------------

struct FDeltaArgs {
  FArgs p;  // first: its members sit at FArgs' offsets
  int32_t d;
};

// D / 4 lanes per (batch, position, head) row, 16 bytes each (the path takes
// strides in multiples of 4 and 16-byte bases); each lane group takes
// kDeltaRowsF rows, 64 / (D / 4) apart, every load issued before the first
// product.  Rows are numbered with the head fastest, so a load instruction
// covers consecutive rows; row numbers fit 32 bits (the builder checks).
constexpr int kDeltaRowsF = 4;

template <int D>
__global__ __launch_bounds__(256) void f32_attn_delta(FDeltaArgs a) {
  constexpr int G = D / 4;   // lanes a row
  constexpr int R = 64 / G;  // rows a wave covers at once
  const FArgs& p = a.p;
  const uint32_t total = (uint32_t)p.batch * p.seq * p.heads;
  const int lane = threadIdx.x % 64, part = lane % G;
  const uint32_t row0 = (blockIdx.x * 4 + threadIdx.x / 64) * (R * kDeltaRowsF) + lane / G;
  auto at_of = [&](uint32_t row) {
    const uint32_t bs = row / (uint32_t)p.heads;
    const int64_t b = bs / (uint32_t)p.seq, s = bs % (uint32_t)p.seq, h = row - bs * (uint32_t)p.heads;
    return b * p.q_sb + h * p.q_sh + s * p.q_ss + 4 * part;
  };
  f32x4 ov[kDeltaRowsF], gv[kDeltaRowsF];
#pragma unroll
  for (int i = 0; i < kDeltaRowsF; ++i) {
    // Rows past the end re-read the last one; nothing is written for them.
    const int64_t at = at_of(min(row0 + R * i, total - 1));
    ov[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.o + at));
    gv[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.dout + at));
  }
  // Every load out before any of their data is used.
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kDeltaRowsF; ++i) {
    float v = ov[i][0] * gv[i][0];
#pragma unroll
    for (int e = 1; e < 4; ++e) v += ov[i][e] * gv[i][e];
#pragma unroll
    for (int m = G / 2; m >= 1; m /= 2) v += __shfl_xor(v, m, G);
    const uint32_t row = row0 + R * i;
    if (row < total && part == 0) p.delta[row] = v;
  }
}

// ---- backward: dK, dV ----------------------------------------------------------------
// A workgroup takes 128 keys (32 a wave).  Per query tile of 64: S (64
// queries x 32 keys) with queries on the registers and keys on the lanes, so
// that P and dS feed the products over queries straight from the
// accumulators.

// Query tiles [qstart, qstop) for the keys of kblk: all (split < 0) or part
// `split`, which leaves its unscaled dK', dV'.
template <int D>
__device__ __forceinline__ void dkdv_block(const FArgs& p, const int kblk, const int hk, const int b, const int split) {
  constexpr int NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  float* stats = flds + 4 * kTileF<D>;  // [stage][lse * log2e (64) | delta (64)]
  const int group = p.heads / p.kv_heads;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lh = lane / 32;
  const int kw0 = kblk * 128, key = kw0 + wave * 32 + lane % 32;
  const int64_t koff = (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  float kf[D / 2], vf[D / 2];
  row_half<D>(p.k + koff + (int64_t)key * p.k_ss, key < p.kv_seq, kf);
  row_half<D>(p.v + koff + (int64_t)key * p.k_ss, key < p.kv_seq, vf);
  f32x16 dk[NB], dv[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) dk[i] = f32x16{}, dv[i] = f32x16{};
  const float c = p.scale * kLog2e;
  auto Q = [&](int s) { return flds + 2 * s * kTileF<D>; };
  auto G = [&](int s) { return flds + (2 * s + 1) * kTileF<D>; };
  auto Ls = [&](int s) { return stats + 128 * s; };
  const int qfirst = p.causal ? kw0 / 64 * 64 : 0;
  const int qstart = split < 0 ? qfirst : qfirst + split * p.span;
  const int qstop = split < 0 ? p.seq : min(p.seq, qstart + p.span);
  const int nsteps = qstart < qstop ? (qstop - qstart + 63) / 64 : 0;
  StageF<D> sq, sg;
  float st = 0.0f;  // threads 0..127: a query's lse * log2e or delta
  auto load = [&](const float* qbase, const float* gbase, int h, int q0) {
    sq.load(qbase, p.q_ss, q0, p.seq);
    sg.load(gbase, p.q_ss, q0, p.seq);
    if (threadIdx.x < 128) {
      const int j = q0 + threadIdx.x % 64;
      const int64_t row = ((int64_t)b * p.seq + j) * p.heads + h;
      st = j < p.seq ? (threadIdx.x < 64 ? p.lse[row] * kLog2e : p.delta[row]) : 0.0f;
    }
  };
  auto store = [&](int s) {
    sq.store(Q(s));
    sg.store(G(s));
    if (threadIdx.x < 128) Ls(s)[threadIdx.x] = st;
  };
  for (int h = hk * group; h < (hk + 1) * group; ++h) {
    const float* qbase = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    const float* gbase = p.dout + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    if (nsteps > 0) {
      load(qbase, gbase, h, qstart);
      store(0);
    }
    __syncthreads();
    for (int j = 0; j < nsteps; ++j) {
      const int cur = j & 1, qq0 = qstart + 64 * j;
      if (j + 1 < nsteps) load(qbase, gbase, h, qq0 + 64);
      const float *Qt = Q(cur), *Gt = G(cur);
      const float* L = Ls(cur);
      const int kw = __builtin_amdgcn_readfirstlane(kw0 + wave * 32);
      const bool edge = qq0 + 64 > p.seq || kw + 32 > p.kv_seq || (p.causal && kw + 31 > qq0);
      // The tile's two halves of 32 queries in turn (half the score
      // accumulators live at once); the next tile goes to LDS after the first.
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        // S = Q K', dP = dO V' (32 queries x 32 keys): query 32 jj + 8 (i / 4) + 4 lh + i % 4 in register i.
        f32x16 s = {}, dp = {};
        over_d<D>(Qt, 32 * jj, kf, s);
        over_d<D>(Gt, 32 * jj, vf, dp);
        // P into s, dS into dp.
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int qi = 32 * jj + 8 * (i / 4) + 4 * lh + i % 4;
          s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -L[qi]));
          dp[i] = s[i] * (dp[i] - L[64 + qi]);
        }
        if (edge) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int query = qq0 + 32 * jj + 8 * (i / 4) + 4 * lh + i % 4;
            const bool seen = query < p.seq && key < p.kv_seq && (!p.causal || key <= query);
            s[i] = seen ? s[i] : 0.0f;
            dp[i] = seen ? dp[i] : 0.0f;
          }
        }
        // dV' (D x 32 keys) += dO' P;  dK' += Q' dS.
        over_positions<D>(Gt, 32 * jj, s, dv);
        over_positions<D>(Qt, 32 * jj, dp, dk);
        // The other stage was last read in step j - 1, before the barrier that ended it.
        if (jj == 0 && j + 1 < nsteps) store(cur ^ 1);
      }
      __syncthreads();
    }
  }
  if (key >= p.kv_seq) return;
  if (split >= 0) {
    const int64_t rows = (int64_t)p.batch * p.kv_seq * p.kv_heads;
    const int64_t row = (((int64_t)split * p.batch + b) * p.kv_seq + key) * p.kv_heads + hk;
    store_rows<D>(p.part + row * D, dk, 1.0f);
    store_rows<D>(p.part + ((int64_t)p.nsplit * rows + row) * D, dv, 1.0f);
    return;
  }
  const int64_t out = koff + (int64_t)key * p.k_ss;
  store_rows<D>(p.dk + out, dk, p.scale);
  store_rows<D>(p.dv + out, dv, 1.0f);
}

// ---- backward: dQ ----------------------------------------------------------------------
// A workgroup takes 128 queries (32 a wave) and sweeps key tiles of 64:
// S' = K Q', dP' = V dO' (keys on the registers, queries on the lanes),
// dS' = P' (dP' - delta), dQ' (D x 32 queries) += K' dS'.

// Keys [k_lo, k_hi) for query block qb: all (split < 0) or part `split`,
// which leaves its unscaled dQ'.
template <int D>
__device__ __forceinline__ void dq_block(const FArgs& p, const int qb, const int h, const int b, const int split) {
  constexpr int NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  const int hk = h / (p.heads / p.kv_heads);
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lane % 32;
  const int64_t qoff = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss;
  const bool live = query < p.seq;
  float qf[D / 2], gf[D / 2];
  row_half<D>(p.q + qoff, live, qf);
  row_half<D>(p.dout + qoff, live, gf);
  const int64_t srow = ((int64_t)b * p.seq + query) * p.heads + h;
  const float l2 = live ? p.lse[srow] * kLog2e : 0.0f;
  const float dl = live ? p.delta[srow] : 0.0f;
  const float c = p.scale * kLog2e;
  const float* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const float* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  f32x16 dq[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) dq[i] = f32x16{};
  const int qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(p.kv_seq, qlast + 1) : p.kv_seq;
  const int k_lo = split < 0 ? 0 : split * p.q_span, k_hi = split < 0 ? kend : min(kend, k_lo + p.q_span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  StageF<D> sk, sv;
  auto K = [&](int s) { return flds + 2 * s * kTileF<D>; };
  auto V = [&](int s) { return flds + (2 * s + 1) * kTileF<D>; };
  if (nsteps > 0) {
    sk.load(kbase, p.k_ss, k_lo, p.kv_seq);
    sv.load(vbase, p.k_ss, k_lo, p.kv_seq);
    sk.store(K(0));
    sv.store(V(0));
  }
  __syncthreads();
  for (int j = 0; j < nsteps; ++j) {
    const int cur = j & 1, k0 = k_lo + 64 * j;
    if (j + 1 < nsteps) {
      sk.load(kbase, p.k_ss, k0 + 64, p.kv_seq);
      sv.load(vbase, p.k_ss, k0 + 64, p.kv_seq);
    }
    // The tile's two halves of 32 keys in turn; the next tile goes to LDS after the first.
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x16 sc = {}, dp = {};
      over_d<D>(K(cur), 32 * kb, qf, sc);
      over_d<D>(V(cur), 32 * kb, gf, dp);
      // dS' into sc.
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sc[i] = __builtin_amdgcn_exp2f(fmaf(sc[i], c, -l2)) * (dp[i] - dl);
      }
      if (k0 + 64 > p.kv_seq || (p.causal && k0 + 63 > q0)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
          sc[i] = key < p.kv_seq && (!p.causal || key <= query) ? sc[i] : 0.0f;
        }
      }
      over_positions<D>(K(cur), 32 * kb, sc, dq);
      if (kb == 0 && j + 1 < nsteps) {
        sk.store(K(cur ^ 1));
        sv.store(V(cur ^ 1));
      }
    }
    __syncthreads();
  }
  if (!live) return;
  if (split >= 0) {
    store_rows<D>(p.q_part + ((((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h) * D, dq, 1.0f);
    return;
  }
  store_rows<D>(p.dq + qoff, dq, p.scale);
}

// ---- the sweeps in bf16 parts -------------------------------------------------------

// The factors' scale, and what takes products of two and three of them back.
constexpr float kUp = 0x1p24f, kDown = 0x1p-24f, kDown2 = 0x1p-48f, kDown3 = 0x1p-72f;
constexpr float kUp2 = 0x1p48f;

// An operand of eight values a lane, in its three parts.
struct Parts {
  bf16x8 of[3];
};
// Eight registers of an accumulator from register `at`.
__device__ __forceinline__ Parts parts_of(const f32x16& x, const int at) {
  u32x4 w[3];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t w0, w1, w2;
    split2(x[at + 2 * e], x[at + 2 * e + 1], w0, w1, w2);
    w[0][e] = w0, w[1][e] = w1, w[2][e] = w2;
  }
  return Parts{{(bf16x8)w[0], (bf16x8)w[1], (bf16x8)w[2]}};
}

// c += a b: the products of parts down to 2^-18 of a b, the least first.
__device__ __forceinline__ f32x16 mfma6(const Parts& a, const Parts& b, f32x16 c) {
  c = mfma(a.of[2], b.of[0], c);
  c = mfma(a.of[1], b.of[1], c);
  c = mfma(a.of[0], b.of[2], c);
  c = mfma(a.of[1], b.of[0], c);
  c = mfma(a.of[0], b.of[1], c);
  return mfma(a.of[0], b.of[0], c);
}

template <int D>
constexpr int kPart = 64 * (D + 8);  // bf16 elements of one part of a tile
template <int D>
constexpr int kTileP = 3 * kPart<D>;

template <int D>
__device__ __forceinline__ Parts rows3(const uint16_t* t, int r0, int ks) {
  return Parts{{frag_rows<D>(t, r0, ks), frag_rows<D>(t + kPart<D>, r0, ks), frag_rows<D>(t + 2 * kPart<D>, r0, ks)}};
}
template <int D>
__device__ __forceinline__ Parts tr3(const uint16_t* t, int d0, int ks) {
  return Parts{{frag_tr<D>(t, d0, ks), frag_tr<D>(t + kPart<D>, d0, ks), frag_tr<D>(t + 2 * kPart<D>, d0, ks)}};
}

// A position's row, times kUp, as the B operand of a product over d: d = 16 ks
// + 8 (lane / 32) + (0..7); zeros for a position past the end.
template <int D>
__device__ __forceinline__ void row_parts(const float* row, bool live, Parts (&f)[D / 16]) {
  const int lh = threadIdx.x % 64 / 32;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    const float* at = row + 16 * ks + 8 * lh;
    const f32x4 lo = live ? *reinterpret_cast<const f32x4*>(at) : f32x4{}, hi = live ? *reinterpret_cast<const f32x4*>(at + 4) : f32x4{};
    u32x4 w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4 x = (e < 2 ? lo : hi) * kUp;
      uint32_t w0, w1, w2;
      split2(x[2 * (e % 2)], x[2 * (e % 2) + 1], w0, w1, w2);
      w[0][e] = w0, w[1][e] = w1, w[2][e] = w2;
    }
    f[ks] = Parts{{(bf16x8)w[0], (bf16x8)w[1], (bf16x8)w[2]}};
  }
}

// A tile loaded into registers (StageF) and stored, times kUp, in its parts.
template <int D>
struct StageP : StageF<D> {
  __device__ void store(uint16_t* t) const {
#pragma unroll
    for (int i = 0; i < StageF<D>::kPer; ++i) {
      const int c = threadIdx.x + 256 * i, row = c / StageF<D>::kChunks, col = c % StageF<D>::kChunks;
      const f32x4 x = this->r[i] * kUp;
      u32x2 w[3];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        uint32_t w0, w1, w2;
        split2(x[2 * e], x[2 * e + 1], w0, w1, w2);
        w[0][e] = w0, w[1][e] = w1, w[2][e] = w2;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x2*>(t + s * kPart<D> + row * (D + 8) + 4 * col) = w[s];
    }
  }
};

// d = 32 db + 8 g + 4 lh + (0..3) of a lane's position: out = x sc.
template <int D>
__device__ __forceinline__ void store_quads(float* row, const f32x16 (&x)[D / 32], float sc) {
  const int lh = threadIdx.x % 64 / 32;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(row + 32 * db + 8 * g + 4 * lh) =
          f32x4{x[db][4 * g], x[db][4 * g + 1], x[db][4 * g + 2], x[db][4 * g + 3]} * sc;
}
template <int N>
__device__ __forceinline__ bool finite(const f32x16 (&x)[N]) {
  bool f = true;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) f = f && fabsf(x[i][e]) < INFINITY;
  return f;
}

// fwd_block in bf16 parts; false, and nothing stored, where it has to be
// computed in fp32 products.
template <int D>
__device__ __forceinline__ bool fwd_parts(const FArgs& p, const int qb, const int b, const int split) {
  constexpr int NS = D / 16, NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  uint16_t* K = reinterpret_cast<uint16_t*>(flds);
  uint16_t* V = K + kTileP<D>;
  const int h = blockIdx.x;
  const int hk = h / (p.heads / p.kv_heads);
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lr = lane % 32, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lr;
  const float* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const float* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  Parts qf[NS];
  row_parts<D>(p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss, query < p.seq, qf);
  f32x16 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) o[i] = f32x16{};
  float m = -INFINITY, l = 0.0f;
  const float c = p.scale * kLog2e * kDown2;  // of scores times kUp2
  const int qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(p.kv_seq, qlast + 1) : p.kv_seq;
  const int k_lo = split < 0 ? 0 : split * p.span, k_hi = split < 0 ? kend : min(kend, k_lo + p.span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  StageP<D> sk, sv;
  if (nsteps > 0) {
    sk.load(kbase, p.k_ss, k_lo, p.kv_seq);
    sv.load(vbase, p.k_ss, k_lo, p.kv_seq);
  }
  for (int j = 0; j < nsteps; ++j) {
    const int k0 = k_lo + 64 * j;
    __syncthreads();  // the previous step's tile is read
    sk.store(K);
    sv.store(V);
    if (j + 1 < nsteps) {
      sk.load(kbase, p.k_ss, k0 + 64, p.kv_seq);
      sv.load(vbase, p.k_ss, k0 + 64, p.kv_seq);
    }
    __syncthreads();
    // S' (64 keys x 32 queries): key 32 kb + 8 (i / 4) + 4 lh + i % 4 in register i.
    f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int ks = 0; ks < NS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] = mfma6(rows3<D>(K, 32 * kb, ks), qf[ks], s[kb]);
    if (k0 + 64 > p.kv_seq || (p.causal && k0 + 63 > q0)) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
          if (key >= p.kv_seq || (p.causal && key > query)) s[kb][i] = -INFINITY;
        }
    }
    float mb = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mb = fmaxf(mb, s[kb][i]);
    mb = fmaxf(mb, other_half(mb)) * c;
    const float mn = fmaxf(m, mb);
    const float shift = isfinite(mn) ? mn : 0.0f;  // lse_shift (folds.jl:194)
    const float alpha = __builtin_amdgcn_exp2f(m - shift);
    l *= alpha;
#pragma unroll
    for (int i = 0; i < NB; ++i) o[i] *= alpha;
    m = mn;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[kb][i] = __builtin_amdgcn_exp2f(fmaf(s[kb][i], c, -shift));
        l += s[kb][i];
      }
      // O' (D x 32 queries) += V' P'.
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const Parts pw = parts_of(s[kb], 8 * half);
#pragma unroll
        for (int db = 0; db < NB; ++db) o[db] = mfma6(tr3<D>(V, 32 * db, 2 * kb + half), pw, o[db]);
      }
    }
  }
  l += other_half(l);
  const bool good = query >= p.seq || (finite(o) && fabsf(l) < INFINITY);
  if (__syncthreads_or(!good)) return false;
  if (query >= p.seq) return true;
  if (split >= 0) {
    const int64_t row = (((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h;
    store_quads<D>(p.part + row * D, o, kDown);
    if (lh == 0) reinterpret_cast<f32x2*>(p.part_ml)[row] = f32x2{m, l};
    return true;
  }
  store_quads<D>(p.o + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss, o, kDown / l);
  if (lh == 0 && p.lse) p.lse[((int64_t)b * p.seq + query) * p.heads + h] = (m + log2f(l)) * kLn2;
  return true;
}

// dkdv_block in bf16 parts; false, and nothing stored, as fwd_parts.
template <int D>
__device__ __forceinline__ bool dkdv_parts(const FArgs& p, const int kblk, const int hk, const int b, const int split) {
  constexpr int NS = D / 16, NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  uint16_t* Q = reinterpret_cast<uint16_t*>(flds);
  uint16_t* G = Q + kTileP<D>;
  float* L = reinterpret_cast<float*>(G + kTileP<D>);  // lse * log2e (64) | delta times kUp2 (64)
  const int group = p.heads / p.kv_heads;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lh = lane / 32;
  const int kw = __builtin_amdgcn_readfirstlane(kblk * 128 + wave * 32), key = kw + lane % 32;
  const int64_t koff = (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  Parts kf[NS], vf[NS];
  row_parts<D>(p.k + koff + (int64_t)key * p.k_ss, key < p.kv_seq, kf);
  row_parts<D>(p.v + koff + (int64_t)key * p.k_ss, key < p.kv_seq, vf);
  f32x16 dk[NB], dv[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) dk[i] = f32x16{}, dv[i] = f32x16{};
  const float c = p.scale * kLog2e * kDown2;  // of scores times kUp2
  const int qfirst = p.causal ? kblk * 128 : 0;
  const int qstart = split < 0 ? qfirst : qfirst + split * p.span;
  const int qstop = split < 0 ? p.seq : min(p.seq, qstart + p.span);
  const int nsteps = qstart < qstop ? (qstop - qstart + 63) / 64 : 0;
  StageP<D> sq, sg;
  float st = 0.0f;  // threads 0..127: a query's lse * log2e or delta, times kUp2
  auto load = [&](int h, int q0) {
    const int64_t qoff = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    sq.load(p.q + qoff, p.q_ss, q0, p.seq);
    sg.load(p.dout + qoff, p.q_ss, q0, p.seq);
    if (threadIdx.x < 128) {
      const int j = q0 + threadIdx.x % 64;
      const int64_t row = ((int64_t)b * p.seq + j) * p.heads + h;
      st = j < p.seq ? (threadIdx.x < 64 ? p.lse[row] * kLog2e : p.delta[row] * kUp2) : 0.0f;
    }
  };
  const int total = nsteps * group;  // steps over the group's query heads
  if (total > 0) load(hk * group, qstart);
  for (int j = 0, q = 0, h = hk * group; j < total; ++j) {
    const int qq0 = qstart + 64 * q;
    if (++q == nsteps) q = 0, ++h;
    __syncthreads();  // the previous step's tile is read
    sq.store(Q);
    sg.store(G);
    if (threadIdx.x < 128) L[threadIdx.x] = st;
    if (j + 1 < total) load(h, qstart + 64 * q);
    __syncthreads();
    const bool edge = qq0 + 64 > p.seq || kw + 32 > p.kv_seq || (p.causal && kw + 31 > qq0);
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      // S = Q K', dP = dO V' (32 queries x 32 keys): query 32 jj + 8 (i / 4) + 4 lh + i % 4 in register i.
      f32x16 s = {}, dp = {};
#pragma unroll
      for (int ks = 0; ks < NS; ++ks) {
        s = mfma6(rows3<D>(Q, 32 * jj, ks), kf[ks], s);
        dp = mfma6(rows3<D>(G, 32 * jj, ks), vf[ks], dp);
      }
      // P into s, dS times kUp2 into dp.
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int qi = 32 * jj + 8 * (i / 4) + 4 * lh + i % 4;
        s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -L[qi]));
        dp[i] = s[i] * (dp[i] - L[64 + qi]);
      }
      if (edge) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int query = qq0 + 32 * jj + 8 * (i / 4) + 4 * lh + i % 4;
          const bool seen = query < p.seq && key < p.kv_seq && (!p.causal || key <= query);
          s[i] = seen ? s[i] : 0.0f;
          dp[i] = seen ? dp[i] : 0.0f;
        }
      }
      // dV' (D x 32 keys) += dO' P;  dK' += Q' dS.
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const Parts pw = parts_of(s, 8 * half), sw = parts_of(dp, 8 * half);
#pragma unroll
        for (int db = 0; db < NB; ++db) {
          dv[db] = mfma6(tr3<D>(G, 32 * db, 2 * jj + half), pw, dv[db]);
          dk[db] = mfma6(tr3<D>(Q, 32 * db, 2 * jj + half), sw, dk[db]);
        }
      }
    }
  }
  const bool good = key >= p.kv_seq || (finite(dk) && finite(dv));
  if (__syncthreads_or(!good)) return false;
  if (key >= p.kv_seq) return true;
  if (split >= 0) {
    const int64_t rows = (int64_t)p.batch * p.kv_seq * p.kv_heads;
    const int64_t row = (((int64_t)split * p.batch + b) * p.kv_seq + key) * p.kv_heads + hk;
    store_quads<D>(p.part + row * D, dk, kDown3);
    store_quads<D>(p.part + ((int64_t)p.nsplit * rows + row) * D, dv, kDown);
    return true;
  }
  const int64_t out = koff + (int64_t)key * p.k_ss;
  store_quads<D>(p.dk + out, dk, p.scale * kDown3);
  store_quads<D>(p.dv + out, dv, kDown);
  return true;
}

// dq_block in bf16 parts; false, and nothing stored, as fwd_parts.
template <int D>
__device__ __forceinline__ bool dq_parts(const FArgs& p, const int qb, const int h, const int b, const int split) {
  constexpr int NS = D / 16, NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float flds[];
  uint16_t* K = reinterpret_cast<uint16_t*>(flds);
  uint16_t* V = K + kTileP<D>;
  const int hk = h / (p.heads / p.kv_heads);
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lane % 32;
  const int64_t qoff = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss;
  const bool live = query < p.seq;
  Parts qf[NS], gf[NS];
  row_parts<D>(p.q + qoff, live, qf);
  row_parts<D>(p.dout + qoff, live, gf);
  const int64_t srow = ((int64_t)b * p.seq + query) * p.heads + h;
  const float l2 = live ? p.lse[srow] * kLog2e : 0.0f;
  const float dl = live ? p.delta[srow] * kUp2 : 0.0f;
  const float c = p.scale * kLog2e * kDown2;  // of scores times kUp2
  const float* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const float* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  f32x16 dq[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) dq[i] = f32x16{};
  const int qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(p.kv_seq, qlast + 1) : p.kv_seq;
  const int k_lo = split < 0 ? 0 : split * p.q_span, k_hi = split < 0 ? kend : min(kend, k_lo + p.q_span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  StageP<D> sk, sv;
  if (nsteps > 0) {
    sk.load(kbase, p.k_ss, k_lo, p.kv_seq);
    sv.load(vbase, p.k_ss, k_lo, p.kv_seq);
  }
  for (int j = 0; j < nsteps; ++j) {
    const int k0 = k_lo + 64 * j;
    __syncthreads();  // the previous step's tile is read
    sk.store(K);
    sv.store(V);
    if (j + 1 < nsteps) {
      sk.load(kbase, p.k_ss, k0 + 64, p.kv_seq);
      sv.load(vbase, p.k_ss, k0 + 64, p.kv_seq);
    }
    __syncthreads();
    const bool edge = k0 + 64 > p.kv_seq || (p.causal && k0 + 63 > q0);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x16 s = {}, dp = {};
#pragma unroll
      for (int ks = 0; ks < NS; ++ks) {
        s = mfma6(rows3<D>(K, 32 * kb, ks), qf[ks], s);
        dp = mfma6(rows3<D>(V, 32 * kb, ks), gf[ks], dp);
      }
      // dS' times kUp2 into s.
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -l2)) * (dp[i] - dl);
      if (edge) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
          s[i] = key < p.kv_seq && (!p.causal || key <= query) ? s[i] : 0.0f;
        }
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const Parts sw = parts_of(s, 8 * half);
#pragma unroll
        for (int db = 0; db < NB; ++db) dq[db] = mfma6(tr3<D>(K, 32 * db, 2 * kb + half), sw, dq[db]);
      }
    }
  }
  if (__syncthreads_or(live && !finite(dq))) return false;
  if (!live) return true;
  if (split >= 0)
    store_quads<D>(p.q_part + ((((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h) * D, dq, kDown3);
  else
    store_quads<D>(p.dq + qoff, dq, p.scale * kDown3);
  return true;
}

// ---- the kernels ----------------------------------------------------------------------

// LDS of either form: two tiles in parts, or two stages of two fp32 tiles.
template <int D>
constexpr size_t kLdsF = (2 * kTileP<D> * sizeof(uint16_t) > 4 * kTileF<D> * sizeof(float) ? 2 * kTileP<D> * sizeof(uint16_t)
                                                                                           : 4 * kTileF<D> * sizeof(float)) +
                         2 * 128 * sizeof(float);

// Scales under this, times kDown3, would lose bits: fp32 products alone.
constexpr float kLeastScale = 0x1p-50f;

template <int D>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void f32_attn_fwd(FArgs p) {
  const bool split = p.nsplit > 1;
  const int z = gridDim.z - 1 - blockIdx.z;  // the last queries first
  const int qb = split ? z / p.nsplit : z, part = split ? z % p.nsplit : -1;
  if (p.scale < kLeastScale || !fwd_parts<D>(p, qb, blockIdx.y, part)) fwd_block<D>(p, qb, blockIdx.y, part);
}

// Both sweeps in one launch: neither needs the other, and alone each leaves
// the device part empty at its end.  dK/dV workgroups, the first keys, the
// longest causal sweeps, first; then the dQ ones, the last queries first.
struct FBwdArgs {
  FArgs p;  // first: its members sit at FArgs' offsets
  uint32_t n_dkdv;
};

// One wave a SIMD: with two, d = 64 spills around its sweeps.  d = 128 spills 43
// registers even so (K and V of a wave's keys take 192 in parts, dK' and dV'
// 128, the next tile 64), 36 of them without the fp32 form beside it.
template <int D>
__global__ __launch_bounds__(256, 1) void f32_attn_bwd(FBwdArgs a) {
  const FArgs& p = a.p;
  if (blockIdx.x < a.n_dkdv) {
    const int hk = blockIdx.x % p.kv_heads, b = blockIdx.x / p.kv_heads % p.batch, z = blockIdx.x / p.kv_heads / p.batch;
    const bool split = p.nsplit > 1;
    const int kblk = split ? z / p.nsplit : z, part = split ? z % p.nsplit : -1;
    if (p.scale < kLeastScale || !dkdv_parts<D>(p, kblk, hk, b, part)) dkdv_block<D>(p, kblk, hk, b, part);
    return;
  }
  const uint32_t i = gridDim.x - 1 - blockIdx.x;  // (from the end: the last queries first)
  const int h = i % p.heads, b = i / p.heads % p.batch, z = i / p.heads / p.batch;
  const bool split = p.q_nsplit > 1;
  const int qb = split ? z / p.q_nsplit : z, part = split ? z % p.q_nsplit : -1;
  if (p.scale < kLeastScale || !dq_parts<D>(p, qb, h, b, part)) dq_block<D>(p, qb, h, b, part);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

FArgs fargs_of(const th_attention_desc* d) {
  FArgs a{};
  a.q = static_cast<const float*>(d->q);
  a.k = static_cast<const float*>(d->k);
  a.v = static_cast<const float*>(d->v);
  a.o = static_cast<float*>(d->o);
  a.lse = d->lse;
  a.dout = static_cast<const float*>(d->dout);
  a.dq = static_cast<float*>(d->dq);
  a.dk = static_cast<float*>(d->dk);
  a.dv = static_cast<float*>(d->dv);
  a.q_sh = d->q_strides[0], a.q_ss = d->q_strides[1], a.q_sb = d->q_strides[2];
  a.k_sh = d->k_strides[0], a.k_ss = d->k_strides[1], a.k_sb = d->k_strides[2];
  a.seq = d->seq;
  a.kv_seq = d->kv_seq > 0 ? d->kv_seq : d->seq;
  a.heads = d->heads, a.kv_heads = d->kv_heads, a.batch = d->batch, a.causal = d->causal;
  a.scale = d->scale > 0 ? d->scale : 1.0f / sqrtf((float)d->head_dim);
  return a;
}

double visible_pairs(const FArgs& a) {
  const double S = a.seq, K = a.kv_seq;
  if (!a.causal) return S * K;
  const double full = std::min(S, K);
  return full * (full + 1) / 2 + std::max(0.0, S - K) * K;
}

template <int D>
int fwd_launch(const th_attention_desc* d, th_launch** out) {
  const size_t lds = kLdsF<D>;
  TH_HIP(hipFuncSetAttribute((const void*)f32_attn_fwd<D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  FArgs a = fargs_of(d);
  const int nqb = (d->seq + 127) / 128;
  const th::Split sp = th::split_of((int64_t)nqb * d->heads * d->batch, a.kv_seq);
  a.nsplit = sp.n, a.span = sp.span;
  th::Builder b("attention_fwd_f32mfma", 7);
  const dim3 grid(d->heads, d->batch, nqb * sp.n);
  int k = b.kernel((const void*)f32_attn_fwd<D>, D == 64 ? "f32_attn_fwd_d64" : "f32_attn_fwd_d128", grid, dim3(256),
                   (uint32_t)lds, a);
  b.ref(0, k, TH_OFFSET(FArgs, q));
  b.ref(1, k, TH_OFFSET(FArgs, k));
  b.ref(2, k, TH_OFFSET(FArgs, v));
  b.ref(3, k, TH_OFFSET(FArgs, o));
  b.ref(4, k, TH_OFFSET(FArgs, lse));
  if (sp.n > 1) {
    const int64_t rows = (int64_t)d->batch * d->seq * d->heads;
    const uint64_t at_o = b.workspace((uint64_t)sp.n * rows * D * sizeof(float));
    const uint64_t at_ml = b.workspace((uint64_t)sp.n * rows * 2 * sizeof(float));
    int kc = b.kernel((const void*)f32_attn_combine, "f32_attn_combine", dim3((unsigned)((rows * (D / 4) + 255) / 256)),
                      dim3(256), 0, FCombineArgs{a, D});
    for (int kk : {k, kc}) {
      b.ws_ref(kk, TH_OFFSET(FArgs, part), at_o);
      b.ws_ref(kk, TH_OFFSET(FArgs, part_ml), at_ml);
    }
    b.ref(3, kc, TH_OFFSET(FArgs, o));
    b.ref(4, kc, TH_OFFSET(FArgs, lse));
  }
  for (int v = 0; v < 4; ++v) b.align(v, 16);
  const double BH = (double)d->batch * d->heads, BHk = (double)d->batch * d->kv_heads;
  b.work(2.0 * BH * a.seq * D * 4 + 2.0 * BHk * a.kv_seq * D * 4 + 4.0 * BH * a.seq, 4.0 * BH * D * visible_pairs(a),
         (int64_t)grid.x * grid.y * grid.z);
  *out = b.release();
  return TH_OK;
}

// The backward's launch: delta, both sweeps, and where small grids split
// them (the dK/dV sweep over queries, the dQ sweep over keys) their sums.
template <int D>
int bwd_launch(const th_attention_desc* d, th_launch** out) {
  const size_t lds = kLdsF<D>;
  const void* fn = (const void*)f32_attn_bwd<D>;
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  FArgs a = fargs_of(d);
  th::Builder b("attention_bwd_f32mfma", 11);
  const int64_t rows = (int64_t)d->batch * d->seq * d->heads;
  const int64_t rows_k = (int64_t)d->batch * a.kv_seq * d->kv_heads;
  TH_REQUIRE(rows < 2147483648LL, "attention: batch x seq x heads must be under 2^31");
  const uint64_t at_delta = b.workspace((uint64_t)rows * sizeof(float));
  const int nkb = (a.kv_seq + 127) / 128, nqb = (d->seq + 127) / 128;
  const int64_t gkv = (int64_t)nkb * d->kv_heads * d->batch, gq = (int64_t)nqb * d->heads * d->batch;
  const th::Split skv = th::split_of(gkv, d->seq, 384), sq = th::split_of(gq, a.kv_seq, 384);
  a.nsplit = skv.n, a.span = skv.span;
  a.q_nsplit = sq.n, a.q_span = sq.span;
  const int64_t n_dkdv = gkv * skv.n, blocks = n_dkdv + gq * sq.n;
  TH_REQUIRE(blocks <= 0x7fffffff, "attention: grid too large");
  constexpr int kDeltaBlockRows = 4 * (64 / (D / 4)) * kDeltaRowsF;  // rows a workgroup
  const int k0 = b.kernel((const void*)f32_attn_delta<D>, "f32_attn_delta",
                          dim3((unsigned)((rows + kDeltaBlockRows - 1) / kDeltaBlockRows)), dim3(256), 0, FDeltaArgs{a, D});
  const int k1 = b.kernel(fn, D == 64 ? "f32_attn_dkdv_d64_f32_attn_dq_d64" : "f32_attn_dkdv_d128_f32_attn_dq_d128",
                          dim3((unsigned)blocks), dim3(256), (uint32_t)lds, FBwdArgs{a, (uint32_t)n_dkdv});
  const size_t offs[9] = {TH_OFFSET(FArgs, q),  TH_OFFSET(FArgs, k),  TH_OFFSET(FArgs, v),
                          TH_OFFSET(FArgs, o),  TH_OFFSET(FArgs, lse), TH_OFFSET(FArgs, dout),
                          TH_OFFSET(FArgs, dq), TH_OFFSET(FArgs, dk),  TH_OFFSET(FArgs, dv)};
  // Both kernels' arguments begin with FArgs: the same offsets.
  for (int kk : {k0, k1}) {
    for (int v = 0; v < 9; ++v) b.ref(v, kk, offs[v]);
    b.ws_ref(kk, TH_OFFSET(FArgs, delta), at_delta);
  }
  for (int v : {0, 1, 2, 3, 5, 6, 7, 8}) b.align(v, 16);
  if (skv.n > 1 || sq.n > 1) {
    FSumArgs s{};
    s.batch = d->batch, s.d = D;
    // The outputs' pointers start as the descriptor's (repointing rewrites them with the others).
    int values[3];
    uint64_t ats[3];
    unsigned total = 0;
    auto add = [&](int value, float* to, const int64_t* strides, int positions, int heads, int parts, float scale,
                   uint64_t at) {
      const unsigned g = (unsigned)(((int64_t)d->batch * positions * heads * (D / 4) + 255) / 256);
      values[s.n] = value, ats[s.n] = at;
      s.of[s.n++] = FSumArgsOne{nullptr, to, strides[0], strides[1], strides[2], positions, heads, parts, scale, g};
      total += g;
    };
    if (skv.n > 1) {
      const uint64_t at = b.workspace((uint64_t)2 * skv.n * rows_k * D * sizeof(float));
      b.ws_ref(k1, TH_OFFSET(FArgs, part), at);
      add(7, a.dk, d->k_strides, a.kv_seq, d->kv_heads, skv.n, a.scale, at);
      add(8, a.dv, d->k_strides, a.kv_seq, d->kv_heads, skv.n, 1.0f, at + (uint64_t)skv.n * rows_k * D * sizeof(float));
    }
    if (sq.n > 1) {
      const uint64_t at = b.workspace((uint64_t)sq.n * rows * D * sizeof(float));
      b.ws_ref(k1, TH_OFFSET(FArgs, q_part), at);
      add(6, a.dq, d->q_strides, d->seq, d->heads, sq.n, a.scale, at);
    }
    const int k2 = b.kernel((const void*)f32_attn_sum,
                            sq.n == 1   ? "f32_attn_sum_dk_dv"
                                                              : skv.n == 1 ? "f32_attn_sum_dq"
                                                                           : "f32_attn_sum_dk_dv_f32_attn_sum_dq",
                            dim3(total), dim3(256), 0, s);
    for (int i = 0; i < s.n; ++i) {
      const size_t one = TH_OFFSET(FSumArgs, of) + i * sizeof(FSumArgsOne);
      b.ref(values[i], k2, one + TH_OFFSET(FSumArgsOne, out));
      b.ws_ref(k2, one + TH_OFFSET(FSumArgsOne, part), ats[i]);
    }
  }
  const double BH = (double)d->batch * d->heads, BHk = (double)d->batch * d->kv_heads;
  b.work(2.0 * BH * a.seq * D * 8 + 2.0 * BHk * a.kv_seq * D * 8 + 8.0 * BH * a.seq,
         2.5 * 4.0 * BH * D * visible_pairs(a), n_dkdv);
  *out = b.release();
  return TH_OK;
}

}  // namespace

namespace th {

// fp32 arrays, head dim 64 or 128, positive lengths, no device-held masks,
// 16-byte aligned operands and rows (strides multiples of 4 floats).
bool f32_attention_takes(const th_attention_desc* d) {
  if (!d || !(d->flags & TH_ATTN_F32) || d->starts || d->lengths) return false;
  if (d->head_dim != 64 && d->head_dim != 128) return false;
  if (d->seq < 1 || d->kv_seq < 0 || d->batch < 1 || d->heads < 1 || d->kv_heads < 1 || d->heads % d->kv_heads)
    return false;
  for (int64_t s : {d->q_strides[0], d->q_strides[1], d->q_strides[2], d->k_strides[0], d->k_strides[1], d->k_strides[2]})
    if (s <= 0 || s % 4) return false;
  for (const void* ptr : {(const void*)d->q, (const void*)d->k, (const void*)d->v, (const void*)d->o,
                          (const void*)d->dout, (const void*)d->dq, (const void*)d->dk, (const void*)d->dv})
    if (!aligned16(ptr)) return false;
  const int64_t kv = d->kv_seq > 0 ? d->kv_seq : d->seq;
  // (Blocks of 128 positions along grid z; sweeps are split only where all the
  // blocks are fewer than 256.)
  return (d->seq + 127) / 128 <= 65535 && (kv + 127) / 128 <= 65535 && d->heads <= 65535 && d->batch <= 65535;
}

int build_attention_f32_fwd(const th_attention_desc* d, th_launch** out) {
  TH_REQUIRE(d->q && d->k && d->v && d->o, "attention: null q, k, v or o");
  return d->head_dim == 64 ? fwd_launch<64>(d, out) : fwd_launch<128>(d, out);
}

int build_attention_f32_bwd(const th_attention_desc* d, th_launch** out) {
  TH_REQUIRE(d->q && d->k && d->v && d->o, "attention: null q, k, v or o");
  TH_REQUIRE(d->lse && d->dout && d->dq && d->dk && d->dv, "attention backward: null lse, dout, dq, dk or dv");
  return d->head_dim == 64 ? bwd_launch<64>(d, out) : bwd_launch<128>(d, out);
}

}  // namespace th
