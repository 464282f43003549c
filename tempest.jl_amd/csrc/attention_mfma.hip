// Op class (c) on the matrix cores at head dims 64, 128 and 256 and any
// lengths: what the tuned kernels of attention.hip (head dim 128, lengths in
// 128s) do not take, short of fp32 arrays (attention_f32.hip).  The reference's cuDNN claim takes half
// precision d <= 256 on tensor cores (ext/cuDNNExt.jl:90-100) and its cuTile
// sweep any tile (ext/cuTileExt/build.jl:326-493); d = 64 and d = 256 are
// the head dims models use beside 128.
//
// bf16 operands, v_mfma_f32_32x32x16_bf16, fp32 statistics; the forms of the
// tuned kernels, simpler: tiles of 64 positions x D in LDS as plain rows of
// D + 8 bf16 (16-byte reads along a row, ds_read_b64_tr_b16 down a column),
// staged through registers one step ahead (zeros past the sequence), one
// barrier a step.
//   forward: a workgroup of four waves per 128 queries, 32 a wave; S' = K Q'
//     (keys on registers, queries on lanes), online softmax in exp2 units,
//     O' += V' P' with P rounded to bf16 (folds.jl:186-222), lse = m + log(l);
//   backward (FA2's formulas, deterministic, no workspace beyond delta):
//     dK, dV: a workgroup per 128 keys (32 a wave, K and V rows in registers)
//     sweeping the query tiles of each query head of its group, S = Q K',
//     dP = dO V', P = exp(S - lse), dS = P (dP - delta), dV' += dO' P,
//     dK' += Q' dS; at d = 256 each workgroup keeps half of dK' and dV'
//     (grid twice as wide, the scores computed by both halves) so that its
//     accumulators fit one wave's registers;
//     dQ: a workgroup per 128 queries sweeping key tiles, S' and dP'
//     recomputed, dQ' += K' dS'.
// Masks: keys past the keys' length and, causal, keys after the query
// (key <= query, positions from 0) weigh 0; queries past the sequence are
// computed on zeros and not stored.
// Device-held masks (M; bf16 at d = 64 and 128, which the general kernels'
// vector ALUs ran before): a first key per query and a key count per sequence.
// A forward or dQ workgroup starts at its queries' least first key, a dK/dV
// workgroup finds the span of queries that see any of its keys, so packed
// documents cost their own pairs and not the sequence's.  The general kernels hold P and dS
// in fp32, so here each is three bf16 parts (split2_towards0) and takes three
// products, on operands that are bf16 already.  Rows may start at any element.
// B2 H12 S2048 d64 in documents of about 256, forward + backward: 5981 us on
// the general kernels, 111 here (99 with P and dS of 16 bits, beside it).
#include <hip/hip_runtime.h>

#include <cmath>

#include "attention_tiles.h"
#include "th_core.h"

namespace {

struct MArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;  // natural log, [b][s][h]
  const uint16_t* dout;
  float* delta;  // backward workspace: rowsum(dO .* O), [b][s][h]
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  int64_t q_sh, q_ss, q_sb;  // strides (elements) of q, o, dout, dq
  int64_t k_sh, k_ss, k_sb;  // strides of k, v, dk, dv
  int32_t seq, kv_seq, heads, kv_heads, batch, causal;
  float scale;
  // A sweep split into parts (small grids): nsplit parts of `span`
  // positions (a multiple of 64) each, fp32 partial results in `part`
  // ([part][b][position][head][d]) and, for the forward, (m, l) in
  // `part_ml`; nsplit <= 1: no split.
  int32_t nsplit, span;
  float* part;
  float* part_ml;
  // The backward's dQ sweep, beside the dK/dV one above.
  int32_t q_nsplit, q_span;
  float* q_part;
  const int32_t* starts;   // M only: (positions, batch), 1-based, or null
  const int32_t* lengths;  // M only: (batch), or null
};

// Global rows of M's arrays start at any element.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef u32x2 u32x2_any __attribute__((aligned(2)));

// The keys of sequence b (M: lengths[b] clamped to the keys' extent).
template <bool M>
__device__ __forceinline__ int keys_of(const MArgs& p, int b) {
  if constexpr (M)
    if (p.lengths) return min(max(p.lengths[b], 0), p.kv_seq);
  return p.kv_seq;
}

// The first key query j < seq of sequence b sees.
__device__ __forceinline__ int first_of(const MArgs& p, int j, int b) {
  return p.starts ? p.starts[(int64_t)j + (int64_t)p.seq * b] - 1 : 0;
}

// The largest of x over the wave's lanes with a query (INT_MAX: none).
__device__ __forceinline__ int most(int x) {
  if (x == 0x7fffffff) x = 0;
#pragma unroll
  for (int i = 1; i < 64; i *= 2) x = max(x, __shfl_xor(x, i, 64));
  return __builtin_amdgcn_readfirstlane(x);
}

// The least of x over the wave's lanes.
__device__ __forceinline__ int fewest(int x) {
#pragma unroll
  for (int i = 1; i < 64; i *= 2) x = min(x, __shfl_xor(x, i, 64));
  return __builtin_amdgcn_readfirstlane(x);
}

// M: whether any of a wave's queries, from q0 on, may see any of the 32 keys from
// k0: none before `first`, its least first key, nor, causal, after its last one.
// Products over keys leave out those of no use, whose values may be anything (a
// weight of 0 times an infinity or a NaN would be a NaN).
__device__ __forceinline__ bool of_use(const MArgs& p, int k0, int first, int q0) {
  return k0 + 32 > first && (!p.causal || k0 < q0 + 32);
}

// The least of x over the workgroup's 256 P threads, through 4 P ints of LDS; a
// barrier on both sides.
template <int P>
__device__ __forceinline__ int least(int x, int* at) {
#pragma unroll
  for (int i = 1; i < 64; i *= 2) x = min(x, __shfl_xor(x, i, 64));
  __syncthreads();
  if (threadIdx.x % 64 == 0) at[threadIdx.x / 64] = x;
  __syncthreads();
  x = at[0];
#pragma unroll
  for (int i = 1; i < 4 * P; ++i) x = min(x, at[i]);
  return x;
}

// P = 2: a workgroup of eight waves whose two halves take the tiles of one
// sweep in turn, each with stages of its own, the second handing its fp32 sums
// to the first through LDS at the end (a lane to the lane of the same place).
// A sweep is a chain of steps, each waiting for the one before (about 1.3 us a
// step of the forward: four take 14.2 us, sixteen 29.6); where the sweeps are of uneven
// length and few, the longest one is the launch's time, and this halves it.
// The host takes it up to these workgroups, us before and after:
//   causal forward whose keys are not split over workgroups, <= 512 (two a CU):
//     B2 H16 S1853 d64 (480) 40.5 -> 35.0, B1 H16 S4000 d128 (512) 118 -> 103;
//     1024: 54.6 -> 74.3, and sweeps of one length (not causal, 480) 45 -> 55.6,
//     already split ones 53.5 -> 58 (with the backward); short
//     sweeps in place of a split: beside the rule;
//   masked forward, <= 512: packed documents B2 H12 S2048 d64 (384), with the
//     backward 114 -> 106; 768 workgroups 110 -> 118;
//   masked backward at d64, <= 1024: the same documents (768) 106 -> 96,
//     1 x 1500 x 8 heads 132 -> 90 in all; 1152 workgroups 133 -> 145.
//   The unmasked backward gains nothing (600 workgroups 181 -> 192), and at d128
//   one wave a SIMD holds a sweep.
constexpr int64_t kFwdHalves = 512, kBwdHalves = 1024;

template <int N>
__device__ __forceinline__ void hand_over(const f32x16 (&x)[N], float* to) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) to[256 * (16 * i + e) + threadIdx.x % 256] = x[i][e];
}
template <int N>
__device__ __forceinline__ void take_over(f32x16 (&x)[N], const float* from) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) x[i][e] += from[256 * (16 * i + e) + threadIdx.x % 256];
}

__device__ __forceinline__ float bf16_float(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// A row of a (position-major) operand as the B operand of a product over d:
// d = 16 ks + 8 (lane / 32) + (0..7); zeros for a position past the end.
template <int D>
__device__ __forceinline__ void row_operand(const uint16_t* row, bool live, bf16x8 (&f)[D / 16]) {
  const int lane = threadIdx.x % 64;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    f[ks] = live ? (bf16x8)(u32x4) * reinterpret_cast<const u32x4_any*>(row + 16 * ks + 8 * (lane / 32)) : bf16x8{};
}

// A 64-position tile of an operand staged through registers: thread t holds
// the 16-byte chunks t + 256 i; rows past `limit` read as zeros.
template <int D>
struct Stage {
  static constexpr int kChunks = D / 8;          // per row
  static constexpr int kPer = 64 * kChunks / 256;  // per thread
  u32x4 r[kPer];
  __device__ void load(const uint16_t* base, int64_t ss, int row0, int limit) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = threadIdx.x % 256 + 256 * i, row = c / kChunks, col = c % kChunks;
      r[i] = row0 + row < limit ? (u32x4) * reinterpret_cast<const u32x4_any*>(base + (int64_t)(row0 + row) * ss + 8 * col)
                                : u32x4{0, 0, 0, 0};
    }
  }
  __device__ void store(uint16_t* t) const {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = threadIdx.x % 256 + 256 * i, row = c / kChunks, col = c % kChunks;
      *reinterpret_cast<u32x4*>(t + row * (D + 8) + 8 * col) = r[i];
    }
  }
};

template <int D>
constexpr int kTile = 64 * (D + 8);  // bf16 elements of a tile in LDS

// The grid is (heads, batch, blocks): blocks slowest, so that under a causal
// mask the longest sweeps start first and the short ones fill in behind them,
// and, (heads x batch) a multiple of 8, a head's blocks share an XCD's L2.
// (Before, a workgroup took a block and its mirror: even work, but half the
// workgroups, and the chip half empty where they are few.)

// ---- forward ---------------------------------------------------------------------

// Keys [k_lo, k_hi) of query block qb: all of them (split < 0), or part
// `split` of the sweep, which leaves its unnormalised O' and (m, l) for the
// combining kernel.
template <int D, bool M, int P>
__device__ __forceinline__ void fwd_block(const MArgs& p, const int qb, const int b, const int split) {
  constexpr int NS = D / 16, NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int h = blockIdx.x;
  const int hk = h / (p.heads / p.kv_heads);
  const int grp = P == 1 ? 0 : threadIdx.x / 256, wave = threadIdx.x / 64 % 4, lane = threadIdx.x % 64, lr = lane % 32, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lr;
  const uint16_t* qbase = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const uint16_t* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const uint16_t* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  bf16x8 qf[NS];
  row_operand<D>(qbase + (int64_t)query * p.q_ss, query < p.seq, qf);
  f32x16 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) o[i] = f32x16{};
  float m = -INFINITY, l = 0.0f;
  const float c = p.scale * kLog2e;
  const int nk = keys_of<M>(p, b), qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(nk, qlast + 1) : nk;
  int k_lo = split < 0 ? 0 : split * p.span, first = 0;
  if constexpr (M) {
    // The sweep starts at the block's least first key, a wave's share of it at the wave's.
    if (p.starts) {
      first = query < p.seq ? first_of(p, query, b) : 0x7fffffff;
      k_lo = max(0, min(least<P>(first, reinterpret_cast<int*>(lds + 4 * P * kTile<D>)), nk)) / 64 * 64;
    }
  }
  const int last_first = M ? most(first) : 0;  // tiles from here on see no first key
  const int least_first = M ? fewest(first) : 0;
  const int k_hi = split < 0 ? kend : min(kend, k_lo + p.span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  Stage<D> sk, sv;
  auto K = [&](int s) { return lds + (4 * grp + 2 * s) * kTile<D>; };
  auto V = [&](int s) { return lds + (4 * grp + 2 * s + 1) * kTile<D>; };
  const int mine = P == 1 ? nsteps : (nsteps + 1 - grp) / 2;  // tiles grp, grp + P, ...
  if (mine > 0) {
    sk.load(kbase, p.k_ss, k_lo + 64 * grp, nk);
    sv.load(vbase, p.k_ss, k_lo + 64 * grp, nk);
    sk.store(K(0));
    sv.store(V(0));
  }
  __syncthreads();
  auto step = [&](int j) {
    const int cur = j & 1, k0 = k_lo + 64 * (P * j + grp);
    if (j + 1 < mine) {
      sk.load(kbase, p.k_ss, k0 + 64 * P, nk);
      sv.load(vbase, p.k_ss, k0 + 64 * P, nk);
    }
    // S' (64 keys x 32 queries): keys 32 kb + 8 (i / 4) + 4 lh + i % 4 in register i.
    f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int ks = 0; ks < NS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] = mfma(frag_rows<D>(K(cur), 32 * kb, ks), qf[ks], s[kb]);
    const bool edge = k0 + 64 > nk || k0 < last_first || (p.causal && k0 + 63 > q0);
    if (edge) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
          if (key >= nk || (M && key < first) || (p.causal && key > query)) s[kb][i] = -INFINITY;
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
    if constexpr (M) {
      // O' (D x 32 queries) += V' P', the weights in three bf16 parts, 32 keys at a time.
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (edge && !of_use(p, k0 + 32 * kb, least_first, q0)) continue;
#pragma unroll
        for (int part = 0; part < 2; ++part) {
          u32x4 w, x, y;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w0 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * part + 2 * e], c, -shift));
            const float w1 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * part + 2 * e + 1], c, -shift));
            l += w0 + w1;
            uint32_t x0, x1, x2;
            split2_towards0(w0, w1, x0, x1, x2);
            w[e] = x0, x[e] = x1, y[e] = x2;
          }
#pragma unroll
          for (int db = 0; db < NB; ++db) {
            const bf16x8 vt = frag_tr<D>(V(cur), 32 * db, 2 * kb + part);
            o[db] = mfma(vt, (bf16x8)y, o[db]);
            o[db] = mfma(vt, (bf16x8)x, o[db]);
            o[db] = mfma(vt, (bf16x8)w, o[db]);
          }
        }
      }
    } else {
      bf16x8 pf[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int part = 0; part < 2; ++part) {
          u32x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w0 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * part + 2 * e], c, -shift));
            const float w1 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * part + 2 * e + 1], c, -shift));
            l += w0 + w1;
            w[e] = pack2(w0, w1);
          }
          pf[2 * kb + part] = (bf16x8)w;
        }
      // O' (D x 32 queries) += V' P', the weights rounded to bf16.
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int db = 0; db < NB; ++db) o[db] = mfma(frag_tr<D>(V(cur), 32 * db, ks), pf[ks], o[db]);
    }
    if (j + 1 < mine) {
      // The other stage was last read in step j - 1, before the barrier that ended it.
      sk.store(K(cur ^ 1));
      sv.store(V(cur ^ 1));
    }
  };
  for (int j = 0; P * j < nsteps; ++j) {
    if (P == 1 || j < mine) step(j);
    __syncthreads();
  }
  if constexpr (P == 2) {
    float* x = reinterpret_cast<float*>(lds);
    float* ml = x + 256 * 16 * NB;
    if (grp == 1) {
      hand_over(o, x);
      ml[threadIdx.x % 256] = m, ml[256 + threadIdx.x % 256] = l;
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = ml[threadIdx.x], mn = fmaxf(m, m1), shift = thd::lse_shift(mn);
    const float a0 = __builtin_amdgcn_exp2f(m - shift), a1 = __builtin_amdgcn_exp2f(m1 - shift);
    l = l * a0 + ml[256 + threadIdx.x] * a1;
    m = mn;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[i][e] = o[i][e] * a0 + x[256 * (16 * i + e) + threadIdx.x] * a1;
  }
  l += other_half(l);
  if (query >= p.seq) return;
  if (split >= 0) {
    // This part's unnormalised O' and (m, l) (m = -inf, l = 0 where it saw no key).
    const int64_t row = (((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h;
    float* po = p.part + row * D;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(po + 32 * db + 8 * g + 4 * lh) =
            f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
    if (lh == 0) reinterpret_cast<f32x2*>(p.part_ml)[row] = f32x2{m, l};
    return;
  }
  const float inv = 1.0f / l;
  uint16_t* obase = p.o + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss;
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * db + 8 * g + 4 * lh;
      *reinterpret_cast<u32x2_any*>(obase + d) =
          u32x2{pack2(o[db][4 * g] * inv, o[db][4 * g + 1] * inv), pack2(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv)};
    }
  if (lh == 0 && p.lse) p.lse[((int64_t)b * p.seq + query) * p.heads + h] = (m + log2f(l)) * kLn2;
}

template <int D, bool M, int P>
__global__ __launch_bounds__(256 * P, D <= 128 ? 2 : 1) void mfma_attn_fwd(MArgs p) {
  const bool split = p.nsplit > 1;
  const int z = gridDim.z - 1 - blockIdx.z;  // the last queries, the longest sweeps, first
  fwd_block<D, M, P>(p, split ? z / p.nsplit : z, blockIdx.y, split ? z % p.nsplit : -1);
}

// The parts of a split forward combined: per (b, query, head) row, M = max
// m_s, L = sum l_s 2^(m_s - M), O = sum O_s 2^(m_s - M) / L in part order;
// lse = (M + log2 L) ln 2.  A thread per four features of a row.
struct CombineArgs {
  MArgs p;  // first: its members sit at MArgs' offsets
  int32_t d;
};

__global__ __launch_bounds__(256) void mfma_attn_combine(CombineArgs a) {
  const MArgs& p = a.p;
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
  const float inv = 1.0f / l;
  *reinterpret_cast<u32x2*>(p.o + b * p.q_sb + h * p.q_sh + pos * p.q_ss + c) =
      u32x2{pack2(acc[0] * inv, acc[1] * inv), pack2(acc[2] * inv, acc[3] * inv)};
  if (c == 0 && p.lse) p.lse[row] = (mx + log2f(l)) * kLn2;
}

// dK, dV and dQ from split sweeps' parts, one launch: out = scale * sum_s
// part_s in part order, rounded to bf16; rows [b][position][head] of `d` features.
struct SumArgsOne {
  const float* part;
  uint16_t* out;
  int64_t sh, ss, sb;
  int32_t positions, heads, nsplit;
  float scale;
  uint32_t blocks;  // workgroups, 256 quads of features each
};
struct SumArgs {
  SumArgsOne of[3];
  int32_t n, batch, d;
};

__global__ __launch_bounds__(256) void mfma_attn_sum(SumArgs all) {
  uint32_t block = blockIdx.x;
  int which = 0;
  while (which + 1 < all.n && block >= all.of[which].blocks) block -= all.of[which++].blocks;
  const SumArgsOne& a = all.of[which];
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
  *reinterpret_cast<u32x2*>(a.out + b * a.sb + h * a.sh + pos * a.ss + c) =
      u32x2{pack2(acc[0], acc[1]), pack2(acc[2], acc[3])};
}

// ---- backward: delta = rowsum(dO .* O) ---------------------------------------------

struct DeltaArgs {
  MArgs p;  // first: its members sit at MArgs' offsets
  int32_t d;
};

// D / 8 lanes per (batch, position, head) row, 16 bytes each; each lane group takes kDeltaRowsM
// rows, 64 / (D / 8) apart, every load issued before the first product.
// Rows are numbered with the head fastest, so a load instruction covers
// consecutive rows; row numbers fit 32 bits (the builder checks).
constexpr int kDeltaRowsM = 4;

template <int D>
__global__ __launch_bounds__(256) void mfma_attn_delta(DeltaArgs a) {
  constexpr int G = D / 8;        // lanes a row
  constexpr int R = 64 / G;       // rows a wave covers at once
  const MArgs& p = a.p;
  const uint32_t total = (uint32_t)p.batch * p.seq * p.heads;
  const int lane = threadIdx.x % 64, part = lane % G;
  const uint32_t row0 = (blockIdx.x * 4 + threadIdx.x / 64) * (R * kDeltaRowsM) + lane / G;
  auto at_of = [&](uint32_t row) {
    const uint32_t bs = row / (uint32_t)p.heads;
    const int64_t b = bs / (uint32_t)p.seq, s = bs % (uint32_t)p.seq, h = row - bs * (uint32_t)p.heads;
    return b * p.q_sb + h * p.q_sh + s * p.q_ss + 8 * part;
  };
  u32x4 ow[kDeltaRowsM], gw[kDeltaRowsM];
#pragma unroll
  for (int i = 0; i < kDeltaRowsM; ++i) {
    // Rows past the end re-read the last one; nothing is written for them.
    const int64_t at = at_of(min(row0 + R * i, total - 1));
    ow[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p.o + at));
    gw[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p.dout + at));
  }
  // Every load out before any of their data is used.
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kDeltaRowsM; ++i) {
    float v = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v += bf16_float((uint16_t)ow[i][e]) * bf16_float((uint16_t)gw[i][e]) +
           bf16_float((uint16_t)(ow[i][e] >> 16)) * bf16_float((uint16_t)(gw[i][e] >> 16));
#pragma unroll
    for (int m = G / 2; m >= 1; m /= 2) v += __shfl_xor(v, m, G);
    const uint32_t row = row0 + R * i;
    if (row < total && part == 0) p.delta[row] = v;
  }
}

// ---- backward: dK, dV ----------------------------------------------------------------
// A workgroup takes 128 keys (32 a wave) and DO of the D features of dK and
// dV (D, or half of 256).  Per query tile of 64: S (64 queries x 32 keys)
// with queries on the registers and keys on the lanes, so that P and dS feed
// the products over queries straight from the accumulators.

// Half a step: 32 queries (half jj of the tile) against the wave's 32 keys.
// `edge`: some pair of them may be masked (compares and selects on every score
// are a quarter of the step's vector work, so whole tiles go without).
template <int D, int DO, bool M>
__device__ __forceinline__ void dkdv_half(const MArgs& p, const uint16_t* Qt, const uint16_t* Gt, const float* L,
                                          const int jj, const bool edge, int qq0, int key, int nk, int dh,
                                          const bf16x8 (&kf)[D / 16], const bf16x8 (&vf)[D / 16],
                                          f32x16 (&dk)[DO / 32], f32x16 (&dv)[DO / 32]) {
  const int lh = threadIdx.x % 64 / 32;
  const float c = p.scale * kLog2e;
  // S = Q K', dP = dO V' (32 queries x 32 keys): query 32 jj + 8 (i / 4) + 4 lh + i % 4 in register i.
  f32x16 s = f32x16{}, dp = f32x16{};
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    s = mfma(frag_rows<D>(Qt, 32 * jj, ks), kf[ks], s);
    dp = mfma(frag_rows<D>(Gt, 32 * jj, ks), vf[ks], dp);
  }
  // P into s, dS into dp.
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int qi = 32 * jj + 8 * (i / 4) + 4 * lh + i % 4;
    s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -L[qi]));
    dp[i] = s[i] * (dp[i] - L[64 + qi]);
    if constexpr (M) dp[i] += 0.0f;  // no -0 (split2_towards0)
  }
  if (edge) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qi = 32 * jj + 8 * (i / 4) + 4 * lh + i % 4, query = qq0 + qi;
      bool seen = query < p.seq && key < nk && (!p.causal || key <= query);
      if constexpr (M) seen = seen && key >= __float_as_int(L[128 + qi]);
      s[i] = seen ? s[i] : 0.0f;
      dp[i] = seen ? dp[i] : 0.0f;
    }
  }
#pragma unroll
  for (int part = 0; part < 2; ++part) {
    u32x4 ph, pm, pl, sh, sm, sl;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 8 * part + 2 * e;
      if constexpr (M) {
        uint32_t x0, x1, x2;
        split2_towards0(s[i], s[i + 1], x0, x1, x2);
        ph[e] = x0, pm[e] = x1, pl[e] = x2;
        split2_towards0(dp[i], dp[i + 1], x0, x1, x2);
        sh[e] = x0, sm[e] = x1, sl[e] = x2;
      } else {
        ph[e] = pack2(s[i], s[i + 1]), sh[e] = pack2(dp[i], dp[i + 1]);
      }
    }
    // dV' (DO features x 32 keys) += dO' P;  dK' += Q' dS.
#pragma unroll
    for (int db = 0; db < DO / 32; ++db) {
      const bf16x8 g = frag_tr<D>(Gt, DO * dh + 32 * db, 2 * jj + part), q = frag_tr<D>(Qt, DO * dh + 32 * db, 2 * jj + part);
      if constexpr (M) {
        dv[db] = mfma(g, (bf16x8)pl, dv[db]);
        dk[db] = mfma(q, (bf16x8)sl, dk[db]);
        dv[db] = mfma(g, (bf16x8)pm, dv[db]);
        dk[db] = mfma(q, (bf16x8)sm, dk[db]);
      }
      dv[db] = mfma(g, (bf16x8)ph, dv[db]);
      dk[db] = mfma(q, (bf16x8)sh, dk[db]);
    }
  }
}

// Query tiles [qstart, qstop) for the keys of kblk: all of them (split <
// 0), or part `split` of the sweep, which leaves its unscaled fp32 dK', dV'.
template <int D, int DO, bool M, int P>
__device__ __forceinline__ void dkdv_block(const MArgs& p, const int kblk, const int dh, const int hk, const int b,
                                           const int split) {
  constexpr int NS = D / 16, NBO = DO / 32;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  constexpr int kStats = M ? 196 : 128;
  // [stage][lse * log2e (64) | delta (64) | M: first keys, as ints (64) | their largest (1) | -]
  float* stats = reinterpret_cast<float*>(lds + 4 * P * kTile<D>);
  const int group = p.heads / p.kv_heads;
  const int grp = P == 1 ? 0 : threadIdx.x / 256, tid = P == 1 ? threadIdx.x : threadIdx.x % 256, wave = tid / 64, lane = threadIdx.x % 64, lr = lane % 32, lh = lane / 32;
  const int kw0 = kblk * 128, key = kw0 + wave * 32 + lr;
  const int64_t koff = (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  bf16x8 kf[NS], vf[NS];
  const int nk = keys_of<M>(p, b);
  row_operand<D>(p.k + koff + (int64_t)key * p.k_ss, key < nk, kf);
  row_operand<D>(p.v + koff + (int64_t)key * p.k_ss, key < nk, vf);
  f32x16 dk[NBO], dv[NBO];
#pragma unroll
  for (int i = 0; i < NBO; ++i) dk[i] = f32x16{}, dv[i] = f32x16{};
  auto Q = [&](int s) { return lds + (4 * grp + 2 * s) * kTile<D>; };
  auto G = [&](int s) { return lds + (4 * grp + 2 * s + 1) * kTile<D>; };
  auto Ls = [&](int s) { return stats + kStats * (2 * grp + s); };
  const int qfirst = p.causal ? kw0 / 64 * 64 : 0;
  int qstart = split < 0 ? qfirst : qfirst + split * p.span;
  int qstop = split < 0 ? p.seq : min(p.seq, qstart + p.span);
  if constexpr (M) {
    if (kw0 >= nk) qstop = qstart;  // no key of the block: zeros
    if (p.starts && kw0 < nk) {
      // The span of queries that see any of the block's keys.
      int lo = 0x7fffffff, hi = 0x7fffffff;  // hi: the least of -j
      for (int j = qstart + threadIdx.x; j < qstop; j += 256 * P)
        if (first_of(p, j, b) < kw0 + 128) lo = min(lo, j), hi = min(hi, -j);
      int* at = reinterpret_cast<int*>(stats + 2 * P * kStats);
      lo = least<P>(lo, at), hi = least<P>(hi, at);
      qstop = lo == 0x7fffffff ? qstart : 1 - hi;
      qstart = lo == 0x7fffffff ? qstart : lo / 64 * 64;
    }
  }
  const int nsteps = qstart < qstop ? (qstop - qstart + 63) / 64 : 0;
  const int mine = P == 1 ? nsteps : (nsteps + 1 - grp) / 2;  // tiles grp, grp + P, ...
  Stage<D> sq, sg;
  int st_most = 0;
  float st = 0.0f;  // threads 0..127: a query's lse * log2e or delta
  auto load = [&](const uint16_t* qbase, const uint16_t* gbase, int h, int q0) {
    sq.load(qbase, p.q_ss, q0, p.seq);
    sg.load(gbase, p.q_ss, q0, p.seq);
    if (tid < 128) {
      const int j = q0 + tid % 64;
      const int64_t row = ((int64_t)b * p.seq + j) * p.heads + h;
      st = j < p.seq ? (tid < 64 ? p.lse[row] * kLog2e : p.delta[row]) : 0.0f;
    } else if (M && tid < 192) {
      const int j = q0 + tid % 64;
      const int f = j < p.seq ? first_of(p, j, b) : 0x7fffffff;
      st = __int_as_float(f), st_most = most(f);
    }
  };
  auto store = [&](int s) {
    sq.store(Q(s));
    sg.store(G(s));
    if (tid < (M ? 192 : 128)) Ls(s)[tid] = st;
    if (M && tid == 128) Ls(s)[192] = __int_as_float(st_most);
  };
  for (int h = hk * group; h < (hk + 1) * group; ++h) {
    const uint16_t* qbase = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    const uint16_t* gbase = p.dout + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    if (mine > 0) {
      load(qbase, gbase, h, qstart + 64 * grp);
      store(0);
    }
    __syncthreads();
    auto step = [&](int j) {
      const int cur = j & 1, qq0 = qstart + 64 * (P * j + grp);
      if (j + 1 < mine) load(qbase, gbase, h, qq0 + 64 * P);
      const uint16_t *Qt = Q(cur), *Gt = G(cur);
      const float* L = Ls(cur);
      const int kw = __builtin_amdgcn_readfirstlane(kw0 + wave * 32);
      bool edge = qq0 + 64 > p.seq || kw + 32 > nk || (p.causal && kw + 31 > qq0);
      if constexpr (M) edge = edge || kw < __builtin_amdgcn_readfirstlane(__float_as_int(L[192]));
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        if (M && p.causal && qq0 + 32 * jj + 31 < kw) continue;  // queries before the wave's keys (as of_use)
        dkdv_half<D, DO, M>(p, Qt, Gt, L, jj, edge, qq0, key, nk, dh, kf, vf, dk, dv);
      }
      if (j + 1 < mine) store(cur ^ 1);
    };
    for (int j = 0; P * j < nsteps; ++j) {
      if (P == 1 || j < mine) step(j);
      __syncthreads();
    }
  }
  if constexpr (P == 2) {
    float* x = reinterpret_cast<float*>(lds);
    if (grp == 1) {
      hand_over(dk, x);
      hand_over(dv, x + 256 * 16 * NBO);
    }
    __syncthreads();
    if (grp == 1) return;
    take_over(dk, x);
    take_over(dv, x + 256 * 16 * NBO);
  }
  // At D = 128 the key as an opaque copy, so that the output addresses below
  // are computed here rather than kept from the sweep's start: measured 4 %
  // faster there; at D = 64 (4 registers spilled around the sweep otherwise)
  // and D = 256 the kept addresses measured faster.
  int ko = key;
  if constexpr (D == 128) asm volatile("" : "+v"(ko));
  if (ko >= p.kv_seq) return;
  if (M && ko >= nk) {  // past the sequence's length: zeros, whatever the gradients are
#pragma unroll
    for (int i = 0; i < NBO; ++i) dk[i] = f32x16{}, dv[i] = f32x16{};
  }
  if (split >= 0) {
    const int64_t rows = (int64_t)p.batch * p.kv_seq * p.kv_heads;
    const int64_t row = (((int64_t)split * p.batch + b) * p.kv_seq + ko) * p.kv_heads + hk;
    float* pk = p.part + row * D;
    float* pv = p.part + ((int64_t)p.nsplit * rows + row) * D;
#pragma unroll
    for (int db = 0; db < NBO; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = DO * dh + 32 * db + 8 * g + 4 * lh;
        *reinterpret_cast<f32x4*>(pk + d) = f32x4{dk[db][4 * g], dk[db][4 * g + 1], dk[db][4 * g + 2], dk[db][4 * g + 3]};
        *reinterpret_cast<f32x4*>(pv + d) = f32x4{dv[db][4 * g], dv[db][4 * g + 1], dv[db][4 * g + 2], dv[db][4 * g + 3]};
      }
    return;
  }
  const int64_t out = koff + (int64_t)ko * p.k_ss;
#pragma unroll
  for (int db = 0; db < NBO; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = DO * dh + 32 * db + 8 * g + 4 * lh;
      const float sc = p.scale;
      *reinterpret_cast<u32x2_any*>(p.dk + out + d) =
          u32x2{pack2(dk[db][4 * g] * sc, dk[db][4 * g + 1] * sc), pack2(dk[db][4 * g + 2] * sc, dk[db][4 * g + 3] * sc)};
      *reinterpret_cast<u32x2_any*>(p.dv + out + d) =
          u32x2{pack2(dv[db][4 * g], dv[db][4 * g + 1]), pack2(dv[db][4 * g + 2], dv[db][4 * g + 3])};
    }
}

// ---- backward: dQ ----------------------------------------------------------------------
// A workgroup takes 128 queries (32 a wave) and sweeps key tiles of 64:
// S' = K Q', dP' = V dO' (keys on the registers, queries on the lanes),
// dS' = P' (dP' - delta), dQ' (D x 32 queries) += K' dS'.

// Keys [k_lo, k_hi) for query block qb: all of them (split < 0), or part
// `split` of the sweep, which leaves its unscaled fp32 dQ'.
template <int D, bool M, int P>
__device__ __forceinline__ void dq_block(const MArgs& p, const int qb, const int h, const int b, const int split) {
  constexpr int NS = D / 16, NB = D / 32;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int hk = h / (p.heads / p.kv_heads);
  const int grp = P == 1 ? 0 : threadIdx.x / 256, wave = threadIdx.x / 64 % 4, lane = threadIdx.x % 64, lr = lane % 32, lh = lane / 32;
  const int q0 = __builtin_amdgcn_readfirstlane(qb * 128 + wave * 32), query = q0 + lr;
  const int64_t qoff = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)query * p.q_ss;
  const bool live = query < p.seq;
  bf16x8 qf[NS], gf[NS];
  row_operand<D>(p.q + qoff, live, qf);
  row_operand<D>(p.dout + qoff, live, gf);
  const int64_t srow = ((int64_t)b * p.seq + query) * p.heads + h;
  const float l2 = live ? p.lse[srow] * kLog2e : 0.0f;
  const float dl = live ? p.delta[srow] : 0.0f;
  const float c = p.scale * kLog2e;
  const uint16_t* kbase = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const uint16_t* vbase = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  f32x16 dq[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) dq[i] = f32x16{};
  const int nk = keys_of<M>(p, b), qlast = min(qb * 128 + 127, p.seq - 1);
  const int kend = p.causal ? min(nk, qlast + 1) : nk;
  int k_lo = split < 0 ? 0 : split * p.q_span, first = 0;
  if constexpr (M) {
    // The sweep starts at the block's least first key, a wave's share of it at the wave's.
    if (p.starts) {
      first = query < p.seq ? first_of(p, query, b) : 0x7fffffff;
      k_lo = max(0, min(least<P>(first, reinterpret_cast<int*>(lds + 4 * P * kTile<D>)), nk)) / 64 * 64;
    }
  }
  const int last_first = M ? most(first) : 0;  // tiles from here on see no first key
  const int least_first = M ? fewest(first) : 0;
  const int k_hi = split < 0 ? kend : min(kend, k_lo + p.q_span);
  const int nsteps = k_hi > k_lo ? (k_hi - k_lo + 63) / 64 : 0;
  Stage<D> sk, sv;
  auto K = [&](int s) { return lds + (4 * grp + 2 * s) * kTile<D>; };
  auto V = [&](int s) { return lds + (4 * grp + 2 * s + 1) * kTile<D>; };
  const int mine = P == 1 ? nsteps : (nsteps + 1 - grp) / 2;  // tiles grp, grp + P, ...
  if (mine > 0) {
    sk.load(kbase, p.k_ss, k_lo + 64 * grp, nk);
    sv.load(vbase, p.k_ss, k_lo + 64 * grp, nk);
    sk.store(K(0));
    sv.store(V(0));
  }
  __syncthreads();
  auto step = [&](int j) {
    const int cur = j & 1, k0 = k_lo + 64 * (P * j + grp);
    if (j + 1 < mine) {
      sk.load(kbase, p.k_ss, k0 + 64 * P, nk);
      sv.load(vbase, p.k_ss, k0 + 64 * P, nk);
    }
    if constexpr (M) {
      // 32 keys at a time, dS in three bf16 parts.
      const bool edge = k0 + 64 > nk || k0 < last_first || (p.causal && k0 + 63 > q0);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (edge && !of_use(p, k0 + 32 * kb, least_first, q0)) continue;
        f32x16 s = {}, dp = {};
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) {
          s = mfma(frag_rows<D>(K(cur), 32 * kb, ks), qf[ks], s);
          dp = mfma(frag_rows<D>(V(cur), 32 * kb, ks), gf[ks], dp);
        }
        // dS' into dp, without a -0 (split2_towards0).
#pragma unroll
        for (int i = 0; i < 16; ++i)
          dp[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c, -l2)) * (dp[i] - dl) + 0.0f;
        if (edge) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
            dp[i] = key < nk && key >= first && (!p.causal || key <= query) ? dp[i] : 0.0f;
          }
        }
#pragma unroll
        for (int part = 0; part < 2; ++part) {
          u32x4 w, x, y;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            uint32_t x0, x1, x2;
            split2_towards0(dp[8 * part + 2 * e], dp[8 * part + 2 * e + 1], x0, x1, x2);
            w[e] = x0, x[e] = x1, y[e] = x2;
          }
#pragma unroll
          for (int db = 0; db < NB; ++db) {
            const bf16x8 kt = frag_tr<D>(K(cur), 32 * db, 2 * kb + part);
            dq[db] = mfma(kt, (bf16x8)y, dq[db]);
            dq[db] = mfma(kt, (bf16x8)x, dq[db]);
            dq[db] = mfma(kt, (bf16x8)w, dq[db]);
          }
        }
      }
    } else {
      f32x16 s[2] = {f32x16{}, f32x16{}}, dp[2] = {f32x16{}, f32x16{}};
#pragma unroll
      for (int ks = 0; ks < NS; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          s[kb] = mfma(frag_rows<D>(K(cur), 32 * kb, ks), qf[ks], s[kb]);
          dp[kb] = mfma(frag_rows<D>(V(cur), 32 * kb, ks), gf[ks], dp[kb]);
        }
      // dS' into dp, masked where the tile needs it.
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          dp[kb][i] = __builtin_amdgcn_exp2f(fmaf(s[kb][i], c, -l2)) * (dp[kb][i] - dl);
      if (k0 + 64 > nk || (p.causal && k0 + 63 > q0)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * kb + 8 * (i / 4) + 4 * lh + i % 4;
            dp[kb][i] = key < nk && (!p.causal || key <= query) ? dp[kb][i] : 0.0f;
          }
      }
      bf16x8 sf[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int part = 0; part < 2; ++part) {
          u32x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = pack2(dp[kb][8 * part + 2 * e], dp[kb][8 * part + 2 * e + 1]);
          sf[2 * kb + part] = (bf16x8)w;
        }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int db = 0; db < NB; ++db) dq[db] = mfma(frag_tr<D>(K(cur), 32 * db, ks), sf[ks], dq[db]);
    }
    if (j + 1 < mine) {
      sk.store(K(cur ^ 1));
      sv.store(V(cur ^ 1));
    }
  };
  for (int j = 0; P * j < nsteps; ++j) {
    if (P == 1 || j < mine) step(j);
    __syncthreads();
  }
  if constexpr (P == 2) {
    float* x = reinterpret_cast<float*>(lds);
    if (grp == 1) hand_over(dq, x);
    __syncthreads();
    if (grp == 1) return;
    take_over(dq, x);
  }
  if (!live) return;
  if (split >= 0) {
    const int64_t row = (((int64_t)split * p.batch + b) * p.seq + query) * p.heads + h;
    float* pq = p.q_part + row * D;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(pq + 32 * db + 8 * g + 4 * lh) =
            f32x4{dq[db][4 * g], dq[db][4 * g + 1], dq[db][4 * g + 2], dq[db][4 * g + 3]};
    return;
  }
  uint16_t* out = p.dq + qoff;
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * db + 8 * g + 4 * lh;
      const float sc = p.scale;
      *reinterpret_cast<u32x2_any*>(out + d) =
          u32x2{pack2(dq[db][4 * g] * sc, dq[db][4 * g + 1] * sc), pack2(dq[db][4 * g + 2] * sc, dq[db][4 * g + 3] * sc)};
    }
}

// Both sweeps in one launch: neither needs the other, and alone each leaves
// the device part empty at its end (and, on small grids, all along).  The
// first p's dK/dV workgroups, the first keys, the longest causal sweeps, first;
// then the dQ ones, the last queries first.
struct BwdArgs {
  MArgs p;  // first: its members sit at MArgs' offsets
  uint32_t n_dkdv;
};

template <int D, int DO, bool M, int P>
__global__ __launch_bounds__(256 * P, D <= 64 ? 2 : 1) void mfma_attn_bwd(BwdArgs a) {
  const MArgs& p = a.p;
  if (blockIdx.x < a.n_dkdv) {
    constexpr int halves = D / DO;
    const int hk = blockIdx.x % p.kv_heads, b = blockIdx.x / p.kv_heads % p.batch, z = blockIdx.x / p.kv_heads / p.batch;
    const bool split = p.nsplit > 1;
    const int x = split ? z / p.nsplit : z;
    dkdv_block<D, DO, M, P>(p, x / halves, x % halves, hk, b, split ? z % p.nsplit : -1);
    return;
  }
  const uint32_t i = gridDim.x - 1 - blockIdx.x;  // (from the end: the last queries first)
  const int h = i % p.heads, b = i / p.heads % p.batch, z = i / p.heads / p.batch;
  const bool split = p.q_nsplit > 1;
  dq_block<D, M, P>(p, split ? z / p.q_nsplit : z, h, b, split ? z % p.q_nsplit : -1);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

MArgs margs_of(const th_attention_desc* d) {
  MArgs a{};
  a.q = static_cast<const uint16_t*>(d->q);
  a.k = static_cast<const uint16_t*>(d->k);
  a.v = static_cast<const uint16_t*>(d->v);
  a.o = static_cast<uint16_t*>(d->o);
  a.lse = d->lse;
  a.dout = static_cast<const uint16_t*>(d->dout);
  a.dq = static_cast<uint16_t*>(d->dq);
  a.dk = static_cast<uint16_t*>(d->dk);
  a.dv = static_cast<uint16_t*>(d->dv);
  a.q_sh = d->q_strides[0], a.q_ss = d->q_strides[1], a.q_sb = d->q_strides[2];
  a.k_sh = d->k_strides[0], a.k_ss = d->k_strides[1], a.k_sb = d->k_strides[2];
  a.seq = d->seq;
  a.kv_seq = d->kv_seq > 0 ? d->kv_seq : d->seq;
  a.heads = d->heads, a.kv_heads = d->kv_heads, a.batch = d->batch, a.causal = d->causal;
  a.scale = d->scale > 0 ? d->scale : 1.0f / sqrtf((float)d->head_dim);
  a.starts = d->starts, a.lengths = d->lengths;
  return a;
}

// (query, key) pairs the mask leaves: the algorithmic work's count.
double visible_pairs(const MArgs& a) {
  const double S = a.seq, K = a.kv_seq;
  if (!a.causal) return S * K;
  // sum over queries q of min(q + 1, K)
  const double full = std::min(S, K);
  return full * (full + 1) / 2 + std::max(0.0, S - K) * K;
}

template <int D>
int fwd_launch(const th_attention_desc* d, th_launch** out) {
  MArgs a = margs_of(d);
  const int nqb = (d->seq + 127) / 128;
  const int64_t groups = (int64_t)nqb * d->heads * d->batch;
  th::Split sp = th::split_of(groups, a.kv_seq);
  bool halves = sp.n == 1 && d->causal && groups <= kFwdHalves;
  // Short sweeps that would be split: halves in place of a twofold split, without its
  // partial results and (whole) its second launch.  us, split alone and so, forward:
  // whole, B2 H8 S512 d64 causal (64 workgroups) 14.4, 11.3; B1 H16 S700 d128 (96)
  // 26.3, 19.7 and not causal 28.8, 21.3; half the parts, B1 H4 S1000 d64 (32) 16.0,
  // 14.5, S2000 19.4, 18.4, B2 H8 S1024 18.4, 18.1.  Longer ones fill the device
  // better split: B1 H2 S8000 d64 46.5, halved 63.7; whole S1024 d128 (24) 18.0, 27.4.
  if (D <= 128 && sp.n > 1 && a.kv_seq <= 768 && groups >= 64) {
    sp = {1, 0}, halves = true;
  } else if (D == 64 && sp.n >= 4 && a.kv_seq <= 2048) {
    const int n = sp.n / 2, span = ((a.kv_seq + n - 1) / n + 63) / 64 * 64;
    sp = {(a.kv_seq + span - 1) / span, span}, halves = true;
  }
  a.nsplit = sp.n, a.span = sp.span;
  th::Builder b("attention_fwd_mfma", 7);
  const dim3 grid(d->heads, d->batch, nqb * sp.n);
  const int P = D <= 128 && halves ? 2 : 1;
  const size_t lds = 4 * P * (size_t)kTile<D> * sizeof(uint16_t);
  const void* fn = P == 2 ? (const void*)mfma_attn_fwd<D, false, D <= 128 ? 2 : 1> : (const void*)mfma_attn_fwd<D, false, 1>;
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  int k = b.kernel(fn, D == 64 ? "mfma_attn_fwd_d64" : D == 128 ? "mfma_attn_fwd_d128"
                                                                                          : "mfma_attn_fwd_d256",
                   grid, dim3(256 * P), (uint32_t)lds, a);
  b.ref(0, k, TH_OFFSET(MArgs, q));
  b.ref(1, k, TH_OFFSET(MArgs, k));
  b.ref(2, k, TH_OFFSET(MArgs, v));
  b.ref(3, k, TH_OFFSET(MArgs, o));
  b.ref(4, k, TH_OFFSET(MArgs, lse));
  if (sp.n > 1) {
    const int64_t rows = (int64_t)d->batch * d->seq * d->heads;
    const uint64_t at_o = b.workspace((uint64_t)sp.n * rows * D * sizeof(float));
    const uint64_t at_ml = b.workspace((uint64_t)sp.n * rows * 2 * sizeof(float));
    int kc = b.kernel((const void*)mfma_attn_combine, "mfma_attn_combine", dim3((unsigned)((rows * (D / 4) + 255) / 256)),
                      dim3(256), 0, CombineArgs{a, D});
    for (int kk : {k, kc}) {
      b.ws_ref(kk, TH_OFFSET(MArgs, part), at_o);
      b.ws_ref(kk, TH_OFFSET(MArgs, part_ml), at_ml);
    }
    b.ref(3, kc, TH_OFFSET(MArgs, o));
    b.ref(4, kc, TH_OFFSET(MArgs, lse));
  }
  for (int v = 0; v < 4; ++v) b.align(v, 16);
  const double BH = (double)d->batch * d->heads, BHk = (double)d->batch * d->kv_heads;
  b.work(2.0 * BH * a.seq * D * 2 + 2.0 * BHk * a.kv_seq * D * 2 + 4.0 * BH * a.seq, 4.0 * BH * D * visible_pairs(a),
         (int64_t)grid.x * grid.y * grid.z);
  *out = b.release();
  return TH_OK;
}

constexpr int kMaskLds = 2 * 196 * sizeof(float) + 16;  // under masks: the dK/dV stages' statistics and four ints

// The backward's launch: delta, both sweeps, and where small grids split
// them (the dK/dV sweep over queries, the dQ sweep over keys) their sums.
template <int D, bool M>
int bwd_launch(const th_attention_desc* d, th_launch** out) {
  constexpr int DO = D == 256 ? 128 : D;
  MArgs a = margs_of(d);
  th::Builder b("attention_bwd_mfma", 11);
  const int64_t rows = (int64_t)d->batch * d->seq * d->heads;
  const int64_t rows_k = (int64_t)d->batch * a.kv_seq * d->kv_heads;
  TH_REQUIRE(rows < 2147483648LL, "attention: batch x seq x heads must be under 2^31");
  const uint64_t at_delta = b.workspace((uint64_t)rows * sizeof(float));
  const int nkb = (a.kv_seq + 127) / 128, nqb = (d->seq + 127) / 128;
  const int64_t gkv = (int64_t)nkb * (D / DO) * d->kv_heads * d->batch, gq = (int64_t)nqb * d->heads * d->batch;
  const th::Split skv = M ? th::Split{1, 0} : th::split_of(gkv, d->seq, 384), sq = M ? th::Split{1, 0} : th::split_of(gq, a.kv_seq, 384);
  a.nsplit = skv.n, a.span = skv.span;
  a.q_nsplit = sq.n, a.q_span = sq.span;
  const int64_t n_dkdv = gkv * skv.n, blocks = n_dkdv + gq * sq.n;
  TH_REQUIRE(blocks <= 0x7fffffff, "attention: grid too large");
  const int P = D == 64 && M && blocks <= kBwdHalves ? 2 : 1;
  const size_t lds = P * (4 * (size_t)kTile<D> * sizeof(uint16_t) + (M ? kMaskLds : 2 * 128 * sizeof(float)));
  const void* fn = P == 2 ? (const void*)mfma_attn_bwd<D, DO, M, D == 64 && M ? 2 : 1> : (const void*)mfma_attn_bwd<D, DO, M, 1>;
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  constexpr int kDeltaBlockRows = 4 * (64 / (D / 8)) * kDeltaRowsM;  // rows a workgroup
  const int k0 = b.kernel((const void*)mfma_attn_delta<D>, "mfma_attn_delta",
                          dim3((unsigned)((rows + kDeltaBlockRows - 1) / kDeltaBlockRows)), dim3(256), 0, DeltaArgs{a, D});
  const char* name = M ? (D == 64 ? "mfma_attn_dkdv_masked_d64_mfma_attn_dq_masked_d64" : "mfma_attn_dkdv_masked_d128_mfma_attn_dq_masked_d128")
                       : D == 64    ? "mfma_attn_dkdv_d64_mfma_attn_dq_d64"
                       : D == 128   ? "mfma_attn_dkdv_d128_mfma_attn_dq_d128"
                                    : "mfma_attn_dkdv_d256_mfma_attn_dq_d256";
  const int k1 = b.kernel(fn, name, dim3((unsigned)blocks), dim3(256 * P), (uint32_t)lds, BwdArgs{a, (uint32_t)n_dkdv});
  const size_t offs[11] = {TH_OFFSET(MArgs, q),      TH_OFFSET(MArgs, k),  TH_OFFSET(MArgs, v),  TH_OFFSET(MArgs, o),
                           TH_OFFSET(MArgs, lse),    TH_OFFSET(MArgs, dout), TH_OFFSET(MArgs, dq), TH_OFFSET(MArgs, dk),
                           TH_OFFSET(MArgs, dv),     TH_OFFSET(MArgs, starts), TH_OFFSET(MArgs, lengths)};
  // Both kernels' arguments begin with MArgs: the same offsets.
  for (int kk : {k0, k1}) {
    for (int v = 0; v < (M ? 11 : 9); ++v) b.ref(v, kk, offs[v]);
    b.ws_ref(kk, TH_OFFSET(MArgs, delta), at_delta);
  }
  if (!M)
    for (int v : {0, 1, 2, 3, 5, 6, 7, 8}) b.align(v, 16);
  if (skv.n > 1 || sq.n > 1) {
    SumArgs s{};
    s.batch = d->batch, s.d = D;
    // The outputs' pointers start as the descriptor's (repointing rewrites them with the others).
    int values[3];
    uint64_t ats[3];
    unsigned total = 0;
    auto add = [&](int value, uint16_t* to, const int64_t* strides, int positions, int heads, int parts, float scale,
                   uint64_t at) {
      const unsigned g = (unsigned)(((int64_t)d->batch * positions * heads * (D / 4) + 255) / 256);
      values[s.n] = value, ats[s.n] = at;
      s.of[s.n++] = SumArgsOne{nullptr, to, strides[0], strides[1], strides[2], positions, heads, parts, scale, g};
      total += g;
    };
    if (skv.n > 1) {
      const uint64_t at = b.workspace((uint64_t)2 * skv.n * rows_k * D * sizeof(float));
      b.ws_ref(k1, TH_OFFSET(MArgs, part), at);
      add(7, a.dk, d->k_strides, a.kv_seq, d->kv_heads, skv.n, a.scale, at);
      add(8, a.dv, d->k_strides, a.kv_seq, d->kv_heads, skv.n, 1.0f, at + (uint64_t)skv.n * rows_k * D * sizeof(float));
    }
    if (sq.n > 1) {
      const uint64_t at = b.workspace((uint64_t)sq.n * rows * D * sizeof(float));
      b.ws_ref(k1, TH_OFFSET(MArgs, q_part), at);
      add(6, a.dq, d->q_strides, d->seq, d->heads, sq.n, a.scale, at);
    }
    const int k2 = b.kernel((const void*)mfma_attn_sum,
                            sq.n == 1   ? "mfma_attn_sum_dk_dv"
                                                              : skv.n == 1 ? "mfma_attn_sum_dq"
                                                                           : "mfma_attn_sum_dk_dv_mfma_attn_sum_dq",
                            dim3(total), dim3(256), 0, s);
    for (int i = 0; i < s.n; ++i) {
      const size_t one = TH_OFFSET(SumArgs, of) + i * sizeof(SumArgsOne);
      b.ref(values[i], k2, one + TH_OFFSET(SumArgsOne, out));
      b.ws_ref(k2, one + TH_OFFSET(SumArgsOne, part), ats[i]);
    }
  }
  const double BH = (double)d->batch * d->heads, BHk = (double)d->batch * d->kv_heads;
  b.work(2.0 * BH * a.seq * D * 4 + 2.0 * BHk * a.kv_seq * D * 4 + 8.0 * BH * a.seq,
         2.5 * 4.0 * BH * D * visible_pairs(a), n_dkdv);
  *out = b.release();
  return TH_OK;
}

// Under device-held masks (or rows the kernels above do not take): whole
// sweeps, a workgroup per block of 128.

template <int D>
int masked_fwd_launch(const th_attention_desc* d, th_launch** out) {
  MArgs a = margs_of(d);
  th::Builder b("attention_fwd_mfma", 7);
  const dim3 grid(d->heads, d->batch, (d->seq + 127) / 128);
  const int P = (int64_t)grid.x * grid.y * grid.z <= kFwdHalves ? 2 : 1;
  const size_t lds = 4 * P * (size_t)kTile<D> * sizeof(uint16_t) + 4 * P * sizeof(int);
  const void* fn = P == 2 ? (const void*)mfma_attn_fwd<D, true, 2> : (const void*)mfma_attn_fwd<D, true, 1>;
  TH_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const int k = b.kernel(fn, D == 64 ? "mfma_attn_fwd_masked_d64" : "mfma_attn_fwd_masked_d128", grid, dim3(256 * P),
                         (uint32_t)lds, a);
  const size_t offs[7] = {TH_OFFSET(MArgs, q),   TH_OFFSET(MArgs, k),      TH_OFFSET(MArgs, v),
                          TH_OFFSET(MArgs, o),   TH_OFFSET(MArgs, lse),    TH_OFFSET(MArgs, starts),
                          TH_OFFSET(MArgs, lengths)};
  for (int v = 0; v < 7; ++v) b.ref(v, k, offs[v]);
  const double BH = (double)d->batch * d->heads, BHk = (double)d->batch * d->kv_heads;
  b.work(2.0 * BH * a.seq * D * 2 + 2.0 * BHk * a.kv_seq * D * 2 + 4.0 * BH * a.seq, 4.0 * BH * D * visible_pairs(a),
         (int64_t)grid.x * grid.y * grid.z);
  *out = b.release();
  return TH_OK;
}

int check_mfma(const th_attention_desc* d, bool backward) {
  TH_REQUIRE(d->q && d->k && d->v && d->o, "attention: null q, k, v or o");
  TH_REQUIRE(aligned16(d->q) && aligned16(d->k) && aligned16(d->v) && aligned16(d->o),
             "attention: q, k, v, o must be 16-byte aligned");
  if (backward) {
    TH_REQUIRE(d->lse && d->dout && d->dq && d->dk && d->dv, "attention backward: null lse, dout, dq, dk or dv");
    TH_REQUIRE(aligned16(d->dout) && aligned16(d->dq) && aligned16(d->dk) && aligned16(d->dv),
               "attention backward: dout, dq, dk, dv must be 16-byte aligned");
  }
  return TH_OK;
}

}  // namespace

namespace th {

// bf16 arrays, head dim 64, 128 or 256, any positive lengths, no
// device-held masks, 16-byte rows, operands and strides.
bool mfma_attention_takes(const th_attention_desc* d) {
  if (!d || (d->flags & TH_ATTN_F32) || d->starts || d->lengths) return false;
  if (d->head_dim != 64 && d->head_dim != 128 && d->head_dim != 256) return false;
  if (d->seq < 1 || d->kv_seq < 0 || d->batch < 1 || d->heads < 1 || d->kv_heads < 1 || d->heads % d->kv_heads)
    return false;
  for (int64_t s : {d->q_strides[0], d->q_strides[1], d->q_strides[2], d->k_strides[0], d->k_strides[1], d->k_strides[2]})
    if (s <= 0 || s % 8) return false;
  const int64_t kv = d->kv_seq > 0 ? d->kv_seq : d->seq;
  // (Blocks of 128 positions along grid z; sweeps are split only where all the
  // blocks are fewer than 256.)
  return (d->seq + 127) / 128 <= 65535 && (kv + 127) / 128 <= 65535 && d->heads <= 65535 && d->batch <= 65535;
}

int build_attention_mfma_fwd(const th_attention_desc* d, th_launch** out) {
  if (int r = check_mfma(d, false)) return r;
  if (decode_attention_takes(d)) return build_attention_decode_fwd(d, 16, false, out);
  switch (d->head_dim) {
    case 64: return fwd_launch<64>(d, out);
    case 128: return fwd_launch<128>(d, out);
    default: return fwd_launch<256>(d, out);
  }
}

int build_attention_mfma_bwd(const th_attention_desc* d, th_launch** out) {
  if (int r = check_mfma(d, true)) return r;
  switch (d->head_dim) {
    case 64: return bwd_launch<64, false>(d, out);
    case 128: return bwd_launch<128, false>(d, out);
    default: return bwd_launch<256, false>(d, out);
  }
}

// bf16 at head dims 64 and 128 under device-held masks, and rows of any
// alignment and strides (descriptors the general kernels' checks passed).
bool masked_attention_takes(const th_attention_desc* d) {
  const int kv = d->kv_seq > 0 ? d->kv_seq : d->seq;
  return !(d->flags & TH_ATTN_F32) && (d->head_dim == 64 || d->head_dim == 128) &&
         (int64_t)d->batch * d->seq * d->heads < 2147483648LL && (d->seq + 127) / 128 <= 65535 && (kv + 127) / 128 <= 65535;
}

int build_attention_masked_fwd(const th_attention_desc* d, th_launch** out) {
  return d->head_dim == 64 ? masked_fwd_launch<64>(d, out) : masked_fwd_launch<128>(d, out);
}

int build_attention_masked_bwd(const th_attention_desc* d, th_launch** out) {
  return d->head_dim == 64 ? bwd_launch<64, true>(d, out) : bwd_launch<128, true>(d, out);
}

}  // namespace th
