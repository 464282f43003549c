// Op class (c), decode: attention forward for a few queries over a long cache
// of keys (bf16, head dims 64 and 128), the masks the device holds included
// (a key count per sequence, a first key per query; test/cuda/attention.jl:254-271).
//
// The work is the cache's bytes: each (sequence, key/value head) reads its K
// and V once for all the query rows that share them, which is seq x (heads /
// kv_heads) rows, at most the 16 columns of one v_mfma_f32_16x16x32_bf16.
// The general kernels give such a call a workgroup a query head, 63 of whose
// 64 query slots are empty, each sweeping the whole cache on the vector ALUs
// and reading K and V once per query head.  Here:
//   - keys are dealt to parts of `span` positions, a workgroup each, about
//     2048 workgroups over the whole cache; a part past its sequence's length
//     ends at once, so sequences of any lengths share the device evenly, and a
//     second kernel folds the parts that exist;
//   - a wave takes every fourth block of 32 keys, the next block's K and V
//     rows (16 KB at d = 128) in flight in registers meanwhile, no LDS and no
//     barrier in the sweep;
//   - S' = K Q' (keys x rows); the score registers of a lane are the B operand
//     of O' += V' P' as they stand, the keys of slot 8 g + j being 4 g + j and
//     16 + 4 g + j - 4; V' comes from whole rows of V (16 lanes of one row a
//     load) by an 8 x 8 transpose of halves inside each lane (v_perm_b32);
//   - the weights are fp32's as in the general kernels: P in three bf16 parts
//     (split2_towards0), three products on V, whose values are bf16 already.
// Rows of q, k, v, o may start at any even address.  B16 H32 KV8, 4096 keys of
// 128 features, lengths of 1/8 to all of it (151 MB on average): 3593 us on the
// general kernels, 45 here (44 with weights of 16 bits), 40 of them this sweep (3.8 TB/s; the copy rate is
// 5.2) and 5 the fold.  Measured and not kept: parts for 1024, 4096 or 8192
// workgroups (50, 52, 52 us), non-temporal loads (46), a lane's four K pieces
// adjacent (46).
#include <hip/hip_runtime.h>

#include <cmath>

#include "attention_tiles.h"
#include "th_core.h"

namespace {

// Rows start where the caller's strides put them: loads and stores of 16 and 8
// bytes that assume the elements' own alignment.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef u32x2 u32x2_any __attribute__((aligned(2)));

constexpr int kRows = 16;    // query rows a workgroup holds
constexpr int kBlock = 32;   // keys a wave takes at a time
constexpr int kStep = 128;   // keys the four waves take at a time

struct DecodeArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;              // natural log, [b][s][h], or null
  const int32_t* starts;   // (positions, batch), 1-based, or null
  const int32_t* lengths;  // (batch), or null
  float* part;             // nparts > 1: unnormalised O, [part][b][s][h][d]
  float* part_ml;          // and (m, l), [part][b][s][h]
  int64_t q_sh, q_ss, q_sb;
  int64_t k_sh, k_ss, k_sb;
  int32_t seq, kv_seq, heads, kv_heads, batch, causal;
  int32_t nparts, span;    // span a multiple of kStep
  float scale;
};

// Sequence b's keys that any of its queries can see: lengths[b] clamped to
// the keys' extent and, causal, the last query's own position.
__device__ __forceinline__ int keys_of(const DecodeArgs& p, int b) {
  int n = p.kv_seq;
  if (p.lengths) n = min(max(p.lengths[b], 0), n);
  return p.causal ? min(n, p.seq) : n;
}

// One block's operands in flight: K as A operands (key l % 16 of each half,
// features 32 s + 8 (l / 16) + (0..7)), V as rows (features E (l % 16) + ..).
template <int D>
struct Block {
  static constexpr int E = D / 16;
  u32x4 k[2][D / 32];
  uint32_t v[8][E / 2];
  // Keys past `last` read the last one again (masked, and their V zeroed, where used).
  __device__ __forceinline__ void load(const uint16_t* kb, const uint16_t* vb, int64_t ss, int key0, int last) {
    const int lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint16_t* row = kb + (int64_t)min(key0 + 16 * t + r, last) * ss + 8 * g;
#pragma unroll
      for (int s = 0; s < D / 32; ++s) k[t][s] = *reinterpret_cast<const u32x4_any*>(row + 32 * s);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint16_t* row = vb + (int64_t)min(key0 + 16 * (j / 4) + 4 * g + j % 4, last) * ss + E * r;
      if constexpr (E == 8) {
        const u32x4 x = *reinterpret_cast<const u32x4_any*>(row);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = x[i];
      } else {
        const u32x2 x = *reinterpret_cast<const u32x2_any*>(row);
        v[j][0] = x[0], v[j][1] = x[1];
      }
    }
  }
};

template <int D>
__global__ __launch_bounds__(256, 2) void mfma_attn_fwd_decode(DecodeArgs p) {
  constexpr int E = D / 16;    // features of V a lane holds of each key
  constexpr int LD = D + 4;    // floats a row of a wave's O in LDS
  __shared__ __attribute__((aligned(16))) float Os[4][kRows][LD];
  __shared__ float Ms[4][kRows], Ls[4][kRows];
  const int part = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const int group = p.heads / p.kv_heads, rows = p.seq * group;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  const int nk = keys_of(p, b), k_lo = part * p.span;
  // A part past the sequence's keys does not exist (the first always does: it
  // stores what a sequence without keys leaves).
  if (part > 0 && k_lo >= nk) return;
  const int k_hi = min(nk, k_lo + p.span);
  // Lane l's row (column of every product): query r / group, head r % group of the group.
  const bool live = r < rows;
  const int j = live ? r / group : 0, h = hk * group + (live ? r % group : 0);
  const int first = p.starts ? p.starts[(int64_t)j + (int64_t)p.seq * b] - 1 : 0;
  const int end = p.causal ? min(nk, j + 1) : nk;
  const float c = p.scale * kLog2e;
  const uint16_t* qrow = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)j * p.q_ss;
  bf16x8 qf[D / 32];
#pragma unroll
  for (int s = 0; s < D / 32; ++s)
    qf[s] = live ? __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4_any*>(qrow + 32 * s + 8 * g)) : bf16x8{};
  const uint16_t* kb = p.k + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  const uint16_t* vb = p.v + (int64_t)b * p.k_sb + (int64_t)hk * p.k_sh;
  f32x4 o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = f32x4{};
  float m = -INFINITY, l = 0.0f;
  // The block of 32 keys from key0.
  auto fold = [&](const Block<D>& x, int key0) {
    f32x4 s[2] = {f32x4{}, f32x4{}};
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x.k[t][i]), qf[i], s[t], 0, 0, 0);
    float mb = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + 16 * t + 4 * g + i;
        s[t][i] = key >= first && key < end ? s[t][i] : -INFINITY;
        mb = fmaxf(mb, s[t][i]);
      }
    mb = fmaxf(mb, __shfl_xor(mb, 16, 64));
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    const float mn = fmaxf(m, mb * c);
    const float shift = thd::lse_shift(mn);
    const float alpha = __builtin_amdgcn_exp2f(m - shift);
    m = mn;
    u32x4 w0, w1, w2;
    float w[8], sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      w[i] = __builtin_amdgcn_exp2f(fmaf(s[i / 4][i % 4], c, -shift));
      sum += w[i];
    }
    l = l * alpha + sum;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t x0, x1, x2;
      split2_towards0(w[2 * i], w[2 * i + 1], x0, x1, x2);
      w0[i] = x0, w1[i] = x1, w2[i] = x2;
    }
    const bool tail = key0 + kBlock > nk;  // keys past the length: V may hold anything there
#pragma unroll
    for (int d2 = 0; d2 < E / 2; ++d2) {
      uint32_t v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = x.v[i][d2];
        if (tail) v[i] = key0 + 16 * (i / 4) + 4 * g + i % 4 < nk ? v[i] : 0u;
      }
      u32x4 even, odd;  // features E (l % 16) + 2 d2 and + 1 of the eight keys
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        even[i] = __builtin_amdgcn_perm(v[2 * i + 1], v[2 * i], 0x05040100u);
        odd[i] = __builtin_amdgcn_perm(v[2 * i + 1], v[2 * i], 0x07060302u);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, u ? odd : even);
        f32x4 t = o[2 * d2 + u] * alpha;
        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, w2), t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, w1), t, 0, 0, 0);
        o[2 * d2 + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, w0), t, 0, 0, 0);
      }
    }
  };
  // Blocks that end before every row's first key see nothing.
  int from = 0;
  if (p.starts) {
    from = live ? first : 0x7fffffff;
#pragma unroll
    for (int x = 1; x < 16; x *= 2) from = min(from, __shfl_xor(from, x, 64));
    from = max(0, min(from, nk) - k_lo);
  }
  const int last = nk - 1;
  int key0 = k_lo + from / kStep * kStep + kBlock * wave;
  if (key0 + kBlock <= k_lo + from) key0 += kStep;
  if (key0 < k_hi) {
    Block<D> even, odd;
    even.load(kb, vb, p.k_ss, key0, last);
    while (true) {
      if (key0 + kStep < k_hi) odd.load(kb, vb, p.k_ss, key0 + kStep, last);
      fold(even, key0);
      key0 += kStep;
      if (key0 >= k_hi) break;
      if (key0 + kStep < k_hi) even.load(kb, vb, p.k_ss, key0 + kStep, last);
      fold(odd, key0);
      key0 += kStep;
      if (key0 >= k_hi) break;
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // Lane l holds row r's features E (4 g + i) + e in o[e][i].
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < E; e += 4)
      *reinterpret_cast<f32x4*>(&Os[wave][r][E * (4 * g + i) + e]) = f32x4{o[e][i], o[e + 1][i], o[e + 2][i], o[e + 3][i]};
  if (g == 0) Ms[wave][r] = m, Ls[wave][r] = l;
  __syncthreads();
  // The four waves' parts in wave order: thread t takes row t / 16, features E (t % 16) + (0..E).
  const int row = threadIdx.x / 16, col = E * (threadIdx.x % 16);
  if (row >= rows) return;
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < 4; ++w) mx = fmaxf(mx, Ms[w][row]);
  const float shift = thd::lse_shift(mx);
  float sum = 0.0f;
  f32x4 acc[E / 4] = {};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float a = __builtin_amdgcn_exp2f(Ms[w][row] - shift);
    sum += a * Ls[w][row];
#pragma unroll
    for (int e = 0; e < E / 4; ++e) acc[e] += a * *reinterpret_cast<const f32x4*>(&Os[w][row][col + 4 * e]);
  }
  const int jo = row / group, ho = hk * group + row % group;
  const int64_t at = ((int64_t)b * p.seq + jo) * p.heads + ho;
  if (p.nparts > 1) {
    const int64_t to = (int64_t)part * p.batch * p.seq * p.heads + at;
#pragma unroll
    for (int e = 0; e < E / 4; ++e) *reinterpret_cast<f32x4*>(p.part + to * D + col + 4 * e) = acc[e];
    if (col == 0) reinterpret_cast<f32x2*>(p.part_ml)[to] = f32x2{mx, sum};
    return;
  }
  const float inv = 1.0f / sum;
  uint16_t* out = p.o + (int64_t)b * p.q_sb + (int64_t)ho * p.q_sh + (int64_t)jo * p.q_ss + col;
#pragma unroll
  for (int e = 0; e < E / 4; ++e)
    *reinterpret_cast<u32x2_any*>(out + 4 * e) = u32x2{pack2(acc[e][0] * inv, acc[e][1] * inv), pack2(acc[e][2] * inv, acc[e][3] * inv)};
  if (col == 0 && p.lse) p.lse[at] = (mx + log2f(sum)) * kLn2;
}

// The parts that exist, folded in part order: a thread per four features of a
// (b, query, head) row, the parts' loads issued eight at a time.
template <int D>
__global__ __launch_bounds__(256) void mfma_attn_decode_combine(DecodeArgs p) {
  constexpr int quads = D / 4;
  const int64_t rows = (int64_t)p.batch * p.seq * p.heads;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= rows * quads) return;
  const int64_t row = t / quads;
  const int c = 4 * (int)(t % quads);
  const int h = (int)(row % p.heads);
  const int64_t pos = (row / p.heads) % p.seq, b = row / ((int64_t)p.heads * p.seq);
  const int n = max(1, (keys_of(p, (int)b) + p.span - 1) / p.span);
  const f32x2* ml = reinterpret_cast<const f32x2*>(p.part_ml) + row;
  const f32x4* po = reinterpret_cast<const f32x4*>(p.part + row * D + c);
  const int64_t step = rows * quads;
  float m = -INFINITY, l = 0.0f;
  f32x4 acc = {};
  for (int s0 = 0; s0 < n; s0 += 8) {
    f32x2 x[8];
    f32x4 y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // a part past the last reads the last again, with no weight
      const int64_t s = min(s0 + u, n - 1);
      x[u] = ml[s * rows];
      y[u] = po[s * step];
    }
    float mn = m;
#pragma unroll
    for (int u = 0; u < 8; ++u) mn = fmaxf(mn, x[u][0]);
    const float shift = thd::lse_shift(mn), alpha = __builtin_amdgcn_exp2f(m - shift);
    l *= alpha;
    acc *= alpha;
    m = mn;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < n) {
        const float w = __builtin_amdgcn_exp2f(x[u][0] - shift);
        l += w * x[u][1];
        acc += w * y[u];
      }
  }
  const float inv = 1.0f / l;
  *reinterpret_cast<u32x2_any*>(p.o + b * p.q_sb + h * p.q_sh + pos * p.q_ss + c) =
      u32x2{pack2(acc[0] * inv, acc[1] * inv), pack2(acc[2] * inv, acc[3] * inv)};
  if (c == 0 && p.lse) p.lse[row] = (m + log2f(l)) * kLn2;
}

// Keys a part: about 2048 workgroups over the whole cache, so that the device
// holds eight waves a SIMD's worth of parts even where most sequences are
// shorter than the cache; at least kStep (each wave one block).
int span_of(const th_attention_desc* d, int64_t keys) {
  const int64_t total = keys * d->kv_heads * d->batch;
  const int64_t span = ((total + 2047) / 2048 + kStep - 1) / kStep * kStep;
  return (int)std::min<int64_t>(span, (keys + kStep - 1) / kStep * kStep);
}

template <int D>
int decode_launch(const th_attention_desc* d, uint32_t align, bool masks, th_launch** out) {
  DecodeArgs a{};
  a.q = static_cast<const uint16_t*>(d->q);
  a.k = static_cast<const uint16_t*>(d->k);
  a.v = static_cast<const uint16_t*>(d->v);
  a.o = static_cast<uint16_t*>(d->o);
  a.lse = d->lse;
  a.starts = d->starts, a.lengths = d->lengths;
  a.q_sh = d->q_strides[0], a.q_ss = d->q_strides[1], a.q_sb = d->q_strides[2];
  a.k_sh = d->k_strides[0], a.k_ss = d->k_strides[1], a.k_sb = d->k_strides[2];
  a.seq = d->seq, a.kv_seq = d->kv_seq > 0 ? d->kv_seq : d->seq;
  a.heads = d->heads, a.kv_heads = d->kv_heads, a.batch = d->batch, a.causal = d->causal;
  a.scale = d->scale > 0 ? d->scale : 1.0f / sqrtf((float)D);
  const int64_t keys = d->causal ? std::min(a.seq, a.kv_seq) : a.kv_seq;
  a.span = span_of(d, keys);
  a.nparts = (int)((keys + a.span - 1) / a.span);
  th::Builder b("attention_fwd_decode", 7);
  const int k = b.kernel((const void*)mfma_attn_fwd_decode<D>, D == 64 ? "mfma_attn_fwd_decode_d64" : "mfma_attn_fwd_decode_d128",
                         dim3(a.nparts, d->kv_heads, d->batch), dim3(256), 0, a);
  int last = k;
  if (a.nparts > 1) {
    const int64_t rows = (int64_t)d->batch * d->seq * d->heads;
    last = b.kernel((const void*)mfma_attn_decode_combine<D>, "mfma_attn_decode_combine",
                    dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0, a);
    const uint64_t at_o = b.workspace((uint64_t)a.nparts * rows * D * sizeof(float));
    const uint64_t at_ml = b.workspace((uint64_t)a.nparts * rows * 2 * sizeof(float));
    for (int kk : {k, last}) {
      b.ws_ref(kk, TH_OFFSET(DecodeArgs, part), at_o);
      b.ws_ref(kk, TH_OFFSET(DecodeArgs, part_ml), at_ml);
    }
  }
  const size_t offs[7] = {TH_OFFSET(DecodeArgs, q),   TH_OFFSET(DecodeArgs, k),      TH_OFFSET(DecodeArgs, v),
                          TH_OFFSET(DecodeArgs, o),   TH_OFFSET(DecodeArgs, lse),    TH_OFFSET(DecodeArgs, starts),
                          TH_OFFSET(DecodeArgs, lengths)};
  for (int v = 0; v < (masks ? 7 : 5); ++v)
    for (int kk = k; kk <= last; ++kk) b.ref(v, kk, offs[v]);
  for (int v = 0; v < 4; ++v) b.align(v, align);
  const double BH = (double)d->batch * d->heads;
  const double pairs = d->causal ? 0.5 * d->seq * (double)keys : (double)d->seq * keys;
  b.work(2.0 * D * (2.0 * BH * d->seq + 2.0 * d->batch * d->kv_heads * (double)a.kv_seq) + 4.0 * BH * d->seq,
         4.0 * BH * pairs * D, (int64_t)a.nparts * d->kv_heads * d->batch);
  *out = b.release();
  return TH_OK;
}

}  // namespace

namespace th {

// bf16, head dim 64 or 128, and no more query rows a key/value head than one
// product has columns: past 16 rows the cache is read again for every 16,
// and the 128-query kernels fill.
bool decode_attention_takes(const th_attention_desc* d) {
  return !(d->flags & TH_ATTN_F32) && (d->head_dim == 64 || d->head_dim == 128) && d->kv_heads > 0 &&
         (int64_t)d->seq * (d->heads / d->kv_heads) <= kRows;
}

int build_attention_decode_fwd(const th_attention_desc* d, uint32_t align, bool masks, th_launch** out) {
  return d->head_dim == 64 ? decode_launch<64>(d, align, masks, out) : decode_launch<128>(d, align, masks, out);
}

}  // namespace th
