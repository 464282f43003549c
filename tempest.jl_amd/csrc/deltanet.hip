// Config 5: chunked gated DeltaNet, forward and gradient (rows a16: the
// reference's scan and recurrence kernels, ext/cuTileExt/build.jl:715-839,
// codegen/scalar.jl:354-440, runtime/stepped.jl, for the program of
// examples/deltanet.jl:58-86).
//
// Per position t of a (batch, head) sequence, S (dk x dv) follows
//   S = exp(a_t) (I - beta_t k_t k_t') S + beta_t k_t v_t',  o_t = S' q_t.
// In chunks of 64 positions (ca = cumsum(a) within the chunk,
// Gamma_ij = exp(ca_i - ca_j)):
//   A = strict lower (beta_i Gamma_ij k_i.k_j),  T = (I + A)^-1,
//   W = T diag(beta e^ca) K,  U~ = T diag(beta) V,
//   P = lower (Gamma_ij q_i.k_j),  Qg = diag(e^ca) Q,  Kd = diag(e^(ca_63 - ca)) K,  g = e^ca_63;
// across chunks:  U = U~ - W S,  O = Qg S + P U,  S <- g S + Kd' U.
//
// Kernels (fp32 arithmetic, every product on the bf16 matrix cores with each
// fp32 operand split into two bf16 halves; inputs bf16 q, k, v and fp32 a, beta):
//   dn_chunk_prep   one workgroup per chunk: ca, A, T (forward substitution,
//                   one lane per column), W, U~.
//   dn_state_scan   one eight-wave workgroup per (sequence, 32 columns of S):
//                   the sequential recurrence, each column block independent;
//                   stores each chunk's starting state and U.
//   dn_output       one workgroup per chunk: P, O.
//   dn_state_grad   one eight-wave workgroup per (sequence, 32 columns): the state
//                   gradient swept back over chunks; stores dU and dS_{n+1}.
//   dn_grad         one workgroup per chunk: the chunk's products' gradients,
//                   the inverse's (dA = -T' dT T'), the decays', a's.
#include <hip/hip_runtime.h>

#include <cmath>

#include "th_core.h"

namespace {

constexpr int kC = 64;    // chunk
constexpr int kD = 128;   // dk = dv
constexpr int kCols = 32; // columns of S per scan workgroup

struct DnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const float* a;
  const float* beta;
  uint16_t* o;
  const uint16_t* dout;
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  float* da;
  float* dbeta;
  // workspace, per chunk c = (b * heads + h) * chunks + n
  float* ca;    // [c][64]
  float* T;     // [c][64][64]
  float* W;     // [c][64][128]
  float* Ut;    // [c][64][128]
  float* S;     // [c][128][128] state at the chunk's start
  float* U;     // [c][64][128]
  float* P;     // [c][64][64]
  float* dU;    // [c][64][128]
  float* dSn;   // [c][128][128] gradient w.r.t. the chunk's end state
  float* dg;    // [c][kDgParts]: <S, dSn> by (column slice, wave) of the state gradient
  int64_t s_h, s_t, s_b;  // strides (elements) of q, k, v, o, dout, dq, dk, dv along head, position, batch
  int64_t g_h, g_t, g_b;  // strides of a, beta, da, dbeta
  int32_t batch, heads, seq, chunks;
};

__device__ __forceinline__ float bf(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t to_bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

struct Chunk {
  int b, h, n;
  int64_t c;       // chunk number
  int64_t row0;    // element offset of position n*64, head h, batch b
  int64_t grow0;   // the same for the gate arrays
};

__device__ __forceinline__ Chunk chunk_of(const DnArgs& p, int64_t c) {
  Chunk k;
  k.c = c;
  k.n = (int)(c % p.chunks);
  const int64_t bh = c / p.chunks;
  k.h = (int)(bh % p.heads);
  k.b = (int)(bh / p.heads);
  k.row0 = k.b * p.s_b + k.h * p.s_h + (int64_t)k.n * kC * p.s_t;
  k.grow0 = k.b * p.g_b + k.h * p.g_h + (int64_t)k.n * kC * p.g_t;
  return k;
}

// Chunk n of the sequence whose first chunk is `first` (its divisions done once).
__device__ __forceinline__ Chunk chunk_at(const DnArgs& p, const Chunk& first, int n) {
  Chunk k = first;
  k.n = n;
  k.c += n;
  k.row0 += (int64_t)n * kC * p.s_t;
  k.grow0 += (int64_t)n * kC * p.g_t;
  return k;
}

// ca = inclusive cumulative sum of a over the chunk (wave 0), into LDS.
__device__ __forceinline__ void cumulative_gates(float* ca, const DnArgs& p, const Chunk& ck) {
  if (threadIdx.x < 64) {
    float x = p.a[ck.grow0 + (int64_t)threadIdx.x * p.g_t];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float y = __shfl_up(x, o, 64);
      if ((int)threadIdx.x >= o) x += y;
    }
    ca[threadIdx.x] = x;
  }
}

// ---- fp32 products on the bf16 matrix cores -----------------------------------------
// Each fp32 operand x is split as hi = bf16(x), lo = bf16(x - hi); a b is
// summed in fp32 as hi hi + hi lo + lo hi on v_mfma_f32_16x16x32_bf16 (the
// lo lo term and lo's rounding leave about 2^-16 of each product; operands
// that are bf16 values, Q K V, have no lo).  The three bf16 products of 32 k
// take 48 matrix-core cycles, the eight fp32 ones (v_mfma_f32_16x16x4_f32)
// for the same k would take 256.
// Operands sit in LDS as rows padded by 16 bytes: the 16-byte pieces of 16
// consecutive rows land on distinct banks.
//
// Lane l = 16 g + r of a 16 x 16 block over 32 consecutive k takes the eight
// k = kb + 8 g + (0..7), each pairing A(i0 + r, k) with B(k, j0 + r); the products'
// k slot g then holds the same k in both operands.  The block
// C(i0 + 4 g + v, j0 + r) sits in register v of lane l.

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef short s16x8v __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4v lds_s16x4v;
constexpr int kLdC = 68;   // LDS row of 64 fp32
constexpr int kLdS = 36;   // LDS row of 32 fp32
constexpr int kLdT = 40;   // LDS row of 32 bf16

__device__ __forceinline__ f32x4v quad(const float* row) { return *reinterpret_cast<const f32x4v*>(row); }

// x, hidden from the compiler's known bits: of a lane number below 16 it would
// make (16 b + x) an `or`, whose rows it then addresses one by one from a
// register each, not from one register and the instruction's offset.
__device__ __forceinline__ int plain(int x) {
  asm("" : "+v"(x));
  return x;
}

// The four k of lane g's quad along a column: X(k, c) at x[k * ld + c].
__device__ __forceinline__ f32x4v column_quad(const float* x, int ld, int k0, int c) {
  return f32x4v{x[k0 * ld + c], x[(k0 + 1) * ld + c], x[(k0 + 2) * ld + c], x[(k0 + 3) * ld + c]};
}

typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

// Two fp32 as a pair of bf16 (nearest even), a in the low half.
__device__ __forceinline__ uint32_t pk2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{a, b}, bf16x2v));
}

// A product operand's eight k (two quads of one row) as bf16 halves: hi the
// nearest bf16, lo the nearest bf16 to the remainder x - hi (exact in fp32),
// so hi + lo holds x to about 2^-16 of it.  kExact: x is a bf16 value, lo is 0.
struct Split8 {
  bf16x8v hi, lo;
};
template <bool kExact>
__device__ __forceinline__ Split8 split8(f32x4v q0, f32x4v q1) {
  const float x[8] = {q0[0], q0[1], q0[2], q0[3], q1[0], q1[1], q1[2], q1[3]};
  u32x4v h, l = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = pk2(x[2 * e], x[2 * e + 1]);
  if constexpr (!kExact) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      l[e] = pk2(x[2 * e] - __uint_as_float(h[e] << 16), x[2 * e + 1] - __uint_as_float(h[e] & 0xffff0000u));
  }
  return Split8{__builtin_bit_cast(bf16x8v, h), __builtin_bit_cast(bf16x8v, l)};
}

// c += a b over 32 k on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16,
// fp32 sums): hi hi + hi lo + lo hi, the lo lo term (about 2^-16 of the
// product) dropped, and the terms of an operand exact in bf16 skipped.
template <bool kExactA, bool kExactB>
__device__ __forceinline__ f32x4v mma_split(const Split8& a, const Split8& b, f32x4v c) {
  if constexpr (!kExactB) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, c, 0, 0, 0);
  if constexpr (!kExactA) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, c, 0, 0, 0);
}

template <int BI, int BJ>
__device__ __forceinline__ void clear(f32x4v (&acc)[BI][BJ]) {
#pragma unroll
  for (int bi = 0; bi < BI; ++bi)
#pragma unroll
    for (int bj = 0; bj < BJ; ++bj) acc[bi][bj] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
}

// Each staging helper issues all of a thread's loads before its first LDS
// store, so their latencies overlap instead of adding up.

// Block (bi, bj) of acc to out (row stride ld), rows i0 + 16 bi + 4 g + v, columns j0 + 16 bj + r, times s.
template <int BI, int BJ>
__device__ __forceinline__ void store_blocks(float* out, int ld, const f32x4v (&acc)[BI][BJ], int i0, int j0, float s) {
  const int r = plain(threadIdx.x % 16), g = plain((threadIdx.x % 64) / 16);
#pragma unroll
  for (int bi = 0; bi < BI; ++bi)
#pragma unroll
    for (int bj = 0; bj < BJ; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) out[(int64_t)(i0 + 16 * bi + 4 * g + v) * ld + j0 + 16 * bj + r] = s * acc[bi][bj][v];
}

// Operand readers for mm_by: block(x0, k0) is the block (x0 .. x0 + 15, k0 .. k0 + 31)
// as this lane l = 16 g + r holds it: (x0 + r, k0 + 8 g .. k0 + 8 g + 7).
// Those over fp32 split it at each read; Planes hold an operand split once
// where it was written (hi and lo as bf16, what split8 gives), read as they are:
// the splits were most of the instructions of a kernel whose waves read each
// operand several times over.
__device__ __forceinline__ int lane_r() { return plain(threadIdx.x % 16); }
__device__ __forceinline__ int lane_g8() { return plain((threadIdx.x % 64) / 16 * 8); }
struct RowF32 {  // (x, k) at p[x * ld + k]
  static constexpr bool kExact = false;
  const float* p;
  int ld;
  __device__ Split8 block(int x0, int k0, int r, int g8) const {
    const float* at = p + (x0 + r) * ld + k0 + g8;
    return split8<kExact>(quad(at), quad(at + 4));
  }
};
struct ColF32 {  // (x, k) at p[k * ld + x]
  static constexpr bool kExact = false;
  const float* p;
  int ld;
  __device__ Split8 block(int x0, int k0, int r, int g8) const {
    return split8<kExact>(column_quad(p, ld, k0 + g8, x0 + r), column_quad(p, ld, k0 + g8 + 4, x0 + r));
  }
};

// Eight bf16 along a row of memory or LDS, 16-byte aligned.
__device__ __forceinline__ bf16x8v row8(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4v*>(p));
}
// Eight rows k0 + g8 .. of column x0 + r of LDS rows of ld bf16:
// ds_read_b64_tr_b16 hands lane i of each 16 element i % 4 of the 8-byte pieces
// that lanes 4 k + i / 4 address; lane j addresses row j / 4, columns
// 4 (j % 4) .., so lane i gets rows 0..3 of column i, and a second read rows 4..7.
__device__ __forceinline__ bf16x8v column8(const uint16_t* p, int ld, int x0, int k0, int r, int g8) {
  const uint16_t* at = p + (k0 + g8 + r / 4) * ld + x0 + 4 * (r % 4);
  const s16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4v*)at);
  const s16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4v*)(at + 4 * ld));
  return __builtin_bit_cast(bf16x8v, s16x8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}
__device__ __forceinline__ bf16x8v none8() { return __builtin_bit_cast(bf16x8v, u32x4v{0u, 0u, 0u, 0u}); }
template <class Ld>
struct RowBf16At {  // (x, k) at bf16 p[x * ld + k]
  static constexpr bool kExact = true;
  const uint16_t* p;
  Ld ld;
  __device__ Split8 block(int x0, int k0, int r, int g8) const { return Split8{row8(p + (x0 + r) * ld + k0 + g8), none8()}; }
};
typedef RowBf16At<int> RowBf16;       // in LDS
typedef RowBf16At<int64_t> RowBf16G;  // in memory
struct ColBf16 {  // (x, k) at bf16 p[k * ld + x], in LDS
  static constexpr bool kExact = true;
  const uint16_t* p;
  int ld;
  __device__ Split8 block(int x0, int k0, int r, int g8) const { return Split8{column8(p, ld, x0, k0, r, g8), none8()}; }
};
struct Planes {  // rows of ld bf16 in LDS, twice
  uint16_t *hi, *lo;
  int ld;
  // Two values, at (i, j) and (i + 1, j).
  __device__ void put_rows(int i, int j, float a, float b) const {
    const uint32_t h = pk2(a, b), l = pk2(a - __uint_as_float(h << 16), b - __uint_as_float(h & 0xffff0000u));
    const int at = i * ld + j;
    hi[at] = (uint16_t)h, hi[at + ld] = (uint16_t)(h >> 16);
    lo[at] = (uint16_t)l, lo[at + ld] = (uint16_t)(l >> 16);
  }
  // Four at (i, j) .. (i, j + 3), j a multiple of 4.
  __device__ void put(int i, int j, f32x4v x) const {
    const u32x2v h = {pk2(x[0], x[1]), pk2(x[2], x[3])};
    const u32x2v l = {pk2(x[0] - __uint_as_float(h[0] << 16), x[1] - __uint_as_float(h[0] & 0xffff0000u)),
                      pk2(x[2] - __uint_as_float(h[1] << 16), x[3] - __uint_as_float(h[1] & 0xffff0000u))};
    *reinterpret_cast<u32x2v*>(hi + i * ld + j) = h;
    *reinterpret_cast<u32x2v*>(lo + i * ld + j) = l;
  }
  // The same at (i, j) and (i, j + 1), j even.
  __device__ void put(int i, int j, float a, float b) const {
    const uint32_t h = pk2(a, b), l = pk2(a - __uint_as_float(h << 16), b - __uint_as_float(h & 0xffff0000u));
    *reinterpret_cast<uint32_t*>(hi + i * ld + j) = h;
    *reinterpret_cast<uint32_t*>(lo + i * ld + j) = l;
  }
};
struct RowPlanes {  // (x, k) at (x, k)
  static constexpr bool kExact = false;
  Planes p;
  __device__ Split8 block(int x0, int k0, int r, int g8) const {
    const int at = (x0 + r) * p.ld + k0 + g8;
    return Split8{row8(p.hi + at), row8(p.lo + at)};
  }
};
struct ColPlanes {  // (x, k) at (k, x)
  static constexpr bool kExact = false;
  Planes p;
  __device__ Split8 block(int x0, int k0, int r, int g8) const {
    return Split8{column8(p.hi, p.ld, x0, k0, r, g8), column8(p.lo, p.ld, x0, k0, r, g8)};
  }
};
// The blocks of acc, rows i0 .. and columns j0 .., times s, to planes.
template <int BI, int BJ>
__device__ __forceinline__ void store_planes(const Planes& to, const f32x4v (&acc)[BI][BJ], int i0, int j0, float s) {
  const int r = lane_r(), g4 = plain((threadIdx.x % 64) / 16 * 4);
#pragma unroll
  for (int bi = 0; bi < BI; ++bi)
#pragma unroll
    for (int bj = 0; bj < BJ; ++bj)
#pragma unroll
      for (int v = 0; v < 4; v += 2)
        to.put_rows(i0 + 16 * bi + g4 + v, j0 + 16 * bj + r, s * acc[bi][bj][v], s * acc[bi][bj][v + 1]);
}

// acc[bi][bj] += X(i0 + 16 bi .., k) Y(k, j0 + 16 bj ..) over k in [0, K).
template <int BI, int BJ, class XR, class YR>
__device__ __forceinline__ void mm_by(f32x4v (&acc)[BI][BJ], const XR& X, int i0, const YR& Y, int j0, int K) {
  const int r = lane_r(), g8 = lane_g8();
  for (int kb = 0; kb < K; kb += 32) {
    Split8 b[BJ];
#pragma unroll
    for (int bj = 0; bj < BJ; ++bj) b[bj] = Y.block(j0 + 16 * bj, kb, r, g8);
    // The rows of X one block at a time: only one of its split blocks live.
#pragma unroll
    for (int bi = 0; bi < BI; ++bi) {
      const Split8 a = X.block(i0 + 16 * bi, kb, r, g8);
#pragma unroll
      for (int bj = 0; bj < BJ; ++bj) acc[bi][bj] = mma_split<XR::kExact, YR::kExact>(a, b[bj], acc[bi][bj]);
    }
  }
}

// Sum over the 16 lanes of a row group (lanes 16 g .. 16 g + 15), a fixed tree
// (1, 2, 4, 8 apart; by then alike within the group of lanes that a mirror swaps).
template <int kDpp>
__device__ __forceinline__ float moved(float x) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), kDpp, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_group_sum(float x) {
  x += moved<0xB1>(x);   // quad_perm 1, 0, 3, 2
  x += moved<0x4E>(x);   // quad_perm 2, 3, 0, 1
  x += moved<0x141>(x);  // row_half_mirror
  x += moved<0x140>(x);  // row_mirror
  return x;
}

constexpr int kLdH = kD + 8;  // bf16 LDS row of Q, K

// ---- forward: the chunk's WY form -------------------------------------------------
// ca, A = strict lower (beta_i Gamma_ij k_i.k_j), T = (I + A)^-1 (forward
// substitution, one lane per column), W = T diag(beta e^ca) K and
// U~ = T diag(beta) V; the products on the matrix cores (split bf16), K and V in
// LDS as bf16.

// Two 64 x 128 bf16 arrays of rows at s_t into LDS rows of kLdH, every load
// issued before the first store.
__device__ __forceinline__ void stage_rows_bf16(uint16_t* dst1, const uint16_t* src1, uint16_t* dst2,
                                                const uint16_t* src2, int64_t s_t) {
  constexpr int n = kC * (kD / 8) / 256;
  uint4 x1[n], x2[n];
#pragma unroll
  for (int u = 0; u < n; ++u) {
    const int e = threadIdx.x + 256 * u, row = e / (kD / 8), c8 = (e % (kD / 8)) * 8;
    x1[u] = *reinterpret_cast<const uint4*>(src1 + row * s_t + c8);
    x2[u] = *reinterpret_cast<const uint4*>(src2 + row * s_t + c8);
  }
#pragma unroll
  for (int u = 0; u < n; ++u) {
    const int e = threadIdx.x + 256 * u, row = e / (kD / 8), c8 = (e % (kD / 8)) * 8;
    *reinterpret_cast<uint4*>(dst1 + row * kLdH + c8) = x1[u];
    *reinterpret_cast<uint4*>(dst2 + row * kLdH + c8) = x2[u];
  }
}

// Under 80 KB, so two workgroups share a CU (one's substitution beside the
// other's loads and products).
constexpr size_t kPrepLds = 2 * kC * kLdH * sizeof(uint16_t) + (2 * kC * kLdC + 2 * kC) * sizeof(float);

__global__ __launch_bounds__(256, 2) void dn_chunk_prep(DnArgs p) {
  extern __shared__ float lds[];
  uint16_t* Kh = reinterpret_cast<uint16_t*>(lds);       // [64][kLdH]
  uint16_t* Vh = Kh + kC * kLdH;                          // [64][kLdH]
  float* AT = reinterpret_cast<float*>(Vh + kC * kLdH);   // [64][kLdC]: A, then T, then T diag(beta)
  float* TX = AT + kC * kLdC;     // [64][kLdC]: T diag(beta e^ca)
  float* TY = AT;                 // each entry rewritten by the thread that read it
  float* ca = TX + kC * kLdC;     // [64]
  float* be = ca + kC;            // [64]
  const Chunk ck = chunk_of(p, blockIdx.x);
  const int t = threadIdx.x, w = t / 64;
  const int r = t % 16, g = (t % 64) / 16;
  stage_rows_bf16(Kh, p.k + ck.row0, Vh, p.v + ck.row0, p.s_t);
  cumulative_gates(ca, p, ck);
  if (t < 64) be[t] = p.beta[ck.grow0 + (int64_t)t * p.g_t];
  __syncthreads();
  if (t < 64) p.ca[ck.c * kC + t] = ca[t];
  // A (64 x 64): wave w takes row block w, blocks at or left of the diagonal.
  {
    const RowBf16 Kr{Kh, kLdH};
    for (int bj = 0; bj < 4; ++bj) {
      f32x4v acc[1][1];
      clear(acc);
      if (bj <= w) mm_by(acc, Kr, 16 * w, Kr, 16 * bj, kD);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * w + 4 * g + v, j = 16 * bj + r;
        AT[i * kLdC + j] = i > j ? be[i] * expf(ca[i] - ca[j]) * acc[0][0][v] : 0.0f;
      }
    }
  }
  __syncthreads();
  // T = (I + A)^-1 by forward substitution: T_ij = -sum_{l<i} A_il T_lj for
  // i > j, T_jj = 1.  Column j = 16 w + (lane / 4) belongs to the four lanes
  // q = lane mod 4 of a quad of wave w: lane q sums the terms l = 4 m + q
  // and keeps T_lj for those l (c[m]), the quad adds its four partial sums
  // ((q0 + q1) + (q2 + q3) in every lane), so all four waves share the
  // 2080 fmas of the sweep.  A_il is 0 for l >= i, so the terms of rows not
  // yet solved (c[m] still 0) add nothing.
  {
    const int q = t % 4, j = 16 * w + (t % 64) / 4;
    float c[kC / 4];
#pragma unroll
    for (int m = 0; m < kC / 4; ++m) c[m] = 0.0f;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      float part = 0.0f;
#pragma unroll
      for (int m = 0; m < (i + 3) / 4; ++m) part = fmaf(AT[i * kLdC + 4 * m + q], c[m], part);
      part += __shfl_xor(part, 1, 64);
      part += __shfl_xor(part, 2, 64);
      const float ti = i == j ? 1.0f : (i < j ? 0.0f : -part);
      if (q == i % 4) c[i / 4] = ti;
    }
    __syncthreads();  // every wave's reads of A precede the writes of T
#pragma unroll
    for (int m = 0; m < kC / 4; ++m) AT[(4 * m + q) * kLdC + j] = c[m];
  }
  __syncthreads();
  {
    float* Tc = p.T + ck.c * kC * kC;
    for (int e = t; e < kC * kC; e += 256) {
      const int i = e / kC, l = e % kC;
      const float tv = AT[i * kLdC + l];
      Tc[e] = tv;
      TX[i * kLdC + l] = tv * be[l] * expf(ca[l]);
      TY[i * kLdC + l] = tv * be[l];
    }
  }
  __syncthreads();
  // W = TX K, U~ = TY V (64 x 128): wave w takes columns 32 w .. 32 w + 31.
  {
    f32x4v wk[4][2], uv[4][2];
    clear(wk);
    clear(uv);
    mm_by(wk, RowF32{TX, kLdC}, 0, ColBf16{Kh, kLdH}, 32 * w, kC);
    mm_by(uv, RowF32{TY, kLdC}, 0, ColBf16{Vh, kLdH}, 32 * w, kC);
    store_blocks(p.W + ck.c * kC * kD, kD, wk, 0, 32 * w, 1.0f);
    store_blocks(p.Ut + ck.c * kC * kD, kD, uv, 0, 32 * w, 1.0f);
  }
}

// ---- forward: the recurrence across chunks, 32 columns of S per workgroup ---------
// Per chunk: the starting state is stored, U = U~ - W S, S <- g S + Kd' U,
// the products on the matrix cores (split bf16).  While a chunk's products run,
// the next chunk's W, U~ columns, K and ca are loaded into registers.

// The two sweeps (this and the state gradient's) are serial chains bound by the
// instructions of a chunk, so each operand is split to bf16 once, as it goes to
// LDS, the state stays in registers (LDS holds its halves for the products, and
// an fp32 copy for 16-byte stores), and a sequence's place is found once, not
// by divisions a chunk: B4 H16 T8192, 128 chunks a sweep, 515 -> 468 us and,
// backward, 810 -> 679 against fp32 operands split at each wave's read.
// Eight waves, two on each SIMD: one workgroup per CU (its LDS), and a
// chunk's serial chain (stage, product, product, update) split eight ways.
constexpr int kScanThreads = 512;
// dg = <S, dSn> of a chunk in partial sums, one per wave of each column
// slice's state-gradient workgroup, folded in a fixed order by their reader.
constexpr int kDgParts = (kD / kCols) * (kScanThreads / 64);

struct ScanInputs {  // one chunk's inputs as this thread loads them
  f32x4v w[4];       // W: 4 x 16 bytes
  f32x4v u;          // U~ columns col0 .. col0 + 31: 16 bytes
  u32x4v k[2];       // K: 2 x 16 bytes (bf16)
  float ca;
};

__device__ __forceinline__ void scan_load(ScanInputs& in, const DnArgs& p, const Chunk& ck, int col0) {
  const int t = threadIdx.x;
  const float* Wc = p.W + ck.c * kC * kD;
  const float* Uc = p.Ut + ck.c * kC * kD;
#pragma unroll
  for (int e = 0; e < 4; ++e) in.w[e] = reinterpret_cast<const f32x4v*>(Wc)[t + kScanThreads * e];
  {
    const int r = t / 8, c = 4 * (t % 8);
    in.u = *reinterpret_cast<const f32x4v*>(Uc + r * kD + col0 + c);
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int x = t + kScanThreads * e, r = x / 16, c = 8 * (x % 16);
    in.k[e] = *reinterpret_cast<const u32x4v*>(p.k + ck.row0 + (int64_t)r * p.s_t + c);
  }
  in.ca = t < kC ? p.ca[ck.c * kC + t] : 0.0f;
}

// The inputs to LDS; K as Kd = diag(e^(ca_63 - ca)) K (ca of the same chunk, already in LDS).
__device__ __forceinline__ void scan_store(const ScanInputs& in, const Planes& W, float* Ut, const Planes& Kd,
                                           const float* ca) {
  const int t = threadIdx.x;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int x = t + kScanThreads * e, r = x / 32, c = 4 * (x % 32);
    W.put(r, c, in.w[e]);
  }
  *reinterpret_cast<f32x4v*>(Ut + (t / 8) * kLdS + 4 * (t % 8)) = in.u;
  const float last = ca[kC - 1];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int x = t + kScanThreads * e, r = x / 16, c = 8 * (x % 16);
    const float ed = expf(last - ca[r]);
    const u32x4v uk = in.k[e];
#pragma unroll
    for (int h = 0; h < 2; ++h)
      Kd.put(r, c + 4 * h, f32x4v{ed * bf((uint16_t)uk[2 * h]), ed * bf((uint16_t)(uk[2 * h] >> 16)), ed * bf((uint16_t)uk[2 * h + 1]),
                 ed * bf((uint16_t)(uk[2 * h + 1] >> 16))});
  }
}

// Scan workgroup b -> (sequence, first column of its slice of S).  The chip
// hands workgroups to its 8 XCDs in turn (b mod 8), each XCD with its own L2;
// the slices of one sequence read the same chunk inputs (W, K, Q, P), so they
// go to one XCD, whose L2 then serves all but the first read: slice j of
// sequence s is workgroup 32 (s / 8) + 8 j + s mod 8 for the sequences in
// whole groups of eight, the rest in order after them.
struct ScanSlot {
  int64_t seq;
  int col0;
};
__device__ __forceinline__ ScanSlot scan_slot() {
  constexpr int kSlices = kD / kCols;
  const int b = blockIdx.x, nseq = gridDim.x / kSlices, whole = nseq / 8 * 8;
  if (b < whole * kSlices) {
    const int q = b / 8;
    return ScanSlot{(int64_t)(q / kSlices) * 8 + b % 8, (q % kSlices) * kCols};
  }
  const int x = b - whole * kSlices;
  return ScanSlot{(int64_t)whole + x / kSlices, (x % kSlices) * kCols};
}

constexpr size_t kScanLds = (2 * kC * kLdH + kC * kLdS + kD * kLdS + kD * kLdT + kC * kLdS + kC * kLdT + kC) * sizeof(float);

__global__ __launch_bounds__(kScanThreads, 1) void dn_state_scan(DnArgs p) {
  extern __shared__ float lds[];
  uint16_t* at = reinterpret_cast<uint16_t*>(lds);
  auto planes = [&](int rows, int ld) {
    const Planes x{at, at + rows * ld, ld};
    at += 2 * rows * ld;
    return x;
  };
  const Planes W = planes(kC, kLdH);   // [64][kLdH]
  const Planes Kd = planes(kC, kLdH);  // [64][kLdH]: diag(e^(ca_63 - ca)) K
  const Planes Sp = planes(kD, kLdT);  // [128][kLdT]: the state's 32 columns
  const Planes Up = planes(kC, kLdT);  // [64][kLdT]: U
  float* Ut = reinterpret_cast<float*>(at);  // [64][kLdS]: U~ columns col0 .. col0 + 31
  float* S = Ut + kC * kLdS;      // [128][kLdS]: the state, as memory takes it
  float* U = S + kD * kLdS;       // [64][kLdS]
  float* ca = U + kC * kLdS;      // [64]
  const int t = threadIdx.x, w = t / 64;
  const int r = plain(t % 16), g4 = plain((t % 64) / 16 * 4);
  const ScanSlot slot = scan_slot();
  const int64_t seq = slot.seq;
  const int col0 = slot.col0;
  for (int e = t; e < kD * kLdS; e += kScanThreads) S[e] = 0.0f;
  for (int e = t; e < kD * kLdT; e += kScanThreads) Sp.hi[e] = 0, Sp.lo[e] = 0;
  f32x4v st[1][2];  // the state: rows 16 w + 4 g + v, columns 16 bj + r
  clear(st);
  const Chunk first = chunk_of(p, seq * p.chunks);
  ScanInputs in;
  scan_load(in, p, first, col0);
  if (t < kC) ca[t] = in.ca;
  __syncthreads();
  scan_store(in, W, Ut, Kd, ca);
  for (int n = 0; n < p.chunks; ++n) {
    const Chunk ck = chunk_at(p, first, n);
    __syncthreads();
    if (n + 1 < p.chunks) scan_load(in, p, chunk_at(p, first, n + 1), col0);
    const float gl = expf(ca[kC - 1]);
    // The chunk's starting state, stored for the output and the backward: read
    // now, written to memory at the chunk's end (and U with it), after the
    // next chunk's inputs are in LDS, whose wait for their loads would also
    // wait for every store issued before it.
    float* Sc = p.S + ck.c * kD * kD;
    f32x4v s_out[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = t + kScanThreads * u, row = e / 8, c = 4 * (e % 8);
      s_out[u] = *reinterpret_cast<const f32x4v*>(S + row * kLdS + c);
    }
    // U = U~ - W S (64 x 32): wave w takes the 16 x 16 block at rows
    // 16 (w mod 4), columns 16 (w / 4).
    {
      f32x4v ws[1][1];
      clear(ws);
      const int i0 = 16 * (w % 4), j0 = 16 * (w / 4);
      mm_by(ws, RowPlanes{W}, i0, ColPlanes{Sp}, j0, kD);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = i0 + g4 + v, j = j0 + r;
        ws[0][0][v] = Ut[i * kLdS + j] - ws[0][0][v];
        U[i * kLdS + j] = ws[0][0][v];
      }
      store_planes(Up, ws, i0, j0, 1.0f);
    }
    __syncthreads();
    // U for memory, 16 bytes a thread.
    const f32x4v u_out = *reinterpret_cast<const f32x4v*>(U + (t / 8) * kLdS + 4 * (t % 8));
    // S <- g S + Kd' U (128 x 32): wave w takes rows 16 w .. 16 w + 15.
    {
      f32x4v ku[1][2];
      clear(ku);
      mm_by(ku, ColPlanes{Kd}, 16 * w, ColPlanes{Up}, 0, kC);
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) st[0][bj][v] = gl * st[0][bj][v] + ku[0][bj][v];
      __syncthreads();  // every wave has read S, U and this chunk's inputs
      store_blocks(S, kLdS, st, 16 * w, 0, 1.0f);
      store_planes(Sp, st, 16 * w, 0, 1.0f);
    }
    if (n + 1 < p.chunks) {
      if (t < kC) ca[t] = in.ca;
      __syncthreads();
      scan_store(in, W, Ut, Kd, ca);
    }
    // S and U of this chunk to memory.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = t + kScanThreads * u, row = e / 8, c = 4 * (e % 8);
      *reinterpret_cast<f32x4v*>(Sc + row * kD + col0 + c) = s_out[u];
    }
    *reinterpret_cast<f32x4v*>(p.U + ck.c * kC * kD + (t / 8) * kD + col0 + 4 * (t % 8)) = u_out;
  }
}

// ---- forward: outputs ----------------------------------------------------------------
// P = lower(Gamma o Q K'), O = diag(e^ca) Q S + P U; the products on the
// matrix cores (split bf16), Q and K in LDS as bf16.

// S and U are read by columns straight from memory (each wave's 32 columns
// once), so only Q, K and P live in LDS and several workgroups share a CU.
constexpr size_t kOutLds = 2 * kC * kLdH * sizeof(uint16_t) + (kC * kLdC + kC) * sizeof(float);

__global__ __launch_bounds__(256, 2) void dn_output(DnArgs p) {
  extern __shared__ float lds[];
  uint16_t* Qh = reinterpret_cast<uint16_t*>(lds);       // [64][kLdH]
  uint16_t* Kh = Qh + kC * kLdH;                          // [64][kLdH]
  float* P = reinterpret_cast<float*>(Kh + kC * kLdH);    // [64][kLdC]
  float* ca = P + kC * kLdC;      // [64]
  const Chunk ck = chunk_of(p, blockIdx.x);
  const int t = threadIdx.x, w = t / 64;
  const int r = t % 16, g = (t % 64) / 16;
  const float* S = p.S + ck.c * kD * kD;  // [128][128]
  const float* U = p.U + ck.c * kC * kD;  // [64][128]
  stage_rows_bf16(Qh, p.q + ck.row0, Kh, p.k + ck.row0, p.s_t);
  if (t < 64) ca[t] = p.ca[ck.c * kC + t];
  __syncthreads();
  const RowBf16 Qr{Qh, kLdH};
  {
    float* Pc = p.P + ck.c * kC * kC;
    for (int bj = 0; bj < 4; ++bj) {
      f32x4v acc[1][1];
      clear(acc);
      if (bj <= w) mm_by(acc, Qr, 16 * w, RowBf16{Kh, kLdH}, 16 * bj, kD);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * w + 4 * g + v, j = 16 * bj + r;
        const float x = i >= j ? expf(ca[i] - ca[j]) * acc[0][0][v] : 0.0f;
        P[i * kLdC + j] = x;
        Pc[i * kC + j] = x;
      }
    }
  }
  __syncthreads();
  // O (64 x 128): wave w takes columns 32 w .. 32 w + 31.
  {
    f32x4v qs[4][2], pu[4][2];
    clear(qs);
    clear(pu);
    mm_by(qs, Qr, 0, ColF32{S, kD}, 32 * w, kD);
    mm_by(pu, RowF32{P, kLdC}, 0, ColF32{U, kD}, 32 * w, kC);
#pragma unroll
    for (int bi = 0; bi < 4; ++bi)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * bi + 4 * g + v;
        const float e = expf(ca[i]);
        uint16_t* orow = p.o + ck.row0 + (int64_t)i * p.s_t + 32 * w + r;
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) orow[16 * bj] = to_bf(e * qs[bi][bj][v] + pu[bi][bj][v]);
      }
  }
}

// ---- backward: the state gradient swept back over chunks -------------------------------
// One workgroup per (sequence, 32 columns of dS), chunks in reverse:
//   dSn_n = dS;  dU = P' dO + diag(e^(last - ca)) K dS;  dS <- Qg' dO + g dS - W' dU,
// the products on the matrix cores (split bf16).  While a chunk's products run,
// the previous chunk's inputs (P, the dO columns, Q, K, W, ca) are loaded
// into registers; they go to LDS once the chunk is done with its own.

constexpr int kLdP = 72;   // LDS row of 64 bf16
constexpr size_t kSgLds = (kC * kLdP + kC * kLdT / 2 + 2 * kC * kLdH + kC * kLdH / 2 + kD * kLdS + kD * kLdT + kC * kLdT + kC) * sizeof(float);

// One chunk's inputs as this thread loads them (plain vector types, so the
// whole set stays in registers).
struct SgInputs {
  f32x4v p[2];     // P: 2 x 16 bytes
  u32x2v d;        // dO columns col0 .. col0 + 31: 8 bytes (bf16)
  u32x4v q[2], k[2];  // Q, K: 2 x 16 bytes each (bf16)
  f32x4v w[4];
  float ca;
};

__device__ __forceinline__ void sg_load(SgInputs& in, const DnArgs& p, const Chunk& ck, int col0) {
  const int t = threadIdx.x;
  const float* Pc = p.P + ck.c * kC * kC;
  const float* Wc = p.W + ck.c * kC * kD;
#pragma unroll
  for (int e = 0; e < 2; ++e) in.p[e] = reinterpret_cast<const f32x4v*>(Pc)[t + kScanThreads * e];
  in.d = *reinterpret_cast<const u32x2v*>(p.dout + ck.row0 + (int64_t)(t / 8) * p.s_t + col0 + 4 * (t % 8));
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int x = t + kScanThreads * e, r = x / 16, c = 8 * (x % 16);
    in.q[e] = *reinterpret_cast<const u32x4v*>(p.q + ck.row0 + (int64_t)r * p.s_t + c);
    in.k[e] = *reinterpret_cast<const u32x4v*>(p.k + ck.row0 + (int64_t)r * p.s_t + c);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) in.w[e] = reinterpret_cast<const f32x4v*>(Wc)[t + kScanThreads * e];
  in.ca = t < kC ? p.ca[ck.c * kC + t] : 0.0f;
}

// The inputs to LDS; Q as Qg = diag(e^ca) Q (ca of the same chunk, already in LDS).
__device__ __forceinline__ void sg_store(const SgInputs& in, const Planes& P, uint16_t* dO, const Planes& Qg, uint16_t* K,
                                         const Planes& W, const float* ca) {
  const int t = threadIdx.x;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int x = t + kScanThreads * e;
    P.put(x / 16, 4 * (x % 16), in.p[e]);
  }
  *reinterpret_cast<u32x2v*>(dO + (t / 8) * kLdT + 4 * (t % 8)) = in.d;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int x = t + kScanThreads * e, r = x / 16, c = 8 * (x % 16);
    const float eq = expf(ca[r]);
    const u32x4v uq = in.q[e];
    *reinterpret_cast<u32x4v*>(K + r * kLdH + c) = in.k[e];
#pragma unroll
    for (int h = 0; h < 2; ++h)
      Qg.put(r, c + 4 * h, f32x4v{eq * bf((uint16_t)uq[2 * h]), eq * bf((uint16_t)(uq[2 * h] >> 16)),
                                  eq * bf((uint16_t)uq[2 * h + 1]), eq * bf((uint16_t)(uq[2 * h + 1] >> 16))});
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int x = t + kScanThreads * e;
    W.put(x / 32, 4 * (x % 32), in.w[e]);
  }
}

__global__ __launch_bounds__(kScanThreads, 1) void dn_state_grad(DnArgs p) {
  extern __shared__ float lds[];
  uint16_t* at = reinterpret_cast<uint16_t*>(lds);
  auto planes = [&](int rows, int ld) {
    const Planes x{at, at + rows * ld, ld};
    at += 2 * rows * ld;
    return x;
  };
  const Planes P = planes(kC, kLdP);    // [64][kLdP]
  const Planes Qg = planes(kC, kLdH);   // [64][kLdH]: diag(e^ca) Q
  const Planes W = planes(kC, kLdH);    // [64][kLdH]
  const Planes dSp = planes(kD, kLdT);  // [128][kLdT]: the state gradient's 32 columns
  const Planes dUp = planes(kC, kLdT);  // [64][kLdT]: dU
  uint16_t* dO = at;                    // [64][kLdT]: columns col0 .. col0 + 31 of dO
  uint16_t* K = dO + kC * kLdT;         // [64][kLdH]
  float* dS = reinterpret_cast<float*>(K + kC * kLdH);  // [128][kLdS]: the state gradient, as memory takes it
  float* ca = dS + kD * kLdS;           // [64]
  const int t = threadIdx.x, w = t / 64;
  const int g4 = plain((t % 64) / 16 * 4);
  const ScanSlot slot = scan_slot();
  const int64_t seq = slot.seq;
  const int col0 = slot.col0;
  for (int e = t; e < kD * kLdS; e += kScanThreads) dS[e] = 0.0f;
  for (int e = t; e < kD * kLdT; e += kScanThreads) dSp.hi[e] = 0, dSp.lo[e] = 0;
  f32x4v st[1][2];  // the state gradient: rows 16 w + 4 g + v, columns 16 bj + r
  clear(st);
  const Chunk first = chunk_of(p, seq * p.chunks);
  SgInputs in;
  {
    const Chunk ck = chunk_at(p, first, p.chunks - 1);
    sg_load(in, p, ck, col0);
    if (t < kC) ca[t] = in.ca;
    __syncthreads();
    sg_store(in, P, dO, Qg, K, W, ca);
  }
  for (int n = p.chunks - 1; n >= 0; --n) {
    const Chunk ck = chunk_at(p, first, n);
    __syncthreads();
    // This chunk's starting state, where this thread's dS values below sit:
    // dg's partial sums take it at the chunk's end.
    f32x4v s_in[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = t + kScanThreads * u, row = e / 8, c = 4 * (e % 8);
      s_in[u] = *reinterpret_cast<const f32x4v*>(p.S + ck.c * kD * kD + row * kD + col0 + c);
    }
    if (n > 0) sg_load(in, p, chunk_at(p, first, n - 1), col0);
    const float last = ca[kC - 1];
    // The gradient at the chunk's end state: read now, written to memory at
    // the chunk's end (and dU with it), after the previous chunk's inputs are
    // in LDS, whose wait for their loads would also wait for every store
    // issued before it.
    float* dSc = p.dSn + ck.c * kD * kD;
    f32x4v ds_out[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = t + kScanThreads * u, row = e / 8, c = 4 * (e % 8);
      ds_out[u] = *reinterpret_cast<const f32x4v*>(dS + row * kLdS + c);
    }
    // dU (64 x 32): wave w takes the 16 x 16 block at rows 16 (w mod 4),
    // columns 16 (w / 4).
    const int i0 = 16 * (w % 4), j0 = 16 * (w / 4);
    f32x4v du[1][1];
    {
      f32x4v kd[1][1];
      clear(du);
      clear(kd);
      mm_by(du, ColPlanes{P}, i0, ColBf16{dO, kLdT}, j0, kC);
      mm_by(kd, RowBf16{K, kLdH}, i0, ColPlanes{dSp}, j0, kD);
#pragma unroll
      for (int v = 0; v < 4; ++v) du[0][0][v] += expf(last - ca[i0 + g4 + v]) * kd[0][0][v];
      store_planes(dUp, du, i0, j0, 1.0f);
    }
    __syncthreads();
    // dS <- Qg' dO + g dS - W' dU (128 x 32): wave w takes rows 16 w .. 16 w + 15.
    {
      f32x4v qd[1][2], wu[1][2];
      clear(qd);
      clear(wu);
      mm_by(qd, ColPlanes{Qg}, 16 * w, ColBf16{dO, kLdT}, 0, kC);
      mm_by(wu, ColPlanes{W}, 16 * w, ColPlanes{dUp}, 0, kC);
      const float gl = expf(last);
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) st[0][bj][v] = qd[0][bj][v] + gl * st[0][bj][v] - wu[0][bj][v];
      __syncthreads();  // every wave has read dS, dU and this chunk's inputs
      store_blocks(dS, kLdS, st, 16 * w, 0, 1.0f);
      store_planes(dSp, st, 16 * w, 0, 1.0f);
    }
    if (n > 0) {
      if (t < kC) ca[t] = in.ca;
      __syncthreads();
      sg_store(in, P, dO, Qg, K, W, ca);
    }
    // dSn and dU of this chunk to memory.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = t + kScanThreads * u, row = e / 8, c = 4 * (e % 8);
      *reinterpret_cast<f32x4v*>(dSc + row * kD + col0 + c) = ds_out[u];
    }
    store_blocks(p.dU + ck.c * kC * kD + col0, kD, du, i0, j0, 1.0f);
    // This wave's part of dg = <S, dSn>.
    float dot = 0.0f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) dot = fmaf(s_in[u][e], ds_out[u][e], dot);
    dot = thd::wave_sum(dot);
    if (t % 64 == 0) p.dg[ck.c * kDgParts + (col0 / kCols) * (kScanThreads / 64) + w] = dot;
  }
}

// ---- backward: the chunk's products, WY form, decays and gates ---------------------
// dQg = dO S', dW = -dU S', dKd = U dSn', dP = lower(dO U'), then everything
// that follows from them: dT, dA = -T' dT T', the gate gradients and dQ, dK, dV.
// Bound by instructions, the splits of fp32 operands and the elementwise work: split
// once where they are written it took 889 us, at each read 1022, for the same
// bytes (a chunk reads 336 KB of states, U, dU, T and arrays and writes 48, 3.3
// TB/s of traffic).  The products stay in the registers that the outputs sum in (dQg
// in dQ's, dKd and T' dW in dK's, dP in the lanes that form dQK), so none of
// them goes through memory; as two kernels that passed dQg, dW, dKd and dP on
// (224 KB a chunk, out and back) the same took 1293 us at B4 H16 T8192.
//
// Every product on the matrix cores, split bf16; dO, Q and K sit in LDS as
// bf16 (their exact values); U, dU and dW take turns in one pair of bf16 planes (hi and
// lo), whose LDS M and N then share; V, T, S and dSn are
// read from memory by the products that use them (S and dSn by rows, each
// wave's 32).  Under 80 KB, so two workgroups share a CU.
// Wave w: columns 32 w .. 32 w + 31 of the 64 x 128 work, rows 16 w .. of the
// 64 x 64 work.  The row sums of the gate gradients are complete within a wave,
// the column work's partials go to LDS by wave and are folded in a fixed
// order, so the result does not depend on timing.

// acc1 += X1 Y, acc2 += X2 Y over k in [0, K): rows i0 .. of X1 and X2, each
// block of Y read once.
template <int BI, int BJ, class X1, class X2, class YR>
__device__ __forceinline__ void mm_by2(f32x4v (&acc1)[BI][BJ], const X1& x1, f32x4v (&acc2)[BI][BJ], const X2& x2,
                                       int i0, const YR& Y, int j0, int K) {
  const int r = lane_r(), g8 = lane_g8();
  for (int kb = 0; kb < K; kb += 32) {
    Split8 b[BJ];
#pragma unroll
    for (int bj = 0; bj < BJ; ++bj) b[bj] = Y.block(j0 + 16 * bj, kb, r, g8);
#pragma unroll
    for (int bi = 0; bi < BI; ++bi) {
      const Split8 a1 = x1.block(i0 + 16 * bi, kb, r, g8), a2 = x2.block(i0 + 16 * bi, kb, r, g8);
#pragma unroll
      for (int bj = 0; bj < BJ; ++bj) {
        acc1[bi][bj] = mma_split<X1::kExact, YR::kExact>(a1, b[bj], acc1[bi][bj]);
        acc2[bi][bj] = mma_split<X2::kExact, YR::kExact>(a2, b[bj], acc2[bi][bj]);
      }
    }
  }
}

// 64 x 128 fp32 rows of memory (stride kD) or bf16 rows (stride s_t), requested
// under the products before the LDS they go to is free.
struct HeldF32 {
  static constexpr int n = kC * 32 / 256;
  f32x4v x[n];
  __device__ void load(const float* src) {
#pragma unroll
    for (int u = 0; u < n; ++u) {
      const int e = threadIdx.x + 256 * u;
      x[u] = quad(src + (e / 32) * kD + 4 * (e % 32));
    }
  }
  __device__ void store(const Planes& to) const {
#pragma unroll
    for (int u = 0; u < n; ++u) {
      const int e = threadIdx.x + 256 * u;
      to.put(e / 32, 4 * (e % 32), x[u]);
    }
  }
};
struct HeldBf16 {
  static constexpr int n = kC * (kD / 8) / 256;
  u32x4v x[n];
  __device__ void load(const uint16_t* src, int64_t s_t) {
#pragma unroll
    for (int u = 0; u < n; ++u) {
      const int e = threadIdx.x + 256 * u;
      x[u] = *reinterpret_cast<const u32x4v*>(src + (e / (kD / 8)) * s_t + 8 * (e % (kD / 8)));
    }
  }
  __device__ void store(uint16_t* dst) const {
#pragma unroll
    for (int u = 0; u < n; ++u) {
      const int e = threadIdx.x + 256 * u;
      *reinterpret_cast<u32x4v*>(dst + (e / (kD / 8)) * kLdH + 8 * (e % (kD / 8))) = x[u];
    }
  }
};

constexpr int kGradX = 2 * kC * kLdP;   // floats: M and N as planes; U, dU and dW take 2 kC kLdH / 2
static_assert(kGradX >= kC * kLdH && kC * kLdP >= kC * kLdC, "");
constexpr size_t kGradLds = 2 * kC * kLdH * sizeof(uint16_t) + kGradX * sizeof(float) +
                            (2 * kC + 5 * 4 * kC + 2 * kC) * sizeof(float);

__global__ __launch_bounds__(256, 2) void dn_grad(DnArgs p) {
  extern __shared__ float lds[];
  uint16_t* Qh = reinterpret_cast<uint16_t*>(lds);       // [64][kLdH]: dO, then Q
  uint16_t* Kh = Qh + kC * kLdH;                          // [64][kLdH]
  uint16_t* x0 = Kh + kC * kLdH;
  const Planes X{x0, x0 + kC * kLdH, kLdH};               // [64][kLdH]: U, then dU, then dW
  const Planes M{x0, x0 + kC * kLdP, kLdP};               // [64][kLdP]: dT, then dG + dG'
  uint16_t* n0 = x0 + 2 * kC * kLdP;
  const Planes Np{n0, n0 + kC * kLdP, kLdP};              // [64][kLdP]: dQK
  float* N = reinterpret_cast<float*>(n0);                // [64][kLdC] before: T' dT, then dG
  float* wrow = reinterpret_cast<float*>(x0) + kGradX;    // [64]: sum_j w_ij
  float* brow = wrow + kC;         // [64]: sum_j dA Gamma G
  float* wcol = brow + kC;         // [4][64]: sum_i w_ij by wave
  float* kx = wcol + 4 * kC;       // [4][64]: k . dX by wave (columns)
  float* vy = kx + 4 * kC;         // [4][64]
  float* qq = vy + 4 * kC;         // [4][64]
  float* kk = qq + 4 * kC;         // [4][64]
  float* ca = kk + 4 * kC;         // [64]
  float* be = ca + kC;             // [64]
  const Chunk ck = chunk_of(p, blockIdx.x);
  const int t = threadIdx.x, w = t / 64;
  const int r = plain(t % 16), g4 = plain((t % 64) / 16 * 4);  // 4 x the row group
  const uint16_t* vg = p.v + ck.row0;
  const float* Tc = p.T + ck.c * kC * kC;  // [64][64]
  const int i0 = 16 * w;  // this wave's rows of the 64 x 64 work
  const int d0 = 32 * w;  // and its columns of the 64 x 128 work
  // This lane's place in block (0, 0) of its wave's columns of an array; the
  // rows of the other blocks are uniform offsets from it.
  const int64_t lane_at = ck.row0 + g4 * p.s_t + d0 + r;
  const uint16_t* vl = p.v + lane_at;
  uint16_t *dql = p.dq + lane_at, *dkl = p.dk + lane_at, *dvl = p.dv + lane_at;
  HeldF32 held;
  held.load(p.U + ck.c * kC * kD);
  stage_rows_bf16(Qh, p.dout + ck.row0, Kh, p.k + ck.row0, p.s_t);
  held.store(X);
  const float dg_part = t < kDgParts ? p.dg[ck.c * kDgParts + t] : 0.0f;
  if (t < 64) {
    ca[t] = p.ca[ck.c * kC + t];
    be[t] = p.beta[ck.grow0 + (int64_t)t * p.g_t];
  }
  __syncthreads();
  const RowBf16 Kr{Kh, kLdH}, Qr{Qh, kLdH};
  const ColBf16 Kc{Kh, kLdH}, Qc{Qh, kLdH};
  const float last = ca[kC - 1];
  const RowPlanes Xr{X};
  const ColPlanes Xc{X};
  const RowBf16 Or{Qh, kLdH};
  // U: dKd = U dSn' (kd; sk = k . dKd a row) and dP = lower(dO U') (this wave's rows).
  f32x4v kd[4][2], dp[1][4];
  clear(kd);
  clear(dp);
  mm_by(kd, Xr, 0, RowF32{p.dSn + ck.c * kD * kD, kD}, d0, kD);
#pragma unroll
  for (int bj = 0; bj < 4; ++bj)
    if (bj <= w) {
      f32x4v a1[1][1];
      clear(a1);
      mm_by(a1, Or, i0, Xr, 16 * bj, kD);
#pragma unroll
      for (int v = 0; v < 4; ++v) dp[0][bj][v] = i0 + g4 + v >= 16 * bj + r ? a1[0][0][v] : 0.0f;
    }
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 16 * bi + g4 + v;
      const float ed = expf(last - ca[i]);
      float sk = 0.0f;
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) {
        sk = fmaf(bf(Kh[i * kLdH + d0 + 16 * bj + r]), kd[bi][bj][v], sk);
        float x = kd[bi][bj][v] * ed;
        asm("" : "+v"(x));  // formed here: put off to its use, it would hold ed and dKd till then
        kd[bi][bj][v] = x;
      }
      sk = row_group_sum(sk);
      if (r == 0) kk[w * kC + i] = sk;
    }
  __syncthreads();
  held.load(p.dU + ck.c * kC * kD);
  held.store(X);
  __syncthreads();
  // dU: dV = beta T' dU~, dU~ V' (this wave's rows), dQg = dO S', dW = -dU S'.
  f32x4v yv[1][4];
  {
    f32x4v dy[4][2];
    clear(dy);
    mm_by(dy, ColF32{Tc, kC}, 0, Xc, d0, kC);
    // In two halves of row blocks: the V values of a half are all read
    // before its first dV store (same element type: loaded in the loop,
    // each read would wait for the previous store).
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      uint32_t vh[2][4];  // the two bf16 of columns d0 + r, d0 + 16 + r
#pragma unroll
      for (int b2 = 0; b2 < 2; ++b2)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const uint16_t* vr = vl + (16 * (2 * hb + b2) + v) * p.s_t;
          vh[b2][v] = (uint32_t)vr[0] | ((uint32_t)vr[16] << 16);
        }
#pragma unroll
      for (int b2 = 0; b2 < 2; ++b2)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int bi = 2 * hb + b2, i = 16 * bi + g4 + v;
          float sv = 0.0f;
#pragma unroll
          for (int bj = 0; bj < 2; ++bj) {
            const float vv = bf((uint16_t)(vh[b2][v] >> (16 * bj))), yv1 = dy[bi][bj][v];
            sv = fmaf(vv, yv1, sv);
            dvl[(16 * bi + v) * p.s_t + 16 * bj] = to_bf(be[i] * yv1);
          }
          sv = row_group_sum(sv);
          if (r == 0) vy[w * kC + i] = sv;
        }
    }
    clear(yv);
    mm_by(yv, Xr, i0, RowBf16G{vg, p.s_t}, 0, kD);
  }
  f32x4v dq[4][2];
  {
    HeldBf16 q;
    f32x4v wq[4][2];
    clear(dq);
    clear(wq);
    mm_by2(dq, Or, wq, Xr, 0, RowF32{p.S + ck.c * kD * kD, kD}, d0, kD);
    __syncthreads();
    store_planes(X, wq, 0, d0, -1.0f);
    q.load(p.q + ck.row0, p.s_t);
    q.store(Qh);
  }
  __syncthreads();
  // dW: dX = T' dW into dK's sum (beta e^ca dX + e^(last - ca) dKd), and
  // dT = dW X' + dU~ Y',  X = diag(beta e^ca) K, Y = diag(beta) V; the row sums q . dQg and k . dX.
  {
    f32x4v dx[4][2];
    clear(dx);
    mm_by(dx, ColF32{Tc, kC}, 0, Xc, d0, kC);
#pragma unroll
    for (int bi = 0; bi < 4; ++bi)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * bi + g4 + v;
        const float e = expf(ca[i]);
        float sq = 0.0f, sx = 0.0f;
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
          const int d = d0 + 16 * bj + r;
          sq = fmaf(bf(Qh[i * kLdH + d]), dq[bi][bj][v], sq);
          sx = fmaf(bf(Kh[i * kLdH + d]), dx[bi][bj][v], sx);
          dq[bi][bj][v] *= e;
          kd[bi][bj][v] = fmaf(be[i] * e, dx[bi][bj][v], kd[bi][bj][v]);
        }
        sq = row_group_sum(sq);
        sx = row_group_sum(sx);
        if (r == 0) qq[w * kC + i] = sq, kx[w * kC + i] = sx;
      }
    f32x4v xk[1][4];
    clear(xk);
    mm_by(xk, Xr, i0, Kr, 0, kD);
    __syncthreads();
#pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
      const float bl = be[16 * bj + r], el = expf(ca[16 * bj + r]);
#pragma unroll
      for (int v = 0; v < 4; ++v) xk[0][bj][v] = bl * (el * xk[0][bj][v] + yv[0][bj][v]);
    }
    store_planes(M, xk, i0, 0, 1.0f);
  }
  __syncthreads();
  // N = T' dT.
  {
    f32x4v acc[1][4];
    clear(acc);
    mm_by(acc, ColF32{Tc, kC}, i0, ColPlanes{M}, 0, kC);
    store_blocks(N, kLdC, acc, i0, 0, 1.0f);
  }
  __syncthreads();
  // dA = -(N T') o strict lower (this wave's rows of N are its own).
  f32x4v dA[1][4];
  clear(dA);
  mm_by(dA, RowF32{N, kLdC}, i0, RowF32{Tc, kC}, 0, kC);
  // With G = K K', QK = Q K', Gamma: dG = dA o beta_i o Gamma (into N);
  // dbeta_i gets sum_j dA Gamma G; w = (dA beta_i G + dP QK) o Gamma gives
  // dca_i += sum_j w_ij - sum_j w_ji.
  {
    f32x4v gk[1][4], qk[1][4];
    clear(gk);
    clear(qk);
#pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
      if (bj <= w) {
        f32x4v a1[1][1], a2[1][1];
        clear(a1);
        clear(a2);
        mm_by(a1, Kr, i0, Kr, 16 * bj, kD);
        mm_by(a2, Qr, i0, Kr, 16 * bj, kD);
        gk[0][bj] = a1[0][0];
        qk[0][bj] = a2[0][0];
      }
    }
    float roww[4] = {0, 0, 0, 0}, rowb[4] = {0, 0, 0, 0};
    float colw[4] = {0, 0, 0, 0};  // column 16 bj + r, this wave's rows
#pragma unroll
    for (int bj = 0; bj < 4; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = i0 + g4 + v, j = 16 * bj + r;
        // (Above the diagonal the exponent is positive: past e^88 it would be
        // an infinity times that 0.)
        const float gam = i >= j ? expf(ca[i] - ca[j]) : 0.0f;
        const float da = i > j ? -dA[0][bj][v] : 0.0f;
        const float gg = bj <= w ? gk[0][bj][v] : 0.0f, q = bj <= w ? qk[0][bj][v] : 0.0f;
        N[i * kLdC + j] = da * be[i] * gam;
        rowb[v] += da * gam * gg;
        const float wv = i >= j ? (da * be[i] * gg + dp[0][bj][v] * q) * gam : 0.0f;
        roww[v] += wv;
        colw[bj] += wv;
        dp[0][bj][v] = i >= j ? dp[0][bj][v] * gam : 0.0f;  // dQK
      }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      roww[v] = row_group_sum(roww[v]);
      rowb[v] = row_group_sum(rowb[v]);
    }
    if (r == 0)
#pragma unroll
      for (int v = 0; v < 4; ++v) wrow[i0 + g4 + v] = roww[v], brow[i0 + g4 + v] = rowb[v];
    // Column sums over this wave's 16 rows: the four row groups g, in order.
#pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
      float x = colw[bj];
      x += __shfl_xor(x, 16, 64);
      x += __shfl_xor(x, 32, 64);
      if (g4 == 0) wcol[w * kC + 16 * bj + r] = x;
    }
  }
  __syncthreads();
  // M <- dG + dG'.
  for (int e = t; e < kC * kC / 2; e += 256) {
    const int i = e / (kC / 2), j = 2 * (e % (kC / 2));
    M.put(i, j, N[i * kLdC + j] + N[j * kLdC + i], N[i * kLdC + j + 1] + N[(j + 1) * kLdC + i]);
  }
  __syncthreads();
  // dQK = dP o Gamma (lower), read by two of the products below along its rows
  // and its columns, into N (free now).
  store_planes(Np, dp, i0, 0, 1.0f);
  __syncthreads();
  // dQ = e^ca dQg + dQK K;  dK = dQK' Q + (dG + dG') K + beta e^ca dX + e^(last - ca) dKd.
  mm_by(dq, RowPlanes{Np}, 0, Kc, d0, kC);
  mm_by(kd, ColPlanes{Np}, 0, Qc, d0, kC);
  mm_by(kd, RowPlanes{M}, 0, Kc, d0, kC);
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) {
        const int64_t at = (16 * bi + v) * p.s_t + 16 * bj;
        dql[at] = to_bf(dq[bi][bj][v]);
        dkl[at] = to_bf(kd[bi][bj][v]);
      }
  // Fold the partials in a fixed order (lane i: row i), then da = the
  // reverse cumulative sum of dca, dca_63 also taking sum kd + dg g.
  if (t < 64) {
    const int i = t;
    float sc = 0.0f, skx = 0.0f, svy = 0.0f, sqq = 0.0f, skk = 0.0f;
    for (int wv = 0; wv < 4; ++wv) {
      sc += wcol[wv * kC + i];
      skx += kx[wv * kC + i];
      svy += vy[wv * kC + i];
      sqq += qq[wv * kC + i];
      skk += kk[wv * kC + i];
    }
    const float sw = wrow[i], sb = brow[i];
    const float e = expf(ca[i]), ed = expf(last - ca[i]);
    const float kd = ed * skk;
    float dca = sw - sc + be[i] * e * skx + e * sqq - kd;
    float kd_all = kd;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kd_all += __shfl_xor(kd_all, o, 64);
    // dg: its kDgParts partial sums, lane q holding part q, a fixed tree.
    float dg = i < kDgParts ? dg_part : 0.0f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dg += __shfl_xor(dg, o, 64);
    if (i == kC - 1) dca += kd_all + dg * expf(last);
    float x = dca;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float y = __shfl_down(x, o, 64);
      if (i + o < 64) x += y;
    }
    p.da[ck.grow0 + (int64_t)i * p.g_t] = x;
    p.dbeta[ck.grow0 + (int64_t)i * p.g_t] = sb + e * skx + svy;
  }
}

bool aligned(const void* q, int bytes) { return (reinterpret_cast<uintptr_t>(q) % bytes) == 0; }

// ca, T, W, Ut, S, U, P; for the backward dU, dSn, dg
constexpr int kSlots = 10;
struct Workspace {
  size_t offs[kSlots];
  size_t bytes;
};

Workspace workspace(int64_t chunks, bool backward) {
  const size_t sizes[kSlots] = {(size_t)kC,      (size_t)kC * kC, (size_t)kC * kD, (size_t)kC * kD, (size_t)kD * kD,
                                (size_t)kC * kD, (size_t)kC * kC, (size_t)kC * kD, (size_t)kD * kD, (size_t)kDgParts};
  Workspace w{};
  size_t at = 0;
  for (int i = 0; i < kSlots; ++i) {
    w.offs[i] = at;
    if (i < 7 || backward) at += ((sizes[i] * chunks * sizeof(float)) + 255) & ~(size_t)255;
  }
  w.bytes = at;
  return w;
}

int check(const th_deltanet_desc* d, bool backward) {
  TH_REQUIRE(d != nullptr, "deltanet: null descriptor");
  TH_REQUIRE(d->dk == kD && d->dv == kD, "deltanet: dk and dv must be 128");
  TH_REQUIRE(d->chunk == kC, "deltanet: the chunk must be 64");
  TH_REQUIRE(d->seq > 0 && d->seq % kC == 0, "deltanet: the sequence length must be a positive multiple of 64");
  TH_REQUIRE(d->batch > 0 && d->heads > 0, "deltanet: batch and heads must be positive");
  TH_REQUIRE(d->q && d->k && d->v && d->a && d->beta && (d->o || backward), "deltanet: null q, k, v, a, beta or o");
  TH_REQUIRE(aligned(d->q, 16) && aligned(d->k, 16) && aligned(d->v, 16) && aligned(d->o, 16),
             "deltanet: q, k, v, o must be 16-byte aligned");
  TH_REQUIRE(d->strides[0] % 8 == 0 && d->strides[1] % 8 == 0 && d->strides[2] % 8 == 0,
             "deltanet: strides must be multiples of 8");
  if (backward) {
    TH_REQUIRE(d->dout && d->dq && d->dk_out && d->dv_out && d->da && d->dbeta, "deltanet backward: null gradient");
    TH_REQUIRE(aligned(d->dout, 16) && aligned(d->dq, 16) && aligned(d->dk_out, 16) && aligned(d->dv_out, 16),
               "deltanet backward: gradients must be 16-byte aligned");
  }
  return TH_OK;
}

int build(const th_deltanet_desc* d, bool backward, th_launch** out) {
  if (int r = th::require_ready()) return r;
  *out = nullptr;
  if (int r = check(d, backward)) return r;
  const int64_t chunks = (int64_t)d->batch * d->heads * (d->seq / kC);
  TH_REQUIRE(chunks <= 0x7fffffff, "deltanet: too many chunks");
  const Workspace w = workspace(chunks, backward);
  DnArgs a{};
  a.q = static_cast<const uint16_t*>(d->q);
  a.k = static_cast<const uint16_t*>(d->k);
  a.v = static_cast<const uint16_t*>(d->v);
  a.a = d->a;
  a.beta = d->beta;
  a.o = static_cast<uint16_t*>(d->o);
  a.dout = static_cast<const uint16_t*>(d->dout);
  a.dq = static_cast<uint16_t*>(d->dq);
  a.dk = static_cast<uint16_t*>(d->dk_out);
  a.dv = static_cast<uint16_t*>(d->dv_out);
  a.da = d->da;
  a.dbeta = d->dbeta;
  // The per-chunk intermediates (ca, T, W, Ut, S, U, P; for the backward dU,
  // dSn, dg) lie in the launch's workspace at w.offs.
  const size_t slot_args[kSlots] = {TH_OFFSET(DnArgs, ca), TH_OFFSET(DnArgs, T),  TH_OFFSET(DnArgs, W),
                                    TH_OFFSET(DnArgs, Ut), TH_OFFSET(DnArgs, S),  TH_OFFSET(DnArgs, U),
                                    TH_OFFSET(DnArgs, P),  TH_OFFSET(DnArgs, dU), TH_OFFSET(DnArgs, dSn),
                                    TH_OFFSET(DnArgs, dg)};
  a.s_h = d->strides[0];
  a.s_t = d->strides[1];
  a.s_b = d->strides[2];
  a.g_h = d->gate_strides[0];
  a.g_t = d->gate_strides[1];
  a.g_b = d->gate_strides[2];
  a.batch = d->batch;
  a.heads = d->heads;
  a.seq = d->seq;
  a.chunks = d->seq / kC;
  const void* fns[5] = {(const void*)dn_chunk_prep, (const void*)dn_state_scan, (const void*)dn_output,
                        (const void*)dn_state_grad, (const void*)dn_grad};
  const size_t ldss[5] = {kPrepLds, kScanLds, kOutLds, kSgLds, kGradLds};
  for (int i = 0; i < 5; ++i) TH_HIP(hipFuncSetAttribute(fns[i], hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldss[i]));
  th::Builder b(backward ? "deltanet_fwd_bwd" : "deltanet_fwd", 12);
  const uint64_t at_ws = b.workspace(w.bytes);
  // A gradient with no o given keeps it in the workspace, at q's strides.
  const bool own_o = d->o == nullptr;
  const uint64_t o_bytes = 2 * ((uint64_t)(d->heads - 1) * d->strides[0] + (uint64_t)(d->seq - 1) * d->strides[1] +
                                (uint64_t)(d->batch - 1) * d->strides[2] + kD);
  const uint64_t at_o = own_o ? b.workspace(o_bytes) : 0;
  const unsigned nchunks = (unsigned)chunks;
  const unsigned scans = (unsigned)((int64_t)d->batch * d->heads * (kD / kCols));
  int ks[5];
  int nk = 0;
  ks[nk++] = b.kernel(fns[0], "dn_chunk_prep", dim3(nchunks), dim3(256), (uint32_t)kPrepLds, a);
  ks[nk++] = b.kernel(fns[1], "dn_state_scan", dim3(scans), dim3(kScanThreads), (uint32_t)kScanLds, a);
  ks[nk++] = b.kernel(fns[2], "dn_output", dim3(nchunks), dim3(256), (uint32_t)kOutLds, a);
  if (backward) {
    ks[nk++] = b.kernel(fns[3], "dn_state_grad", dim3(scans), dim3(kScanThreads), (uint32_t)kSgLds, a);
    ks[nk++] = b.kernel(fns[4], "dn_grad", dim3(nchunks), dim3(256), (uint32_t)kGradLds, a);
  }
  const size_t offs[12] = {TH_OFFSET(DnArgs, q),  TH_OFFSET(DnArgs, k),  TH_OFFSET(DnArgs, v),     TH_OFFSET(DnArgs, a),
                           TH_OFFSET(DnArgs, beta), TH_OFFSET(DnArgs, o), TH_OFFSET(DnArgs, dout), TH_OFFSET(DnArgs, dq),
                           TH_OFFSET(DnArgs, dk), TH_OFFSET(DnArgs, dv), TH_OFFSET(DnArgs, da),  TH_OFFSET(DnArgs, dbeta)};
  for (int v = 0; v < 12; ++v)
    if (!(own_o && v == 5))
      for (int i = 0; i < nk; ++i) b.ref(v, ks[i], offs[v]);
  if (own_o)
    for (int i = 0; i < nk; ++i) b.ws_ref(ks[i], offs[5], at_o);
  for (int j = 0; j < kSlots; ++j)
    if (j < 7 || backward)
      for (int i = 0; i < nk; ++i) b.ws_ref(ks[i], slot_args[j], at_ws + w.offs[j]);
  for (int v : {0, 1, 2, 5, 6, 7, 8, 9}) b.align(v, 16);
  // Algorithmic work: per chunk, forward ~ C^2 dk (A) + C^3/3 (T) + 2 C^2 d (W, U~) + C^2 dk (P)
  // + 2 C dk dv (W S, Qg S) + C^2 dv (P U) + C dk dv (Kd' U) multiply-adds; the backward ~2.3x.
  const double C = kC, D = kD;
  const double fwd = 2.0 * (C * C * D + C * C * C / 3 + 2 * C * C * D + C * C * D + 3 * C * D * D + C * C * D);
  const double bytes_fwd = 2.0 * (4 * C * D) + 8.0 * C;  // q, k, v read, o written (bf16); a, beta
  b.work(chunks * (backward ? fwd * 3.3 : fwd), chunks * (backward ? 2 * bytes_fwd + 2.0 * 4 * C * D : bytes_fwd),
         chunks);
  th_launch* l = b.release();
  l->work.bytes = chunks * (backward ? 2 * bytes_fwd + 2.0 * 4 * C * D : bytes_fwd);
  l->work.flops = chunks * (backward ? fwd * 3.3 : fwd);
  *out = l;
  return TH_OK;
}

}  // namespace

extern "C" int th_build_deltanet_fwd(const th_deltanet_desc* d, th_launch** out) { return build(d, false, out); }

extern "C" int th_build_deltanet(const th_deltanet_desc* d, th_launch** out) { return build(d, true, out); }
