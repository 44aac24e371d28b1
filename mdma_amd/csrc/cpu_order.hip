// The CPU-order mode (MDMA_ACT_F32_CPU): the quantized matmul and the ops
// around it computed in the reference CPU backend's arithmetic order, so
// their results are the CPU backend's bit for bit.
//
// CpuBackend::qmatmul (/root/reference/src/backend/cpu.rs:46-48,335-368):
// each row is dequantized to f32 (candle's to_float, called from
// src/backend/cpu/dequant.rs:36) and every output is a sequential f32 sum,
// starting from -0.0, of the f32-rounded products w_i * x_i, never fused
// into an FMA. A sum in that order is one dependent chain, so here one lane
// owns one output row (and up to 8 tokens' chains of it); rows run in
// parallel, the columns of a row in order.
//
// The dequantized weights are exact products (the values match candle's in
// any evaluation order): Q8_0 q * d has 8 + 11 significant bits; Q6_K
// (d * sc) * q at most 11 + 7 + 5 < 24; Q4_K d * sc and dmin * m have at most
// 17 bits and (d * sc) * q 21, so only the final subtraction d*sc*q - dmin*m
// rounds, once.
//
// rmsnorm (cpu.rs:388-402), silu_mul (:447-458) and attention (:530-590,
// softmax_inplace :50-60) follow the CPU's sequence of roundings too:
// sequential sums, correctly rounded division and square root (formed in
// double and rounded once to f32, which for one operation on f32 operands
// gives the correctly rounded f32 result), and the C library's expf
// (libm_expf.h). The file is compiled with `fp contract(off)`: no f32
// multiply-add is fused.
#include <algorithm>

#include "internal.h"
#include "kernels.h"
#include "libm_expf.h"

// No f32 multiply and add in this file is fused into an FMA.
#pragma clang fp contract(off)

namespace mdma {
namespace {

// Correctly rounded f32 division and square root.
__device__ __forceinline__ float div_rn(float a, float b) { return (float)((double)a / (double)b); }
__device__ __forceinline__ float sqrt_rn(float a) { return (float)__builtin_sqrt((double)a); }

__device__ __forceinline__ uint32_t byte_of(uint32_t w, int k) { return (w >> (8 * k)) & 0xffu; }

// One group of a row's weights in registers, in GGUF byte order whatever
// the buffer's layout (layout.cpp's planes are gathered back), and its
// dequantized element e. GC: columns per group.
template <int DT>
struct Group;

template <>
struct Group<DT_Q4_K> {
  static constexpr int GC = 256;
  uint4 hd;       // f16 d, f16 dmin, 12 scale bytes
  uint32_t q[32];  // 128 quant bytes
  float d1[8], m1[8];
  __device__ __forceinline__ void load(const uint8_t *wr, uint32_t nb, uint32_t b, bool prepared) {
    if (prepared) {
      const uint32_t U = 4 * nb;
#pragma unroll
      for (int p = 0; p < 4; p++) {
        const uint4 a = ldx16(wr + 16 * (4 * b + p)), c = ldx16(wr + 16 * (U + 4 * b + p));
        q[8 * p + 0] = a.x, q[8 * p + 1] = a.y, q[8 * p + 2] = a.z, q[8 * p + 3] = a.w;
        q[8 * p + 4] = c.x, q[8 * p + 5] = c.y, q[8 * p + 6] = c.z, q[8 * p + 7] = c.w;
      }
      hd = ldx16(wr + 32 * U + 16 * b);
    } else {
      const uint8_t *blk = wr + 144 * (size_t)b;
      hd = ldx16(blk);
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint4 a = ldx16(blk + 16 + 16 * k);
        q[4 * k + 0] = a.x, q[4 * k + 1] = a.y, q[4 * k + 2] = a.z, q[4 * k + 3] = a.w;
      }
    }
    const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
#pragma unroll
    for (int p = 0; p < 4; p++) {
      int sca, scb, ma, mb;
      q4k_scales_i(hd, p, sca, scb, ma, mb);
      d1[2 * p] = d * (float)sca, m1[2 * p] = dmin * (float)ma;
      d1[2 * p + 1] = d * (float)scb, m1[2 * p + 1] = dmin * (float)mb;
    }
  }
  // Column e: sub-block s = e / 32, pair j = e / 64, byte 32 j + e % 32,
  // the low nibble for even s, the high one for odd.
  __device__ __forceinline__ float deq(int e) const {
#pragma clang fp contract(off)
    const int s = e / 32, j = e / 64, byte = 32 * j + e % 32;
    const uint32_t qv = (byte_of(q[byte / 4], byte % 4) >> (4 * (s & 1))) & 0xF;
    const float t = d1[s] * (float)qv;
    return t - m1[s];
  }
};

template <>
struct Group<DT_Q6_K> {
  static constexpr int GC = 256;
  uint32_t ql[32], qh[16];
  uint32_t scw[2][2];  // scw[n][h] byte r: the scale of quarter r, columns 128 n + 32 r + 16 h ..
  float d;
  __device__ __forceinline__ void load(const uint8_t *wr, uint32_t nb, uint32_t b, bool prepared) {
    if (prepared) {
      const uint32_t U = 4 * nb;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int n = k >> 1, h = k & 1;
        const uint32_t u = 4 * b + k;
        const uint4 a = ldx16(wr + 16 * u), c = ldx16(wr + 16 * (U + u)), e = ldx16(wr + 16 * (2 * U + u));
        const int qa = 16 * n + 4 * h, qb = 16 * n + 8 + 4 * h, hh = 8 * n + 4 * h;
        ql[qa] = a.x, ql[qa + 1] = a.y, ql[qa + 2] = a.z, ql[qa + 3] = a.w;
        ql[qb] = c.x, ql[qb + 1] = c.y, ql[qb + 2] = c.z, ql[qb + 3] = c.w;
        qh[hh] = e.x, qh[hh + 1] = e.y, qh[hh + 2] = e.z, qh[hh + 3] = e.w;
        scw[n][h] = *reinterpret_cast<const uint32_t *>(wr + 48 * U + 4 * u);
      }
      d = h2f(ldu16(wr + 52 * U + 2 * b));
    } else {
      const uint8_t *blk = wr + 210 * (size_t)b;  // 2-byte aligned
#pragma unroll
      for (int k = 0; k < 32; k++) ql[k] = ld2x16(blk + 4 * k);
#pragma unroll
      for (int k = 0; k < 16; k++) qh[k] = ld2x16(blk + 128 + 4 * k);
      uint32_t sc[4];
#pragma unroll
      for (int k = 0; k < 4; k++) sc[k] = ld2x16(blk + 192 + 4 * k);
      // scw[n][h] byte r = sc[8 n + 2 r + h]
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          uint32_t w = 0;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int i = 8 * n + 2 * r + h;
            w |= byte_of(sc[i / 4], i % 4) << (8 * r);
          }
          scw[n][h] = w;
        }
      d = h2f(ldu16(blk + 208));
    }
  }
  // Column e = 128 n + 32 r + l: low 4 bits from ql[64 n + 32 (r & 1) + l]
  // (low nibble for r < 2), high 2 bits from qh[32 n + l] >> 2 r, scale
  // sc[8 n + 2 r + l / 16]; the value (d * sc) * (q - 32).
  __device__ __forceinline__ float deq(int e) const {
#pragma clang fp contract(off)
    const int n = e / 128, r = (e % 128) / 32, l = e % 32, h = l / 16;
    const int lb = 64 * n + 32 * (r & 1) + l, hb = 32 * n + l;
    const uint32_t low = (byte_of(ql[lb / 4], lb % 4) >> (r < 2 ? 0 : 4)) & 0xF;
    const uint32_t high = (byte_of(qh[hb / 4], hb % 4) >> (2 * r)) & 3;
    const int qv = (int)(low | (high << 4)) - 32;
    const int sc = (int)(int8_t)byte_of(scw[n][h], r);
    const float ds = d * (float)sc;
    return ds * (float)qv;
  }
};

template <>
struct Group<DT_Q8_0> {
  static constexpr int GC = 32;
  uint32_t q[8];
  float d;
  __device__ __forceinline__ void load(const uint8_t *wr, uint32_t nb, uint32_t b, bool prepared) {
    if (prepared) {
      const uint4 a = ldx16(wr + 16 * b), c = ldx16(wr + 16 * (nb + b));
      q[0] = a.x, q[1] = a.y, q[2] = a.z, q[3] = a.w, q[4] = c.x, q[5] = c.y, q[6] = c.z, q[7] = c.w;
      d = h2f(ldu16(wr + 32 * nb + 2 * b));
    } else {
      const uint8_t *blk = wr + 34 * (size_t)b;  // 2-byte aligned
#pragma unroll
      for (int k = 0; k < 8; k++) q[k] = ld2x16(blk + 2 + 4 * k);
      d = h2f(ldu16(blk));
    }
  }
  __device__ __forceinline__ float deq(int e) const {
#pragma clang fp contract(off)
    const int qv = (int)(int8_t)byte_of(q[e / 4], e % 4);
    return (float)qv * d;
  }
};

constexpr int SEQ_TT = 8;  // token chains per lane for calls of more than one token

// y[t, row] for rows blockIdx.x * 64 + lane and tokens blockIdx.y * TT ..:
// the sequential sums. x is staged one group at a time into LDS (every lane
// then reads the same word: a broadcast).
template <int DT, int TT>
__global__ __launch_bounds__(64) void gemv_seq_kernel(const uint8_t *__restrict__ w, uint64_t row_bytes,
                                                      uint32_t n_out, uint32_t n_in, bool prepared,
                                                      const float *__restrict__ x, uint32_t T,
                                                      float *__restrict__ y) {
#pragma clang fp contract(off)
  constexpr int GC = Group<DT>::GC;
  __shared__ __attribute__((aligned(16))) float xs[TT][GC];
  const uint32_t lane = threadIdx.x, row = blockIdx.x * 64 + lane, t0 = blockIdx.y * TT;
  const uint8_t *wr = w + (size_t)min(row, n_out - 1) * row_bytes;
  const uint32_t ng = n_in / GC;
  float s[TT];
#pragma unroll
  for (int k = 0; k < TT; k++) s[k] = -0.0f;
  for (uint32_t g = 0; g < ng; g++) {
    Group<DT> grp;
    grp.load(wr, ng, g, prepared);
    __syncthreads();  // the previous group's reads of xs are done
    for (uint32_t i = lane; i < TT * GC / 4; i += 64) {
      const uint32_t k = i / (GC / 4), c = i % (GC / 4), t = min(t0 + k, T - 1);
      *reinterpret_cast<float4 *>(&xs[k][4 * c]) =
          *reinterpret_cast<const float4 *>(x + (size_t)t * n_in + (size_t)g * GC + 4 * c);
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < GC; e++) {
      const float wv = grp.deq(e);
#pragma unroll
      for (int k = 0; k < TT; k++) {
        const float p = wv * xs[k][e];
        s[k] = s[k] + p;
      }
    }
  }
  if (row < n_out) {
#pragma unroll
    for (int k = 0; k < TT; k++)
      if (t0 + k < T) y[(size_t)(t0 + k) * n_out + row] = s[k];
  }
}

// s plus n4 float4 of LDS (a multiple of 8), in order, one dependent
// addition each: the next 8 reads are in flight while 8 are added. On gfx950
// a dependent f32 addition takes 8.4 cycles (measured), so 4096 of them take
// about 15 us whatever feeds them.
typedef float v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float chain8(float s, const v4f (&v)[8]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int k = 0; k < 8; k++) {
    s = s + v[k].x;
    s = s + v[k].y;
    s = s + v[k].z;
    s = s + v[k].w;
  }
  return s;
}
template <class Read>
__device__ __forceinline__ float chain_add(float s, uint32_t n4, Read &&rd) {
  v4f v[8], w[8];
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = rd(k);
  for (uint32_t g = 0; g < n4; g += 16) {
    const uint32_t g1 = g + 8 < n4 ? g + 8 : g, g2 = g + 16 < n4 ? g + 16 : g;  // (past the end: read, not added)
#pragma unroll
    for (int k = 0; k < 8; k++) w[k] = rd(g1 + k);
    s = chain8(s, v);
    if (g + 8 >= n4) break;
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = rd(g2 + k);
    s = chain8(s, w);
  }
  return s;
}

// ---- few tiles over prepared rows: dequantization and chains apart ----
// (4 tokens and 16 rows a workgroup, the groups of tokens in the grid)
// With one lane doing everything for its row, the chain's next addition waits
// for the column's whole dequantization (about 11 VALU instructions a
// column), on one wave per SIMD. Here NP producer waves dequantize, multiply
// by x and leave the f32-rounded products in LDS, and chain waves (one lane
// per row and token) only add them, in column order: the same operations on
// the same operands, so the same bits. What bounds it is the chain, one
// dependent f32 addition per column, where the rows leave CUs free (one token,
// 4096x4096 20.5 us of which 15 are additions, 4096x14336 57 of 52), and the
// producers' VALU and LDS traffic where they do not.
//
// A stage is NP * 64 / R units of a row (UC columns each) for R rows; its
// products sit in LDS as [column / 4][token][row] float4, double-buffered: the
// producers fill stage s while the chains add stage s - 1. The next stage's
// weights and x are in flight across the barrier (lds_barrier).
struct SeqJob {
  const uint8_t *w;
  float *y;
  uint32_t n_out, tiles;
};
struct SeqSet {
  SeqJob j[3];
};

// One unit of a prepared row (layout.cpp): its bytes, and its weights
// four columns at a time: quad i covers columns col(u, i) .. + 3 of the stage.
template <int DT>
struct SeqUnit;

template <>
struct SeqUnit<DT_Q4_K> {
  static constexpr uint32_t UC = 64;
  uint4 a, b, hd;
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t u, uint32_t U) {
    a = ldx16(row + 16 * (size_t)u);
    b = ldx16(row + 16 * (size_t)(U + u));
    hd = ldx16(row + 32 * (size_t)U + 16 * (size_t)(u >> 2));
  }
  struct Scales {
    float d[2], m[2];
  };
  __device__ __forceinline__ Scales scales(uint32_t u) const {
    int sca, scb, ma, mb;
    q4k_scales_i(hd, u & 3, sca, scb, ma, mb);
    const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
    return Scales{{d * (float)sca, d * (float)scb}, {dmin * (float)ma, dmin * (float)mb}};
  }
  __device__ static __forceinline__ uint32_t col(uint32_t u, int i) { return 64 * u + 4 * i; }
  // fma: d1 * q is exact (17 + 4 bits), so it rounds once, as t - m1 does.
  __device__ __forceinline__ void weights(const Scales &s, int i, float *o) const {
    const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const uint32_t v = (i < 8 ? q[i & 7] : q[i & 7] >> 4) & 0x0F0F0F0Fu;
    const float d = s.d[i >> 3], m = s.m[i >> 3];
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = __builtin_fmaf(d, (float)byte_of(v, k), -m);
  }
};

template <>
struct SeqUnit<DT_Q6_K> {
  static constexpr uint32_t UC = 64;
  uint4 a, b, q;
  uint32_t sc, d;
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t u, uint32_t U) {
    a = ldx16(row + 16 * (size_t)u);
    b = ldx16(row + 16 * (size_t)(U + u));
    q = ldx16(row + 16 * (size_t)(2 * U + u));
    sc = *reinterpret_cast<const uint32_t *>(row + 48 * (size_t)U + 4 * (size_t)u);
    d = ldu16(row + 52 * (size_t)U + 2 * (size_t)(u >> 2));
  }
  struct Scales {
    float d[4];
  };
  __device__ __forceinline__ Scales scales(uint32_t) const {
    Scales s;
    const float df = h2f(d);
#pragma unroll
    for (int r = 0; r < 4; r++) s.d[r] = df * (float)(int)(int8_t)byte_of(sc, r);
    return s;
  }
  // Quad i: quarter i / 4, columns 4 (i % 4) of the unit's 16.
  __device__ static __forceinline__ uint32_t col(uint32_t u, int i) {
    return 256 * (u >> 2) + 128 * ((u >> 1) & 1) + 32 * (i >> 2) + 16 * (u & 1) + 4 * (i & 3);
  }
  __device__ __forceinline__ void weights(const Scales &s, int i, float *o) const {
    const uint32_t qa[4] = {a.x, a.y, a.z, a.w}, qb[4] = {b.x, b.y, b.z, b.w}, qh[4] = {q.x, q.y, q.z, q.w};
    const int r = i >> 2, k4 = i & 3;
    const uint32_t low = (r & 1 ? qb[k4] : qa[k4]) >> (r < 2 ? 0 : 4) & 0x0F0F0F0Fu;
    const uint32_t h = r == 0 ? qh[k4] << 4 : r == 1 ? qh[k4] << 2 : r == 2 ? qh[k4] : qh[k4] >> 2;
    const uint32_t v = low | (h & 0x30303030u);
    // (q - 32) first, exact: a zero weight keeps the sign (d * sc) * 0 has.
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = s.d[r] * ((float)byte_of(v, k) - 32.0f);
  }
};

template <>
struct SeqUnit<DT_Q8_0> {
  static constexpr uint32_t UC = 32;
  uint4 a, b;
  uint32_t d;
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t u, uint32_t U) {
    a = ldx16(row + 16 * (size_t)u);
    b = ldx16(row + 16 * (size_t)(U + u));
    d = ldu16(row + 32 * (size_t)U + 2 * (size_t)u);
  }
  struct Scales {
    float d;
  };
  __device__ __forceinline__ Scales scales(uint32_t) const { return Scales{h2f(d)}; }
  __device__ static __forceinline__ uint32_t col(uint32_t u, int i) { return 32 * u + 4 * i; }
  __device__ __forceinline__ void weights(const Scales &s, int i, float *o) const {
    const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const uint32_t v = q[i] ^ 0x80808080u;
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = ((float)byte_of(v, k) - 128.0f) * s.d;
  }
};

template <int DT, int R, int NP, int TT>
__global__ __launch_bounds__(64 * (NP + (R * TT + 63) / 64)) void gemv_seq_pipe_kernel(
    SeqSet js, uint32_t n_in, uint64_t row_bytes, const float *__restrict__ x, uint32_t T) {
#pragma clang fp contract(off)
  // Tokens TT blockIdx.y and up; T: those left.
  x += (size_t)TT * blockIdx.y * n_in;
  const uint32_t t0 = TT * blockIdx.y;
  T -= t0;
  using Unit = SeqUnit<DT>;
  constexpr int UC = Unit::UC, NC = (R * TT + 63) / 64, UPW = 64 / R, UPS = NP * UPW;
  constexpr int SC = UPS * UC;          // columns of a stage
  constexpr int LANES = R * TT;         // chains
  constexpr int X4 = TT * SC / 4;       // float4 of x per stage
  constexpr int XN = (X4 + 64 * NP - 1) / (64 * NP);
  __shared__ __attribute__((aligned(16))) v4f prod[2][SC / 4][LANES];
  __shared__ __attribute__((aligned(16))) v4f xs[2][TT][SC / 4];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t tile = blockIdx.x, ji = 0;
  while (ji < 2 && tile >= js.j[ji].tiles) tile -= js.j[ji].tiles, ji++;
  const uint8_t *w = ji == 0 ? js.j[0].w : ji == 1 ? js.j[1].w : js.j[2].w;
  float *y = ji == 0 ? js.j[0].y : ji == 1 ? js.j[1].y : js.j[2].y;
  const uint32_t n_out = ji == 0 ? js.j[0].n_out : ji == 1 ? js.j[1].n_out : js.j[2].n_out;
  const uint32_t U = n_in / UC, S = (U + UPS - 1) / UPS, n4 = n_in / 4;
  if (wave < NC) {  // chains
    const uint32_t c = min(wave * 64 + lane, (uint32_t)LANES - 1);
    float s = -0.0f;
    lds_barrier();  // the first stage's x
    for (uint32_t st = 0; st < S; st++) {
      lds_barrier();  // stage st's products
      const v4f(*pb)[LANES] = prod[st & 1];
      const uint32_t q4 = min((uint32_t)SC / 4, n4 - st * (SC / 4));  // a multiple of 8
      s = chain_add(s, q4, [&](uint32_t k) { return pb[k][c]; });
    }
    const uint32_t row = tile * R + c % R, t = c / R;
    if (wave * 64 + lane < LANES && row < n_out && t < T) y[(size_t)(t0 + t) * n_out + row] = s;
    return;
  }
  const uint32_t p = wave - NC, ptid = p * 64 + lane, r = lane % R, uu = p * UPW + lane / R;
  const uint8_t *wr = w + (size_t)min(tile * R + r, n_out - 1) * row_bytes;
  auto load_x = [&](uint32_t st, v4f (&o)[XN]) {
#pragma unroll
    for (int i = 0; i < XN; i++) {
      const uint32_t e = ptid + 64 * NP * i, t = min(e / (SC / 4), T - 1), c4 = min(st * (SC / 4) + e % (SC / 4), n4 - 1);
      o[i] = *reinterpret_cast<const v4f *>(x + (size_t)t * n_in + 4 * (size_t)c4);
    }
  };
  auto store_x = [&](uint32_t st, const v4f (&v)[XN]) {
#pragma unroll
    for (int i = 0; i < XN; i++) {
      const uint32_t e = ptid + 64 * NP * i;
      if (X4 % (64 * NP) == 0 || e < X4) xs[st & 1][e / (SC / 4)][e % (SC / 4)] = v[i];
    }
  };
  auto compute = [&](uint32_t st, const Unit &un) {
    const uint32_t u = st * UPS + uu;
    const typename Unit::Scales sc = un.scales(u);
    const v4f(*xb)[SC / 4] = xs[st & 1];
    v4f(*pb)[LANES] = prod[st & 1];
#pragma unroll
    for (int i = 0; i < UC / 4; i++) {
      float wv[4];
      un.weights(sc, i, wv);
      const uint32_t c4 = Unit::col(uu, i) / 4;  // (a stage is whole blocks)
#pragma unroll
      for (int t = 0; t < TT; t++) {
        const v4f xv = xb[t][c4];
        pb[c4][t * R + r] = v4f{wv[0] * xv.x, wv[1] * xv.y, wv[2] * xv.z, wv[3] * xv.w};
      }
    }
  };
  auto unit_at = [&](uint32_t st) { return min(st * UPS + uu, U - 1); };
  // D stages' weights and x in flight: a stage is 0.5 to 2 us of chain, a
  // load from HBM about 1 us. S + 1 barriers in all, as in the chain waves.
  constexpr int D = R == 64 ? 4 : 2;
  Unit u0, u1, u2, u3;
  v4f x0[XN], x1[XN], x2[XN], x3[XN];
  load_x(0, x0);
  u0.load(wr, unit_at(0), U);
  store_x(0, x0);
  load_x(1, x1);
  u1.load(wr, unit_at(1), U);
  if constexpr (D == 4) {
    load_x(2, x2);
    u2.load(wr, unit_at(2), U);
    load_x(3, x3);
    u3.load(wr, unit_at(3), U);
    load_x(4, x0);
  } else {
    load_x(2, x0);
  }
  lds_barrier();
  auto stage = [&](uint32_t st, Unit &un, v4f (&xn)[XN]) {
    if (st >= S) return;
    compute(st, un);
    store_x(st + 1, xn);
    load_x(st + 1 + D, xn);
    un.load(wr, unit_at(st + D), U);
    lds_barrier();
  };
  for (uint32_t st = 0; st < S; st += D) {
    if constexpr (D == 4) {
      stage(st, u0, x1);
      stage(st + 1, u1, x2);
      stage(st + 2, u2, x3);
      stage(st + 3, u3, x0);
    } else {
      stage(st, u0, x1);
      stage(st + 1, u1, x0);
    }
  }
}

// Float weights (F32, F16): the row read element by element, x from global
// memory (uniform addresses).
template <int DT, int TT>
__global__ __launch_bounds__(64) void gemv_seq_float_kernel(const uint8_t *__restrict__ w, uint32_t n_out,
                                                            uint32_t n_in, const float *__restrict__ x, uint32_t T,
                                                            float *__restrict__ y) {
#pragma clang fp contract(off)
  const uint32_t lane = threadIdx.x, row = blockIdx.x * 64 + lane, t0 = blockIdx.y * TT;
  const size_t r = min(row, n_out - 1);
  float s[TT];
  const float *xr[TT];
#pragma unroll
  for (int k = 0; k < TT; k++) s[k] = -0.0f, xr[k] = x + (size_t)min(t0 + k, T - 1) * n_in;
  for (uint32_t i = 0; i < n_in; i++) {
    const float wv = DT == DT_F32 ? reinterpret_cast<const float *>(w)[r * n_in + i]
                                  : h2f(reinterpret_cast<const uint16_t *>(w)[r * n_in + i]);
#pragma unroll
    for (int k = 0; k < TT; k++) {
      const float p = wv * xr[k][i];
      s[k] = s[k] + p;
    }
  }
  if (row < n_out) {
#pragma unroll
    for (int k = 0; k < TT; k++)
      if (t0 + k < T) y[(size_t)(t0 + k) * n_out + row] = s[k];
  }
}

// rmsnorm (cpu.rs:388-402) of one row per workgroup, optionally after the
// residual add (Backend::add_rmsnorm default, src/backend.rs:502-513: sum =
// a + b, then rmsnorm of the sum): the rounded squares go to LDS in parallel
// and wave 0 adds them in order (dot(row, row), from -0.0), then every lane
// forms its outputs (row[i] * scale) * w[i] with scale = 1 / sqrt(mean + eps).
__global__ __launch_bounds__(1024) void rmsnorm_seq_kernel(const float *__restrict__ w, uint32_t dim,
                                                          const float *__restrict__ a, const float *__restrict__ b,
                                                          float *__restrict__ sum, float *__restrict__ y, float eps) {
#pragma clang fp contract(off)
  constexpr uint32_t CHUNK = 8192;  // squares in LDS at a time
  __shared__ __attribute__((aligned(16))) float sq[CHUNK];
  __shared__ float scale_sh;
  const size_t base = (size_t)blockIdx.x * dim;
  const float *ar = a + base, *br = b ? b + base : nullptr;
  float ss = -0.0f;
  for (uint32_t c0 = 0; c0 < dim; c0 += CHUNK) {
    const uint32_t n = min(CHUNK, dim - c0);
    if (c0) __syncthreads();  // the previous chunk is added
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < n; i += 1024) {
      const float v = br ? ar[c0 + i] + br[c0 + i] : ar[c0 + i];
      sq[i] = v * v;
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // the chain, the same in every lane of wave 0
      uint32_t i = n / 32 * 32;
      if (i) ss = chain_add(ss, i / 4, [&](uint32_t k) { return reinterpret_cast<const v4f *>(sq)[k]; });
      for (; i < n; i++) ss = ss + sq[i];
    }
  }
  if (threadIdx.x == 0) {
    const float mean = div_rn(ss, (float)dim);
    scale_sh = div_rn(1.0f, sqrt_rn(mean + eps));
  }
  __syncthreads();
  const float scale = scale_sh;
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < dim; i += 1024) {
    const float v = br ? ar[i] + br[i] : ar[i];
    if (sum) sum[base + i] = v;
    const float t = v * scale;
    y[base + i] = t * w[i];
  }
}

// silu_mul (cpu.rs:447-458): y = (g / (1 + exp(-g))) * u.
__global__ void silu_mul_seq_kernel(const float *__restrict__ g, const float *__restrict__ u, float *__restrict__ y,
                                    size_t n) {
#pragma clang fp contract(off)
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float gv = g[i];
    const float den = 1.0f + libm_expf(-gv);
    const float s = div_rn(gv, den);
    y[i] = s * u[i];
  }
}

// Attention (cpu.rs:437-445,530-590 with softmax_inplace :50-60) of one
// (query, query head) per workgroup over the f16 cache (its values widen to
// f32 exactly): scores[t] = dot(q, k_t) * scale (sequential over head_dim,
// from -0.0); mx = max over the scores from -inf (a maximum in any order);
// e_t = expf(s_t - mx); their sum from +0.0 in key order (one lane); p_t =
// e_t / sum; o[d] = the sequential sum from +0.0 of p_t * v_t[d] in key
// order (one lane per dim). The scores live in `sc`, a slice of kv_cap
// floats per (query, head). pos_dev (a captured decode step): one query per
// sequence at position *pos_dev, which sees keys [0, *pos_dev].
__global__ __launch_bounds__(256) void attn_seq_kernel(const float *__restrict__ q, const uint16_t *__restrict__ K,
                                                       const uint16_t *__restrict__ V, float *__restrict__ o,
                                                       float *__restrict__ sc, uint32_t kv_cap, uint32_t prefix,
                                                       uint32_t hd, uint32_t n_q_heads, uint32_t n_kv_heads,
                                                       float scale, uint64_t seq_stride,
                                                       const uint32_t *__restrict__ pos_dev) {
#pragma clang fp contract(off)
  __shared__ float qs[256];
  __shared__ float red[4];
  __shared__ float sum_sh;
  const uint32_t qh = blockIdx.x, i = blockIdx.y, tid = threadIdx.x;
  if (pos_dev) prefix = *pos_dev;
  const uint32_t kvh = qh / (n_q_heads / n_kv_heads), kv_row = n_kv_heads * hd;
  const uint32_t visible = seq_stride ? prefix + 1 : prefix + i + 1;
  K += (size_t)i * seq_stride + (size_t)kvh * hd;
  V += (size_t)i * seq_stride + (size_t)kvh * hd;
  float *s = sc + ((size_t)i * n_q_heads + qh) * kv_cap;
  const float *qv = q + ((size_t)i * n_q_heads + qh) * hd;
  for (uint32_t d = tid; d < hd; d += 256) qs[d] = qv[d];
  __syncthreads();
  float mx = -INFINITY;
  for (uint32_t t = tid; t < visible; t += 256) {
    const uint16_t *kr = K + (size_t)t * kv_row;
    float acc = -0.0f;
    for (uint32_t d = 0; d < hd; d++) {
      const float p = qs[d] * h2f(kr[d]);
      acc = acc + p;
    }
    const float v = acc * scale;
    s[t] = v;
    mx = fmaxf(mx, v);
  }
  // The maximum over the block (fmaxf is exact and ignores NaN in any order).
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  for (uint32_t t = tid; t < visible; t += 256) s[t] = libm_expf(s[t] - mx);
  __syncthreads();
  if (tid == 0) {
    float total = 0.0f;
    for (uint32_t t = 0; t < visible; t++) total = total + s[t];
    sum_sh = total;
  }
  __syncthreads();
  const float total = sum_sh;
  for (uint32_t t = tid; t < visible; t += 256) s[t] = div_rn(s[t], total);
  __syncthreads();
  for (uint32_t d = tid; d < hd; d += 256) {
    float acc = 0.0f;
    for (uint32_t t = 0; t < visible; t++) {
      const float p = s[t] * h2f(V[(size_t)t * kv_row + d]);
      acc = acc + p;
    }
    o[((size_t)i * n_q_heads + qh) * hd + d] = acc;
  }
}

}  // namespace

namespace {
// One token: rows past this take 64-row workgroups (a chain wave's lanes all
// used), fewer take 16-row ones, which spread over every CU. The fused
// 28672-row gate/up 45.9 us in 64-row workgroups; 4096 rows of 4096 columns
// 20.5 us in 16-row ones (64-row ones would use 64 of the 256 CUs).
constexpr uint64_t SEQ_WIDE_ROWS = 16384;
// Tiles of 16 rows and 4 tokens up to which the split kernel is the faster
// one, per job: past them the launch is bound by its products' VALU work
// (0.145, 0.159, 0.088 us a tile of 4096 columns for Q4_K, Q6_K, Q8_0, and a
// part that does not fall with the columns), which the 8-token kernel, whose
// time is its chain's, spends less of per token; several jobs are as many of its
// launches. us, split / 8-token kernel, 4096 columns: Q6_K 4096 rows T = 40
// (2560 tiles) 408 / 421, 44 (2816) 447 / 421; Q4_K 28672 rows T = 4 (1792) 260 /
// 275, 4096 rows T = 36 (2304) 330 / 272; Q8_0 4096 rows T = 40 223 / 251, 56
// (3584) 307 / 265; Q4_K 512 rows of 2048, T = 200 (1600) 137 / 133; Q8_0 768
// rows of 288, T = 200 (2400) 29.3 / 24.6, 288 rows (900) 15.2 / 22.2.
uint64_t seq_pipe_tiles(int32_t dt, uint64_t n_in) {
  const uint64_t top = dt == DT_Q4_K ? 2170 : dt == DT_Q6_K ? 2700 : 2850, fill = dt == DT_Q4_K ? 850 : 200;
  return top * n_in / (n_in + fill);
}

template <int DT, int R, int NP, int TT>
void seq_pipe(mdma_ctx *ctx, const GemvJob *jobs, int n, uint64_t row_bytes, const float *x, uint64_t T) {
  SeqSet js{};
  uint64_t tiles = 0;
  for (int i = 0; i < 3; i++) {
    js.j[i] = i < n ? SeqJob{jobs[i].w, jobs[i].y, (uint32_t)jobs[i].n_out, (uint32_t)((jobs[i].n_out + R - 1) / R)}
                    : SeqJob{nullptr, nullptr, 0, 0};
    tiles += js.j[i].tiles;
  }
  const dim3 grid((uint32_t)tiles, (uint32_t)((T + TT - 1) / TT));
  gemv_seq_pipe_kernel<DT, R, NP, TT><<<grid, dim3(64 * (NP + (R * TT + 63) / 64)), 0, ctx->stream>>>(
      js, (uint32_t)jobs[0].n_in, row_bytes, x, (uint32_t)T);
  hip_check(hipGetLastError(), "gemv_seq_pipe launch");
}
template <int DT>
void seq_pipe_t(mdma_ctx *ctx, const GemvJob *jobs, int n, uint64_t row_bytes, const float *x, uint64_t T) {
  uint64_t rows = 0;
  for (int i = 0; i < n; i++) rows += jobs[i].n_out;
  if (T == 1 && rows > SEQ_WIDE_ROWS)
    // (Two producers need a stage of half a block, which Q6_K's interleaved
    // columns do not have.)
    seq_pipe<DT, 64, DT == DT_Q4_K ? 2 : 4, 1>(ctx, jobs, n, row_bytes, x, T);
  else if (T == 1)
    seq_pipe<DT, 16, 2, 1>(ctx, jobs, n, row_bytes, x, T);
  else if (T == 2)
    seq_pipe<DT, 16, 1, 2>(ctx, jobs, n, row_bytes, x, T);
  else
    seq_pipe<DT, 16, 1, 4>(ctx, jobs, n, row_bytes, x, T);
}
}  // namespace

void launch_gemv_seq(mdma_ctx *ctx, const GemvJob *jobs, int n, const float *x, uint64_t T) {
  const GemvJob &j = jobs[0];
  bool one = T > 0 && n <= 3 && j.layout == MDMA_LAYOUT_GFX950 && j.n_in % block_size(j.dtype) == 0 &&
             j.n_in > 0 && j.n_in <= 0xffffffffull;
  uint64_t tiles = 0;
  for (int i = 0; i < n; i++) {
    one = one && jobs[i].layout == j.layout && jobs[i].dtype == j.dtype && jobs[i].n_in == j.n_in && jobs[i].n_out > 0;
    tiles += (jobs[i].n_out + 15) / 16;
  }
  // (One token has no such limit; two take half a tile's products.)
  if (!one || tiles > 0x7ffffffull ||
      (T > 1 && (T == 2 ? tiles / 2 : (T + 3) / 4 * tiles) > n * seq_pipe_tiles(j.dtype, j.n_in))) {
    for (int i = 0; i < n; i++) launch_gemv_seq(ctx, jobs[i], x, T);
    return;
  }
  const uint64_t rb = gfx950_row_bytes(j.dtype, j.n_in);
  if (j.dtype == DT_Q4_K) seq_pipe_t<DT_Q4_K>(ctx, jobs, n, rb, x, T);
  else if (j.dtype == DT_Q6_K) seq_pipe_t<DT_Q6_K>(ctx, jobs, n, rb, x, T);
  else seq_pipe_t<DT_Q8_0>(ctx, jobs, n, rb, x, T);
}

void launch_gemv_seq(mdma_ctx *ctx, const GemvJob &j, const float *x, uint64_t T) {
  if (!T || !j.n_out) return;
  if (j.n_out > 0xffffffffull || j.n_in > 0xffffffffull || T > 0xffffffffull)
    shape_fail("qmatmul (cpu order): dimensions past 32 bits");
  const bool prepared = j.layout == MDMA_LAYOUT_GFX950;
  const uint64_t row_bytes = prepared ? gfx950_row_bytes(j.dtype, j.n_in)
                                      : j.n_in / block_size(j.dtype) * type_size(j.dtype);
  const uint32_t gx = (uint32_t)((j.n_out + 63) / 64);
  const uint32_t n_out = (uint32_t)j.n_out, n_in = (uint32_t)j.n_in, t = (uint32_t)T;
#define MDMA_SEQ_GO(KERNEL, TT, ...)                                                                          \
  KERNEL<<<dim3(gx, (uint32_t)((T + TT - 1) / TT)), dim3(64), 0, ctx->stream>>>(__VA_ARGS__)
#define MDMA_SEQ_Q(DT)                                                                                     \
  do {                                                                                                     \
    if ((DT == DT_Q8_0 ? j.n_in % 32 : j.n_in % 256) || (j.n_in % 4))                                     \
      shape_fail("qmatmul (cpu order): rows must be whole blocks");                                        \
    if (T == 1) MDMA_SEQ_GO((gemv_seq_kernel<DT, 1>), 1, j.w, row_bytes, n_out, n_in, prepared, x, t, j.y); \
    else MDMA_SEQ_GO((gemv_seq_kernel<DT, SEQ_TT>), SEQ_TT, j.w, row_bytes, n_out, n_in, prepared, x, t, j.y); \
  } while (0)
  switch (j.dtype) {
    case DT_Q4_K: MDMA_SEQ_Q(DT_Q4_K); break;
    case DT_Q6_K: MDMA_SEQ_Q(DT_Q6_K); break;
    case DT_Q8_0: MDMA_SEQ_Q(DT_Q8_0); break;
    case DT_F32:
      if (T == 1) MDMA_SEQ_GO((gemv_seq_float_kernel<DT_F32, 1>), 1, j.w, n_out, n_in, x, t, j.y);
      else MDMA_SEQ_GO((gemv_seq_float_kernel<DT_F32, SEQ_TT>), SEQ_TT, j.w, n_out, n_in, x, t, j.y);
      break;
    case DT_F16:
      if (T == 1) MDMA_SEQ_GO((gemv_seq_float_kernel<DT_F16, 1>), 1, j.w, n_out, n_in, x, t, j.y);
      else MDMA_SEQ_GO((gemv_seq_float_kernel<DT_F16, SEQ_TT>), SEQ_TT, j.w, n_out, n_in, x, t, j.y);
      break;
    default: fail(MDMA_ERR_NOT_IMPLEMENTED, "qmatmul (cpu order): unsupported weight dtype");
  }
#undef MDMA_SEQ_Q
#undef MDMA_SEQ_GO
  hip_check(hipGetLastError(), "gemv_seq launch");
}

void launch_rmsnorm_seq(mdma_ctx *ctx, const float *w, uint64_t dim, const float *a, const float *b, float *sum,
                        float *y, uint64_t rows, float eps) {
  if (!rows) return;
  rmsnorm_seq_kernel<<<dim3((uint32_t)rows), dim3(1024), 0, ctx->stream>>>(w, (uint32_t)dim, a, b, sum, y, eps);
  hip_check(hipGetLastError(), "rmsnorm_seq launch");
}

void launch_silu_mul_seq(mdma_ctx *ctx, const float *g, const float *u, float *y, uint64_t n) {
  if (!n) return;
  const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 65536);
  silu_mul_seq_kernel<<<dim3((uint32_t)blocks), dim3(256), 0, ctx->stream>>>(g, u, y, n);
  hip_check(hipGetLastError(), "silu_mul_seq launch");
}

void launch_attn_seq(mdma_ctx *ctx, const float *q, const uint16_t *k, const uint16_t *v, float *o, uint64_t n_q,
                     uint64_t kv_len, uint64_t hd, uint64_t n_q_heads, uint64_t n_kv_heads, uint64_t seq_stride,
                     const uint32_t *pos_dev) {
  if (!n_q) return;
  if (hd > 256 || n_q > 65535 || n_q_heads > 0xffffffffull || kv_len > 0xffffffffull)
    shape_fail("attn (cpu order): head_dim past 256 or too many queries");
  float *sc = reinterpret_cast<float *>(scratch(ctx, n_q * n_q_heads * kv_len * 4));
  const float scale = 1.0f / sqrtf((float)hd);
  const uint32_t prefix = (uint32_t)(seq_stride ? kv_len - 1 : kv_len - n_q);
  attn_seq_kernel<<<dim3((uint32_t)n_q_heads, (uint32_t)n_q), dim3(256), 0, ctx->stream>>>(
      q, k, v, o, sc, (uint32_t)kv_len, prefix, (uint32_t)hd, (uint32_t)n_q_heads, (uint32_t)n_kv_heads, scale,
      seq_stride, pos_dev);
  hip_check(hipGetLastError(), "attn_seq launch");
}

}  // namespace mdma
