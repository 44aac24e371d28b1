// f32-activation GEMM of several tokens on the f64 matrix cores, over the
// prepared Q4_K / Q6_K / Q8_0 layouts (layout.cpp).
//
// y[t, r] = sum_i deq(W)[r, i] * x[t, i], the reference's Backend::qmatmul
// (/root/reference/src/backend.rs:469) with the f32 mode's arithmetic: every
// weight a double formed from its quant byte (byte_f64 and one FMA), every
// product exact in the double it is added in, one f32 rounding at the end.
//
// What bounds it is v_mfma_f64_16x16x4 itself: 64 cycles for 2048
// operations, 70 TFLOP/s on the whole chip (measured); the row teams it
// replaces did the same sums in 8-token launches on the VALU, 6.5 TFLOP/s
// (300 tokens: gate/up 2x14336x4096 Q4_K 9.88 -> 1.25 ms, 4096x14336 Q6_K
// 5.13 -> 0.66 ms, 53 to 56 TFLOP/s of the operations asked for).
// So the design keeps the rest out of the matrix core's way:
//  - Weights go from HBM to registers to operands, no LDS: lane l supplies
//    row l % 16 of a 16-row tile for the k group g = l / 16, and since a sum
//    over k may be taken in any order, group g simply walks the 64 columns
//    of unit g of the 256-column block: 16-byte plane loads, and per weight
//    one v_perm_b32 and one f64 FMA, issued under the MFMAs.
//  - x goes to LDS by DMA as f32, one token row of 256 columns per wave
//    instruction, double-buffered by block, and is read 4 columns at a time
//    and converted as it is read.
//  - A block takes a wave 3.5 us per 16-token tile, so one wave per SIMD
//    hides every load of the next block behind the current one.
//  - The (tile, block) pairs of the whole launch are dealt out evenly in one
//    contiguous run per workgroup, so every CU stays busy to the end whatever
//    the rows and tokens; a tile cut by a run's end is left as f64 partials
//    that a second kernel adds in run order (fixed order: the same bits every
//    time). A tile is 64 us to 1 ms of work, its partials 64 KB.
#include <algorithm>

#include "kernels.h"

namespace mdma {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr uint32_t BK = 256;           // columns of a block
constexpr uint32_t XP = BK + 4;        // LDS pitch of a token's block (floats): 16 tokens on distinct banks
constexpr int RW = 2;                  // 16-row tiles per wave
constexpr uint32_t TR = 4 * RW * 16;   // rows of a workgroup's tile (gated: half gate, half up)
constexpr uint64_t F64_LOOP_TOKENS = 128;  // most tokens taken 8 at a time where there is no space for partials

struct F64Args {
  const uint8_t *w[3];
  float *y[3];
  uint32_t n_out[3];
  uint32_t tiles[3];  // row tiles of each job
  const float *x;
  uint64_t row_bytes;
  uint32_t n_in, T, nb, nt;  // nb: blocks of a row; nt: token tiles
  uint32_t per_q, per_r;     // run of workgroup w: [w per_q + min(w, per_r), ...)
  uint32_t units;            // tiles * nb
  double *part;              // [workgroup][2][RW * TW * 4][256], or null: runs are whole tiles
};

// A lane's 64 columns of a 256-column block: raw bytes, their quads (4
// columns each) and the coefficients of w = c1 (2 + byte / 2048) + c0.
template <int DT>
struct Unit64;

template <>
struct Unit64<DT_Q4_K> {
  uint4 a, b, hd;
  double c1[2], c0[2];
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t b0, uint32_t g, uint32_t n_in) {
    const uint32_t U = n_in / 64, u = 4 * b0 + g;
    a = ld16(row + 16 * (size_t)u);
    b = ld16(row + 16 * (size_t)(U + u));
    hd = ldx16(row + 32 * (size_t)U + 16 * (size_t)b0);
  }
  __device__ __forceinline__ void coef(uint32_t, uint32_t g, uint32_t) {
    int s[2], m[2];
    q4k_scales_i(hd, g, s[0], s[1], m[0], m[1]);
    const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const double ds = (double)(d * (float)s[i]), dm = (double)(dmin * (float)m[i]);
      c1[i] = 2048.0 * ds;
      c0[i] = -fma(4096.0, ds, dm);
    }
  }
  __device__ static __forceinline__ int part(int i) { return i >> 3; }
  __device__ static __forceinline__ uint32_t col(uint32_t g, int i) { return 64 * g + 4 * i; }
  __device__ __forceinline__ uint32_t quad(int i) const {
    const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    return (i < 8 ? q[i & 7] : q[i & 7] >> 4) & 0x0F0F0F0Fu;
  }
};

template <>
struct Unit64<DT_Q6_K> {
  uint4 a, b, q;
  uint32_t sc, d;
  double c1[4], c0[4];
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t b0, uint32_t g, uint32_t n_in) {
    const uint32_t U = n_in / 64, u = 4 * b0 + g;
    a = ld16(row + 16 * (size_t)u);
    b = ld16(row + 16 * (size_t)(U + u));
    q = ld16(row + 16 * (size_t)(2 * U + u));
    sc = *reinterpret_cast<const uint32_t *>(row + 48 * (size_t)U + 4 * (size_t)u);
    d = ldu16(row + 52 * (size_t)U + 2 * (size_t)b0);
  }
  __device__ __forceinline__ void coef(uint32_t, uint32_t, uint32_t) {
    const double df = (double)h2f(d);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const double ds = df * (double)(int)(int8_t)((sc >> (8 * r)) & 0xff);
      c1[r] = 2048.0 * ds;
      c0[r] = -4128.0 * ds;
    }
  }
  __device__ static __forceinline__ int part(int i) { return i >> 2; }
  __device__ static __forceinline__ uint32_t col(uint32_t g, int i) {
    return 128 * (g >> 1) + 16 * (g & 1) + 32 * (i >> 2) + 4 * (i & 3);
  }
  __device__ __forceinline__ uint32_t quad(int i) const {
    const uint32_t qa[4] = {a.x, a.y, a.z, a.w}, qb[4] = {b.x, b.y, b.z, b.w}, qh[4] = {q.x, q.y, q.z, q.w};
    const int r = i >> 2, k = i & 3;
    const uint32_t low = ((r & 1 ? qb[k] : qa[k]) >> (r < 2 ? 0 : 4)) & 0x0F0F0F0Fu;
    const uint32_t h = r == 0 ? qh[k] << 4 : r == 1 ? qh[k] << 2 : r == 2 ? qh[k] : qh[k] >> 2;
    return low | (h & 0x30303030u);
  }
};

// Q8_0: units (blocks) g and g + 4 of the 8 in a 256-column block; units
// past the row's end count as zero weights, and zero x (zero_tail).
template <>
struct Unit64<DT_Q8_0> {
  uint4 a[2], b[2];
  uint32_t d[2];
  double c1[2], c0[2];
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t b0, uint32_t g, uint32_t n_in) {
    const uint32_t U = n_in / 32;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t u = min(8 * b0 + g + 4 * i, U - 1);
      a[i] = ld16(row + 16 * (size_t)u);
      b[i] = ld16(row + 16 * (size_t)(U + u));
      d[i] = ldu16(row + 32 * (size_t)U + 2 * (size_t)u);
    }
  }
  __device__ __forceinline__ void coef(uint32_t b0, uint32_t g, uint32_t n_in) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const double ds = 8 * b0 + g + 4 * i < n_in / 32 ? (double)h2f(d[i]) : 0.0;
      c1[i] = 2048.0 * ds;
      c0[i] = -4224.0 * ds;
    }
  }
  __device__ static __forceinline__ int part(int i) { return i >> 3; }
  __device__ static __forceinline__ uint32_t col(uint32_t g, int i) { return 32 * g + 128 * (i >> 3) + 4 * (i & 7); }
  __device__ __forceinline__ uint32_t quad(int i) const {
    const int h = i >> 3;
    const uint32_t q[8] = {a[h].x, a[h].y, a[h].z, a[h].w, b[h].x, b[h].y, b[h].z, b[h].w};
    return q[i & 7] ^ 0x80808080u;
  }
};

// A tile's place: its job, first row and first token.
template <int TW>
struct Place {
  const uint8_t *w;
  float *y;
  uint32_t n_out, row0, tok0;
};
template <int TW, bool GLU>
__device__ __forceinline__ Place<TW> place(const F64Args &a, uint32_t tile) {
  uint32_t rt = tile / a.nt;
  const uint32_t tok0 = (tile - rt * a.nt) * (16 * TW);
  const int j = GLU || rt < a.tiles[0] ? 0 : rt < a.tiles[0] + a.tiles[1] ? 1 : 2;
  rt -= j > 0 ? a.tiles[0] : 0;
  rt -= j > 1 ? a.tiles[1] : 0;
  return Place<TW>{j == 0 ? a.w[0] : j == 1 ? a.w[1] : a.w[2], j == 0 ? a.y[0] : j == 1 ? a.y[1] : a.y[2],
                   j == 0 ? a.n_out[0] : j == 1 ? a.n_out[1] : a.n_out[2], rt * (GLU ? TR / 2 : TR), tok0};
}

// The accumulators of v_mfma_f64_16x16x4 with x as A and w as B: element r
// of lane l is token 4 r + l / 16, row l % 16 of the 16x16 tile.
template <int TW, bool GLU>
__device__ __forceinline__ void store_tile(const F64Args &a, const Place<TW> &p, const v4d (&acc)[RW][TW], float *yg,
                                           uint32_t wave, uint32_t lane) {
#pragma unroll
  for (int t = 0; t < TW; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t tok = p.tok0 + 16 * t + 4 * r + lane / 16;
      if (tok >= a.T) continue;
      if (GLU) {
        const uint32_t row = p.row0 + 16 * wave + lane % 16;
        if (row < p.n_out) yg[(size_t)tok * p.n_out + row] = silu_mul1((float)acc[0][t][r], (float)acc[1][t][r]);
      } else {
#pragma unroll
        for (int i = 0; i < RW; i++) {
          const uint32_t row = p.row0 + 16 * (RW * wave + i) + lane % 16;
          if (row < p.n_out) p.y[(size_t)tok * p.n_out + row] = (float)acc[i][t][r];
        }
      }
    }
}

// x past the row's end of its last, partial block (Q8_0 only): zeroes over
// what the DMA read there (the row's last columns again), which a zero weight
// would turn into NaN where it is infinite.
template <int DT, int N>
__device__ __forceinline__ void zero_tail(float (*xb)[XP], uint32_t b, uint32_t n_in, uint32_t lane) {
  if (DT != DT_Q8_0 || (b + 1) * BK <= n_in) return;
  if (b * BK + 4 * lane < n_in) return;
#pragma unroll
  for (int r = 0; r < N; r++) *reinterpret_cast<v4f *>(&xb[r][4 * lane]) = v4f{0, 0, 0, 0};
}

__device__ __forceinline__ uint32_t run_start(const F64Args &a, uint32_t w) { return w * a.per_q + min(w, a.per_r); }

template <int DT, int TW, bool GLU>
__global__ __launch_bounds__(256, TW <= 2 ? 2 : 1) void gemm_f64_kernel(F64Args a, float *yg) {
  __shared__ __attribute__((aligned(16))) float xs[2][16 * TW][XP];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g = lane / 16, l16 = lane % 16;
  // Contiguous runs on one XCD (workgroups go to the 8 XCDs round-robin), so
  // neighbouring tiles share their weights and x in its L2.
  const uint32_t G = gridDim.x, wg = G % 8 ? blockIdx.x : (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  uint32_t u = run_start(a, wg);
  const uint32_t u_end = min(run_start(a, wg + 1), a.units);
  bool first = true;
  while (u < u_end) {
    const uint32_t tile = u / a.nb, b0 = u - tile * a.nb, b1 = min(a.nb, b0 + (u_end - u));
    const Place<TW> p = place<TW, GLU>(a, tile);
    const uint8_t *wr[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) {
      const uint32_t row = GLU ? p.row0 + 16 * wave + l16 : p.row0 + 16 * (RW * wave + i) + l16;
      wr[i] = (GLU && i ? a.w[1] : p.w) + (size_t)min(row, p.n_out - 1) * a.row_bytes;
    }
    // x of a block: one DMA per token row, the wave's rows wave * 4 TW ..
    auto load_x = [&](uint32_t b, uint32_t buf) {
      const uint32_t col = min(b * BK + 4 * lane, a.n_in - 4);
#pragma unroll
      for (int i = 0; i < 4 * TW; i++) {
        const uint32_t r = wave * (4 * TW) + i, tok = min(p.tok0 + r, a.T - 1);
        lds_dma16(a.x + (size_t)tok * a.n_in, 4 * col, &xs[buf][r][0]);
      }
    };
    v4d acc[RW][TW];
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
      for (int t = 0; t < TW; t++) acc[i][t] = v4d{0, 0, 0, 0};
    Unit64<DT> cur[RW], nxt[RW];
    lds_barrier();  // the previous tile's reads of xs are done
    load_x(b0, b0 & 1);
#pragma unroll
    for (int i = 0; i < RW; i++) nxt[i].load(wr[i], b0, g, a.n_in);
    for (uint32_t b = b0; b < b1; b++) {
#pragma unroll
      for (int i = 0; i < RW; i++) {
        cur[i] = nxt[i];
        cur[i].coef(b, g, a.n_in);
      }
      lds_wait_dma();
      zero_tail<DT, 4 * TW>(&xs[b & 1][wave * (4 * TW)], b, a.n_in, lane);
      lds_barrier();  // every wave's x of block b is in LDS; block b - 1's reads are done
      if (b + 1 < b1) {
        load_x(b + 1, (b + 1) & 1);
#pragma unroll
        for (int i = 0; i < RW; i++) nxt[i].load(wr[i], b + 1, g, a.n_in);
      }
      const float(*xb)[XP] = xs[b & 1];
#pragma unroll
      for (int s = 0; s < 16; s++) {
        v4f xv[TW];
#pragma unroll
        for (int t = 0; t < TW; t++)
          xv[t] = *reinterpret_cast<const v4f *>(&xb[16 * t + l16][Unit64<DT>::col(g, s)]);
        uint32_t q[RW];
#pragma unroll
        for (int i = 0; i < RW; i++) q[i] = cur[i].quad(s);
        const int c = Unit64<DT>::part(s);
#define MDMA_F64_STEP(K)                                                                        \
  {                                                                                             \
    double wv[RW];                                                                              \
    _Pragma("unroll") for (int i = 0; i < RW; i++)                                              \
        wv[i] = fma(cur[i].c1[c], byte_f64<K>(q[i]), cur[i].c0[c]);                             \
    _Pragma("unroll") for (int t = 0; t < TW; t++) {                                            \
      const double xd = (double)xv[t][K];                                                       \
      _Pragma("unroll") for (int i = 0; i < RW; i++)                                            \
          acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(xd, wv[i], acc[i][t], 0, 0, 0);      \
    }                                                                                           \
  }
        MDMA_F64_STEP(0)
        MDMA_F64_STEP(1)
        MDMA_F64_STEP(2)
        MDMA_F64_STEP(3)
#undef MDMA_F64_STEP
      }
    }
    if (b0 == 0 && b1 == a.nb) {
      store_tile<TW, GLU>(a, p, acc, yg, wave, lane);
    } else {  // (only with a.part: a run's first or last tile)
      double *o = a.part + (size_t)(2 * wg + (first ? 0 : 1)) * (RW * TW * 4) * 256 + threadIdx.x;
#pragma unroll
      for (int i = 0; i < RW; i++)
#pragma unroll
        for (int t = 0; t < TW; t++)
#pragma unroll
          for (int r = 0; r < 4; r++) o[((i * TW + t) * 4 + r) * 256] = acc[i][t][r];
    }
    first = false;
    u += b1 - b0;
  }
}

// One workgroup per tile: the tiles that two or more runs share, their
// partials added in run order.
template <int TW, bool GLU>
__global__ __launch_bounds__(256) void gemm_f64_merge_kernel(F64Args a, uint32_t G, float *yg) {
  const uint32_t tile = blockIdx.x, ub = tile * a.nb, ue = ub + a.nb;
  // The run holding unit u.
  auto run_of = [&](uint32_t u) {
    const uint32_t big = a.per_r * (a.per_q + 1);
    return u < big ? u / (a.per_q + 1) : a.per_r + (u - big) / a.per_q;
  };
  const uint32_t w0 = run_of(ub), w1 = run_of(ue - 1);
  if (w0 == w1) return;
  const Place<TW> p = place<TW, GLU>(a, tile);
  v4d acc[RW][TW];
  for (uint32_t w = w0; w <= w1; w++) {
    // The run's first piece is its slot 0, a later one (its last) slot 1.
    const double *o = a.part + (size_t)(2 * w + (run_start(a, w) >= ub ? 0 : 1)) * (RW * TW * 4) * 256 + threadIdx.x;
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
      for (int t = 0; t < TW; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const double v = o[((i * TW + t) * 4 + r) * 256];
          acc[i][t][r] = w == w0 ? v : acc[i][t][r] + v;
        }
  }
  store_tile<TW, GLU>(a, p, acc, yg, threadIdx.x >> 6, threadIdx.x & 63);
}

// Workgroups over a.units (tile, block) pairs, and the bytes of their partials.
uint32_t grid_of(mdma_ctx *ctx, int tw, uint32_t units) {
  return std::min(units, (uint32_t)ctx->cu_count * (tw <= 2 ? 2 : 1));
}
uint64_t part_bytes(uint32_t G, int tw) { return (uint64_t)G * 2 * RW * tw * 4 * 256 * 8; }

template <int DT, int TW, bool GLU>
void launch(mdma_ctx *ctx, F64Args &a, uint32_t tiles, float *yg) {
  uint32_t G = grid_of(ctx, TW, a.units);
  if (a.part) {
    a.per_q = a.units / G, a.per_r = a.units % G;
  } else {  // runs of whole tiles
    const uint32_t n = (tiles + G - 1) / G;
    G = (tiles + n - 1) / n;
    a.per_q = n * a.nb, a.per_r = 0;
  }
  const TimeEvents ev(ctx);
  launch_timed(gemm_f64_kernel<DT, TW, GLU>, dim3(G), dim3(256), ctx->stream, ev.start, a.part ? nullptr : ev.stop, a,
               yg);
  hip_check(hipGetLastError(), "gemm_f64 launch");
  if (a.part) {
    launch_timed(gemm_f64_merge_kernel<TW, GLU>, dim3(tiles), dim3(256), ctx->stream, nullptr, ev.stop, a, G, yg);
    hip_check(hipGetLastError(), "gemm_f64 merge launch");
  }
}

template <int DT, bool GLU>
void launch_tw(mdma_ctx *ctx, F64Args &a, int tw, uint32_t tiles, float *yg) {
  switch (tw) {
    case 1: launch<DT, 1, GLU>(ctx, a, tiles, yg); break;
    case 2: launch<DT, 2, GLU>(ctx, a, tiles, yg); break;
    case 3: launch<DT, 3, GLU>(ctx, a, tiles, yg); break;
    default: launch<DT, 4, GLU>(ctx, a, tiles, yg); break;
  }
}

// ---- 2 to 8 tokens ----
// v_mfma_f64_4x4x4 does four 4x4x4 products in 18 cycles (measured, 62
// TFLOP/s): its four blocks take the same 4 tokens and 4 rows each of a
// 16-row tile, so up to 4 tokens cost about a third of the 16-token tile. It
// does not overlap with the VALU (also measured: an MFMA and a v_perm_b32
// take the sum of their times), so the products and the weights' two VALU
// operations bound the kernel together, about 33 cycles per 64 weights and 4
// tokens. us, row teams / here: gate/up 2x14336x4096 Q4_K T = 2: 73 / 38.7,
// 4: 135 / 41, 8: 267 / 62 (the 16-token tile: 83); 4096x14336 Q6_K 40 / 24.4,
// 66 / 26.6, 134 / 41.5. Lane l supplies
// row l % 16 of the tile and token l % 4, both for k group l / 16, as above,
// and holds the sum of token l / 16, row l % 16.
//
// The NW waves of a workgroup take the blocks of a 16-row tile (gated: 16
// rows of gate and the same of up) in turn, so that neighbouring waves read
// neighbouring 64 bytes of a row, and add their sums in wave order through
// LDS. x comes by DMA into the wave's own double buffer: no barrier but the
// one per tile (a second where the sums have one buffer: gated 3 and 4 tokens,
// for which a second workgroup fits the CU's LDS then, gate/up 2x14336x4096 at 4
// tokens 45.7 -> 41.2 us, 2x5632x2048 14.5 -> 12.1). The next block's loads
// are in flight behind the current one's products, across tiles too.
constexpr int f64_waves(int TT) { return TT <= 4 ? 16 : 8; }  // on a CU
template <int DT, int TT, bool GLU, int NW>
__global__ __launch_bounds__(64 * NW, f64_waves(TT) / 4) void gemv_f64_kernel(F64Args a, float *yg) {
  constexpr int R = GLU ? 2 : 1, NT = (TT + 3) / 4, RB = TT <= 4 && !(GLU && TT == 4) ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float xs[NW][2][TT][XP];
  __shared__ __attribute__((aligned(16))) double red[RB][NW][R * NT][64];
  // As many workgroups on a CU as launch_small's grid counts on.
  static_assert((sizeof(xs) + sizeof(red)) * (f64_waves(TT) / NW) <= 160 * 1024, "LDS");
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g = lane / 16, l16 = lane % 16;
  const uint32_t tiles = a.units;
  struct At {
    const uint8_t *w;
    float *y;
    uint32_t n_out, row0;
  };
  auto at = [&](uint32_t rt) {
    const int j = GLU || rt < a.tiles[0] ? 0 : rt < a.tiles[0] + a.tiles[1] ? 1 : 2;
    rt -= j > 0 ? a.tiles[0] : 0;
    rt -= j > 1 ? a.tiles[1] : 0;
    return At{j == 0 ? a.w[0] : j == 1 ? a.w[1] : a.w[2], j == 0 ? a.y[0] : j == 1 ? a.y[1] : a.y[2],
              j == 0 ? a.n_out[0] : j == 1 ? a.n_out[1] : a.n_out[2], 16 * rt};
  };
  Unit64<DT> cur[R], nxt[R];
  auto issue = [&](uint32_t tile, uint32_t b, uint32_t buf) {
    const At p = at(tile);
    const size_t off = (size_t)min(p.row0 + l16, p.n_out - 1) * a.row_bytes;
#pragma unroll
    for (int i = 0; i < R; i++) nxt[i].load((i ? a.w[1] : p.w) + off, b, g, a.n_in);
    const uint32_t col = min(b * BK + 4 * lane, a.n_in - 4);
#pragma unroll
    for (int t = 0; t < TT; t++) lds_dma16(a.x + (size_t)min((uint32_t)t, a.T - 1) * a.n_in, 4 * col, &xs[wave][buf][t][0]);
  };
  uint32_t tile = blockIdx.x, buf = 0, par = 0;
  if (wave < a.nb) issue(tile, wave, 0);
  for (; tile < tiles; tile += gridDim.x) {
    double acc[R][NT];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[i][t] = 0.0;
    for (uint32_t b = wave; b < a.nb; b += NW) {
      lds_wait_dma();
      zero_tail<DT, TT>(xs[wave][buf], b, a.n_in, lane);
#pragma unroll
      for (int i = 0; i < R; i++) {
        cur[i] = nxt[i];
        cur[i].coef(b, g, a.n_in);
      }
      const bool more = b + NW < a.nb;
      const uint32_t tn = more ? tile : tile + gridDim.x;
      if (tn < tiles) issue(tn, more ? b + NW : wave, buf ^ 1);
      const float(*xb)[XP] = xs[wave][buf];
#pragma unroll
      for (int s = 0; s < 16; s++) {
        v4f xv[NT];
#pragma unroll
        for (int t = 0; t < NT; t++)
          xv[t] = *reinterpret_cast<const v4f *>(&xb[TT == 2 ? lane & 1 : 4 * t + (lane & 3)]
                                                   [Unit64<DT>::col(g, s)]);
        uint32_t q[R];
#pragma unroll
        for (int i = 0; i < R; i++) q[i] = cur[i].quad(s);
        const int c = Unit64<DT>::part(s);
#define MDMA_F64_STEP(K)                                                                   \
  {                                                                                        \
    double wv[R];                                                                          \
    _Pragma("unroll") for (int i = 0; i < R; i++)                                          \
        wv[i] = fma(cur[i].c1[c], byte_f64<K>(q[i]), cur[i].c0[c]);                        \
    _Pragma("unroll") for (int t = 0; t < NT; t++) {                                       \
      const double xd = (double)xv[t][K];                                                  \
      _Pragma("unroll") for (int i = 0; i < R; i++)                                        \
          acc[i][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(xd, wv[i], acc[i][t], 0, 0, 0);   \
    }                                                                                      \
  }
        MDMA_F64_STEP(0)
        MDMA_F64_STEP(1)
        MDMA_F64_STEP(2)
        MDMA_F64_STEP(3)
#undef MDMA_F64_STEP
      }
      buf ^= 1;
    }
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int t = 0; t < NT; t++) red[par][wave][i * NT + t][lane] = acc[i][t];
    lds_barrier();
    if (wave < NT) {
      double s[R];
#pragma unroll
      for (int i = 0; i < R; i++) {
        s[i] = red[par][0][i * NT + wave][lane];
#pragma unroll
        for (int w = 1; w < NW; w++) s[i] += red[par][w][i * NT + wave][lane];
      }
      const At p = at(tile);
      const uint32_t tok = 4 * wave + g, row = p.row0 + l16;
      if (tok < a.T && row < p.n_out) {
        if (GLU) yg[(size_t)tok * p.n_out + row] = silu_mul1((float)s[0], (float)s[R - 1]);
        else p.y[(size_t)tok * p.n_out + row] = (float)s[0];
      }
    }
    if (RB == 2) par ^= 1;
    else lds_barrier();
  }
}

template <int DT, int TT, bool GLU, int NW>
void launch_small(mdma_ctx *ctx, F64Args &a, float *yg) {
  const uint32_t G = std::min(a.units, (uint32_t)ctx->cu_count * f64_waves(TT) / NW);
  const TimeEvents ev(ctx);
  launch_timed(gemv_f64_kernel<DT, TT, GLU, NW>, dim3(G), dim3(64 * NW), ctx->stream, ev.start, ev.stop, a, yg);
  hip_check(hipGetLastError(), "gemv_f64 launch");
}
template <int DT, bool GLU>
void launch_small_t(mdma_ctx *ctx, F64Args &a, float *yg) {
  const bool wide = a.nb >= 8;
#define MDMA_F64_T(TT)                                                    \
  if (wide) launch_small<DT, TT, GLU, TT <= 4 ? 8 : 4>(ctx, a, yg);       \
  else launch_small<DT, TT, GLU, 4>(ctx, a, yg)
  if (a.T <= 2) { MDMA_F64_T(2); }
  else if (a.T <= 4) { MDMA_F64_T(4); }
  else { MDMA_F64_T(8); }
#undef MDMA_F64_T
}

}  // namespace

bool launch_gemm_f64(mdma_ctx *ctx, const GemvJob *jobs, int n_jobs, const float *x, uint64_t T, float *glu_y) {
  const GemvJob &j0 = jobs[0];
  const bool glu = glu_y != nullptr;
  if (T < F64_MIN_TOKENS || T > 1u << 20 || n_jobs < 1 || n_jobs > 3 || !j0.n_in || j0.n_in > 1u << 20 ||
      j0.layout != MDMA_LAYOUT_GFX950 || j0.n_in % block_size(j0.dtype))
    return false;
  F64Args a{};
  uint64_t row_tiles = 0;
  for (int i = 0; i < n_jobs; i++) {
    if (jobs[i].layout != j0.layout || jobs[i].dtype != j0.dtype || jobs[i].n_in != j0.n_in || !jobs[i].n_out ||
        jobs[i].n_out > 1u << 24 || (glu && jobs[i].n_out != j0.n_out))
      return false;
    a.w[i] = jobs[i].w;
    a.y[i] = jobs[i].y;
    a.n_out[i] = (uint32_t)jobs[i].n_out;
    a.tiles[i] = (uint32_t)((jobs[i].n_out + (glu ? TR / 2 : TR) - 1) / (glu ? TR / 2 : TR));
    if (!glu || i == 0) row_tiles += a.tiles[i];
  }
  a.nb = (uint32_t)((j0.n_in + BK - 1) / BK);
  a.x = x;
  a.row_bytes = gfx950_row_bytes(j0.dtype, j0.n_in);
  a.n_in = (uint32_t)j0.n_in;
  a.T = (uint32_t)T;
#define MDMA_F64_DT(GO)                            \
  if (j0.dtype == DT_Q4_K) { GO(DT_Q4_K); }        \
  else if (j0.dtype == DT_Q6_K) { GO(DT_Q6_K); }   \
  else { GO(DT_Q8_0); }
  if (T <= 8) {
    a.units = 0;
    for (int i = 0; i < (glu ? 1 : n_jobs); i++) a.units += a.tiles[i] = (a.n_out[i] + 15) / 16;
#define MDMA_F64_GO(DT)                                  \
  if (glu) launch_small_t<DT, true>(ctx, a, glu_y);      \
  else launch_small_t<DT, false>(ctx, a, nullptr)
    MDMA_F64_DT(MDMA_F64_GO)
#undef MDMA_F64_GO
    return true;
  }
  // Token tiles of 16 tw tokens, tw <= 4: as few as cover T, then as narrow
  // as still do (the 16-token tiles past T are the only padding).
  const uint64_t t16 = (T + 15) / 16;
  a.nt = (uint32_t)((t16 + 3) / 4);
  const int tw = (int)((t16 + a.nt - 1) / a.nt);
  if (row_tiles * a.nt * a.nb > 0x7fffffffull) return false;
  const uint32_t tiles = (uint32_t)row_tiles * a.nt, G = grid_of(ctx, tw, a.units = tiles * a.nb);
  if (tiles % G) {
    a.part = static_cast<double *>(split_parts(ctx, part_bytes(G, tw)));
    // No space for partials and tiles for less than half the CUs: 8 tokens at
    // a time, whose kernel needs none. us, 8-token launches / whole tiles:
    // 4096x4096 Q6_K T = 9: 20.3 / 94, 64 (32 tiles): 104 / 288; 4096x14336 T =
    // 16: 82 / 349; gate/up 2x14336x4096 Q4_K (224 tiles) T = 16: 119 / 90. From
    // about 200 tokens the launches add up to a tile's time even over few rows.
    if (!a.part && T <= F64_LOOP_TOKENS && 2 * (uint64_t)tiles < (uint64_t)ctx->cu_count) {
      for (uint64_t t0 = 0; t0 < T; t0 += 8) {
        const uint64_t tn = std::min<uint64_t>(8, T - t0);
        GemvJob js[3];
        for (int i = 0; i < n_jobs; i++) js[i] = jobs[i], js[i].y += js[i].y ? t0 * js[i].n_out : 0;
        if (glu) launch_gemv_f32_gated(ctx, js[0], js[1], x + t0 * j0.n_in, tn, glu_y + t0 * j0.n_out);
        else launch_gemv_f32(ctx, js, n_jobs, x + t0 * j0.n_in, tn);
      }
      return true;
    }
  }
#define MDMA_F64_GO(DT)                                 \
  if (glu) launch_tw<DT, true>(ctx, a, tw, tiles, glu_y); \
  else launch_tw<DT, false>(ctx, a, tw, tiles, nullptr)
  MDMA_F64_DT(MDMA_F64_GO)
#undef MDMA_F64_GO
#undef MDMA_F64_DT
  return true;
}

}  // namespace mdma
