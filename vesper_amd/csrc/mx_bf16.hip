// The BF16-activation MXFP4 expert: y = W2 . (silu(W1 . x) * (W3 . x)) with BF16 activations, FP32
// accumulation, no activation quantization and no clamp (the benchmark's configuration 0), on the same tiled
// expert bytes the decode layer streams (mx_tile_expert).
//
// The reference's expert (ExpertExecutor.execute, src/vesper/expert.py:51-79) quantizes x and the down
// input to E4M3 per 32-block and feeds scaled MFMAs; this profile keeps the activations exact, so the
// products run on the BF16 MFMA (V_MFMA_F32_16X16X32_BF16, FP32 accumulation) with the weights converted
// exactly: each E2M1 value times its block's E8M0 scale has at most two significant bits, so
// V_CVT_SCALEF32_PK_BF16_FP4 gives it exactly in BF16 (the scale operand's exponent field is the E8M0 code;
// checked on gfx950 for every code and value, code 255 giving NaN as the format defines).
//
// MFMA mapping (measured on gfx950): A lane l = row l % 16, K 8 (l / 16) + 0..7; B lane l = column l % 16,
// same K; D lane l register i = row 4 (l / 16) + i, column l % 16. A is 16 weight rows, B is up to 16 tokens (exchanged
// for few tokens: kFewTokens).
// In the tiled layout a lane (m, q) of tile t holds the 32 E2M1 values of row m, K block 4c + q as four
// 32-bit words; MFMA r of chunk c takes word r of every lane, i.e. K = 32 (4c + q) + 8r + 0..7 at lane group
// q, and the activations are read with the same map, so every product pairs the right operands.
//
// Two launches on the caller's stream:
//   gate/up + SwiGLU (I/8 tiles, 8 waves each): workgroup j owns gate/up tile j (8 W1 rows and the same 8
//     W3 rows) over all of K, the waves taking contiguous eighths of the chunks, all tokens in one
//     pass; the eight partial tiles are added through LDS in wave order, and the workgroup finishes its 8 intermediate positions: h = silu(g) * u (* route weight) in FP32 (optionally written out with g
//     and u), and h as two BF16 terms hi + lo for the down product (hi = bf16(h), lo = bf16(h - hi): their
//     sum holds h to about 16 significant bits);
//   down (H/32 row pairs of tiles, 8 waves): W2 rows against hi and lo (two MFMAs per step), the eight waves'
//     sums added in wave order and rounded once to BF16.
// Every sum runs in a fixed order (an MFMA chain per word and wave, words, waves), independent of T and of scheduling, so
// a token's result does not depend on the batch it runs in.
#include <algorithm>
#include <cmath>

#include "mx_device.h"
#include "mx_internal.h"
#include "mx_numerics.h"

namespace {

using mxd::ldg128;
using mxd::ldg128_nt;
using mxd::ldg32_nt;
using mxd::tiled_offsets;
using mxd::TiledOffsets;

constexpr int kMaxTokens = 16;
constexpr int kGuWaves = 8;      // gate/up: waves per tile, each a contiguous eighth of K
constexpr int kMaxHidden = 8192;
constexpr int kMaxInter = 4096;

// Up to kFewTokens tokens the MFMA's operands are exchanged: A is the activations, its row 4 t + r word r's K range of
// token t, so ONE 16-byte load per lane serves the four MFMAs of a chunk, and B is the weights (column n = weight row
// n). MFMA r multiplies word r; of its D (lane (n, g) register i = activation row 4 g + i = token g, word i) register r
// is the product wanted and the other three are dropped. With a column per token the four operand loads a chunk and
// term were 4 KB through the CU's load path beside 1 KB of a tile's weights (8 KB beside 2 in down), whatever the
// number of tokens. Both forms keep one MFMA chain per word and add the four at the end, so a token's result is the
// same in either. The 7168 x 2048 expert, us a call at 1 / 3 / 4 / 5 / 16 tokens: 12.0 / 12.1 / 12.4 / 12.3 / 17.4 with a
// column per token at any count, 9.5 / 9.8 / 9.9 / 12.2 / 17.4 with the exchange (a gate/up ring of 4 chunks; of 8, the
// whole of a wave's K, 10.0 / - / 10.1). What is left is the two launches' ramps and drains: 23.4 MB take 3.4 us at the
// rate of a plain read.
constexpr int kFewTokens = 4;

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
using mxd::v4f;

struct GateUpArgs {
  const uint8_t* blob;
  const uint16_t* x;      // [T][H] BF16
  const float* route_w;   // [T] or null
  float* h;               // [T][I] or null
  float* gu;              // [T][2I] or null
  uint16_t* hs;           // [2][T][I] BF16: hi, then lo
  int H, I, T;
};

struct DownArgs {
  const uint8_t* blob;
  const uint16_t* hs;   // [2][T][I]
  uint16_t* y;          // [T][H]
  int H, I, T;
};

// Word r of a lane's 16-byte block (8 E2M1 values) times 2^(code - 127), as the 8 BF16 values of an MFMA
// operand (exact).
__device__ __forceinline__ v8bf fp4_word_bf16(uint32_t word, uint32_t code) {
  const float scale = __uint_as_float(code << 23);
  const v2bf p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 0);
  const v2bf p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 1);
  const v2bf p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 2);
  const v2bf p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 3);
  return v8bf{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

__device__ __forceinline__ uint32_t word_of(const uint4 v, int r) {
  return r == 0 ? v.x : r == 1 ? v.y : r == 2 ? v.z : v.w;
}

// One 128-wide K chunk of one tile: MFMA r multiplies word r of the lane's 16 weight bytes w (E8M0 code `code`) into
// acc[r]. xv: the activations, kFew one operand for all four words, else one per word and 16 tokens.
template <bool kFew>
__device__ __forceinline__ void tile_chunk_mfma(const uint4& w, uint32_t code, const uint4 (&xv)[kFew ? 1 : 4],
                                                v4f (&acc)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const v8bf m = fp4_word_bf16(word_of(w, r), code);
    if constexpr (kFew) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, xv[0]), m, acc[r], 0, 0, 0);
    else acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(m, __builtin_bit_cast(v8bf, xv[r]), acc[r], 0, 0, 0);
  }
}

// A wave's sums of a tile, the four words' chains added in word order: lane (n, q) holds weight row n of token q in
// element 0 (kFew), or weight rows 4 q + 0..3 of token n.
template <bool kFew>
struct TileSum {
  float v[kFew ? 1 : 4];
};

template <bool kFew>
__device__ __forceinline__ TileSum<kFew> tile_sum(const v4f (&acc)[4]) {
  TileSum<kFew> s;
  if constexpr (kFew) {
    s.v[0] = ((acc[0][0] + acc[1][1]) + acc[2][2]) + acc[3][3];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) s.v[i] = ((acc[0][i] + acc[1][i]) + acc[2][i]) + acc[3][i];
  }
  return s;
}

// Chunks [c0, c1) through a register ring of R: load(k, c) fills slot k, mma(k) multiplies it. kFew: no load is under a
// branch of its own, those past the end repeat the last chunk -- where paths with and without a load meet, the
// compiler waits for every load in flight before the next product. For more tokens, whose operand loads fill the load
// path, the repeated chunks cost more (19.0 us a call against 17.4 at 16 tokens). Reading chunk c0 is safe where the
// range is empty: it is a chunk of the tile.
template <int R, bool kFew, typename Load, typename Mma>
__device__ __forceinline__ void stream_ring(int c0, int c1, Load load, Mma mma) {
  const int n = c1 - c0;
  if constexpr (kFew) {
    const int last = max(n - 1, 0);
#pragma unroll
    for (int k = 0; k < R; ++k) load(k, c0 + min(k, last));
    int i = 0;
    for (; i + R < n; i += R) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        mma(k);
        load(k, c0 + min(i + k + R, last));
        __builtin_amdgcn_sched_barrier(0);   // keeps the refills between the products
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (i + k < n) mma(k);
  } else {
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k < n) load(k, c0 + k);
    for (int i = 0; i < n; i += R) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        if (i + k < n) {
          mma(k);
          if (i + k + R < n) load(k, c0 + i + k + R);
        }
      }
    }
  }
}

// Where a lane's activation operand of word 0 (kFew: its only one) starts in a token's row, and its token.
template <bool kFew>
__device__ __forceinline__ int operand_token(int lane, int T) {
  return min(kFew ? (lane & 15) >> 2 : lane & 15, T - 1);
}
template <bool kFew>
__device__ __forceinline__ int operand_offset(int lane) {
  return 64 * (lane >> 4) + (kFew ? 16 * (lane & 3) : 0);
}

// grid (I/8), 64 kGuWaves threads. Tile j = 4 g + t of row group g: MFMA rows 0-7 are W1 rows 8j + 0..7, rows
// 8-15 the same W3 rows; chunk c of the tile at (g C + c) 4096 + 1024 t, its codes byte t of the chunk's scale
// words. Wave w streams chunks [C w / 8, C (w + 1) / 8) through a register ring.
template <bool kFew>
__global__ __launch_bounds__(64 * kGuWaves) void bf16_gateup_swiglu_kernel(GateUpArgs a) {
  constexpr int kRing = kFew ? 4 : 3, kX = kFew ? 1 : 4;
  __shared__ TileSum<kFew> red[kGuWaves][64];
  __shared__ float tile[16][kMaxTokens + 1];
  const int j = blockIdx.x, g = j >> 2, t = j & 3;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.H, I = a.I;
  const int chunks = H / 128;
  const int c0 = chunks * wave / kGuWaves, c1 = chunks * (wave + 1) / kGuWaves;
  const int q = lane >> 4, tok = operand_token<kFew>(lane, a.T);
  const uint8_t* wp = a.blob + (size_t)g * chunks * 4096 + t * 1024 + 16 * lane;
  const uint8_t* sp = a.blob + tiled_offsets(H, I).gu_s + (size_t)g * chunks * 256 + 4 * lane;
  const uint8_t* xrow = reinterpret_cast<const uint8_t*>(a.x + (size_t)tok * H) + operand_offset<kFew>(lane);
  uint4 w[kRing];
  uint32_t sw[kRing];
  uint4 xv[kRing][kX];
  auto load = [&](int k, int c) {
    w[k] = ldg128_nt(wp + (size_t)c * 4096);
    sw[k] = ldg32_nt(sp + (size_t)c * 256);
#pragma unroll
    for (int r = 0; r < kX; ++r) xv[k][r] = ldg128(xrow + (size_t)c * 256 + 16 * r);
  };
  v4f acc[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = v4f{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](int k) { tile_chunk_mfma<kFew>(w[k], (sw[k] >> (8 * t)) & 0xFF, xv[k], acc); };
  stream_ring<kRing, kFew>(c0, c1, load, mma);
  red[wave][lane] = tile_sum<kFew>(acc);
  __syncthreads();
  if (wave == 0) {
    // the waves' tiles added in wave order
    TileSum<kFew> s = red[0][lane];
    const int n = lane & 15;
#pragma unroll
    for (int i = 0; i < kX; ++i) {
#pragma unroll
      for (int v = 1; v < kGuWaves; ++v) s.v[i] = s.v[i] + red[v][lane].v[i];
      if constexpr (kFew) tile[n][q] = s.v[i];
      else tile[4 * q + i][n] = s.v[i];
    }
  }
  __syncthreads();
  // thread (token, i): intermediate position 8 j + i, gate row i and up row 8 + i of the tile
  if (tid >= 8 * a.T) return;
  const int n = tid >> 3, i = tid & 7, pos = 8 * j + i;
  const float gv = tile[i][n], uv = tile[8 + i][n];
  float h = gv / (1.0f + expf(-gv)) * uv;
  if (a.route_w) h *= a.route_w[n];
  const size_t idx = (size_t)n * I + pos;
  if (a.h) a.h[idx] = h;
  if (a.gu) {
    a.gu[(size_t)n * 2 * I + pos] = gv;
    a.gu[(size_t)n * 2 * I + I + pos] = uv;
  }
  const uint32_t hi = mx::bf16_bits(h);
  const float rest = h - __uint_as_float(hi << 16);
  a.hs[idx] = (uint16_t)hi;
  a.hs[(size_t)a.T * I + idx] = (uint16_t)mx::bf16_bits(rest);
}

// grid (H / 16 / kDownTiles), 64 kDownWaves threads. A workgroup owns kDownTiles consecutive 16-row tiles of one 64-row
// group (tile t's MFMA rows are W2 rows 64b + 16t + 0..15) over all of K; the I/128 chunks are shared out over the waves,
// each wave's in flight together (kDownRing of them), and the waves' sums added in wave order.
// The launch is bound by its memory round trips, not by its bytes (7.8 MB at 7168 x 2048): us a call (both launches, a
// column per token at any count) at 1 / 4 / 16 tokens with 2 tiles x 8 waves 12.5 / 13.4 / 17.4, 4 tiles x 4 waves (two round trips a wave) 12.9-13.7 /
// 13.4-14.2 / 18.4, 1 tile x 8 waves 14.0 / 14.9 / 21.0, 2 x 4 12.8 / 13.6 / 17.5, 2 x 16 12.4 / 13.4 / 18.8.
constexpr int kDownTiles = 2, kDownWaves = 8, kDownRing = 2;

template <bool kFew>
__global__ __launch_bounds__(64 * kDownWaves) void bf16_down_kernel(DownArgs a) {
  constexpr int kX = kFew ? 1 : 4;
  __shared__ TileSum<kFew> red[kDownWaves][kDownTiles][64];
  const int b = blockIdx.x * kDownTiles / 4, t0 = blockIdx.x * kDownTiles % 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.H, I = a.I;
  const int chunks = I / 128;
  const int c0 = chunks * wave / kDownWaves, c1 = chunks * (wave + 1) / kDownWaves;
  const int q = lane >> 4, tok = operand_token<kFew>(lane, a.T);
  const TiledOffsets off = tiled_offsets(H, I);
  const uint8_t* wp = a.blob + off.dn_w + (size_t)b * chunks * 4096 + 1024 * t0 + 16 * lane;
  const uint8_t* sp = a.blob + off.dn_s + (size_t)b * chunks * 256 + 4 * lane;
  const uint8_t* hrow = reinterpret_cast<const uint8_t*>(a.hs + (size_t)tok * I) + operand_offset<kFew>(lane);
  const size_t lo = (size_t)a.T * I * 2;   // bytes from the hi term to the lo term
  uint4 w[kDownRing][kDownTiles], xv[kDownRing][2][kX];
  uint32_t sw[kDownRing];
  auto load = [&](int k, int c) {
#pragma unroll
    for (int t = 0; t < kDownTiles; ++t) w[k][t] = ldg128_nt(wp + (size_t)c * 4096 + 1024 * t);
    sw[k] = ldg32_nt(sp + (size_t)c * 256);
#pragma unroll
    for (int term = 0; term < 2; ++term)
#pragma unroll
      for (int r = 0; r < kX; ++r) xv[k][term][r] = ldg128(hrow + term * lo + (size_t)c * 256 + 16 * r);
  };
  v4f acc[kDownTiles][4];
#pragma unroll
  for (int t = 0; t < kDownTiles; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[t][r] = v4f{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](int k) {
#pragma unroll
    for (int t = 0; t < kDownTiles; ++t)
#pragma unroll
      for (int term = 0; term < 2; ++term)
        tile_chunk_mfma<kFew>(w[k][t], (sw[k] >> (8 * (t0 + t))) & 0xFF, xv[k][term], acc[t]);
  };
  stream_ring<kDownRing, kFew>(c0, c1, load, mma);
#pragma unroll
  for (int t = 0; t < kDownTiles; ++t) red[wave][t][lane] = tile_sum<kFew>(acc[t]);
  __syncthreads();
  const int n = lane & 15;
  if (wave < kDownTiles && (kFew ? q : n) < a.T) {   // wave t finishes tile t
    TileSum<kFew> s = red[0][wave][lane];
#pragma unroll
    for (int i = 0; i < kX; ++i)
#pragma unroll
      for (int v = 1; v < kDownWaves; ++v) s.v[i] = s.v[i] + red[v][wave][lane].v[i];
    uint16_t* y = a.y + (size_t)(kFew ? q : n) * H + 64 * b + 16 * (t0 + wave);
    if constexpr (kFew) {
      y[n] = (uint16_t)mx::bf16_bits(s.v[0]);
    } else {
      uint2 packed;
      packed.x = mx::bf16_bits(s.v[0]) | (mx::bf16_bits(s.v[1]) << 16);
      packed.y = mx::bf16_bits(s.v[2]) | (mx::bf16_bits(s.v[3]) << 16);
      *reinterpret_cast<uint2*>(y + 4 * q) = packed;
    }
  }
}

bool is_aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

}  // namespace

using mxi::as_stream;
using mxi::use;

static uint64_t bf16_scratch_bytes(int32_t I, int32_t T) { return (uint64_t)2 * T * I * sizeof(uint16_t); }

int mx_expert_forward_bf16(mx_ctx* ctx, const void* tiled, int32_t H, int32_t I, const uint16_t* x, int32_t T,
                           const float* route_w, float* h, float* gu, uint16_t* y, void* stream) {
  if (int s = use(ctx)) return s;
  MX_REQUIRE(tiled != nullptr && is_aligned(tiled, 256), "mx_expert_forward_bf16: 256-byte aligned tiled expert required");
  MX_REQUIRE(H > 0 && H % 128 == 0 && H <= kMaxHidden && I > 0 && I % 128 == 0 && I <= kMaxInter,
             "mx_expert_forward_bf16: H and I must be positive multiples of 128, H <= %d and I <= %d", kMaxHidden,
             kMaxInter);
  MX_REQUIRE(T >= 0 && T <= kMaxTokens, "token count %d outside [0, %d]", T, kMaxTokens);
  if (T == 0) return MX_OK;
  MX_REQUIRE(x && y && is_aligned(x, 16) && is_aligned(y, 8), "mx_expert_forward_bf16: x (16-byte) and y (8-byte) required");
  MX_REQUIRE(!h || is_aligned(h, 4), "mx_expert_forward_bf16: h must be 4-byte aligned");
  hipStream_t st = as_stream(stream);
  void* base = nullptr;
  if (int s = mxi::scratch(ctx, bf16_scratch_bytes(I, T), &base)) return s;
  uint16_t* hs = (uint16_t*)base;
  GateUpArgs ga{(const uint8_t*)tiled, x, route_w, h, gu, hs, H, I, T};
  const bool few = T <= kFewTokens;
  hipLaunchKernelGGL(few ? bf16_gateup_swiglu_kernel<true> : bf16_gateup_swiglu_kernel<false>, dim3(I / 8), dim3(64 * kGuWaves), 0, st, ga);
  MX_LAUNCH_CHECK("bf16_gateup_swiglu_kernel");
  DownArgs da{(const uint8_t*)tiled, hs, y, H, I, T};
  hipLaunchKernelGGL(few ? bf16_down_kernel<true> : bf16_down_kernel<false>, dim3(H / 16 / kDownTiles), dim3(64 * kDownWaves), 0, st, da);
  MX_LAUNCH_CHECK("bf16_down_kernel");
  return MX_OK;
}
