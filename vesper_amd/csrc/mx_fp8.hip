// FP8 E4M3 block-scaled projections on gfx950 (NativeProjections.fp8, src/vesper/projections.py:135-154;
// projection_probe.cu:9-51).
//
// Two scale profiles, one kernel body:
//   block 32  (the reference's projection): weight E8M0 per 32 x 32 block [N/32][K/32], activations
//             per-32 E8M0 (the activation32 quantizer). Both scales are powers of two and are fed to the
//             scaled MFMA, which applies them exactly.
//   block 128 (DeepSeek-style FP32 scales): weight FP32 per 128 x 128 block
//             [ceil(N/128)][K/128], activations per-token per-128 FP32. Per 128-wide chunk the MFMA gives
//             the block dot d (unit scales) and the kernel accumulates acc = fma(d, f32(sa * sw), acc):
//             one rounding per output and chunk. (The reference's only FP8 projection has power-of-two
//             block-32 scales, where every order gives the same sums; this profile's order is this
//             build's own.)
//
// Weights are held in a device-native tiled layout (mx_fp8_tile): for each group of 64 rows and each
// 128-wide K chunk, 4 tiles of 16 rows x 2 KB, each stored as two 1 KB halves of 16 bytes per lane in
// MFMA operand order, so every wave load reads 1 KB of contiguous HBM.
#include <algorithm>
#include <cmath>

#include "mx_device.h"
#include "mx_internal.h"
#include "mx_numerics.h"

namespace {

using mxd::ldg128;
using mxd::ldg128_nt;
using mxd::ldg32;
using mxd::ldgf;
using mxd::mfma_fp8_fp8;
using mxd::v4f;
using mxi::fail;

constexpr int kTiles = 4;   // 16-row MFMA tiles per workgroup: 64 weight rows
constexpr int kTok = 16;    // token columns per MFMA
constexpr int kGemvMaxTokens = 32;   // above this the tiled GEMM reuses each weight tile for 128 tokens
struct Fp8Blob {
  size_t scales;   // byte offset of the scale section
  size_t total;    // blob bytes (256-byte multiple)
};

__host__ __device__ inline Fp8Blob fp8_blob(int N, int K, int block) {
  const size_t w = (size_t)N * K;
  const size_t s = block == 32 ? w / 32 : (size_t)((N + 127) / 128) * (size_t)(K / 128) * 4;
  Fp8Blob b;
  b.scales = w;
  b.total = (w + s + 255) & ~(size_t)255;
  return b;
}

// Reference layout -> tiled blob. Weight piece i (16 bytes): lane l = i % 64, half h, tile t, chunk c,
// row group g; row 64g + 16t + l % 16, K 128c + 64h + 16 (l / 16). Block-32 scale word (g, c, l): byte t is
// the E8M0 code of (row block (64g + 16t) / 32, K block 4c + l / 16). Block-128 scales are copied as is.
__global__ void fp8_tile_kernel(const uint8_t* __restrict__ w, const void* __restrict__ sw, uint8_t* __restrict__ blob,
                                int N, int K, int block) {
  const int64_t C = K / 128;
  const int64_t pieces = (int64_t)N * K / 16;
  const int64_t words = block == 32 ? (int64_t)(N / 64) * C * 64 : 0;
  const int64_t fscales = block == 32 ? 0 : (int64_t)((N + 127) / 128) * C;
  const Fp8Blob off = fp8_blob(N, K, block);
  const int64_t total = pieces + words + fscales;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    if (i < pieces) {
      const int l = (int)(i & 63), h = (int)((i >> 6) & 1), t = (int)((i >> 7) & 3);
      const int64_t rest = i >> 9, c = rest % C, g = rest / C;
      const int64_t row = 64 * g + 16 * t + (l & 15);
      const int64_t k0 = 128 * c + 64 * h + 16 * (l >> 4);
      *reinterpret_cast<uint4*>(blob + i * 16) = *reinterpret_cast<const uint4*>(w + row * K + k0);
    } else if (i < pieces + words) {
      const int64_t j = i - pieces;
      const int l = (int)(j & 63);
      const int64_t rest = j >> 6, c = rest % C, g = rest / C;
      const uint8_t* s8 = (const uint8_t*)sw;
      uint32_t word = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) word |= (uint32_t)s8[((64 * g + 16 * t) / 32) * (K / 32) + 4 * c + (l >> 4)] << (8 * t);
      *reinterpret_cast<uint32_t*>(blob + off.scales + j * 4) = word;
    } else {
      const int64_t j = i - pieces - words;
      reinterpret_cast<float*>(blob + off.scales)[j] = ((const float*)sw)[j];
    }
  }
}

// Per-token per-128 FP32-scale quantizer: one wave per 128-wide block, 2 values per lane.
__global__ __launch_bounds__(256) void act_quant128_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ q,
                                                           float* __restrict__ s, int64_t blocks) {
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= blocks) return;
  const uint32_t pair = reinterpret_cast<const uint32_t*>(x + b * 128)[lane];
  const float v0 = mx::bf16_value(pair & 0xFFFFu), v1 = mx::bf16_value(pair >> 16);
  float amax = fmaxf(fabsf(v0), fabsf(v1));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) amax = fmaxf(amax, __shfl_xor(amax, m, 64));
  const float sc = mx::act128_scale(amax);
  const uint32_t c0 = mx::act_quant_value(v0, sc), c1 = mx::act_quant_value(v1, sc);
  reinterpret_cast<uint16_t*>(q + b * 128)[lane] = (uint16_t)(c0 | (c1 << 8));
  if (lane == 0) s[b] = sc;
}

// E4M3 codes of 8 values over their block-128 scale sc: the quotients x / sc by mx::act128_quotient (one
// reciprocal per block, then a multiply and two fused multiply-adds per value instead of an IEEE division;
// the codes equal those of the division on every input), packed by mxd::e4m3x4 (equal to the encoder on
// every input).
__device__ __forceinline__ uint2 act128_codes8(const float (&v)[8], float sc) {
  const float inv = 1.0f / sc;
  uint2 c;
  c.x = mxd::e4m3x4(mx::act128_quotient(v[0], sc, inv), mx::act128_quotient(v[1], sc, inv),
                    mx::act128_quotient(v[2], sc, inv), mx::act128_quotient(v[3], sc, inv));
  c.y = mxd::e4m3x4(mx::act128_quotient(v[4], sc, inv), mx::act128_quotient(v[5], sc, inv),
                    mx::act128_quotient(v[6], sc, inv), mx::act128_quotient(v[7], sc, inv));
  return c;
}

// The same quantizer with 8 values per lane (16-byte loads, 8-byte stores), 16 lanes per block, blocks in
// a grid-stride loop; x 16-byte and q 8-byte aligned.
__global__ __launch_bounds__(256) void act_quant128_v8_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ q,
                                                              float* __restrict__ s, int64_t blocks) {
  const int sub = threadIdx.x & 15;
  for (int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4; b < blocks;
       b += ((int64_t)gridDim.x * blockDim.x) >> 4) {
    const uint4 raw = *reinterpret_cast<const uint4*>(x + b * 128 + 8 * sub);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    float v[8];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = mx::bf16_value(w[i] & 0xFFFFu);
      v[2 * i + 1] = mx::bf16_value(w[i] >> 16);
      amax = fmaxf(amax, fmaxf(fabsf(v[2 * i]), fabsf(v[2 * i + 1])));
    }
    amax = mxd::row16_max(amax);
    const float sc = mx::act128_scale(amax);
    *reinterpret_cast<uint2*>(q + b * 128 + 8 * sub) = act128_codes8(v, sc);
    if (sub == 0) s[b] = sc;
  }
}

// The 8 codes of this lane's values `raw` (one 128-value block per 16 lanes, sub = lane % 16) with the quantizer
// launches' arithmetic, and their scale: block 32 the E8M0 code (the four lanes of a quad hold one), block 128 the
// FP32 bits.
template <int kBlock>
__device__ __forceinline__ uint2 quantize8(const uint4& raw, uint32_t& scale) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
  float v[8];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = mx::bf16_value(w[i] & 0xFFFFu);
    v[2 * i + 1] = mx::bf16_value(w[i] >> 16);
    amax = fmaxf(amax, fmaxf(fabsf(v[2 * i]), fabsf(v[2 * i + 1])));
  }
  if constexpr (kBlock == 32) {
    amax = fmaxf(mxd::quad_max(amax), mx::u2f(mx::kAmaxFloorBits));
    scale = mx::act_scale_code(amax);
    const float r = 1.0f / mx::e8m0_value(scale);   // exact: a power of two
    return make_uint2(mxd::e4m3x4(v[0] * r, v[1] * r, v[2] * r, v[3] * r),
                      mxd::e4m3x4(v[4] * r, v[5] * r, v[6] * r, v[7] * r));
  } else {
    const float sc = mx::act128_scale(mxd::row16_max(amax));
    scale = __float_as_uint(sc);
    return act128_codes8(v, sc);
  }
}

// Quantizer of the decode GEMV's own input: codes in the order in which its waves load them, so that a chunk's
// operand of 16 tokens is two linear 1 KB loads instead of 32 row pieces of 64 bytes, and its scales 64 contiguous
// bytes instead of 16 rows. Token tile tt (16 tokens), chunk c: half h of lane (q, n) -- token 16 tt + n, K 64 h + 16 q
// + 0..15 of the chunk -- at (tt C + c) 2048 + 1024 h + 16 (16 q + n); the scales (block 32: four E8M0 codes, block 128:
// FP32) at (tt C + c) 64 + 4 n. 16 lanes per (token, chunk). kRows: q_rows, s_rows (either nullable) get the codes and
// scales as rows, too, for a caller that asks for them -- the same bytes as the quantizer launches write.
template <int kBlock, bool kRows>
__global__ __launch_bounds__(256) void fp8_quant_ordered_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ q,
                                                                uint8_t* __restrict__ s, uint8_t* __restrict__ q_rows,
                                                                uint8_t* __restrict__ s_rows, int T, int C) {
  const int b = (int)(blockIdx.x * 16 + (threadIdx.x >> 4)), sub = threadIdx.x & 15;
  if (b >= T * C) return;   // whole groups of 16 lanes
  const int t = b / C, c = b - t * C, n = t & 15;
  uint32_t scale;
  const uint2 codes =
      quantize8<kBlock>(ldg128(reinterpret_cast<const uint8_t*>(x + ((size_t)t * C + c) * 128 + 8 * sub)), scale);
  const size_t at = (size_t)(t >> 4) * C + c;
  // values 8 sub .. 8 sub + 7: half sub / 8, lane group (sub / 2) % 4, upper or lower 8 bytes by sub % 2
  *reinterpret_cast<uint2*>(q + at * 2048 + 1024 * (sub >> 3) + 16 * (16 * ((sub >> 1) & 3) + n) + 8 * (sub & 1)) = codes;
  if constexpr (kBlock == 32) {
    if ((sub & 3) == 0) {
      s[at * 64 + 4 * n + (sub >> 2)] = (uint8_t)scale;
      if (kRows && s_rows) s_rows[(size_t)b * 4 + (sub >> 2)] = (uint8_t)scale;
    }
  } else {
    if (sub == 0) {
      *reinterpret_cast<uint32_t*>(s + at * 64 + 4 * n) = scale;
      if (kRows && s_rows) *reinterpret_cast<uint32_t*>(s_rows + (size_t)b * 4) = scale;
    }
  }
  if (kRows && q_rows) *reinterpret_cast<uint2*>(q_rows + (size_t)b * 128 + 8 * sub) = codes;
}

struct Fp8Args {
  const uint8_t* blob;
  int N, K, T;
  const uint8_t* xq;   // [T][K] E4M3
  const void* xs;      // block 32: uint8 [T][K/32]; block 128: float [T][K/128]
  uint16_t* y;         // [T][N] BF16
  float* trace;        // [T][N] FP32 sums, nullable
  float* partial;      // split K: [splits][T][N] FP32 partial sums (written instead of y)
  const uint16_t* x;   // fused GEMV (few tokens): the BF16 input [T][K], quantized in the kernel
  int ordered;         // GEMV: xq and xs as fp8_quant_ordered_kernel writes them, else [T][K] rows
  int64_t x_stride;    // activation elements per token: K, or groups x K when grouped
  int x_group_rows;    // grouped activations (block-32 GEMV, rows): weight rows [g R, (g + 1) R) multiply
                       // activation group g, codes at xq + tok x_stride + g K; 0 = one group
  // gate/up pair (kPair): blob is W1 and blob2 W3, y and y3 (nullable) their BF16 outputs
  const uint8_t* blob2;
  uint16_t* y3;
  uint16_t* din;         // [T][N] BF16: silu(W1 x) * (W3 x) [* route_w], clamped
  float* swiglu_trace;   // [T][N][5], nullable
  const float* route_w;  // [T] or null
  float limit;
};

// Decode GEMV over 16-row MFMA tiles for up to 16 NT tokens. A workgroup of W waves owns M tile sets of TM
// consecutive tiles over all of K: wave w takes set w % M and the (w / M)-th of W / M contiguous K parts, streams its
// chunks (2 KB of weights per tile and chunk, non-temporal loads, each chunk's activation operands loaded once for its
// TM tiles) through a register ring of row_ring chunks, and the K parts' partial tiles are added through LDS in
// K-part order. K is shared between workgroups only where few rows and a long K would leave most of the chip
// idle (RowShape::S): elsewhere no partial sums leave the workgroup and there is no reduce launch.
// Bound by the weight stream and, for several tokens, by the requests that the activations add to it: a chunk's codes
// of 16 tokens as row pieces were 32 requests and their scales 16, beside 16 for a tile's weights, so a wave takes two
// tiles where there are enough and the codes come in load order (fp8_quant_ordered_kernel). 16 tokens, us a call:
// 7168 x 16384 32.4 -> 23.4, 24576 x 1536 14.3 -> 10.7, 2112 x 7168 13.4 -> 9.9 against 64-row groups with K split over
// workgroups, and 44.8 -> 28.1 / 19.3 -> 12.5 / 16.4 -> 12.2 at 32 tokens, whose weights are read once (NT = 2).
// Fused (few tokens): the M waves of a K part first quantize its chunks of the call's tokens (P passes of 4 blocks
// of 128 values each) into the part's LDS rows with the quantizer launches' arithmetic, so the call needs none.
// Pair: the two tiles of a set are the same 16 rows of W1 and W3, and the workgroup finishes with SwiGLU.
constexpr int kFusedMaxTokens = 4;
constexpr int kFusedRow = 144;    // an LDS row: 128 codes + 16 bytes of padding
constexpr int kTileQRows = 16;    // fused: at most 4 passes of 4 blocks per wave

__host__ __device__ constexpr int row_ring(int TM) { return TM == 1 ? 4 : 3; }

template <int TM, int NT>
struct RowChunk {
  uint4 a[TM][2];   // weights: a tile's two 1 KB halves of the chunk, 16 bytes per lane
  uint32_t sw[2];   // block 32: the chunk's weight scale word (byte t = tile t of the row group); pair: W3's, too
  uint4 b[NT][2];   // activation codes (unfused)
  uint32_t sx[NT];  // unfused: block 32 the token's 4 E8M0 codes of the chunk, block 128 its FP32 scale's bits
};

// Where a lane reads its operands; chunk c's are at fixed strides from these.
template <int TM, int NT>
struct RowSource {
  const uint8_t* w[TM];    // tile t's halves of chunk c at + 8192 c and + 8192 c + 1024
  const uint8_t* sw[TM];   // block 32: the scale words at + 256 c (one word serves the tiles of one row group)
  const uint8_t* x[NT];    // the lane's codes: 16 bytes at + x_chunk c and x_half further
  const uint8_t* xs[NT];   // and its token's scales, chunk c's 4 bytes at + xs_chunk c
  int x_chunk, x_half, xs_chunk;
};

template <int kBlock, bool kFused, int TM, int NT, bool kPair>
__device__ __forceinline__ void row_load(RowChunk<TM, NT>& r, const RowSource<TM, NT>& s, int c) {
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    r.a[t][0] = ldg128_nt(s.w[t] + (size_t)c * 8192);
    r.a[t][1] = ldg128_nt(s.w[t] + (size_t)c * 8192 + 1024);
  }
  if constexpr (kBlock == 32) {
    r.sw[0] = ldg32(s.sw[0] + (size_t)c * 256);
    if constexpr (kPair) r.sw[1] = ldg32(s.sw[TM - 1] + (size_t)c * 256);
  }
  if constexpr (!kFused) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const uint8_t* x = s.x[u] + (size_t)c * s.x_chunk;
      r.b[u][0] = ldg128(x);
      r.b[u][1] = ldg128(x + s.x_half);
      r.sx[u] = ldg32(s.xs[u] + (size_t)c * s.xs_chunk);
    }
  }
}

__device__ __forceinline__ float chunk_scale(float swl, int i) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(swl), i));
}

// One chunk into the accumulators. tsel: the first tile's index in its row group (its scale byte); swf: block 128,
// the chunk's weight block scale; keep[u]: all ones where this lane's token of tile u is in use, else zero; row / qs:
// fused, this lane's token's LDS row and scale word.
template <int kBlock, bool kFused, int TM, int NT, bool kPair>
__device__ __forceinline__ void row_mma(const RowChunk<TM, NT>& r, v4f (&acc)[NT][TM], int q,
                                        const uint32_t (&keep)[NT], int tsel, float swf, const uint8_t* row,
                                        const uint32_t* qs) {
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    uint4 b0 = r.b[u][0], b1 = r.b[u][1];
    uint32_t sx = r.sx[u];
    if constexpr (kFused) {
      b0 = *reinterpret_cast<const uint4*>(row + 16 * q);
      b1 = *reinterpret_cast<const uint4*>(row + 64 + 16 * q);
      sx = *qs;
    }
    b0 = make_uint4(b0.x & keep[u], b0.y & keep[u], b0.z & keep[u], b0.w & keep[u]);
    b1 = make_uint4(b1.x & keep[u], b1.y & keep[u], b1.z & keep[u], b1.w & keep[u]);
    if constexpr (kBlock == 32) {
      const int xb = (int)((sx >> (8 * q)) & 0xFF);
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        const int ws = (int)((r.sw[kPair && t ? 1 : 0] >> (8 * (kPair ? tsel : tsel + t))) & 0xFF);
        acc[u][t] = mfma_fp8_fp8(r.a[t][0], r.a[t][1], b0, b1, acc[u][t], ws, xb);
      }
    } else {
      const float s = __uint_as_float(sx) * swf;
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        const v4f d = mfma_fp8_fp8(r.a[t][0], r.a[t][1], b0, b1, v4f{0.f, 0.f, 0.f, 0.f}, 127, 127);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][t][i] = fmaf(d[i], s, acc[u][t][i]);
      }
    }
  }
}

// grid (ceil(tile sets / M), ceil(T / (16 NT)), kSplit: K splits), 64 W threads. kSplit: a workgroup writes its FP32 sums
// to a.partial (fp8_splitk_reduce_kernel adds them in split order). A template argument: with the grid's size read in
// every kernel the launches of a few us each took 0.2 us longer (shared expert of four layers 52.2 -> 53.7 us).
template <int kBlock, bool kFused, int W, int M, int TM, int NT, int P, bool kPair, bool kSplit>
__global__ __launch_bounds__(64 * W) void fp8_row_gemv_kernel(Fp8Args a) {
  static_assert(W % M == 0 && 4 * P * M <= kTileQRows && M * TM * NT <= W && (NT == 1 || !kFused) &&
                    (!kPair || (TM == 2 && NT == 1 && M == 1 && kBlock == 32)),
                "row GEMV shape");
  constexpr int KP = W / M, R = row_ring(TM);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kp = w / M, sets = kPair ? a.N / 16 : a.N / 16 / TM;
  const int set_raw = blockIdx.x * M + w % M, set = min(set_raw, sets - 1);   // a set past the last repeats it
  const int tile = kPair ? set : set * TM;
  const int q = lane >> 4, nn = lane & 15;
  const int tok0 = blockIdx.y * (kTok * NT);
  const int ntok = min(kTok * NT, a.T - tok0);   // the workgroup's tokens; token tile u holds tok0 + 16 u ..
  const int C = a.K / 128, g = tile >> 2;
  const Fp8Blob off = fp8_blob(a.N, a.K, kBlock);
  const float* swrow = reinterpret_cast<const float*>(a.blob + off.scales) + (size_t)(tile >> 3) * C;
  // grouped activations: a set's rows lie in one activation group (x_group_rows % 64 == 0)
  const int xgroup = a.x_group_rows ? (16 * tile) / a.x_group_rows : 0;
  RowSource<TM, NT> src;
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const uint8_t* blob = kPair && t ? a.blob2 : a.blob;
    const int tl = kPair ? tile : tile + t;
    src.w[t] = blob + (size_t)g * C * 8192 + (tl & 3) * 2048 + 16 * lane;
    src.sw[t] = blob + off.scales + (size_t)g * C * 256 + 4 * lane;
  }
  uint32_t keep[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    // idle columns read the last token's bytes
    const int local = min(16 * u + nn, ntok - 1);
    keep[u] = 16 * u + nn < ntok ? 0xFFFFFFFFu : 0u;
    if (a.ordered) {
      const size_t tt = (size_t)((tok0 + local) >> 4) * C;
      src.x[u] = a.xq + tt * 2048 + 16 * (16 * q + (local & 15));
      src.xs[u] = (const uint8_t*)a.xs + tt * 64 + 4 * (local & 15);
    } else {
      const size_t at = (size_t)(tok0 + local) * a.x_stride + (size_t)xgroup * a.K;
      src.x[u] = a.xq + at + 16 * q;
      src.xs[u] = (const uint8_t*)a.xs + at / 32;
    }
  }
  src.x_chunk = a.ordered ? 2048 : 128;
  src.x_half = a.ordered ? 1024 : 64;
  src.xs_chunk = a.ordered ? 64 : 4;
  // the workgroup's chunks: all of K, or its share of them (blockIdx.z of gridDim.z)
  int cb = 0, cw = C;
  if constexpr (kSplit) {
    const int z = blockIdx.z, S = gridDim.z;   // at most 16: C z fits 32 bits
    cb = C * z / S;
    cw = C * (z + 1) / S - cb;
  }
  const int c0 = cb + (cw * kp) / KP, n = (cw * (kp + 1)) / KP - (cw * kp) / KP;
  // fused: K part kp's rows, block b = i ntok + token (chunk c0 + i), 128 codes + 16 bytes of padding each,
  // quantized by the part's M waves together (wave w % M takes blocks 4 P (w % M) + 0 .. 4 P - 1), then one
  // spare row per wave that takes the stores of lanes past the part's blocks (no branch around the math:
  // branches would make the compiler wait for the weight loads before quantizing). qsc: a row's scales, block 32
  // four E8M0 bytes, block 128 one FP32
  constexpr int kPartRows = 4 * P * M;
  __shared__ __attribute__((aligned(16))) uint8_t qx[kFused ? (KP * kPartRows + W) * kFusedRow : 16];
  __shared__ uint32_t qsc[kFused ? KP * kPartRows + W : 1];
  const int sub = lane & 15, grp = lane >> 4;
  const int nb = n * ntok, nl = max(n - 1, 0), b0 = 4 * P * (w % M);
  uint4 xv[kFused ? P : 1];
  if constexpr (kFused) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int b = min(b0 + 4 * p + grp, max(nb - 1, 0));
      xv[p] = ldg128(reinterpret_cast<const uint8_t*>(a.x + (size_t)(tok0 + b % ntok) * a.K +
                                                      (size_t)(c0 + b / ntok) * 128 + 8 * sub));
    }
  }
  // the activation loads first, then the ring, then the quantization: loads return in order, so quantizing
  // waits for the activations alone (scheduling barriers keep the compiler from interleaving the three)
  __builtin_amdgcn_sched_barrier(0);
  // block 128: the wave's weight block scales, lane i holding chunk c0 + sw0 + i's; each chunk's is read out with
  // v_readlane into a scalar register
  int sw0 = 0;
  float swl = 0.f;
  if constexpr (kBlock == 128) swl = ldgf(swrow + c0 + min(lane, nl));
  auto next_scales = [&](int i) {
    sw0 = i;
    swl = ldgf(swrow + c0 + min(sw0 + lane, nl));
    asm volatile("" : "+v"(swl));   // waited for here, not where the paths with and without this load meet
  };
  RowChunk<TM, NT> buf[R];
#pragma unroll
  for (int j = 0; j < R; ++j) row_load<kBlock, kFused, TM, NT, kPair>(buf[j], src, c0 + min(j, nl));
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (kFused) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int b = b0 + 4 * p + grp;
      const int row = b < nb ? kp * kPartRows + b : KP * kPartRows + w;
      uint32_t scale;
      const uint2 codes = quantize8<kBlock>(xv[p], scale);
      if constexpr (kBlock == 32) {
        if ((sub & 3) == 0) reinterpret_cast<uint8_t*>(qsc + row)[sub >> 2] = (uint8_t)scale;
      } else {
        if (sub == 0) qsc[row] = scale;
      }
      *reinterpret_cast<uint2*>(qx + row * kFusedRow + 8 * sub) = codes;
    }
    if constexpr (M == 1) {
      // the rows are this wave's own: its LDS writes complete before its reads (no workgroup barrier)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      mxd::lds_barrier();   // the part's rows come from M waves; LDS only, the weight loads stay in flight
    }
  }
  v4f acc[NT][TM];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[u][t] = v4f{0.f, 0.f, 0.f, 0.f};
  const int qtok = kFused ? min(nn, ntok - 1) : 0;
  const uint8_t* qrow = qx + (kp * kPartRows + qtok) * kFusedRow;
  const uint32_t* qs = qsc + kp * kPartRows + qtok;
  int i = 0;
  for (; i + R < n; i += R) {
    if constexpr (kBlock == 128)
      if (i + R > sw0 + 64) next_scales(i);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      // a ring: chunk i + j is multiplied, then its slot is refilled with chunk i + j + R before the next chunk is
      // waited for (the barrier keeps the compiler from batching the loads after all of them)
      row_mma<kBlock, kFused, TM, NT, kPair>(buf[j], acc, q, keep, tile & 3,
                                             kBlock == 128 ? chunk_scale(swl, i + j - sw0) : 0.f,
                                             qrow + (i + j) * ntok * kFusedRow, qs + (i + j) * ntok);
      row_load<kBlock, kFused, TM, NT, kPair>(buf[j], src, c0 + min(i + j + R, nl));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (kBlock == 128)
    if (i + R > sw0 + 64) next_scales(i);
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (i + j < n)
      row_mma<kBlock, kFused, TM, NT, kPair>(buf[j], acc, q, keep, tile & 3,
                                             kBlock == 128 ? chunk_scale(swl, i + j - sw0) : 0.f,
                                             qrow + (i + j) * ntok * kFusedRow, qs + (i + j) * ntok);
  __shared__ float4 red[W][TM * NT][64];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < TM; ++t)
      red[w][TM * u + t][lane] = make_float4(acc[u][t][0], acc[u][t][1], acc[u][t][2], acc[u][t][3]);
  __syncthreads();
  // wave w < M TM NT finishes tile (w / M) % TM of set w % M for token tile w / (M TM): K-part order, over the parts
  // that own chunks (KP > C leaves some without)
  float4 o4 = make_float4(0.f, 0.f, 0.f, 0.f);
  const int ft = w / M;
  if (w < M * TM * NT) {
    bool first = true;
#pragma unroll
    for (int v = 0; v < KP; ++v) {
      if ((cw * (v + 1)) / KP == (cw * v) / KP) continue;
      const float4 r = red[w % M + M * v][ft][lane];
      if (first) {
        o4 = r;
        first = false;
      } else {
        o4.x = o4.x + r.x;
        o4.y = o4.y + r.y;
        o4.z = o4.z + r.z;
        o4.w = o4.w + r.w;
      }
    }
  }
  if constexpr (kPair) {
    // element (token, row) per thread: gate and up of it from LDS
    __shared__ float pair[2][kTok][16 + 1];
    if (w < 2 && nn < ntok) {
      const float v[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) pair[w][nn][4 * q + e] = v[e];
    }
    __syncthreads();
    for (int p = tid; p < 16 * ntok; p += 64 * W) {
      const int pt = p >> 4, row = p & 15;
      const size_t o = (size_t)(tok0 + pt) * a.N + 16 * tile + row;
      const uint32_t b1 = mx::bf16_bits(pair[0][pt][row]), b3 = mx::bf16_bits(pair[1][pt][row]);
      const float v = mxd::swiglu_element(b1, b3, a.limit, a.route_w != nullptr, a.route_w ? a.route_w[tok0 + pt] : 1.f,
                                          a.swiglu_trace ? a.swiglu_trace + o * 5 : nullptr);
      if (a.y) a.y[o] = (uint16_t)b1;
      if (a.y3) a.y3[o] = (uint16_t)b3;
      a.din[o] = (uint16_t)mx::bf16_bits(v);   // last: a caller may keep it where W1's or W3's output was
    }
    return;
  }
  const int local = 16 * (ft / TM) + nn;
  if (w >= M * TM * NT || local >= ntok || set_raw >= sets) return;
  const size_t o = (size_t)(tok0 + local) * a.N + 16 * (tile + ft % TM) + 4 * q;
  if constexpr (kSplit) {
    *reinterpret_cast<float4*>(a.partial + (size_t)blockIdx.z * a.T * a.N + o) = o4;
    return;
  }
  uint2 packed;
  packed.x = mx::bf16_bits(o4.x) | (mx::bf16_bits(o4.y) << 16);
  packed.y = mx::bf16_bits(o4.z) | (mx::bf16_bits(o4.w) << 16);
  *reinterpret_cast<uint2*>(a.y + o) = packed;
  if (a.trace) *reinterpret_cast<float4*>(a.trace + o) = o4;
}

// Split-K epilogue: y = BF16(sum over splits in order), 4 outputs per thread.
__global__ void fp8_splitk_reduce_kernel(const float* __restrict__ partial, int splits, int64_t count,
                                         uint16_t* __restrict__ y, float* __restrict__ trace) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= count) return;
  float4 s = *reinterpret_cast<const float4*>(partial + i);
  for (int z = 1; z < splits; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(partial + (size_t)z * count + i);
    s.x = s.x + v.x;
    s.y = s.y + v.y;
    s.z = s.z + v.z;
    s.w = s.w + v.w;
  }
  uint2 packed;
  packed.x = mx::bf16_bits(s.x) | (mx::bf16_bits(s.y) << 16);
  packed.y = mx::bf16_bits(s.z) | (mx::bf16_bits(s.w) << 16);
  *reinterpret_cast<uint2*>(y + i) = packed;
  if (trace) *reinterpret_cast<float4*>(trace + i) = s;
}

// ---- GEMM for many tokens ------------------------------------------------------------------------
//
// grid (ceil(N / 256), ceil(T / 128), K splits), 768 threads = 12 waves. Waves 0-7 multiply: wave w owns
// the 64-row group 4 * blockIdx.x + (w % 4) and the token half w / 4 (64 tokens), 4 row tiles x 4 token
// tiles of 16 x 16. Waves 8-11 only copy operands global -> LDS (direct copies, no registers) into a
// 3-stage ring, two chunks ahead. Measured on MI355X: a CU moves at most 64 bytes per clock from L2 into
// LDS, and while a chunk is still on its way from HBM (the first workgroup of an XCD to ask for it, and
// every workgroup asking at the same time) a wave issuing copies stalls for most of their latency. When
// the multiplying waves issue the copies themselves, each 128-wide chunk takes about 2,700 clocks: the
// stalled copies hold up the MFMAs behind them. In waves of their own the stalls hold up no MFMA, since
// each SIMD issues from whichever of its waves is ready; the copy waves then set the pace (about 1,900
// clocks per chunk for the o projection at T = 2048, 1,000 when every chunk is already in L2) against
// about 1,450 for the multiplying waves. Stage layout: the 4 row groups' weight chunks
// (32 KB, piece 8 g + 2 t + h in the tiled blob's MFMA operand order), the 128 tokens' activation codes
// (16 KB, block 2 u + h holding at lane (q, n) bytes 64 h + 16 q .. of token 16 u + n: the B operand of
// token tile u), their scales (512 B) and the 4 row groups' weight-scale words (1 KB, 256 B each). Step
// c: the multiplying waves read chunk c from its stage and multiply; the copy waves issue chunk c + 2 into
// the stage chunk c - 1 left and wait for chunk c + 1; one barrier ends the step. The loops have no
// compiler-visible global loads (the copies are inline assembly), so the compiler adds no vmcnt waits.
constexpr int kGemmTok = 128;                 // tokens per workgroup
constexpr int kWaveTiles = 4;                 // token tiles per multiplying wave
constexpr int kGemmThreads = 768;
constexpr int kGemmA = 32768;
constexpr int kGemmB = 16384;
constexpr int kGemmSA = 512;
constexpr int kGemmSW = 1024;
constexpr int kGemmStage = kGemmA + kGemmB + kGemmSA + kGemmSW;
constexpr int kGemmStages = 3;
constexpr int kGemmCopies = 14;   // per copy wave and chunk: 8 weight, 4 activation, 1 + 1 scale
static_assert(kGemmStages * kGemmStage <= 160 * 1024, "GEMM LDS ring");

template <int kBlock>
__global__ __launch_bounds__(kGemmThreads) void fp8_gemm_kernel(Fp8Args a) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kGemmStages * kGemmStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, n = lane & 15;
  const int chunks = a.K / 128, per = (chunks + gridDim.z - 1) / gridDim.z;
  const int c0 = blockIdx.z * per;
  const int C = min(per, chunks - c0);
  const int groups = a.N / 64;
  const int bx = blockIdx.x;
  const int m0 = blockIdx.y * kGemmTok;
  const Fp8Blob off = fp8_blob(a.N, a.K, kBlock);
  const uint32_t lds0 = mxd::lds_addr(lds);

  if (wave >= 8) {
    // copy wave p: row group p's 8 weight pieces and scale word(s), activation tiles 2p and 2p + 1 (both
    // blocks of each), the scales of tokens 32p .. 32p + 31. Rows past N and tokens past T repeat valid ones.
    const int p = wave - 8;
    const int gp = min(bx * 4 + p, groups - 1);
    const uint8_t* wsrc = a.blob + (size_t)gp * chunks * 8192 + 16 * lane;
    const uint8_t* bsrc0 = a.xq + (size_t)min(m0 + 32 * p + n, a.T - 1) * a.K + 16 * q;
    const uint8_t* bsrc1 = a.xq + (size_t)min(m0 + 32 * p + 16 + n, a.T - 1) * a.K + 16 * q;
    const int stok = min(m0 + 32 * p + (lane & 31), a.T - 1);
    const uint8_t* sasrc = kBlock == 32 ? (const uint8_t*)a.xs + (size_t)stok * (a.K / 32)
                                        : (const uint8_t*)a.xs + (size_t)stok * chunks * 4;
    const uint8_t* swsrc = kBlock == 32 ? a.blob + off.scales + (size_t)gp * chunks * 256 + 4 * lane
                                        : a.blob + off.scales + ((size_t)((64 * gp) / 128) * chunks) * 4;
    auto copy = [&](int cl) {
      const int c = c0 + cl;
      const uint32_t st = lds0 + (uint32_t)(cl % kGemmStages) * kGemmStage;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mxd::global_to_lds16(wsrc + (size_t)c * 8192 + i * 1024, __builtin_amdgcn_readfirstlane(st + (8 * p + i) * 1024));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        mxd::global_to_lds16(bsrc0 + (size_t)c * 128 + 64 * h,
                             __builtin_amdgcn_readfirstlane(st + kGemmA + (4 * p + h) * 1024));
        mxd::global_to_lds16(bsrc1 + (size_t)c * 128 + 64 * h,
                             __builtin_amdgcn_readfirstlane(st + kGemmA + (4 * p + 2 + h) * 1024));
      }
      const uint32_t sa_lds = __builtin_amdgcn_readfirstlane(st + kGemmA + kGemmB + 128 * p);
      if (lane < 32) mxd::global_to_lds4(sasrc + (size_t)c * 4, sa_lds);
      const uint32_t sw_lds = __builtin_amdgcn_readfirstlane(st + kGemmA + kGemmB + kGemmSA + 256 * p);
      if (kBlock == 32 || lane == 0) mxd::global_to_lds4(swsrc + (size_t)c * (kBlock == 32 ? 256 : 4), sw_lds);
    };
    copy(0);
    if (C > 1) {
      copy(1);
      __builtin_amdgcn_s_waitcnt(mxd::vm_wait_imm(kGemmCopies));
    } else {
      __builtin_amdgcn_s_waitcnt(mxd::vm_wait_imm(0));
    }
    mxd::copy_barrier();
    for (int c = 0; c < C; ++c) {
      if (c + 2 < C) {
        copy(c + 2);
        __builtin_amdgcn_s_waitcnt(mxd::vm_wait_imm(kGemmCopies));   // chunk c + 1 has landed
      } else {
        __builtin_amdgcn_s_waitcnt(mxd::vm_wait_imm(0));
      }
      mxd::copy_barrier();
    }
    return;
  }

  const int g_raw = bx * 4 + (wave & 3);
  const bool has_rows = g_raw < groups;
  const int g = has_rows ? g_raw : groups - 1;
  const int u0 = (wave >> 2) * kWaveTiles;
  v4f acc[kTiles][kWaveTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int u = 0; u < kWaveTiles; ++u) acc[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
  mxd::copy_barrier();
  for (int c = 0; c < C; ++c) {
    const uint8_t* st = lds + (c % kGemmStages) * kGemmStage;
    uint4 am[kTiles][2], b[kWaveTiles][2];
    float sx[kWaveTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        am[t][h] = *reinterpret_cast<const uint4*>(st + (8 * (wave & 3) + 2 * t + h) * 1024 + 16 * lane);
#pragma unroll
    for (int u = 0; u < kWaveTiles; ++u) {
      const int tile = u0 + u;
      b[u][0] = *reinterpret_cast<const uint4*>(st + kGemmA + (2 * tile) * 1024 + 16 * lane);
      b[u][1] = *reinterpret_cast<const uint4*>(st + kGemmA + (2 * tile + 1) * 1024 + 16 * lane);
      sx[u] = *reinterpret_cast<const float*>(st + kGemmA + kGemmB + 4 * (16 * tile + n));
    }
    const uint32_t swv = *reinterpret_cast<const uint32_t*>(st + kGemmA + kGemmB + kGemmSA + 256 * (wave & 3) +
                                                            (kBlock == 32 ? 4 * lane : 0));
    if constexpr (kBlock == 32) {
#pragma unroll
      for (int u = 0; u < kWaveTiles; ++u) {
        const int sxb = (int)((__float_as_uint(sx[u]) >> (8 * q)) & 0xFF);
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
          acc[t][u] = mfma_fp8_fp8(am[t][0], am[t][1], b[u][0], b[u][1], acc[t][u], (int)((swv >> (8 * t)) & 0xFF),
                                   sxb);
      }
    } else {
      const float swf = __uint_as_float(swv);
      constexpr int kSteps = kTiles * kWaveTiles;
      v4f d[2];
      d[0] = mfma_fp8_fp8(am[0][0], am[0][1], b[0][0], b[0][1], v4f{0.f, 0.f, 0.f, 0.f}, 127, 127);
#pragma unroll
      for (int k = 0; k < kSteps; ++k) {
        const int t = k % kTiles, u = k / kTiles;
        if (k + 1 < kSteps) {
          const int t1 = (k + 1) % kTiles, u1 = (k + 1) / kTiles;
          d[(k + 1) & 1] = mfma_fp8_fp8(am[t1][0], am[t1][1], b[u1][0], b[u1][1], v4f{0.f, 0.f, 0.f, 0.f}, 127, 127);
        }
        __builtin_amdgcn_sched_barrier(0);
        const float sc = sx[u] * swf;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][u][i] = fmaf(d[k & 1][i], sc, acc[t][u][i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    mxd::copy_barrier();
  }
  if (!has_rows) return;
#pragma unroll
  for (int u = 0; u < kWaveTiles; ++u) {
    const int tok = m0 + 16 * (u0 + u) + n;
    if (tok >= a.T) continue;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const size_t o = (size_t)tok * a.N + 64 * g + 16 * t + 4 * q;
      const float4 v = make_float4(acc[t][u][0], acc[t][u][1], acc[t][u][2], acc[t][u][3]);
      if (gridDim.z > 1) {
        *reinterpret_cast<float4*>(a.partial + (size_t)blockIdx.z * a.T * a.N + o) = v;
        continue;
      }
      uint2 packed;
      packed.x = mx::bf16_bits(v.x) | (mx::bf16_bits(v.y) << 16);
      packed.y = mx::bf16_bits(v.z) | (mx::bf16_bits(v.w) << 16);
      *reinterpret_cast<uint2*>(a.y + o) = packed;
      if (a.trace) *reinterpret_cast<float4*>(a.trace + o) = v;
    }
  }
}

int check_fp8_shape(int N, int K, int block, const char* who) {
  MX_REQUIRE(block == 32 || block == 128, "%s: block must be 32 or 128", who);
  MX_REQUIRE(N > 0 && N % 64 == 0 && K > 0 && K % 128 == 0, "%s: rows must be a multiple of 64 and width of 128",
             who);
  return MX_OK;
}

// K splits of the GEMM: only when the rows and tokens alone give fewer workgroups than half the CUs (the partial
// sums cost a write and a read of splits x T x N floats and a reduce launch), then about 512, every split keeping 8
// chunks. 2112 x 7168 at T = 2048 (144 workgroups) ran 97 us per call unsplit against 110 us with 4 splits (MI355X,
// quantizer included).
int fp8_gemm_splits(int N, int K, int T) {
  const int base_wgs = ((N / 64 + 3) / 4) * ((T + kGemmTok - 1) / kGemmTok);
  if (base_wgs >= 128) return 1;
  return std::max(1, std::min({8, (K / 128) / 8, (512 + base_wgs - 1) / base_wgs}));
}

// Shape of the decode GEMV: W waves a workgroup, M tile sets of TM tiles, K split over S workgroups.
struct RowShape {
  int W, M, TM, S = 1;
  int parts() const { return W / M; }   // K parts of a workgroup
};

// Gate/up of the FP8 expert. The 5120 x 2304 expert (two / three / four launches), us at 1 / 4 / 16 tokens: 13.7 / 17.8 / 20.4
// with 8 waves, 14.7 / 17.8 / 21.2 with 16, 14.1 / 18.2 / 20.0 with 4; 31.6 / 33.0 / 34.7 as six launches (quantizer,
// W1, W3, SwiGLU, quantizer, W2). Two launches of about 6 us for 35 MB: their ramps and drains bound it now.
constexpr RowShape kPairShape{8, 1, 2};

// Whether `parts` K parts of C chunks can quantize T tokens themselves: a part's chunks x tokens fit its LDS rows.
bool fp8_fits(int parts, int C, int T) { return T <= kFusedMaxTokens && (C + parts - 1) / parts * T <= kTileQRows; }

RowShape fp8_row_shape(int N, int K, int T) {
  // us per call (quantizer launch included where there is one), weights rotated, W x M x TM, block 32 unless said.
  // * up to 4 chunks, more than 256 tiles or 16 tokens: no K parts, four tiles a workgroup. A part without a chunk is
  //   launched, and waits, for nothing: 12288 x 128 at 4 / 8 / 32 tokens 7.1 / 6.4 / 6.9 with the shapes below, 3.3 / 5.5 /
  //   6.1 so; 24576 x 512 6.9 / 8.8 / 11.3 and 5.0 / 7.2 / 8.7. Few tiles and tokens are the faster for the parts (512 rows
  //   block 128, 4 tokens 3.2 / 3.5).
  // * up to 256 tiles: one tile a workgroup, 4 K parts; 8 where those quantize the call and 4 cannot, or where they
  //   shorten the chains and the quantization enough. 2112 rows, 4 parts / 8 parts: 1 token of 32 / 40 / 56 / 64 chunks 4.8
  //   / 4.9, 6.0 / 6.2, 6.9 / 6.7, 7.3 / 7.1 (block 128 4.8 / 5.0, 6.1 / 5.8, 6.8 / 6.0, 7.1 / 6.5), 72 10.2 / 7.7; 2 tokens
  //   of 20 / 24 / 32 / 40 5.1 / 5.1, 5.2 / 4.9, 5.5 / 5.2, 7.9 / 6.7, of 72 10.4 / 11.2; 3 of 20 5.1 / 5.8, 4 of 16 4.6 /
  //   4.7, of 20 6.8 / 5.9, of 40 7.9 / 8.8; 16 of 56 9.9 / 10.1.
  // * between: two tiles of 4 K parts where those quantize the call, else of 8 where those do, else two tiles a wave, so
  //   that each activation operand is loaded for two products. 7168 rows, 8 x 2 x 1 / 16 x 2 x 1 / 4 x 1 x 2: 1 token of 32
  //   / 64 / 72 / 128 chunks 7.7 / 8.3 / 7.9, 12.3 / 12.4 / 12.9, 15.8 / 14.1 / 15.1, 23.3 / 21.5 / 23.8; 2 of 32 / 40 / 72
  //   7.9 / 8.2 / 8.4, 11.5 / 10.3 / 11.3, 15.9 / 17.6 / 15.2; 4 of 16 / 20 / 32 / 40 5.4 / 6.4 / 6.1, 8.7 / 7.2 / 8.1, 10.1
  //   / 8.5 / 10.4, 11.5 / 13.2 / 11.3.
  // * from 1024 tiles: two tiles a wave, 4 K parts, but for 3 or 4 tokens that 4 parts quantize two sets a workgroup (the
  //   two waves of a part share that), of two tiles up to 12 chunks (a part's chunks are its ring) and of one above, and
  //   for up to 4 tokens quantized before from 32 chunks two sets of one tile. 24576 rows, 4 x 1 x 2 / 8 x 2 x 2 / 8 x 2 x
  //   1 at 4 tokens of 10 / 12 / 16 chunks 9.3 / 8.8 / 8.9, 9.9 / 9.3 / 9.5, 12.7 / 13.2 / 11.1, and, quantized before, of
  //   18 / 24 / 32 / 40 14.6 / 15.5 / 15.3, 16.7 / 17.5 / 18.2, 21.6 / 21.9 / 20.7, 25.1 / 26.8 / 24.9 (block 128 of 32 20.7
  //   / 22.1 / 19.7; 16384 x 8192 at 2 tokens 26.4 with the first, 24.4 with the last).
  const int tiles = N / 16, C = K / 128;
  if (C <= 4 && (tiles > 256 || T > kTok)) return {4, 4, 1};
  if (tiles <= 256) {
    RowShape sh{fp8_fits(8, C, T) && (!fp8_fits(4, C, T) || (T <= 2 && C * T >= 56)) ? 8 : 4, 1, 1};
    // Where the tiles leave CUs idle and a part would run through more than 16 chunks, K is split over as many workgroups
    // as fill the 256 CUs, 32 chunks or more each, and a second launch adds the splits (about 2.5 us). Block 32, us without
    // / with, at 1 / 8 / 32 tokens: 512 x 12288 - / 10.8 -> 9.5 / 16.1 -> 11.9, 512 x 16384 - / 12.4 -> 9.7 / 19.0 -> 12.2,
    // 512 x 65536 34.6 -> 12.0 / 34.2 -> 15.6 / 59.4 -> 21.5, 1280 x 32768 21.0 -> 14.6 / 20.8 -> 15.1 / 34.6 -> 22.1. With
    // 16 chunks a part the second launch costs as much as it saves: 64 x 16384 8.4 -> 7.6 at one token, 512 x 8192 8.5 ->
    // 8.8 at 8; with tiles for more than half the CUs it loses: 2112 x 16384 10.1 -> 13.0 and 13.7 -> 16.2.
    if (C > 16 * sh.W) sh.S = std::max(1, std::min({16, 256 / tiles, C / 32}));
    return sh;
  }
  if (tiles >= 1024) {
    if (!fp8_fits(4, C, T)) return T <= kFusedMaxTokens && C >= 32 ? RowShape{8, 2, 1} : RowShape{4, 1, 2};
    if (T < 3) return {4, 1, 2};
    return {8, 2, C <= 12 ? 2 : 1};
  }
  if (fp8_fits(4, C, T)) return {8, 2, 1};
  if (fp8_fits(8, C, T)) return {16, 2, 1};
  return {4, 1, 2};
}

// K splits of a call, and the bytes of their partial sums.
int fp8_splits(int N, int K, int T) {
  return T <= kGemvMaxTokens ? fp8_row_shape(N, K, T).S : fp8_gemm_splits(N, K, T);
}
uint64_t fp8_partial_bytes(int N, int K, int T) {
  const int splits = fp8_splits(N, K, T);
  return splits > 1 ? (uint64_t)splits * T * N * sizeof(float) : 0;
}

// Fused quantization passes (4 blocks of 128 each per wave) for a K part's chunks x the tokens, shared by the
// part's M waves: 1, 2 or 4, or 0 when they exceed the part's LDS rows (the call then quantizes in its own
// launch).
int fp8_fused_passes(const RowShape& sh, int K, int T) {
  if (T > kFusedMaxTokens) return 0;
  const int parts = sh.parts() * sh.S, blocks = ((K / 128 + parts - 1) / parts) * T;
  if (blocks > kTileQRows) return 0;
  const int per_wave = (blocks + sh.M - 1) / sh.M;
  return per_wave <= 4 ? 1 : per_wave <= 8 ? 2 : 4;
}

// fp8_row_gemv_kernel of shape (W, M, TM): P fused quantization passes, or P = 0 when x comes quantized. A combination
// that fp8_row_shape does not make has no kernel and is an error, not a call that leaves y as it was.
template <int kBlock, int W, int M, int TM, bool kPair = false, bool kSplit = false>
int launch_row_gemv(const Fp8Args& a, int P, hipStream_t st, int S = 1) {
  const int sets = kPair ? a.N / 16 : a.N / 16 / TM;
  auto go = [&](auto kernel, int tokens = kTok) {
    hipLaunchKernelGGL(kernel, dim3((sets + M - 1) / M, (a.T + tokens - 1) / tokens, S), dim3(64 * W), 0, st, a);
    MX_LAUNCH_CHECK("fp8_row_gemv_kernel");
    return MX_OK;
  };
  // More than 16 tokens: both token tiles in a workgroup, so that the weights are read once -- but in two workgroups
  // where the codes come as rows (16 pieces of 64 bytes an operand) and two workgroups a tile still fit the CUs: the
  // grouped product of 8 x 64 / 8 x 256 rows of 4096 at 32 tokens 9.0 / 9.2 us in one, 6.3 / 6.5 in two (8 x 512 9.9 and
  // 11.1, 8 x 1024 12.8 and 14.7).
  if constexpr (W == 4 && M == 1)
    if (P == 0 && a.T > kTok && (a.ordered || a.N > 2048))
      return go(fp8_row_gemv_kernel<kBlock, false, W, M, TM, 2, 1, false, kSplit>, 2 * kTok);
  if (P == 0) return go(fp8_row_gemv_kernel<kBlock, false, W, M, TM, 1, 1, kPair, kSplit>);
  if constexpr (W / M < 8 || kPair)   // 8 parts are only chosen for more blocks than one pass takes
    if (P == 1) return go(fp8_row_gemv_kernel<kBlock, true, W, M, TM, 1, 1, kPair, kSplit>);
  if constexpr (8 * M <= kTileQRows)
    if (P == 2) return go(fp8_row_gemv_kernel<kBlock, true, W, M, TM, 1, 2, kPair, kSplit>);
  if constexpr (16 * M <= kTileQRows)
    if (P == 4) return go(fp8_row_gemv_kernel<kBlock, true, W, M, TM, 1, 4, kPair, kSplit>);
  return fail(MX_ERR_STATE, "FP8 GEMV: %d passes of the %d x %d x %d shape have no kernel", P, W, M, TM);
}

template <int kBlock>
int launch_row_gemv(const RowShape& sh, const Fp8Args& a, int P, hipStream_t st) {
  const int shape = 100 * sh.W + 10 * sh.M + sh.TM;
  if (sh.S > 1) {
    if (shape == 411) return launch_row_gemv<kBlock, 4, 1, 1, false, true>(a, P, st, sh.S);
    return fail(MX_ERR_STATE, "FP8 GEMV: shape %d does not split K", shape);
  }
  switch (shape) {
    case 411: return launch_row_gemv<kBlock, 4, 1, 1>(a, P, st);
    case 811: return launch_row_gemv<kBlock, 8, 1, 1>(a, P, st);
    case 412: return launch_row_gemv<kBlock, 4, 1, 2>(a, P, st);
    case 441: return launch_row_gemv<kBlock, 4, 4, 1>(a, P, st);
    case 821: return launch_row_gemv<kBlock, 8, 2, 1>(a, P, st);
    case 822: return launch_row_gemv<kBlock, 8, 2, 2>(a, P, st);
    case 1621: return launch_row_gemv<kBlock, 16, 2, 1>(a, P, st);
  }
  return fail(MX_ERR_STATE, "FP8 GEMV: shape %d has no kernel", shape);
}

// Whether a[0 .. na) and b[0 .. nb) share bytes (a null pointer shares none). A launch that quantizes its own input
// reads it while other workgroups already write their outputs: where the two share bytes (a projection in place, a down
// input kept in y), a quantizer launch of its own reads it first.
bool overlap(const void* a, uint64_t na, const void* b, uint64_t nb) {
  return a && b && (uintptr_t)a < (uintptr_t)b + nb && (uintptr_t)b < (uintptr_t)a + na;
}

// Whether the GEMV quantizes a plain call's activations itself (fp8_row_gemv_kernel, few tokens).
bool fp8_fused_ok(int N, int K, int T) { return T <= kFusedMaxTokens && fp8_fused_passes(fp8_row_shape(N, K, T), K, T) > 0; }

// fp8_quant_ordered_kernel: T tokens' codes and scales into buffers of T rounded up to 16 rows.
int launch_quant_ordered(int block, const uint16_t* x, uint8_t* q, void* s, int T, int K, hipStream_t st,
                         uint8_t* q_rows = nullptr, void* s_rows = nullptr) {
  const int C = K / 128;
  const dim3 grid((unsigned)(((int64_t)T * C + 15) / 16));
  const bool rows = q_rows || s_rows;
  auto kernel = block == 32 ? (rows ? fp8_quant_ordered_kernel<32, true> : fp8_quant_ordered_kernel<32, false>)
                            : (rows ? fp8_quant_ordered_kernel<128, true> : fp8_quant_ordered_kernel<128, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, x, q, (uint8_t*)s, q_rows, (uint8_t*)s_rows, T, C);
  MX_LAUNCH_CHECK("fp8_quant_ordered_kernel");
  return MX_OK;
}

// The product on quantized activations: the row GEMV (T <= 32) or the tiled GEMM, with K split over fp8_splits(N, K, T)
// workgroups whose FP32 partial sums go to `partial` (fp8_partial_bytes) and are added in split order by
// fp8_splitk_reduce_kernel.
// x_fused: the BF16 input when the GEMV quantizes it itself (fp8_fused_ok), else null (q and sc given); ordered: q
// and sc as launch_quant_ordered wrote them.
int launch_fp8_product(const uint8_t* blob, int N, int K, int block, const uint8_t* q, const void* sc, int T,
                       uint16_t* y, float* trace, float* partial, hipStream_t st, const uint16_t* x_fused = nullptr,
                       bool ordered = false, int x_group_rows = 0) {
  Fp8Args a{};
  a.blob = blob;
  a.N = N;
  a.K = K;
  a.T = T;
  a.x_group_rows = x_group_rows;
  a.x_stride = x_group_rows ? (int64_t)K * (N / x_group_rows) : K;
  a.xq = q;
  a.xs = sc;
  a.y = y;
  a.trace = trace;
  a.partial = partial;
  a.x = x_fused;
  a.ordered = ordered;
  const int splits = fp8_splits(N, K, T);
  if (T <= kGemvMaxTokens) {
    const RowShape sh = fp8_row_shape(N, K, T);
    const int P = x_fused ? fp8_fused_passes(sh, K, T) : 0;
    if (int s = block == 32 ? launch_row_gemv<32>(sh, a, P, st) : launch_row_gemv<128>(sh, a, P, st)) return s;
  } else {
    const dim3 grid((N / 64 + 3) / 4, (T + kGemmTok - 1) / kGemmTok, splits);
    if (block == 32) hipLaunchKernelGGL(fp8_gemm_kernel<32>, grid, dim3(kGemmThreads), 0, st, a);
    else hipLaunchKernelGGL(fp8_gemm_kernel<128>, grid, dim3(kGemmThreads), 0, st, a);
    MX_LAUNCH_CHECK("fp8_gemm_kernel");
  }
  if (splits > 1) {
    const int64_t count = (int64_t)T * N;
    hipLaunchKernelGGL(fp8_splitk_reduce_kernel, dim3((unsigned)((count / 4 + 255) / 256)), dim3(256), 0, st,
                       (const float*)partial, splits, count, y, trace);
    MX_LAUNCH_CHECK("fp8_splitk_reduce_kernel");
  }
  return MX_OK;
}

}  // namespace

using namespace mxi;

extern "C" {

uint64_t mx_fp8_tiled_bytes(int32_t N, int32_t K, int32_t block) {
  if ((block != 32 && block != 128) || N <= 0 || N % 64 || K <= 0 || K % 128) return 0;
  return fp8_blob(N, K, block).total;
}

int mx_fp8_tile(mx_ctx* ctx, const uint8_t* w, const void* sw, int32_t N, int32_t K, int32_t block, void* tiled,
                void* stream) {
  if (int s = use(ctx)) return s;
  if (int s = check_fp8_shape(N, K, block, "mx_fp8_tile")) return s;
  MX_REQUIRE(w && sw && tiled, "mx_fp8_tile: null pointer");
  MX_REQUIRE(((uintptr_t)w & 15) == 0 && ((uintptr_t)tiled & 255) == 0 && ((uintptr_t)sw & 3) == 0,
             "mx_fp8_tile: weights 16-byte, scales 4-byte and the tiled blob 256-byte aligned");
  hipLaunchKernelGGL(fp8_tile_kernel, dim3(2048), dim3(256), 0, as_stream(stream), w, sw, (uint8_t*)tiled, N, K,
                     block);
  MX_LAUNCH_CHECK("fp8_tile_kernel");
  return MX_OK;
}

int mx_act_quant128(mx_ctx* ctx, const uint16_t* x, uint8_t* q, float* s, int64_t rows, int64_t width, void* stream) {
  if (int s2 = use(ctx)) return s2;
  MX_REQUIRE(rows >= 0 && width > 0 && width % 128 == 0, "mx_act_quant128: width must be a positive multiple of 128");
  if (!rows) return MX_OK;
  MX_REQUIRE(x && q && s && ((uintptr_t)x & 3) == 0 && ((uintptr_t)q & 1) == 0,
             "mx_act_quant128: null or misaligned pointer");
  const int64_t blocks = rows * (width / 128);
  if (((uintptr_t)x & 15) == 0 && ((uintptr_t)q & 7) == 0) {
    const int64_t want = (blocks + 15) / 16;   // 16 blocks per 256-thread workgroup and pass
    hipLaunchKernelGGL(act_quant128_v8_kernel, dim3((unsigned)(want < 8192 ? want : 8192)), dim3(256), 0,
                       as_stream(stream), x, q, s, blocks);
    MX_LAUNCH_CHECK("act_quant128_v8_kernel");
    return MX_OK;
  }
  MX_REQUIRE(blocks <= (int64_t)(1u << 31) * 4 - 4, "mx_act_quant128: too many blocks for one launch");
  hipLaunchKernelGGL(act_quant128_kernel, dim3((unsigned)((blocks + 3) / 4)), dim3(256), 0, as_stream(stream), x, q, s,
                     blocks);
  MX_LAUNCH_CHECK("act_quant128_kernel");
  return MX_OK;
}

int mx_fp8_projection(mx_ctx* ctx, const void* tiled, int32_t N, int32_t K, int32_t block, const uint16_t* x,
                      int32_t T, uint16_t* y, float* trace, uint8_t* q_out, void* s_out, void* stream) {
  if (int s = use(ctx)) return s;
  if (int s = check_fp8_shape(N, K, block, "mx_fp8_projection")) return s;
  MX_REQUIRE(T >= 0, "mx_fp8_projection: negative token count");
  if (!T) return MX_OK;
  MX_REQUIRE(tiled && x && y, "mx_fp8_projection: null pointer");
  MX_REQUIRE(((uintptr_t)tiled & 255) == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)y & 7) == 0 &&
                 ((uintptr_t)trace & 15) == 0,
             "mx_fp8_projection: tiled 256-byte, x 16-byte, y 8-byte and trace 16-byte alignment required");
  hipStream_t st = as_stream(stream);
  MX_REQUIRE(((uintptr_t)q_out & 15) == 0 && ((uintptr_t)s_out & 3) == 0,
             "mx_fp8_projection: q 16-byte, s 4-byte aligned");
  // The decode GEMV's codes come in its load order, in whole tiles of 16 tokens, and the rows that a caller asks for are
  // written beside them; up to 4 tokens' rows are read as they are (us, rows / load order: 2112 x 7168 block 128 at one
  // token 8.7 / 9.1, block 32 at 16 12.4 / 10.6, 512 x 7168 at 32 17.8 / 11.9, 7168 x 16384 at 32 43.3 / 29.5).
  const bool codes = q_out || s_out;
  const bool ordered = T <= kGemvMaxTokens && (!codes || T > kFusedMaxTokens);
  const uint64_t rows = ordered ? (T + kTok - 1) / kTok * kTok : T;
  const uint64_t q_b = (rows * K + 255) & ~255ull, s_b = (rows * (K / 32) + 255) & ~255ull;   // 4 scale bytes a chunk
  void* base = nullptr;
  if (int s = scratch(ctx, q_b + s_b + fp8_partial_bytes(N, K, T) + 256, &base)) return s;
  uint8_t* q = q_out && !ordered ? q_out : (uint8_t*)base;
  void* sc = s_out && !ordered ? s_out : (void*)((uint8_t*)base + q_b);
  float* partial = (float*)((uint8_t*)base + q_b + s_b);
  const uint64_t x_b = (uint64_t)T * K * 2, y_b = (uint64_t)T * N * 2;
  if (!codes && fp8_fused_ok(N, K, T) && !overlap(x, x_b, y, y_b) &&
      !overlap(x, x_b, trace, 2 * y_b))   // the GEMV quantizes x itself
    return launch_fp8_product((const uint8_t*)tiled, N, K, block, nullptr, nullptr, T, y, trace, partial, st, x);
  if (ordered) {
    if (int s = launch_quant_ordered(block, x, q, sc, T, K, st, q_out, s_out)) return s;
  } else if (block == 32) {
    if (int s = mx_act_quant32(ctx, x, q, (uint8_t*)sc, T, K, stream)) return s;
  } else {
    if (int s = mx_act_quant128(ctx, x, q, (float*)sc, T, K, stream)) return s;
  }
  return launch_fp8_product((const uint8_t*)tiled, N, K, block, q, sc, T, y, trace, partial, st, nullptr, ordered);
}

int mx_fp8_grouped_projection(mx_ctx* ctx, const void* tiled, int32_t groups, int32_t rows, int32_t K,
                              const uint8_t* q, const uint8_t* s, int32_t T, uint16_t* y, float* trace, void* stream) {
  if (int st = use(ctx)) return st;
  MX_REQUIRE(groups >= 1 && groups <= 64 && rows > 0 && rows % 64 == 0 && rows <= (1 << 20),
             "mx_fp8_grouped_projection: 1 to 64 groups of a positive multiple of 64 rows required");
  const int N = groups * rows;
  if (int st = check_fp8_shape(N, K, 32, "mx_fp8_grouped_projection")) return st;
  MX_REQUIRE(T >= 0 && T <= kGemvMaxTokens, "mx_fp8_grouped_projection: token count %d outside [0, %d]", T,
             kGemvMaxTokens);
  if (!T) return MX_OK;
  MX_REQUIRE(tiled && q && s && y, "mx_fp8_grouped_projection: null pointer");
  MX_REQUIRE(((uintptr_t)tiled & 255) == 0 && ((uintptr_t)q & 15) == 0 && ((uintptr_t)s & 3) == 0 &&
                 ((uintptr_t)y & 7) == 0 && ((uintptr_t)trace & 15) == 0,
             "mx_fp8_grouped_projection: tiled 256-byte, q 16-byte, s 4-byte, y 8-byte, trace 16-byte alignment");
  void* partial = nullptr;
  if (int st = scratch(ctx, fp8_partial_bytes(N, K, T), &partial)) return st;
  return launch_fp8_product((const uint8_t*)tiled, N, K, 32, q, s, T, y, trace, (float*)partial, as_stream(stream),
                            nullptr, false, rows);
}

int mx_fp8_expert_forward(mx_ctx* ctx, const void* w1, const void* w3, const void* w2, int32_t H, int32_t I,
                          const uint16_t* x, int32_t T, float limit, const float* route_w, uint16_t* y,
                          const mx_expert_stages* stages, void* stream) {
  if (int s = use(ctx)) return s;
  MX_REQUIRE(w1 && w3 && w2, "mx_fp8_expert_forward: null tiled weight");
  MX_REQUIRE(((uintptr_t)w1 & 255) == 0 && ((uintptr_t)w3 & 255) == 0 && ((uintptr_t)w2 & 255) == 0,
             "mx_fp8_expert_forward: tiled weights must be 256-byte aligned");
  MX_REQUIRE(H > 0 && H % 128 == 0 && I > 0 && I % 128 == 0, "expert shapes must be positive multiples of 128");
  MX_REQUIRE(T >= 0 && T <= kTok, "token count %d outside [0, %d]", T, kTok);
  MX_REQUIRE(std::isfinite(limit) && limit >= 0.f, "Invalid SwiGLU limit");
  if (!T) return MX_OK;
  MX_REQUIRE(x && y && ((uintptr_t)x & 15) == 0 && ((uintptr_t)y & 15) == 0,
             "x and y must be 16-byte aligned device pointers");
  hipStream_t st = as_stream(stream);
  auto r256 = [](uint64_t b) { return (b + 255) & ~255ull; };
  const uint64_t sizes[5] = {r256((uint64_t)kTok * H), r256((uint64_t)kTok * H / 32), r256((uint64_t)T * I * 2),
                             r256((uint64_t)kTok * I), r256((uint64_t)kTok * I / 32)};
  uint64_t total = fp8_partial_bytes(H, I, T);
  for (uint64_t b : sizes) total += b;
  void* base = nullptr;
  if (int s = scratch(ctx, total, &base)) return s;
  uint8_t* cur = (uint8_t*)base;
  uint8_t* buf[5];
  for (int i = 0; i < 5; ++i) {
    buf[i] = cur;
    cur += sizes[i];
  }
  float* partial = (float*)cur;   // of the down product
  uint8_t* q = (stages && stages->q) ? stages->q : buf[0];
  uint8_t* s = (stages && stages->s) ? stages->s : buf[1];
  uint16_t* din = (stages && stages->down_input) ? stages->down_input : (uint16_t*)buf[2];
  uint8_t* dq = (stages && stages->down_q) ? stages->down_q : buf[3];
  uint8_t* ds = (stages && stages->down_s) ? stages->down_s : buf[4];
  Fp8Args a{};
  a.blob = (const uint8_t*)w1;
  a.blob2 = (const uint8_t*)w3;
  a.N = I;
  a.K = H;
  a.T = T;
  a.xq = q;
  a.xs = s;
  a.x_stride = H;
  a.y = stages ? stages->w1 : nullptr;
  a.y3 = stages ? stages->w3 : nullptr;
  a.din = din;
  a.swiglu_trace = stages ? stages->trace : nullptr;
  a.route_w = route_w;
  a.limit = limit;
  MX_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)dq & 15) == 0 && ((uintptr_t)a.y & 7) == 0 &&
                 ((uintptr_t)a.y3 & 7) == 0 && ((uintptr_t)din & 3) == 0 && ((uintptr_t)s & 3) == 0 &&
                 ((uintptr_t)ds & 3) == 0,
             "stage buffers: q/down_q 16-byte, w1/w3 8-byte, scales and down_input 4-byte aligned");
  // few tokens: each launch quantizes its own input, unless the caller asks for those codes or gives an output that
  // shares bytes with it (or, for the down input, a buffer that 16-byte loads cannot read); more tokens: codes in the
  // GEMV's load order
  const uint64_t xh = (uint64_t)T * H * 2, xi = (uint64_t)T * I * 2;   // bytes of [T][H] and of [T][I]
  const bool own_q = !stages || (!stages->q && !stages->s);
  const bool shared_x = overlap(x, xh, din, xi) || overlap(x, xh, a.y, xi) || overlap(x, xh, a.y3, xi) ||
                        overlap(x, xh, a.swiglu_trace, 10 * xi);   // 5 floats an element
  const int p1 = own_q && !shared_x ? fp8_fused_passes(kPairShape, H, T) : 0;
  a.ordered = own_q;
  if (p1) a.x = x;
  else if (int e = own_q ? launch_quant_ordered(32, x, q, s, T, H, st) : mx_act_quant32(ctx, x, q, s, T, H, stream))
    return e;
  if (int e = launch_row_gemv<32, kPairShape.W, 1, 2, true>(a, p1, st)) return e;
  const bool own_dq = (!stages || (!stages->down_q && !stages->down_s)) && ((uintptr_t)din & 15) == 0;
  if (own_dq && fp8_fused_ok(H, I, T) && !overlap(din, xi, y, xh))
    return launch_fp8_product((const uint8_t*)w2, H, I, 32, nullptr, nullptr, T, y, nullptr, partial, st, din);
  if (int e = own_dq ? launch_quant_ordered(32, din, dq, ds, T, I, st) : mx_act_quant32(ctx, din, dq, ds, T, I, stream))
    return e;
  return launch_fp8_product((const uint8_t*)w2, H, I, 32, dq, ds, T, y, nullptr, partial, st, nullptr, own_dq);
}

}  // extern "C"
