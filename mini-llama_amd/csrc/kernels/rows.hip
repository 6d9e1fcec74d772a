// Linear of a few activation rows on gfx950: y[m, n] = sum_k W[n, k] x[m, k]
// for m = 2..16 with x resident in LDS.
//
// A workgroup per weight tile has to fetch and convert x anew for every tile:
// 16 rows x 4096 are 256 KiB of fp32 per workgroup against 68 KiB of q8_0
// weights, so a 28672-row gate|up projection moved 470 MB of x from L2 for
// 117 MB of weights (49 us; 4 rows of q4_1 73 MB in 35 us). Here the grid is
// one workgroup per CU: it converts x once into MFMA fragments in LDS, then
// streams its share of the weight tiles past them, bound by the weight reads.
//  - A workgroup owns consecutive tiles; its 16 waves split the tiles' units
//    (16 rows x 128 k, the contiguous lines of mlq_layout.h) into equal
//    consecutive runs, whatever the tile count: a wave streams one
//    contiguous byte range, kDepth units in flight in a register ring. Tiles
//    that a wave covers whole it finishes itself; the first and last, partial
//    ones go through LDS and are added in wave order (deterministic). No
//    integer division by a runtime value anywhere: dealing units out with
//    them cost 5 us a launch.
//  - Up to 8 rows (HL): fp32-class, as the decode GEMV. Activations as fp16
//    hi + lo pairs (x to ~2^-22, MFMA rows 2r and 2r + 1), codes decoded
//    exactly, each block's sum scaled by its fp16 scale in fp32 (q4_1: plus
//    its min times the block's fp32 sum of x).
//  - 9..16 rows: activations rounded to fp16, weights d * q (+ m) rounded to
//    fp16, the MFMA accumulating over a 128-k group, as the skinny GEMM.
//  - Raw GGUF blocks (launch_aos_gemv; the reference's `const void*` device
//    weight, src/cuda_quant.cu:300-361) stream the same way for up to 8 rows:
//    only the loads differ (see AosUnit). Staged through LDS and multiplied
//    element by element in fp32 they were bound by ~5 VALU per weight: one
//    row of 18944 x 3584 q4_0 25.4 -> 13.1 us, q8_0 24.2 -> 15.8, q4_1 24.0 ->
//    13.9; four rows 88.5 -> 14.1.
//  - Up to 8 rows longer than the LDS on at most a tile per CU (down
//    projections): x in pieces, a wave's sums staying in registers.
//  - Each (row, 128-k group) is scaled by its own power of two (the group's
//    largest |x| into [2^14, 2^15)) before it becomes fp16, and the group's
//    sums are scaled back in fp32: any finite x, and no dependence on how
//    units are dealt to waves.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../mlq_layout.h"
#include "device_common.h"
#include "launch.h"
#include "weight_decode.h"

namespace mlq {
namespace {


// Sixteen waves with two units in flight each: 4 layers of an 8B model in
// q8_0 at 16 rows took 277.7 us, eight waves with four in flight 279.3, with
// six 281.9; sixteen with four 328.1 (its registers spill past 128).
constexpr int W = 16, D = 2;

constexpr uint32_t kPast = 0x80000000u;  // an offset past every buffer

// Where the codes come from: the tiled layout, or GGUF blocks as they lie in
// the file (kAos4: base and rows start on 4-byte boundaries; kAos2: on 2-byte
// ones).
enum Source { kTiled, kAos4, kAos2 };

struct RowsArgs {
  const uint8_t* qs;  // kAos*: the GGUF blocks, rows of row_bytes
  const uint8_t* d;
  const uint8_t* mn;
  const float* x;
  float* y;
  int m, n, k, g, ny;
  int nb, row_bytes;  // kAos*
  int tiles, extra;  // tiles per workgroup; the first `extra` have one more
  int phase;         // groups staged at a time (all of them, or one tile per workgroup)
  Epilogue epi;
};

// LDS of a workgroup: fragments, 2^-e per (group, row), block sums (HL q4_1);
// reused at the end for two partial tiles per wave.
template <int QT, int RP, bool HL>
struct Lds {
  static constexpr int kRows = HL ? 2 * RP : RP;    // MFMA rows stored
  static constexpr int kGroup = kRows * kGroupK * 2;
  static constexpr int kScale = RP * 4;
  static constexpr int kSums = HL && QT == MLQ_Q4_1 ? kGroupBlocks * RP * 4 : 0;
  static constexpr int kPart = W * 2 * 64 * (HL ? 8 : 16);
  static size_t bytes(int g) {
    return std::max((size_t)g * (kGroup + kScale + kSums), (size_t)kPart);
  }
};

// GGUF blocks: lane (row lane % 16, quarter kq = lane / 16) reads, of each of
// the unit's four blocks, the 12 bytes from the 4-byte boundary at or below
// the block (q8_0: plus 8 kq, q4: plus 8 (kq % 2)). They hold the lane's 8
// code bytes, 2 or 4 bytes in, and in quarter 0 (q4: also 2) the scale (and
// min) ahead of them; no window passes the 4-byte boundary behind its block.
// q4_1 blocks (20 bytes) all share one phase; off a 4-byte boundary they take
// 16 bytes.
struct AosUnit {
  uint4 w4[4];
};
// One unit's weights as loaded by a lane: lines of the tiled layout, or blocks.
struct TiledUnit {
  uint4 q, q2;
  uint2 d, m;
};
template <int SRC>
using Unit = std::conditional_t<SRC == kTiled, TiledUnit, AosUnit>;

template <int QT>
__device__ __host__ constexpr int aos_block_bytes() {
  return QT == MLQ_Q8_0 ? 34 : QT == MLQ_Q4_0 ? 18 : 20;
}

// 8 code bytes (q4: already masked nibbles; q8_0: signed) -> exact fp16.
template <int QT>
__device__ __forceinline__ h8_t bytes_exact(uint32_t c0, uint32_t c1) {
  if constexpr (QT == MLQ_Q8_0) {
    c0 ^= 0x80808080u;
    c1 ^= 0x80808080u;
  }
  const float bias = QT == MLQ_Q8_0 ? 1152.0f : QT == MLQ_Q4_0 ? 1032.0f : 1024.0f;
  const h2_t b2 = {(_Float16)bias, (_Float16)bias};
  uint4 o;
  o.x = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, c0, 0x04010400u)) - b2);
  o.y = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, c0, 0x04030402u)) - b2);
  o.z = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, c1, 0x04010400u)) - b2);
  o.w = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, c1, 0x04030402u)) - b2);
  return __builtin_bit_cast(h8_t, o);
}

// Largest of a non-negative float over the N-lane groups of a wave, compared
// as integers: NaN propagates (its bits exceed infinity's).
template <int N>
__device__ __forceinline__ float group_max_nonneg(float v) {
  static_assert(N == 4 || N == 8 || N == 16 || N == 32, "lanes per row");
  int b = __builtin_bit_cast(int, v);
  b = max(b, __builtin_amdgcn_mov_dpp(b, kDppXor1, 0xF, 0xF, false));
  b = max(b, __builtin_amdgcn_mov_dpp(b, kDppXor2, 0xF, 0xF, false));
  if constexpr (N >= 8) b = max(b, __builtin_amdgcn_mov_dpp(b, kDppHalfMirror, 0xF, 0xF, false));
  if constexpr (N >= 16) b = max(b, __builtin_amdgcn_mov_dpp(b, kDppMirror, 0xF, 0xF, false));
  if constexpr (N >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
    b = max((int)r[0], (int)r[1]);
  }
  return __builtin_bit_cast(float, b);
}

// PH: x in pieces of a.phase groups, one tile per workgroup.
template <int QT, int RP, bool HL, int SRC, bool PH>
__global__ __launch_bounds__(64 * W) void rows_kernel(RowsArgs a) {
  using L = Lds<QT, RP, HL>;
  constexpr int MR = L::kRows;
  constexpr int LPR = RP == 1 ? 32 : 64 / RP;  // lanes per row of a load
  constexpr int GL = RP == 1 ? 2 : 1;  // groups per load
  constexpr int NL = 32 / LPR;         // 16-byte loads per group
  constexpr int BG = 2;                // groups a wave stages at a time
  constexpr int AC = HL ? 2 : 4;       // accumulators per lane
  constexpr bool SUMS = HL && QT == MLQ_Q4_1;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* frag = smem;
  float* scale = (float*)(smem + (size_t)a.phase * L::kGroup);
  float* sums = (float*)((uint8_t*)scale + (size_t)a.phase * L::kScale);
  float* part = (float*)smem;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.g;
  // this workgroup's tiles and this wave's run of their units
  const int T = a.tiles + ((int)blockIdx.x < a.extra ? 1 : 0);
  const int t0 = (int)blockIdx.x * a.tiles + min((int)blockIdx.x, a.extra);
  const int U = PH ? a.phase : T * G;
  int u0 = wave * U / W, u1 = (wave + 1) * U / W, n = u1 - u0;
  int gb = 0, ge = G;  // the groups in LDS

  using U1 = Unit<SRC>;
  constexpr uint32_t QB = QT == MLQ_Q8_0 ? 2048u : 1024u;
  constexpr int BS = aos_block_bytes<QT>();
  size_t unit0 = (size_t)t0 * G + u0;
  const size_t rows0 = (size_t)t0 * kTileRows;
  const uint8_t* aos = a.qs + rows0 * a.row_bytes;  // (kAos*)
  const int lead = SRC == kAos2 ? (int)((uintptr_t)aos & 3) : 0;
  rsrc_t rq =
      SRC == kTiled ? make_rsrc(a.qs + unit0 * QB, (uint32_t)n * QB)
                    : make_rsrc(aos - lead, (uint32_t)((lead + (size_t)min((size_t)T * kTileRows, a.n - rows0) * a.row_bytes + 3) & ~(size_t)3));
  rsrc_t rd = SRC == kTiled ? make_rsrc(a.d + unit0 * 128, (uint32_t)n * 128u) : rq;
  rsrc_t rm = SRC == kTiled && QT == MLQ_Q4_1
                        ? make_rsrc(a.mn + unit0 * 128, (uint32_t)n * 128u) : rd;
  const uint32_t qoff = (uint32_t)lane * 16u, soff = (uint32_t)(lane & 15) * 8u;
  // (kAos*) byte offset of the lane's row and the quarter's eight code bytes
  const uint32_t arow = (uint32_t)(lead + (lane & 15) * a.row_bytes);
  const uint32_t aq = QT == MLQ_Q8_0 ? 8u * (lane >> 4) : 8u * ((lane >> 4) & 1);
  // the next unit to load, as (tile, group)
  const int first = wave * T / W;  // = u0 / G
  int ltile = first, lg = u0 - first * G;
  // unit j of the run, in order (zeros past it)
  auto load = [&](U1& s, int j) __attribute__((always_inline)) {
    if constexpr (SRC == kTiled) {
      s.q = buf_load16_stream(rq, qoff, (uint32_t)j * QB);
      if (QT == MLQ_Q8_0) s.q2 = buf_load16_stream(rq, qoff, (uint32_t)j * QB + 1024u);
      s.d = buf_load8(rd, soff, (uint32_t)j * 128u);
      if (QT == MLQ_Q4_1) s.m = buf_load8(rm, soff, (uint32_t)j * 128u);
    } else {
      const uint32_t su =
          j < n ? (uint32_t)(ltile * kTileRows * a.row_bytes + lg * (kGroupBlocks * BS)) : kPast;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint32_t at = arow + (uint32_t)(b * BS);
        const int w0 = (int)((at & ~3u) + aq);
        if constexpr (QT == MLQ_Q4_1 && SRC == kAos2) {
          s.w4[b] = buf_load16(rq, (uint32_t)w0, su);
        } else {
          const auto v = __builtin_amdgcn_raw_buffer_load_b96(rq, w0, (int)su, 0);
          s.w4[b] = make_uint4(v[0], v[1], v[2], 0u);
        }
      }
      if (++lg == G) {
        lg = 0;
        ++ltile;
      }
    }
  };
  // block b of a unit of group g: its exact codes, scale and min
  auto block = [&](const U1& s, int b, int g, float& d, float& mn) __attribute__((always_inline)) {
    mn = 0.0f;
    if constexpr (SRC == kTiled) {
      d = (float)half_at(s.d, b);
      if constexpr (QT == MLQ_Q4_1) mn = (float)half_at(s.m, b);
      return decode_exact<QT>(s.q, s.q2, b);
    } else {
      uint32_t c0, c1;
      const uint4 v = s.w4[b];
      if constexpr (QT == MLQ_Q4_1) {
        // one phase for every block: the base's
        const bool half = SRC == kAos2 && lead != 0;
        c0 = half ? __builtin_amdgcn_alignbit(v.z, v.y, 16) : v.y;
        c1 = half ? __builtin_amdgcn_alignbit(v.w, v.z, 16) : v.z;
        const uint32_t dm = half ? __builtin_amdgcn_alignbit(v.y, v.x, 16) : v.x;
        const uint32_t row = __builtin_bit_cast(
            uint32_t, xor16_pair(__builtin_bit_cast(float, dm)).lo);
        d = half_bits_to_float((uint16_t)row);
        mn = half_bits_to_float((uint16_t)(row >> 16));
      } else {
        const bool odd = SRC == kAos4 ? (b & 1) != 0 : ((arow + (uint32_t)(b * BS)) & 2u) != 0;
        c0 = odd ? v.y : __builtin_amdgcn_alignbit(v.y, v.x, 16);
        c1 = odd ? v.z : __builtin_amdgcn_alignbit(v.z, v.y, 16);
        // the scale sits in quarter 0 (q4_0: and 2): to the row's other quarters
        d = xor16_pair(half_bits_to_float((uint16_t)(odd ? v.x >> 16 : v.x))).lo;
        if constexpr (QT == MLQ_Q8_0) d = xor32_pair(d).lo;
      }
      // blocks past the row belong to the next one
      if (g * kGroupBlocks + b >= a.nb) d = mn = 0.0f;
      if constexpr (QT != MLQ_Q8_0) {
        const uint32_t sh = 4u * (uint32_t)(lane >> 5);  // elements 16..31: high nibbles
        c0 = (c0 >> sh) & 0x0F0F0F0Fu;
        c1 = (c1 >> sh) & 0x0F0F0F0Fu;
      }
      return bytes_exact<QT>(c0, c1);
    }
  };

  // ---- x -> fragments. Lane group rho of LPR lanes reads row rho of a 128-k
  // group, lane q of it the float4s q, q + LPR, ...; rows past m and columns
  // past k read as zero through offsets past the buffer.
  const rsrc_t rx = make_rsrc(a.x, (uint32_t)((size_t)a.m * a.k * 4));
  const int rho = RP == 1 ? 0 : lane / LPR, q = lane % LPR;
  const int gl = RP == 1 ? lane / LPR : 0;  // the lane's group of a load
  const bool vec = SRC == kTiled || (a.k & 3) == 0;
  struct Batch {
    float4 v[BG / GL][NL];
  };
  auto load_x = [&](Batch& b, int g0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BG / GL; ++i)
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int col = (g0 + i * GL + gl) * kGroupK + 4 * (j * LPR + q);
        const uint32_t off = rho < a.m && col < a.k ? (uint32_t)(rho * a.k + col) * 4u : kPast;
        if (vec) {
          b.v[i][j] = __builtin_bit_cast(float4, buf_load16(rx, off, 0));
        } else {  // the row's end falls inside a float4
          b.v[i][j].x = __builtin_bit_cast(float, buf_load4(rx, off, 0));
          b.v[i][j].y = __builtin_bit_cast(float, buf_load4(rx, col + 1 < a.k ? off + 4u : kPast, 0));
          b.v[i][j].z = __builtin_bit_cast(float, buf_load4(rx, col + 2 < a.k ? off + 8u : kPast, 0));
          b.v[i][j].w = __builtin_bit_cast(float, buf_load4(rx, col + 3 < a.k ? off + 12u : kPast, 0));
        }
      }
  };
  auto stage = [&](const Batch& b, int g0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BG / GL; ++i) {
      const int g = g0 + i * GL + gl;
      float mx = 0.0f;
#pragma unroll
      for (int j = 0; j < NL; ++j) mx = abs_maximum4(mx, b.v[i][j]);
      // 2^e must be a finite float: groups whose largest |x| is below 2^-112
      // keep e = 127 (they land below 2^15, coarser but finite)
      const int e = min(pow2_scale_exp(group_max_nonneg<LPR>(mx)), 127);
      const float sc = ldexp_f(1.0f, e);
      if (g >= ge) continue;
      const int at = PH ? g - gb : g;
      if (q == 0) scale[at * RP + rho] = ldexp_f(1.0f, -e);
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int f = j * LPR + q;  // float4 of the group: block f / 8, quarter (f / 2) % 4
        uint8_t* p = frag + (size_t)at * L::kGroup +
                     (((f >> 3) * 4 + ((f >> 1) & 3)) * MR) * 16 + (f & 1) * 8;
        float4 v = b.v[i][j];
        v.x *= sc;
        v.y *= sc;
        v.z *= sc;
        v.w *= sc;
        if constexpr (HL) {
          uint2 hi, lo;
          split2(v.x, v.y, hi.x, lo.x);
          split2(v.z, v.w, hi.y, lo.y);
          *(uint2*)(p + (2 * rho) * 16) = hi;
          *(uint2*)(p + (2 * rho + 1) * 16) = lo;
          if constexpr (SUMS) {
            // (the lanes of a block share their group, so all of them are here)
            const float s = row_sum<8>((v.x + v.y) + (v.z + v.w));
            if ((f & 7) == 0) sums[(at * kGroupBlocks + (f >> 3)) * RP + rho] = s;
          }
        } else {
          *(uint2*)(p + rho * 16) = make_uint2(pack_h2(v.x, v.y), pack_h2(v.z, v.w));
        }
      }
    }
  };
  // x is requested ahead of the weights (loads return in order and x mostly
  // hits L2); groups past the first 32 are staged behind them
  Batch b0;
  U1 ring[D];
  auto fill = [&]() __attribute__((always_inline)) {
    const int gs = gb + wave * BG;
    load_x(b0, gs);
#pragma unroll
    for (int i = 0; i < D; ++i) load(ring[i], i);
    stage(b0, gs);
    for (int g = gs + W * BG; g < ge; g += W * BG) {
      load_x(b0, g);
      stage(b0, g);
    }
    __syncthreads();
  };
  if constexpr (PH) ge = min(G, a.phase);
  fill();

  // ---- the wave's units
  float acc[AC], head[AC];  // running; the run's first tile if not whole
#pragma unroll
  for (int i = 0; i < AC; ++i) acc[i] = head[i] = 0.0f;
  const uint8_t* af0 = frag + ((lane >> 4) * MR + (lane & 15) % MR) * 16;
  const int r0 = AC * (lane >> 4) % RP;  // this lane's first row (repeated past RP)
  int tile = first, g = u0 - first * G;
  // the output of `v` (this lane's AC rows of weight row lane % 16)
  auto store_tile = [&](const float (&v)[AC], int t) __attribute__((always_inline)) {
    const int row = (t0 + t) * kTileRows + (lane & 15);
    const int r = AC * (lane >> 4);
    if (a.epi.act == kEpiSwiGLU) {
#pragma unroll
      for (int i = 0; i < AC; ++i) {
        const float p = add_bias(a.epi, v[i], row);  // n % 16 == 0: every row exists
        const float up = dpp<kDppRor8>(p);
        if ((lane & 8) == 0 && r + i < a.m)
          a.y[(size_t)(r + i) * a.ny + glu_col(row)] = silu_f(p) * up;
      }
    } else if (row < a.n) {
#pragma unroll
      for (int i = 0; i < AC; ++i)
        if (r + i < a.m) a.y[(size_t)(r + i) * a.n + row] = add_bias(a.epi, v[i], row);
    }
  };
  auto flush = [&]() __attribute__((always_inline)) {
    if (tile * G >= u0 && (tile + 1) * G <= u1) {
      store_tile(acc, tile);
    } else {  // (the last tile of the run stays in acc, see below)
#pragma unroll
      for (int i = 0; i < AC; ++i) head[i] = acc[i];
    }
#pragma unroll
    for (int i = 0; i < AC; ++i) acc[i] = 0.0f;
  };
  // this lane's two rows of p's RP values (one row: its value and nothing past
  // it, which would be off an 8-byte boundary and, at the end, outside the LDS)
  auto row_pair = [&](const float* p) __attribute__((always_inline)) {
    if constexpr (RP == 1) return make_float2(p[0], 0.0f);
    else return *(const float2*)(p + r0);
  };
  auto run = [&](const U1& s) __attribute__((always_inline)) {
    const uint8_t* af = af0 + (size_t)g * L::kGroup;
    if constexpr (HL) {
      float t[2] = {0.0f, 0.0f};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const h8_t av = __builtin_bit_cast(h8_t, *(const uint4*)(af + b * 4 * MR * 16));
        float d, mb;
        const h8_t bv = block(s, b, g, d, mb);
        const f4_t z = {0.f, 0.f, 0.f, 0.f};
        const f4_t p = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, z, 0, 0, 0);
        t[0] += d * (p[0] + p[1]);
        t[1] += d * (p[2] + p[3]);
        if constexpr (SUMS) {
          const float2 sx = row_pair(sums + (g * kGroupBlocks + b) * RP);
          t[0] += mb * sx.x;
          t[1] += mb * sx.y;
        }
      }
      const float2 sc = row_pair(scale + g * RP);
      acc[0] += t[0] * sc.x;
      acc[1] += t[1] * sc.y;
    } else {
      f4_t p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const h8_t av = __builtin_bit_cast(h8_t, *(const uint4*)(af + b * 4 * MR * 16));
        const h8_t bv = decode_scaled<QT>(s.q, s.q2, s.d, s.m, b);
        p = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, p, 0, 0, 0);
      }
      const f4_t sc = *(const f4_t*)(scale + g * RP + r0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += p[i] * sc[i];
    }
    ++g;
    if constexpr (!PH) {
      if (g == G) {
        flush();
        g = 0;
        ++tile;
      }
    }
  };
  auto stream = [&]() __attribute__((always_inline)) {
    int j = 0;
    for (; j + D <= n; j += D) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        run(ring[i]);
        load(ring[i], j + D + i);
      }
    }
#pragma unroll
    for (int i = 0; i < D; ++i)
      if (j + i < n) run(ring[i]);
  };
  stream();
  if constexpr (PH) {
    // the tile's next groups; each wave keeps its sums
    for (gb = a.phase; gb < G; gb += a.phase) {
      ge = min(G, gb + a.phase);
      const int c = ge - gb;
      u0 = wave * c / W;
      u1 = (wave + 1) * c / W;
      n = u1 - u0;
      g = u0;
      unit0 = (size_t)t0 * G + gb + u0;
      rq = make_rsrc(a.qs + unit0 * QB, (uint32_t)n * QB);
      rd = make_rsrc(a.d + unit0 * 128, (uint32_t)n * 128u);
      rm = QT == MLQ_Q4_1 ? make_rsrc(a.mn + unit0 * 128, (uint32_t)n * 128u) : rd;
      __syncthreads();  // every wave is done with the fragments
      fill();
      stream();
    }
  }
  // A run's partial tiles: the first one (head, or acc if the run ends inside
  // it) in slot 0, the last one in slot 1.
  __syncthreads();  // every wave is done with the fragments
  {
    float* p = part + (wave * 2 * 64 + lane) * AC;
#pragma unroll
    for (int i = 0; i < AC; ++i) {
      p[i] = tile == first ? acc[i] : head[i];
      p[64 * AC + i] = acc[i];
    }
  }
  __syncthreads();

  // ---- tiles shared by several waves, added in wave order
  if constexpr (PH) {
    if (wave != 0) return;
    float v[AC];
#pragma unroll
    for (int i = 0; i < AC; ++i) v[i] = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w)
#pragma unroll
      for (int i = 0; i < AC; ++i) v[i] += part[(w * 2 * 64 + lane) * AC + i];
    store_tile(v, 0);
    return;
  }
  for (int t = wave; t < T; t += W) {
    const int wlo = t * W / T, whi = ((t + 1) * W - 1) / T;  // waves whose runs may meet it
    float v[AC];
#pragma unroll
    for (int i = 0; i < AC; ++i) v[i] = 0.0f;
    bool whole = false;  // one wave had all of it and stored it
#pragma unroll 4
    for (int w = wlo; w <= whi; ++w) {
      const int lo = w * U / W, hi = (w + 1) * U / W;
      if (max(lo, t * G) >= min(hi, (t + 1) * G)) continue;
      whole |= lo <= t * G && hi >= (t + 1) * G;
      const float* p = part + ((w * 2 + (lo >= t * G ? 0 : 1)) * 64 + lane) * AC;
#pragma unroll
      for (int i = 0; i < AC; ++i) v[i] += p[i];
    }
    if (!whole) store_tile(v, t);
  }
}

size_t lds_limit();

template <int QT, int RP, bool HL, int SRC = kTiled>
hipError_t launch_rp(RowsArgs a, int nt, hipStream_t stream) {
  using L = Lds<QT, RP, HL>;
  const int grid = std::min(nt, device_cus());
  a.tiles = nt / grid;
  a.extra = nt % grid;
  a.phase = a.g;
  void (*kernel)(RowsArgs) = rows_kernel<QT, RP, HL, SRC, false>;
  if constexpr (SRC == kTiled && HL) {
    if (L::bytes(a.g) > lds_limit()) {  // (one tile per workgroup, rows_supported)
      const int most = (int)(lds_limit() / (L::bytes(64) / 64)), pieces = (a.g + most - 1) / most;
      a.phase = (a.g + pieces - 1) / pieces;
      kernel = rows_kernel<QT, RP, HL, SRC, true>;
    }
  }
  const size_t lds = L::bytes(a.phase);
  const hipError_t e = allow_dynamic_lds((const void*)kernel, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * W), lds, stream, a);
  return hipGetLastError();
}

template <int QT>
hipError_t launch_qt(const RowsArgs& a, int nt, hipStream_t stream) {
  if (a.m <= 2) return launch_rp<QT, 2, true>(a, nt, stream);
  if (a.m <= 4) return launch_rp<QT, 4, true>(a, nt, stream);
  if (a.m <= 8) return launch_rp<QT, 8, true>(a, nt, stream);
  return launch_rp<QT, 16, false>(a, nt, stream);
}

template <int QT>
size_t lds_qt(int m, int g) {
  return m <= 2   ? Lds<QT, 2, true>::bytes(g)
         : m <= 4 ? Lds<QT, 4, true>::bytes(g)
         : m <= 8 ? Lds<QT, 8, true>::bytes(g)
                  : Lds<QT, 16, false>::bytes(g);
}

template <int QT, int SRC>
hipError_t launch_aos_src(const RowsArgs& a, int nt, hipStream_t stream) {
  if (a.m == 1) return launch_rp<QT, 1, true, SRC>(a, nt, stream);
  if (a.m == 2) return launch_rp<QT, 2, true, SRC>(a, nt, stream);
  if (a.m <= 4) return launch_rp<QT, 4, true, SRC>(a, nt, stream);
  return launch_rp<QT, 8, true, SRC>(a, nt, stream);
}

template <int QT>
hipError_t launch_aos_qt(const RowsArgs& a, int nt, hipStream_t stream) {
  const bool four = ((uintptr_t)a.qs & 3) == 0 && a.row_bytes % 4 == 0;
  return four ? launch_aos_src<QT, kAos4>(a, nt, stream) : launch_aos_src<QT, kAos2>(a, nt, stream);
}

size_t lds_limit() {
  static const size_t limit = [] {
    int dev = 0, bytes = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) !=
            hipSuccess ||
        bytes <= 0)
      return (size_t)64 * 1024;
    return (size_t)bytes;
  }();
  return limit;
}
}  // namespace

// Where streaming past a resident x beats a workgroup per tile (4 layers of a
// 7B model, us, workgroup per tile against this kernel for the shapes past
// the line): it starts later (all of x is converted before the first unit),
// so with few tiles the others win (288 and 224 tiles, 4 rows of q4_0: 206
// with them left to the GEMV, 217 without).
//  - 5..16 rows: more than 5/4 tiles per CU (8 rows of q4_0 578 -> 233, 16 rows
//    of q8_0 501 -> 338; at hidden 2048, FFN 5632, 704 tiles, 115 -> 109 and
//    191 -> 153).
//  - 2..4 rows, whose x is small: 128 units per CU (4 rows of q4_0 307 -> 206;
//    the 704-tile projections of hidden 2048 take 91.5 against 93.2).
bool rows_faster(int m, int n, int k) {
  const Geometry geo = geometry(n, k);
  if (m <= 4) return (int64_t)geo.nt * geo.g >= 128 * (int64_t)device_cus();
  return 4 * (int64_t)geo.nt > 5 * (int64_t)device_cus();
}

bool rows_supported(int type, int m, int n, int k) {
  if (m < 2 || m > 16 || k % 4 != 0) return false;
  // 32-bit buffer offsets into x (2^31 marks out of range)
  if ((uint64_t)m * k * 4 >= (1ull << 31)) return false;
  const int g = geometry(n, k).g;
  const size_t lds = type == MLQ_Q8_0   ? lds_qt<MLQ_Q8_0>(m, g)
                     : type == MLQ_Q4_0 ? lds_qt<MLQ_Q4_0>(m, g)
                                        : lds_qt<MLQ_Q4_1>(m, g);
  // Up to 8 rows on at most a tile per CU take a longer x in pieces (4 rows
  // of 4096 x 14336 q4_1, 4 layers with it 214 us, 202 in pieces; before that
  // these ran on fp16 activations; 9..16 rows lose: 16 of 4096 x 14336 q8_0
  // 288 with the fp16 copy, 302 in pieces).
  return lds <= lds_limit() || (m <= 8 && geometry(n, k).nt <= device_cus());
}

hipError_t launch_rows(const mlq_weight& w, const float* x, float* y, int m, hipStream_t stream,
                       const Epilogue& epi) {
  const Geometry geo = geometry(w.n, w.k);
  RowsArgs a = {};
  a.qs = (const uint8_t*)w.base + w.qs_off;
  a.d = (const uint8_t*)w.base + w.d_off;
  a.mn = w.type == MLQ_Q4_1 ? (const uint8_t*)w.base + w.m_off : nullptr;
  a.x = x;
  a.y = y;
  a.m = m;
  a.n = w.n;
  a.k = w.k;
  a.g = geo.g;
  a.ny = epi.act == kEpiSwiGLU ? w.n / 2 : w.n;
  a.epi = epi;
  switch (w.type) {
    case MLQ_Q8_0: return launch_qt<MLQ_Q8_0>(a, geo.nt, stream);
    case MLQ_Q4_0: return launch_qt<MLQ_Q4_0>(a, geo.nt, stream);
    default: return launch_qt<MLQ_Q4_1>(a, geo.nt, stream);
  }
}

// The row counts and lengths that need no workspace: rows of x padded to 1,
// 2, 4 or 8, at 144 bytes per 32 elements, beside 48 KiB in the LDS. (The
// fragments take less: 137 bytes at most.)
bool aos_gemv_supported(int type, int m, int n, int k) {
  if (m < 1 || m > 8 || n < 1 || k < 1) return false;
  if (type != MLQ_Q8_0 && type != MLQ_Q4_0 && type != MLQ_Q4_1) return false;
  const size_t rows = m == 1 ? 1 : m == 2 ? 2 : m <= 4 ? 4 : 8;
  const size_t nb = (size_t)((k + kQK - 1) / kQK);
  return ((rows * nb * 144 + 255) & ~(size_t)255) + 48 * 1024 <= lds_limit();
}

hipError_t launch_aos_gemv(int type, const void* aos, int n, int k, const float* x, float* y,
                           int m, hipStream_t stream) {
  if (!aos_gemv_supported(type, m, n, k) || ((uintptr_t)aos & 1) != 0) return hipErrorInvalidValue;
  const Geometry geo = geometry(n, k);
  RowsArgs a = {};
  a.qs = (const uint8_t*)aos;
  a.x = x;
  a.y = y;
  a.m = m;
  a.n = n;
  a.k = k;
  a.g = geo.g;
  a.nb = geo.nb;
  a.ny = n;
  a.row_bytes = geo.nb * (type == MLQ_Q8_0 ? 34 : type == MLQ_Q4_0 ? 18 : 20);
  switch (type) {
    case MLQ_Q8_0: return launch_aos_qt<MLQ_Q8_0>(a, geo.nt, stream);
    case MLQ_Q4_0: return launch_aos_qt<MLQ_Q4_0>(a, geo.nt, stream);
    default: return launch_aos_qt<MLQ_Q4_1>(a, geo.nt, stream);
  }
}

}  // namespace mlq
