// GEMV on raw GGUF blocks, many weight tiles or 3..8 rows of x:
// y[r][n] = sum_k W[n][k] x[r][k], every weight byte read from HBM once. (Few
// tiles and one or two rows: aos_gemv.hip, whose workgroups hold 8 weight rows
// each and stage x anew for them.)
//
// The arithmetic is the reference's per-element dequantization in fp32
// (src/quant.cc:477-503): every weight becomes the fp32 value d * q, d * (q - 8)
// (both exact) or d * q + m (rounded once) and meets the fp32 activation in an
// fp32 multiply-add. fp16 hi + lo pairs of x at the fp16 matrix rate are faster
// (one row of 18944 x 3584 q4_0 13.1 us) but lose what lies 2^-39 below the
// largest x of its 128 columns and infinite activations, and for q4_1 (block sums
// and min apart) round further than the kernel for few tiles.
//  - One workgroup of 8 waves per CU owns consecutive tiles of 16 rows; the
//    tiles' units (16 rows x 128 k) are split into equal consecutive runs, one
//    per wave, kDepth units in flight. Tiles that a wave covers whole it stores
//    itself, shared ones go through LDS and are added in wave order
//    (deterministic). x goes to LDS once per workgroup as it is, one barrier.
//    (16 waves: 19.2 us against 18.5 for 18944 x 3584 q8_0; one unit in flight
//    21.7, three 19.1.)
//  - A lane's weight row is lane % 16 and its quarter of each GGUF block (8
//    elements) lane / 16, for the loads, the decode and the products alike.
//  - 3..8 rows: v_mfma_f32_4x4x1_16b_f32, exact products and fp32 sums, whose 16
//    blocks are four rows of x against four weight rows each, the four quarters in
//    different blocks; a lane's accumulators are the rows of x. (16 x 16 x 4 would
//    do four times the work for four rows.) One or two rows: fp32 FMA (one row
//    15.8 us against 21.3 on the MFMA).
//  - Sums: chains of 16 products, two added per unit, units in order, then the
//    four quarters. Relative error against 64 bits, K = 3584 1.1e-7 (few-tile
//    kernel 1.5e-7), 18944 1.3e-7 (3.1e-7).
// Bound by VALU: two to three instructions a weight to make the fp32 values, one
// more per row; the row-strided 12-byte loads cost ~18 address cycles each. us,
// few-tile kernel -> this one, 18944 x 3584: one row q4_0 25.9 -> 15.6, q8_0 25.9 ->
// 19.4, two rows of q4_0 36.5 -> 18.8, four 89.0 -> 22.3; 8 rows of 18944 x 2080 q4_1
// 112 -> 22.0.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../mlq_layout.h"
#include "device_common.h"
#include "launch.h"

namespace mlq {
namespace {

constexpr int kWaves = 8;
constexpr int kDepth = 2;                 // units in flight per wave
constexpr uint32_t kPast = 0x80000000u;   // an offset past every buffer

struct AosArgs {
  const uint8_t* w;  // GGUF blocks, row n at w + n * row_bytes
  const float* x;    // [m][k]
  float* y;          // [m][n]
  int m, n, k, nb, g;
  int row_bytes;
  int tiles, extra;  // tiles per workgroup; the first `extra` have one more
};

template <int QT>
__device__ __host__ constexpr int aos_block_bytes() {
  return QT == MLQ_Q8_0 ? 34 : QT == MLQ_Q4_0 ? 18 : 20;
}

// A lane reads, of each of the unit's four blocks, a window from the 4-byte
// boundary at or below the block (q8_0: plus 8 quarter, q4: plus 8 (quarter %
// 2)): its 8 code bytes lie 2 or 4 bytes behind the block's phase in it, and in
// quarter 0 (q4: also 2) the scale (and min) ahead of them. Windows of 12 bytes
// where every row and the base start on 4-byte boundaries (FOUR: the phase of
// block b is then known), else of 16; what passes the 4-byte boundary behind the
// workgroup's rows reads as zero.
struct Unit {
  uint4 v[4];
};

// 8 code bytes (q4: already one nibble each) -> q (q4_0: q - 8) in fp32, exact.
template <int QT>
__device__ __forceinline__ void codes_f32(uint32_t c0, uint32_t c1, float (&q)[8]) {
  if constexpr (QT == MLQ_Q4_0) {  // n - 8 as a signed byte
    c0 = (c0 + 0x78787878u) ^ 0x80808080u;
    c1 = (c1 + 0x78787878u) ^ 0x80808080u;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t b = (j < 4 ? c0 : c1) >> (8 * (j & 3));
    q[j] = QT == MLQ_Q4_1 ? (float)(uint8_t)b : (float)(int8_t)b;
  }
}

template <int QT, int MR, bool FOUR>
__global__ __launch_bounds__(64 * kWaves) void aos_tiles_kernel(AosArgs a) {
  constexpr int W = kWaves, BS = aos_block_bytes<QT>();
  constexpr int NA = MR == 8 ? 2 : 1;     // accumulator quads (4 rows of x each)
  constexpr int XR = MR < 4 ? MR : 4;     // rows of x of a quad that exist
  constexpr int kPartTile = 64 * NA;      // (rows past XR are never written nor stored)
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  f4_t* xs = (f4_t*)smem;                 // [k / 4][MR], four columns each
  // at the end: two partial tiles per wave, [row of x][weight row]
  float* part = (float*)(xs + a.g * (kGroupK / 4) * MR);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.g;

  // this workgroup's tiles and this wave's run of their units
  const int T = a.tiles + ((int)blockIdx.x < a.extra ? 1 : 0);
  const int t0 = (int)blockIdx.x * a.tiles + min((int)blockIdx.x, a.extra);
  const int U = T * G;
  const int u0 = wave * U / W, u1 = (wave + 1) * U / W, n = u1 - u0;
  const int first = wave * T / W;  // = u0 / G
  const int rows0 = t0 * kTileRows;
  const uint8_t* base = a.w + (size_t)rows0 * a.row_bytes;
  const int lead = FOUR ? 0 : (int)((uintptr_t)base & 3);
  const rsrc_t rw = make_rsrc(
      base - lead,
      (uint32_t)((lead + (size_t)min(T * kTileRows, a.n - rows0) * a.row_bytes + 3) & ~(size_t)3));
  const uint32_t arow = (uint32_t)(lead + (lane & 15) * a.row_bytes);
  const uint32_t aq = QT == MLQ_Q8_0 ? 8u * (lane >> 4) : 8u * ((lane >> 4) & 1);

  int ltile = first, lg = u0 - first * G;  // the next unit to load
  auto load = [&](Unit& s) __attribute__((always_inline)) {
    const uint32_t su = (uint32_t)(ltile * kTileRows * a.row_bytes + lg * (kGroupBlocks * BS));
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t at = arow + (uint32_t)(b * BS);
      const int off = (int)((at & ~3u) + aq);
      if constexpr (FOUR) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(rw, off, (int)su, 0);
        s.v[b] = make_uint4(v[0], v[1], v[2], 0u);
      } else {
        s.v[b] = buf_load16(rw, (uint32_t)off, su);
      }
    }
    if (++lg == G) {
      lg = 0;
      ++ltile;
    }
  };
  // block b of a unit of group g as fp32 weights
  auto weights = [&](const Unit& s, int b, int g, float (&w)[8]) __attribute__((always_inline)) {
    uint4 v = s.v[b];
    uint32_t head, c0, c1;  // the block's first bytes (scale, min); the lane's codes
    if constexpr (FOUR) {
      const bool odd = QT != MLQ_Q4_1 && (b & 1) != 0;  // 34 b and 18 b bytes: phase 2
      head = odd ? v.x >> 16 : v.x;
      if constexpr (QT == MLQ_Q4_1) {
        c0 = v.y;
        c1 = v.z;
      } else {
        c0 = odd ? v.y : __builtin_amdgcn_alignbit(v.y, v.x, 16);
        c1 = odd ? v.z : __builtin_amdgcn_alignbit(v.z, v.y, 16);
      }
    } else {
      const uint32_t phase = (arow + (uint32_t)(b * BS)) & 3u;
      head = __builtin_amdgcn_alignbyte(v.y, v.x, phase);
      const uint32_t p1 = __builtin_amdgcn_alignbyte(v.z, v.y, phase);
      const uint32_t p2 = __builtin_amdgcn_alignbyte(v.w, v.z, phase);
      c0 = QT == MLQ_Q4_1 ? p1 : __builtin_amdgcn_alignbit(p1, head, 16);
      c1 = QT == MLQ_Q4_1 ? p2 : __builtin_amdgcn_alignbit(p2, p1, 16);
    }
    // the scale sits in quarter 0 (q4: and 2): to the row's other quarters
    float h = xor16_pair(__builtin_bit_cast(float, head)).lo;
    if constexpr (QT == MLQ_Q8_0) h = xor32_pair(h).lo;
    const uint32_t bits = __builtin_bit_cast(uint32_t, h);
    float d = half_bits_to_float((uint16_t)bits);
    float mn = QT == MLQ_Q4_1 ? half_bits_to_float((uint16_t)(bits >> 16)) : 0.0f;
    if (g * kGroupBlocks + b >= a.nb) d = mn = 0.0f;  // past the row: the next row's blocks
    if constexpr (QT != MLQ_Q8_0) {
      const uint32_t sh = 4u * (uint32_t)(lane >> 5);  // elements 16..31: high nibbles
      c0 = (c0 >> sh) & 0x0F0F0F0Fu;
      c1 = (c1 >> sh) & 0x0F0F0F0Fu;
    }
    codes_f32<QT>(c0, c1, w);
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = QT == MLQ_Q4_1 ? __builtin_fmaf(d, w[j], mn) : d * w[j];
  };

  // ---- x into LDS (zeros past m and past k), requested ahead of the weights
  const rsrc_t rx = make_rsrc(a.x, (uint32_t)((size_t)a.m * a.k * 4));
  const bool vec = (a.k & 3) == 0;
  const int quads = G * (kGroupK / 4);
  auto load_x = [&](f4_t (&v)[MR], int c) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < MR; ++r) {
      const uint32_t off = (uint32_t)(r * a.k + 4 * c) * 4u;
      if (vec) {
        v[r] = __builtin_bit_cast(f4_t, buf_load16(rx, r < a.m && 4 * c < a.k ? off : kPast, 0));
      } else {  // the row's end may fall inside a quad
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[r][i] = __builtin_bit_cast(
              float, buf_load4(rx, r < a.m && 4 * c + i < a.k ? off + 4u * i : kPast, 0));
      }
    }
  };
  auto store_x = [&](const f4_t (&v)[MR], int c) __attribute__((always_inline)) {
    if (c >= quads) return;
#pragma unroll
    for (int r = 0; r < MR; ++r) xs[c * MR + r] = v[r];
  };
  Unit ring[kDepth];
  f4_t xv[MR];
  load_x(xv, threadIdx.x);
  if (n >= kDepth) {
#pragma unroll
    for (int i = 0; i < kDepth; ++i) load(ring[i]);
  } else if (n > 0) {
    load(ring[0]);
  }
  store_x(xv, threadIdx.x);
  for (int c = 64 * W; c < quads; c += 64 * W) {
    load_x(xv, c + threadIdx.x);
    store_x(xv, c + threadIdx.x);
  }
  __syncthreads();

  // ---- the wave's units
  f4_t acc[NA], head[NA];  // running; the run's first tile if not whole
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i] = head[i] = (f4_t){0.f, 0.f, 0.f, 0.f};
  const f4_t* xl = xs + 2 * (lane >> 4) * MR + (MR <= 2 ? 0 : lane & 3);
  int tile = first, g = u0 - first * G;
  // v[r / 4][r % 4] (row r of x, weight row lane % 16) over the four quarters
  auto quarters = [&](f4_t (&v)[NA]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int r = 0; r < XR; ++r) v[i][r] = xor32_sum(xor16_sum(v[i][r]));
  };
  // output of row 4 i + lane / 16 of x and weight row lane % 16 of tile t
  auto store = [&](float v, int i, int t) __attribute__((always_inline)) {
    const int row = (t0 + t) * kTileRows + (lane & 15), r = 4 * i + (lane >> 4);
    if (row < a.n && r < a.m) a.y[(size_t)r * a.n + row] = v;
  };
  auto flush = [&]() __attribute__((always_inline)) {
    quarters(acc);
    if (tile * G >= u0 && (tile + 1) * G <= u1) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const f4_t v = acc[i];
        const int r = lane >> 4;
        store(XR == 1 || r == 0 ? v[0] : XR == 2 || r == 1 ? v[1] : r == 2 ? v[2] : v[3], i, tile);
      }
    } else {  // (the run's last tile stays in acc)
#pragma unroll
      for (int i = 0; i < NA; ++i) head[i] = acc[i];
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[i] = (f4_t){0.f, 0.f, 0.f, 0.f};
  };
  auto run = [&](const Unit& s) __attribute__((always_inline)) {
    f4_t c[NA][2];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float w[8];
      weights(s, b, g, w);
      const f4_t* xp = xl + (g * 32 + b * 8) * MR;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        f4_t& ch = c[i][b >> 1];
        if ((b & 1) == 0) ch = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (MR <= 2) {
#pragma unroll
            for (int r = 0; r < MR; ++r) {
              const f4_t x4 = xp[h * MR + r];
#pragma unroll
              for (int j = 0; j < 4; ++j) ch[r] = __builtin_fmaf(x4[j], w[4 * h + j], ch[r]);
            }
            continue;
          }
          const f4_t x4 = xp[h * MR + 4 * i];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            ch = __builtin_amdgcn_mfma_f32_4x4x1f32(x4[j], w[4 * h + j], ch, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int r = 0; r < XR; ++r) acc[i][r] += c[i][0][r] + c[i][1][r];
    if (++g == G) {
      flush();
      g = 0;
      ++tile;
    }
  };
  // No load past the run's end: the 16 waves' would cost a microsecond of
  // address cycles.
  int j = 0;
  for (; j + 2 * kDepth <= n; j += kDepth) {
#pragma unroll
    for (int i = 0; i < kDepth; ++i) {
      run(ring[i]);
      load(ring[i]);
    }
  }
  const int left = n - j;  // fewer than 2 kDepth, kDepth of them loaded
#pragma unroll
  for (int i = 0; i < kDepth; ++i) {
    if (i < left) run(ring[i]);
    if (i + kDepth < left) load(ring[i]);
  }
#pragma unroll
  for (int i = 0; i < kDepth; ++i)
    if (i + kDepth < left) run(ring[i]);

  // ---- partial tiles: a run's first one (head, or acc if the run ends inside
  // it) in slot 0, its last in slot 1; added in wave order
  quarters(acc);
  if (lane < 16) {
    float* p = part + wave * 2 * kPartTile + lane;
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int r = 0; r < XR; ++r) {
        p[(4 * i + r) * 16] = tile == first ? acc[i][r] : head[i][r];
        p[kPartTile + (4 * i + r) * 16] = acc[i][r];
      }
  }
  __syncthreads();
  for (int t = wave; t < T; t += W) {
    float v[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) v[i] = 0.0f;
    bool whole = false;  // one wave had all of it and stored it
    // (over all waves: the reads are in flight together, and finding the first
    // and last one that met the tile takes two divisions)
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int lo = w * U / W, hi = (w + 1) * U / W;
      const bool met = max(lo, t * G) < min(hi, (t + 1) * G);
      whole |= lo <= t * G && hi >= (t + 1) * G;
      const float* p = part + (w * 2 + (lo >= t * G ? 0 : 1)) * kPartTile + lane;
#pragma unroll
      for (int i = 0; i < NA; ++i) v[i] += met ? p[64 * i] : 0.0f;
    }
    if (!whole) {
#pragma unroll
      for (int i = 0; i < NA; ++i) store(v[i], i, t);
    }
  }
}

template <int QT, int MR, bool FOUR>
hipError_t launch_mr(const AosArgs& a, int grid, hipStream_t stream) {
  constexpr size_t kParts = (size_t)kWaves * 2 * 64 * (MR == 8 ? 2 : 1) * sizeof(float);
  const size_t lds = (size_t)a.g * kGroupK * MR * sizeof(float) + kParts;
  const auto kernel = aos_tiles_kernel<QT, MR, FOUR>;
  const hipError_t e = allow_dynamic_lds((const void*)kernel, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kWaves), lds, stream, a);
  return hipGetLastError();
}

template <int QT, bool FOUR>
hipError_t launch_rows_of(const AosArgs& a, int grid, hipStream_t stream) {
  if (a.m == 1) return launch_mr<QT, 1, FOUR>(a, grid, stream);
  if (a.m == 2) return launch_mr<QT, 2, FOUR>(a, grid, stream);
  if (a.m <= 4) return launch_mr<QT, 4, FOUR>(a, grid, stream);
  return launch_mr<QT, 8, FOUR>(a, grid, stream);
}

template <int QT>
hipError_t launch_typed(const AosArgs& a, int grid, hipStream_t stream) {
  const bool four = ((uintptr_t)a.w & 3) == 0 && a.row_bytes % 4 == 0;
  return four ? launch_rows_of<QT, true>(a, grid, stream)
              : launch_rows_of<QT, false>(a, grid, stream);
}

}  // namespace

hipError_t launch_aos_tiles(int type, const void* aos, int n, int k, const float* x, float* y,
                            int m, hipStream_t stream) {
  const Geometry geo = geometry(n, k);
  const int grid = std::min(geo.nt, device_cus());
  AosArgs a = {};
  a.w = (const uint8_t*)aos;
  a.x = x;
  a.y = y;
  a.m = m;
  a.n = n;
  a.k = k;
  a.nb = geo.nb;
  a.g = geo.g;
  a.tiles = geo.nt / grid;
  a.extra = geo.nt % grid;
  switch (type) {
    case MLQ_Q8_0: a.row_bytes = geo.nb * 34; return launch_typed<MLQ_Q8_0>(a, grid, stream);
    case MLQ_Q4_0: a.row_bytes = geo.nb * 18; return launch_typed<MLQ_Q4_0>(a, grid, stream);
    default: a.row_bytes = geo.nb * 20; return launch_typed<MLQ_Q4_1>(a, grid, stream);
  }
}

}  // namespace mlq
