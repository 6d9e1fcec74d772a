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
//    contiguous byte range, D units in flight in a register ring. Tiles
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
//  - Up to 8 rows longer than the LDS on at most a tile per CU (down
//    projections): x in pieces, a wave's sums staying in registers.
//  - Each (row, 128-k group) is scaled by its own power of two (the group's
//    largest |x| into [2^14, 2^15)) before it becomes fp16, and the group's
//    sums are scaled back in fp32: any finite x, and no dependence on how
//    units are dealt to waves.
#include <hip/hip_runtime.h>

#include <algorithm>

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

struct RowsArgs {
  const uint8_t* qs;
  const uint8_t* d;
  const uint8_t* mn;
  const float* x;
  float* y;
  int m, n, k, g, ny;
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

// One unit's weights as loaded by a lane.
struct Unit {
  uint4 q, q2;
  uint2 d, m;
};

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
template <int QT, int RP, bool HL, bool PH>
__global__ __launch_bounds__(64 * W) void rows_kernel(RowsArgs a) {
  using L = Lds<QT, RP, HL>;
  constexpr int MR = L::kRows;
  constexpr int LPR = 64 / RP;         // lanes per row of a load
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

  constexpr uint32_t QB = QT == MLQ_Q8_0 ? 2048u : 1024u;
  size_t unit0 = (size_t)t0 * G + u0;
  rsrc_t rq = make_rsrc(a.qs + unit0 * QB, (uint32_t)n * QB);
  rsrc_t rd = make_rsrc(a.d + unit0 * 128, (uint32_t)n * 128u);
  rsrc_t rm = QT == MLQ_Q4_1 ? make_rsrc(a.mn + unit0 * 128, (uint32_t)n * 128u) : rd;
  const uint32_t qoff = (uint32_t)lane * 16u, soff = (uint32_t)(lane & 15) * 8u;
  const int first = wave * T / W;  // = u0 / G
  // unit j of the run, in order (zeros past it)
  auto load = [&](Unit& s, int j) __attribute__((always_inline)) {
    s.q = buf_load16_stream(rq, qoff, (uint32_t)j * QB);
    if (QT == MLQ_Q8_0) s.q2 = buf_load16_stream(rq, qoff, (uint32_t)j * QB + 1024u);
    s.d = buf_load8(rd, soff, (uint32_t)j * 128u);
    if (QT == MLQ_Q4_1) s.m = buf_load8(rm, soff, (uint32_t)j * 128u);
  };

  // ---- x -> fragments. Lane group rho of LPR lanes reads row rho of a 128-k
  // group, lane q of it the float4s q, q + LPR, ...; rows past m and columns
  // past k read as zero through offsets past the buffer.
  const rsrc_t rx = make_rsrc(a.x, (uint32_t)((size_t)a.m * a.k * 4));
  const int rho = lane / LPR, q = lane % LPR;
  struct Batch {
    float4 v[BG][NL];
  };
  auto load_x = [&](Batch& b, int g0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BG; ++i)
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int col = (g0 + i) * kGroupK + 4 * (j * LPR + q);
        const uint32_t off = rho < a.m && col < a.k ? (uint32_t)(rho * a.k + col) * 4u : kPast;
        b.v[i][j] = __builtin_bit_cast(float4, buf_load16(rx, off, 0));
      }
  };
  auto stage = [&](const Batch& b, int g0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BG; ++i) {
      const int g = g0 + i;
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
  Unit ring[D];
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
  auto run = [&](const Unit& s) __attribute__((always_inline)) {
    const uint8_t* af = af0 + (size_t)g * L::kGroup;
    if constexpr (HL) {
      float t[2] = {0.0f, 0.0f};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const h8_t av = __builtin_bit_cast(h8_t, *(const uint4*)(af + b * 4 * MR * 16));
        const h8_t bv = decode_exact<QT>(s.q, s.q2, b);
        const float d = (float)half_at(s.d, b);
        const f4_t z = {0.f, 0.f, 0.f, 0.f};
        const f4_t p = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, z, 0, 0, 0);
        t[0] += d * (p[0] + p[1]);
        t[1] += d * (p[2] + p[3]);
        if constexpr (SUMS) {
          const float mb = (float)half_at(s.m, b);
          const float2 sx = *(const float2*)(sums + (g * kGroupBlocks + b) * RP + r0);
          t[0] += mb * sx.x;
          t[1] += mb * sx.y;
        }
      }
      const float2 sc = *(const float2*)(scale + g * RP + r0);
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

template <int QT, int RP, bool HL>
hipError_t launch_rp(RowsArgs a, int nt, hipStream_t stream) {
  using L = Lds<QT, RP, HL>;
  const int grid = std::min(nt, device_cus());
  a.tiles = nt / grid;
  a.extra = nt % grid;
  a.phase = a.g;
  void (*kernel)(RowsArgs) = rows_kernel<QT, RP, HL, false>;
  if constexpr (HL) {
    if (L::bytes(a.g) > lds_limit()) {  // (one tile per workgroup, rows_supported)
      const int most = (int)(lds_limit() / (L::bytes(64) / 64)), pieces = (a.g + most - 1) / most;
      a.phase = (a.g + pieces - 1) / pieces;
      kernel = rows_kernel<QT, RP, HL, true>;
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

// Where streaming past a resident x beats a workgroup per tile. It starts later
// (all of x is converted before the first unit), so a CU needs work enough to make
// up for that. Both measured for 512..152064 weight rows and K 256..18944 (time
// here over the workgroup per tile's, q8_0 / q4_0 / q4_1):
//  - 2..4 rows, whose x is small: 128 units per CU (4 rows 0.7 to 1.0 there, of
//    28672 x 4096 0.78 / 0.65 / 0.51). Not two rows of at most 8 groups (152064 x
//    896 1.20 / 1.00 / 1.13), nor two or three of q8_0 where the GEMV's 16 waves
//    share K evenly (two rows of 8192 x 8192 1.13, 65536 x 2048 1.22; 18944 x 3584
//    0.94, 13824 x 5120 0.72).
//  - 5..8 rows: more than 5/4 tiles per CU and 56 units per CU (6 rows 48, more
//    40): 5 rows of 20480 x 1024, 40 units, 1.15 / 1.17 / 1.02, of 29000 x 896, 50,
//    1.04 / 0.98 / 0.90; 8 rows of 8192 x 2048, 32, 1.07 / 1.00 / 0.89, of 14336 x
//    1536, 42, 0.80 / 0.74 / 0.66, of 28672 x 4096 0.46 / 0.34 / 0.45.
//  - 9..16 rows: more than 5/4 tiles per CU (16 of 5184 x 256 0.56 / 0.74 / 0.54, of
//    18944 x 3584 0.50 / 0.59 / 0.49); in q4_0, whose skinny kernel runs two tiles per
//    CU in one round, more than two of them past K 2048 (16 of 6144 x 4096 1.18, x
//    2048 0.85, 11008 x 4096 0.74).
bool rows_faster(int type, int m, int n, int k) {
  const Geometry geo = geometry(n, k);
  const int64_t cus = device_cus(), units = (int64_t)geo.nt * geo.g;
  if (m <= 4)
    return units >= 128 * cus && !(m == 2 && geo.g <= 8) &&
           !(m <= 3 && type == MLQ_Q8_0 && geo.g % 16 == 0);
  if (4 * (int64_t)geo.nt <= 5 * cus) return false;
  if (m <= 8) return units >= std::max(40, 8 * (12 - m)) * cus;
  return type != MLQ_Q4_0 || geo.nt > 2 * cus || geo.g <= 16;
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

}  // namespace mlq
