// F32 Linear: y[r][row] = sum_k x[r][k] * W[row][k] + epilogue, W fp32
// [n][k] row-major (cudaLinearDeviceInput, src/cuda_matmul.cc:205-241, which
// calls cuBLAS Sgemm; also the F32 arm of forwardLinearDevice,
// src/forward.cc:206-209). The reference's F32 weights are the unquantized
// model's projections and the tied lm_head.
//
// Up to 8 rows of x: HBM-streaming GEMV. One workgroup (4 waves) per 16-row
// tile, 4 rows per wave; lanes stride K with float4 loads, so every W element
// is read once (non-temporal: W is streamed, x stays cached). Under the
// SwiGLU epilogue a wave takes two gate rows and their two up rows (rows
// 16t+j and 16t+8+j of the interleaved tile), so both operands of an output
// meet in one wave.
//
// More rows: fp32 MFMA (v_mfma_f32_*_f32: exact fp32 products, fp32
// accumulation). In passes of 8 rows the GEMV reads W m/8 times and issues
// 2 VALU lanes' worth of work per product pair: 200 x 4096 x 4096 took
// 977 us (6.9 TFLOP/s), bound by FMA issue and by 25 sweeps over W. Two
// kernels, chosen by the number of 64 x 64 output tiles (linear_f32_tiled):
//  - gemm_f32_kernel: 64 x 64 tiles, x and W staged through LDS in 32-k
//    stages; bound by the fp32 matrix rate (128 multiply-adds per clock and
//    CU).
//  - skinny_f32_kernel: few tiles; a workgroup per 16 W rows and up to 64
//    rows of x, its 8 waves splitting K, fragments straight from memory;
//    bound by the reads of W (and of x from L2).
// An MFMA adds to its accumulator in k order, so one chain over all of K
// would round K times (about 1.5e-6 relative at K = 4096, where the GEMV's 64
// interleaved lanes and their tree give 1.6e-7). Both kernels therefore run
// short chains from zero and add them as trees: of 4 k, as the GEMV's lanes at
// K = 256; in the tiled kernel of 16 k from K = 1536 and of 32 k from K = 3072,
// where the GEMV's own chains have grown past them (every chain that is cut
// costs 16 additions per lane: 200 x 4096 x 4096 takes 91 us in chains of 8).
// Measured error against 64 bits (normal inputs, 4096 W rows), GEMV against tiled
// and skinny: K = 64 6.77e-8, 6.76e-8, 6.77e-8; 256 7.79e-8, 7.79e-8, 7.80e-8; 512
// 8.57e-8, 8.36e-8, 8.24e-8; 1536 1.12e-7, 1.03e-7, 9.2e-8; 3072 1.42e-7, 1.27e-7,
// 1.03e-7; 4096 1.59e-7, 1.30e-7, 1.10e-7; 15000 2.83e-7, 1.57e-7, 1.62e-7 (chains of
// 32 k modelled 1.2e-7 at 256 and 512).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace mlq {
namespace {

constexpr int kF32MaxRows = 8;

struct F32Args {
  const float* w;
  const float* x;
  float* y;
  int m, n, k, ny;
  Epilogue epi;
};

template <int MR, bool VEC>
__global__ __launch_bounds__(256) void linear_f32_kernel(F32Args a) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const bool glu = a.epi.act == kEpiSwiGLU;
  int rows[4];
  const float* wr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int off = glu ? (i < 2 ? 2 * wave + i : 8 + 2 * wave + (i - 2)) : 4 * wave + i;
    rows[i] = 16 * (int)blockIdx.x + off;
    wr[i] = a.w + (size_t)min(rows[i], a.n - 1) * a.k;
  }
  float acc[4][MR];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < MR; ++r) acc[i][r] = 0.0f;

  if constexpr (VEC) {
#pragma unroll 2
    for (int kk = lane * 4; kk < a.k; kk += 256) {
      f4_t wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) wv[i] = __builtin_nontemporal_load((const f4_t*)(wr[i] + kk));
#pragma unroll
      for (int r = 0; r < MR; ++r) {
        const f4_t xv = *(const f4_t*)(a.x + (size_t)r * a.k + kk);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[i][r] += wv[i].x * xv.x;
          acc[i][r] += wv[i].y * xv.y;
          acc[i][r] += wv[i].z * xv.z;
          acc[i][r] += wv[i].w * xv.w;
        }
      }
    }
  } else {
    for (int kk = lane; kk < a.k; kk += 64) {
      float wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) wv[i] = wr[i][kk];
#pragma unroll
      for (int r = 0; r < MR; ++r) {
        const float xv = a.x[(size_t)r * a.k + kk];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][r] += wv[i] * xv;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < MR; ++r) acc[i][r] = wave_sum(acc[i][r]);
  if (lane != 0) return;
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    float* yr = a.y + (size_t)r * a.ny;
    if (glu) {
      // n % 16 == 0 under SwiGLU, so every row of the tile exists
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float g = add_bias(a.epi, acc[i][r], rows[i]);
        const float u = add_bias(a.epi, acc[i + 2][r], rows[i + 2]);
        yr[glu_col(rows[i])] = silu_f(g) * u;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (rows[i] < a.n) yr[rows[i]] = add_bias(a.epi, acc[i][r], rows[i]);
    }
  }
}

typedef float f16v_t __attribute__((ext_vector_type(16)));

// Four consecutive floats of a row at column col (columns at or past `end`
// read as zero; rows past the buffer range too). VEC: the row starts on a
// 16-byte boundary and end % 4 == 0.
constexpr uint32_t kPastRange = 0x80000000u;
template <bool VEC>
__device__ __forceinline__ f4_t load_row4(rsrc_t r, uint32_t row_off, int col, int end) {
  if constexpr (VEC) {
    const uint32_t off = col < end ? row_off + (uint32_t)col * 4 : kPastRange;
    return __builtin_bit_cast(f4_t, buf_load16(r, off, 0));
  } else {
    f4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t off = col + i < end ? row_off + (uint32_t)(col + i) * 4 : kPastRange;
      v[i] = __builtin_bit_cast(float, buf_load4(r, off, 0));
    }
    return v;
  }
}

// ---- 64 x 64 output tiles ---------------------------------------------------
// KS groups of four waves; group ks takes the ks-th part of K, its waves the
// tile's four 32 x 32 quarters (v_mfma_f32_32x32x2_f32). A stage is 32 k of 64
// x rows and 64 W rows, 16-byte loads of 128 contiguous bytes per row, two
// stages ahead in registers (one stage's MFMAs, ~0.5 us, are shorter than a
// trip to HBM: 95 us with one at 200 x 4096 x 4096, 77 with two), two LDS
// slabs, one barrier per stage. Lane half h
// of a fragment reads k = 8j + 4h .. +3 as one 16-byte LDS read and feeds
// four MFMAs, whose k pair is (8j + i, 8j + 4 + i): any pairing covers the
// sum. Rows are padded to 36 floats, which spreads those reads over the banks.
constexpr int kTile = 64, kStageK = 32, kLdsRow = kStageK + 4;

template <int KS>
constexpr int gemm_f32_lds() { return KS * 2 * 2 * kTile * kLdsRow * (int)sizeof(float); }

// CH: k of a chain (4, 16 or 32).
template <int KS, bool VEC, int CH>
__global__ __launch_bounds__(256 * KS) void gemm_f32_kernel(F32Args a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
  // Hardware places workgroup b on XCD b % 8: each XCD takes a contiguous
  // run of tiles, row tiles fastest, so the row tiles of one W tile share
  // its L2.
  const int mt = (a.m + kTile - 1) / kTile, nt = (a.n + kTile - 1) / kTile;
  const int per = (mt * nt + 7) / 8;
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= mt * nt) return;
  const int m0 = (tile % mt) * kTile, n0 = (tile / mt) * kTile;
  const rsrc_t rx = make_rsrc(a.x + (size_t)m0 * a.k,
                              (uint32_t)((size_t)min(kTile, a.m - m0) * a.k * 4));
  const rsrc_t rw = make_rsrc(a.w + (size_t)n0 * a.k,
                              (uint32_t)((size_t)min(kTile, a.n - n0) * a.k * 4));
  const int stages = (a.k + kStageK - 1) / kStageK;
  const int per_ks = (stages + KS - 1) / KS;
  const int k0 = ks * per_ks * kStageK;
  const int kend = min(a.k, k0 + per_ks * kStageK);

  const int t = tid & 255;
  const int lrow = t >> 3, lcol = 4 * (t & 7);
  float* slab = smem + ks * 2 * 2 * kTile * kLdsRow;
  f4_t even[4], odd[4];
  auto load = [&](f4_t (&pre)[4], int s) __attribute__((always_inline)) {
    const int col = k0 + s * kStageK + lcol;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      pre[i] = load_row4<VEC>(i < 2 ? rx : rw,
                              (uint32_t)(((i & 1) * 32 + lrow) * a.k) * 4, col, kend);
  };
  auto store = [&](const f4_t (&pre)[4], int buf) __attribute__((always_inline)) {
    float* p = slab + buf * 2 * kTile * kLdsRow;
#pragma unroll
    for (int i = 0; i < 4; ++i) *(f4_t*)(p + (i * 32 + lrow) * kLdsRow + lcol) = pre[i];
  };
  f16v_t sum = {}, mid = {};
  const int frag = (lane & 31) * kLdsRow + 4 * (lane >> 5);
  const int arow = 32 * wm * kLdsRow + frag, brow = (kTile + 32 * wn) * kLdsRow + frag;
  auto run = [&](int buf) __attribute__((always_inline)) {
    const float* p = slab + buf * 2 * kTile * kLdsRow;
    // MFMA u takes two k: the chain it belongs to starts every CH / 2
    f4_t av, bv;
    f16v_t c[32 / CH];
#pragma unroll
    for (int u = 0; u < kStageK / 2; ++u) {
      if (u % 4 == 0) {
        av = *(const f4_t*)(p + arow + 2 * u);
        bv = *(const f4_t*)(p + brow + 2 * u);
      }
      f16v_t& in = c[u / (CH / 2)];
      if (u % (CH / 2) == 0) in = (f16v_t){};
      in = __builtin_amdgcn_mfma_f32_32x32x2f32(av[u % 4], bv[u % 4], in, 0, 0, 0);
    }
    if constexpr (CH == 4) {
      c[0] = (c[0] + c[1]) + (c[2] + c[3]);
      c[1] = (c[4] + c[5]) + (c[6] + c[7]);
    }
    if constexpr (CH < 32) c[0] += c[1];
    return c[0];
  };
  // stages past the part's end (an odd count, or the last prefetches) load
  // zeros and add nothing
  load(even, 0);
  load(odd, 1);
  store(even, 0);
  for (int s = 0; s < per_ks; s += 2) {
    load(even, s + 2);
    __syncthreads();
    f16v_t two = run(0);
    store(odd, 1);
    load(odd, s + 3);
    __syncthreads();
    two += run(1);
    store(even, 0);
    mid += two;
    if ((s & 6) == 6) {
      sum += mid;
      mid = (f16v_t){};
    }
  }
  sum += mid;
  // K parts in order through LDS: 32 x 32 floats per wave, lane-contiguous
  if constexpr (KS > 1) {
    __syncthreads();
    float* part = smem + wave * 1024;
#pragma unroll
    for (int i = 0; i < 16; ++i) part[i * 64 + lane] = sum[i];
    __syncthreads();
    if (ks != 0) return;
#pragma unroll
    for (int q = 1; q < KS; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[i] += smem[(wave + 4 * q) * 1024 + i * 64 + lane];
  }
  // lane holds row 8 (i / 4) + 4 (lane / 32) + i % 4 of column lane % 32
  const int row = n0 + 32 * wn + (lane & 31);
  const int r0 = m0 + 32 * wm + 4 * (lane >> 5);
  if (a.epi.act == kEpiSwiGLU) {
    // gate lanes (bit 3 clear) and their up lanes 8 further on
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float v = row < a.n ? add_bias(a.epi, sum[i], row) : 0.0f;
      const float u = dpp<kDppRor8>(v);
      const int r = r0 + 8 * (i >> 2) + (i & 3);
      if ((lane & 8) == 0 && row < a.n && r < a.m)
        a.y[(size_t)r * a.ny + glu_col(row)] = silu_f(v) * u;
    }
  } else if (row < a.n) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = r0 + 8 * (i >> 2) + (i & 3);
      if (r < a.m) a.y[(size_t)r * a.n + row] = add_bias(a.epi, sum[i], row);
    }
  }
}

// ---- few tiles: 16 W rows x up to 16 MB rows of x per workgroup ---------------
// v_mfma_f32_16x16x4_f32: lane l reads row l % 16 at k = 4 (l / 16) .. +3 of a
// 16-k step as one 16-byte load (16 rows x 64 contiguous bytes) and feeds four
// MFMAs. A wave has two blocks of 32 k in flight.
constexpr int kSkinnyF32Waves = 8;

template <int MB, bool VEC>
__global__ __launch_bounds__(64 * kSkinnyF32Waves) void skinny_f32_kernel(F32Args a) {
  __shared__ float part[kSkinnyF32Waves * 16 * MB * 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (int)blockIdx.x * 16, m0 = (int)blockIdx.y * 16 * MB;
  const int mr = min(16 * MB, a.m - m0);
  const rsrc_t rx = make_rsrc(a.x + (size_t)m0 * a.k, (uint32_t)((size_t)mr * a.k * 4));
  const rsrc_t rw = make_rsrc(a.w + (size_t)n0 * a.k,
                              (uint32_t)((size_t)min(16, a.n - n0) * a.k * 4));
  const int blocks = (a.k + 31) / 32;
  const int per = (blocks + kSkinnyF32Waves - 1) / kSkinnyF32Waves;
  const int k0 = wave * per * 32, kend = min(a.k, k0 + per * 32);
  const uint32_t roff = (uint32_t)((lane & 15) * a.k) * 4;
  const int lcol = 4 * (lane >> 4);
  struct Block {
    f4_t w[2], x[MB][2];
  };
  auto load = [&](Block& b, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int col = k0 + 32 * i + 16 * h + lcol;
      b.w[h] = load_row4<VEC>(rw, roff, col, kend);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        b.x[mb][h] = load_row4<VEC>(rx, roff + (uint32_t)(16 * mb * a.k) * 4, col, kend);
    }
  };
  f4_t acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = (f4_t){0.f, 0.f, 0.f, 0.f};
  auto run = [&](const Block& b) __attribute__((always_inline)) {
    const f4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      f4_t in[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          in[h][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.x[mb][h][i], b.w[h][i], z, 0, 0, 0);
      acc[mb] += ((in[0][0] + in[0][1]) + (in[0][2] + in[0][3])) +
                 ((in[1][0] + in[1][1]) + (in[1][2] + in[1][3]));
    }
  };
  Block b0, b1;
  load(b0, 0);
  load(b1, 1);
  for (int i = 0; i < per; i += 2) {
    run(b0);
    load(b0, i + 2);
    run(b1);
    load(b1, i + 3);
  }
  // lane holds rows 4 (lane / 16) + i of W row lane % 16
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      part[((wave * MB + mb) * 16 + 4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[mb][i];
  __syncthreads();
  auto total = [&](int r, int c) {
    static_assert(kSkinnyF32Waves == 8, "a tree of eight");
    auto at = [&](int w) { return part[(w * 16 * MB + r) * 16 + c]; };
    return ((at(0) + at(1)) + (at(2) + at(3))) + ((at(4) + at(5)) + (at(6) + at(7)));
  };
  if (a.epi.act == kEpiSwiGLU) {
    for (int o = tid; o < mr * 8; o += 64 * kSkinnyF32Waves) {
      const int r = o >> 3, c = o & 7;
      // n % 16 == 0 under SwiGLU, so every row of the tile exists
      const float g = add_bias(a.epi, total(r, c), n0 + c);
      const float u = add_bias(a.epi, total(r, c + 8), n0 + c + 8);
      a.y[(size_t)(m0 + r) * a.ny + glu_col(n0 + c)] = silu_f(g) * u;
    }
  } else {
    for (int o = tid; o < mr * 16; o += 64 * kSkinnyF32Waves) {
      const int r = o >> 4, row = n0 + (o & 15);
      if (row < a.n) a.y[(size_t)(m0 + r) * a.n + row] = add_bias(a.epi, total(r, o & 15), row);
    }
  }
}

// 64 x 64 tiles when they fill most of the chip's CUs; K is split over two
// groups of waves (two waves per SIMD hide the stage barrier).
bool linear_f32_tiled(int m, int n) {
  return (int64_t)((m + kTile - 1) / kTile) * ((n + kTile - 1) / kTile) >= 192;
}

template <bool VEC>
hipError_t launch_mfma_f32(const F32Args& a, hipStream_t s) {
  if (linear_f32_tiled(a.m, a.n)) {
    const int tiles = ((a.m + kTile - 1) / kTile) * ((a.n + kTile - 1) / kTile);
    constexpr int KS = 2;
    const auto kernel = a.k < 1536   ? gemm_f32_kernel<KS, VEC, 4>
                        : a.k < 3072 ? gemm_f32_kernel<KS, VEC, 16>
                                     : gemm_f32_kernel<KS, VEC, 32>;
    const hipError_t e = allow_dynamic_lds((const void*)kernel, gemm_f32_lds<KS>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3((tiles + 7) / 8 * 8), dim3(256 * KS), gemm_f32_lds<KS>(), s, a);
    return hipGetLastError();
  }
  const int mb = a.m <= 16 ? 1 : a.m <= 32 ? 2 : 4;
  const dim3 grid((a.n + 15) / 16, (a.m + 16 * mb - 1) / (16 * mb)), block(64 * kSkinnyF32Waves);
  switch (mb) {
    case 1: hipLaunchKernelGGL((skinny_f32_kernel<1, VEC>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((skinny_f32_kernel<2, VEC>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((skinny_f32_kernel<4, VEC>), grid, block, 0, s, a); break;
  }
  return hipGetLastError();
}

template <bool VEC>
void launch_rows(const F32Args& a, int mr, hipStream_t s) {
  const dim3 grid((a.n + 15) / 16), block(256);
  switch (mr) {
    case 1: hipLaunchKernelGGL((linear_f32_kernel<1, VEC>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((linear_f32_kernel<2, VEC>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((linear_f32_kernel<3, VEC>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((linear_f32_kernel<4, VEC>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((linear_f32_kernel<5, VEC>), grid, block, 0, s, a); break;
    case 6: hipLaunchKernelGGL((linear_f32_kernel<6, VEC>), grid, block, 0, s, a); break;
    case 7: hipLaunchKernelGGL((linear_f32_kernel<7, VEC>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((linear_f32_kernel<8, VEC>), grid, block, 0, s, a); break;
  }
}

}  // namespace

hipError_t launch_linear_f32(const float* w, int n, int k, const float* x, float* y, int m,
                             hipStream_t stream, const Epilogue& epi) {
  F32Args a;
  a.w = w;
  a.x = x;
  a.y = y;
  a.m = m;
  a.n = n;
  a.k = k;
  a.ny = epi.act == kEpiSwiGLU ? n / 2 : n;
  a.epi = epi;
  const bool vec = k % 4 == 0 && ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0;
  // the MFMA kernels address 64 rows of K floats by 31-bit byte offsets, and
  // the skinny one puts 64-row blocks on a grid dimension
  if (m > kF32MaxRows && k <= (1 << 22) && m <= (1 << 20))
    return vec ? launch_mfma_f32<true>(a, stream) : launch_mfma_f32<false>(a, stream);
  for (int r0 = 0; r0 < m; r0 += kF32MaxRows) {
    const int mr = m - r0 < kF32MaxRows ? m - r0 : kF32MaxRows;
    a.x = x + (size_t)r0 * k;
    a.y = y + (size_t)r0 * a.ny;
    if (vec) launch_rows<true>(a, mr, stream);
    else launch_rows<false>(a, mr, stream);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace mlq
