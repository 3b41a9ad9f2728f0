// bf16-activation contractions for every shape that does not fill the CUs with
// the large tiles of l2c_qgemm_ks.hip and l2c_bfgemm.hip (decode batches, short
// vocabularies, ragged sizes): out[b][r] = sum_k X[b][k] * deq(W)[r][k] with
// MXFP4, per-row-scaled fp8 or bf16 weights, in the layouts those kernels take,
// for any K % 32 == 0.
//
//  * The k-split tiles of l2c_gemm_ksplit.hip on v_mfma_f32_16x16x32_bf16: every
//    wave computes the whole 16 MF x 16 NF tile over its own k-steps (step s on
//    wave s % WAVES) from its own two LDS stages, waiting for nothing but its
//    own DMA; the waves' partial tiles are added in wave order at the end.
//  * A step is 64 k (fp8, bf16) or 128 k (MXFP4): 128 or 256 bytes of an X row and
//    64 or 128 of a W row, moved by 16-byte LDS DMAs whose chunks are
//    XOR-swizzled by row bits on the source side. MXFP4 scales come as one-byte
//    DMAs, lane (r, q) = (l % 16, l / 16) fetching the byte of the block it
//    multiplies: a byte lands zero-extended in the lane's own LDS word.
//  * A lane's 16-byte W chunk holds the codes of 1, 2 or 4 MFMAs (8 bf16, 16 fp8
//    or 32 E2M1 codes: one whole MXFP4 block), and its X chunks are those of the
//    same k: within a window lane quarter q takes k = q w .. q w + w - 1, w = 8,
//    16 or 32 (k is summed over, so its order is free). Codes are converted
//    exactly to bf16 by the scaled conversions, as in the large kernels.
//  * The rest of K past the last whole step goes in 32-deep units, one wave each,
//    straight from memory.
//  * Rows past the operands are clamped to the last row and not stored.
//  * Bounds: staging from L2 (X again for every weight tile) while few rows of
//    either operand are in a tile, HBM for W below; at K = 4096, one box, before
//    against now, us: 16 x 11008 MXFP4 44.4 / 10.5, fp8 38.2 / 10.0, bf16 45.7 /
//    16.9 (5.4 TB/s of W); 40 x 8004 41.5 / 9.9, 39.7 / 10.2, 36.0 / 12.9;
//    64 x 8192 41.9 / 11.2, 41.8 / 10.9, 37.1 / 13.9; 11 x 12032 x 2048
//    103 / 8.0, 90 / 8.1, 89 / 9.9.
#include <cmath>

#include "l2c_common.h"
#include "l2c_ksplit.h"
#include "../../include/l2c.h"

namespace {

using l2c::f32x4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_ptr;

constexpr int kFmtBf16 = 2;  // bf16 weights; `scales` is the device alpha or null
constexpr int kStages = 2;

// At most N of this wave's memory instructions are outstanding after it.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, unsigned char *dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr *)dst, 16, voffset, soffset, 0, 0);
}
__device__ __forceinline__ void dma1(__amdgpu_buffer_rsrc_t rsrc, unsigned char *dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr *)dst, 1, voffset, soffset, 0, 0);
}

// Geometry of one step of KS k.
template <int FMT, int MF, int NF>
struct Shape {
  static constexpr int KS = FMT == L2C_Q_MXFP4 ? 128 : 64;
  static constexpr bool kMx = FMT == L2C_Q_MXFP4;
  static constexpr int kBM = 16 * MF, kBN = 16 * NF, kTile = kBM * kBN;
  static constexpr int kPerChunk = kMx ? 4 : FMT == L2C_Q_FP8 ? 2 : 1;  // MFMAs a 16-byte W chunk feeds
  static constexpr int kWindows = KS / (32 * kPerChunk);                 // W chunks a lane takes a step
  static constexpr int kXRow = 2 * KS, kWRow = 64 * kWindows;            // bytes of a row and step
  static constexpr int kXRowsPerDma = 1024 / kXRow, kWRowsPerDma = 1024 / kWRow;
  static constexpr int kXDma = kBM / kXRowsPerDma, kWDma = kBN / kWRowsPerDma;
  static constexpr int kSDma = kMx ? NF * kWindows : 0;
  static constexpr int kWOff = kBM * kXRow, kSOff = kWOff + kBN * kWRow;
  static constexpr int kStage = kSOff + kSDma * 256;
  static constexpr int kDma = kXDma + kWDma + kSDma;
  // The waves' stages, which their partial sums take over at the end.
  static constexpr int lds(int waves) { return waves * (kStages * kStage > kTile * 4 ? kStages * kStage : kTile * 4); }
  static_assert(kXDma * kXRowsPerDma == kBM && kWDma * kWRowsPerDma == kBN, "whole instructions");
};

// 16-byte chunk swizzle of a row of `bytes` bytes: 16 rows reading one chunk
// touch all 64 banks.
template <int BYTES>
__device__ __forceinline__ int swizzle(int row) {
  if constexpr (BYTES == 64) return (row >> 2) & 3;
  if constexpr (BYTES == 128) return (row >> 1) & 7;
  return row & 15;
}

template <int FMT>
__device__ __forceinline__ bf16x8 convert(const unsigned *w, float scale) {
  unsigned d[4];
  if constexpr (FMT == L2C_Q_MXFP4) {
    d[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[0], scale, 0));
    d[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[0], scale, 1));
    d[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[0], scale, 2));
    d[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[0], scale, 3));
  } else if constexpr (FMT == L2C_Q_FP8) {
    d[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.0f, false));
    d[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.0f, true));
    d[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.0f, false));
    d[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.0f, true));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = w[i];
  }
  return __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3]));
}

template <int FMT, int MF, int NF, int WAVES>
__global__ __launch_bounds__(WAVES *L2C_WAVE) void qgemm_ksplit_kernel(float *__restrict__ out,
                                                                       const uint16_t *__restrict__ X,
                                                                       const uint8_t *__restrict__ Wq,
                                                                       const void *__restrict__ scales, int M, int N,
                                                                       int K) {
  using S = Shape<FMT, MF, NF>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S::lds(WAVES)];
  const int tile = l2c::xcd_tile(blockIdx.x, gridDim.x);
  const int mtiles = (M + S::kBM - 1) / S::kBM;
  const int m0 = (tile % mtiles) * S::kBM, n0 = (tile / mtiles) * S::kBN;
  const int mrows = min(S::kBM, M - m0), nrows = min(S::kBN, N - n0);
  const int tid = threadIdx.x, lane = tid % L2C_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / L2C_WAVE);
  const int r = lane % 16, q = lane / 16;
  const int xrb = 2 * K, wrb = S::kMx ? K / 2 : FMT == L2C_Q_FP8 ? K : 2 * K, srb = K / 32;
  const uint8_t *const wbase = Wq + static_cast<size_t>(n0) * wrb;
  const uint8_t *const sbase = static_cast<const uint8_t *>(scales) + static_cast<size_t>(n0) * srb;
  const __amdgpu_buffer_rsrc_t rx =
      l2c::buffer_rsrc(X + static_cast<size_t>(m0) * K, static_cast<uint32_t>(mrows) * xrb);
  const __amdgpu_buffer_rsrc_t rw = l2c::buffer_rsrc(wbase, static_cast<uint32_t>(nrows) * wrb);
  const __amdgpu_buffer_rsrc_t rs = S::kMx ? l2c::buffer_rsrc(sbase, static_cast<uint32_t>(nrows) * srb) : rw;

  int xsrc[S::kXDma], wsrc[S::kWDma], ssrc[NF];
#pragma unroll
  for (int i = 0; i < S::kXDma; ++i) {
    constexpr int slots = S::kXRow / 16;
    const int row = S::kXRowsPerDma * i + lane / slots;
    xsrc[i] = min(row, mrows - 1) * xrb + 16 * ((lane % slots) ^ swizzle<S::kXRow>(row));
  }
#pragma unroll
  for (int j = 0; j < S::kWDma; ++j) {
    constexpr int slots = S::kWRow / 16;
    const int row = S::kWRowsPerDma * j + lane / slots;
    wsrc[j] = min(row, nrows - 1) * wrb + 16 * ((lane % slots) ^ swizzle<S::kWRow>(row));
  }
#pragma unroll
  for (int j = 0; j < NF; ++j) ssrc[j] = min(16 * j + r, nrows - 1) * srb + q;

  unsigned char *const base = lds + wave * (kStages * S::kStage);
  auto dma = [&](int stage, int s) __attribute__((always_inline)) {
    unsigned char *d = base + stage * S::kStage;
#pragma unroll
    for (int j = 0; j < S::kWDma; ++j)
      dma16(rw, d + S::kWOff + 1024 * j, wsrc[j], S::kWRow * s);
    if constexpr (S::kMx) {
#pragma unroll
      for (int v = 0; v < S::kWindows; ++v)
#pragma unroll
        for (int j = 0; j < NF; ++j)
          dma1(rs, d + S::kSOff + 256 * (v * NF + j), ssrc[j], S::KS / 32 * s + 4 * v);
    }
#pragma unroll
    for (int i = 0; i < S::kXDma; ++i)
      dma16(rx, d + 1024 * i, xsrc[i], S::kXRow * s);
  };
  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int stage) __attribute__((always_inline)) {
    const unsigned char *d = base + stage * S::kStage;
#pragma unroll
    for (int v = 0; v < S::kWindows; ++v) {
      u32x4 w[NF], x[MF][S::kPerChunk];
      float scale[NF];
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int row = 16 * j + r;
        w[j] = *reinterpret_cast<const u32x4 *>(d + S::kWOff + row * S::kWRow +
                                                16 * ((4 * v + q) ^ swizzle<S::kWRow>(row)));
        scale[j] = 1.0f;
        if constexpr (S::kMx)
          scale[j] = __uint_as_float(*reinterpret_cast<const unsigned *>(d + S::kSOff + 256 * (v * NF + j) + 4 * lane)
                                     << 23);
      }
#pragma unroll
      for (int t = 0; t < S::kPerChunk; ++t)
#pragma unroll
        for (int i = 0; i < MF; ++i) {
          const int row = 16 * i + r;
          x[i][t] = *reinterpret_cast<const u32x4 *>(
              d + row * S::kXRow + 16 * ((S::kPerChunk * (4 * v + q) + t) ^ swizzle<S::kXRow>(row)));
        }
#pragma unroll
      for (int t = 0; t < S::kPerChunk; ++t) {
        bf16x8 b[NF];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
          unsigned part[4];
#pragma unroll
          for (int c = 0; c < 4 / S::kPerChunk; ++c) part[c] = w[j][4 / S::kPerChunk * t + c];
          b[j] = convert<FMT>(part, scale[j]);
        }
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int j = 0; j < NF; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[i][t]), b[j], acc[i][j],
                                                                0, 0, 0);
      }
    }
  };

  // What the sums of the lane's columns are multiplied by, loaded ahead of the DMAs:
  // loads and stores complete in order, and a load between the epilogue's stores
  // waits for them.
  float factor[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) factor[j] = 1.0f;
  if constexpr (FMT == kFmtBf16) {
    if (scales) {
      const float alpha = *static_cast<const float *>(scales);
#pragma unroll
      for (int j = 0; j < NF; ++j) factor[j] = alpha;
    }
  } else if constexpr (FMT == L2C_Q_FP8) {
#pragma unroll
    for (int j = 0; j < NF; ++j)
      factor[j] = static_cast<const float *>(scales)[n0 + min(16 * j + r, nrows - 1)];
  }
  const int steps = K / S::KS;
  if (wave < steps) {
    const int last = wave + (steps - 1 - wave) / WAVES * WAVES;
    dma(0, wave);
    int cur = 0;
    for (int s = wave; s <= last; s += WAVES) {
      __builtin_amdgcn_sched_barrier(0);
      dma(cur ^ 1, min(s + WAVES, last));
      wait_vmcnt<S::kDma>();
      multiply(cur);
      cur ^= 1;
    }
    wait_vmcnt<0>();
  }
  // The rest of K in 32-deep units, one wave each, straight from memory.
  for (int u = (wave + WAVES - steps % WAVES) % WAVES; steps * S::KS + 32 * u < K; u += WAVES) {
    const int k0 = steps * S::KS + 32 * u;
    bf16x8 b[NF];
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int row = min(16 * j + r, nrows - 1);
      unsigned part[4];
      float scale = 1.0f;
      if constexpr (S::kMx) {
        part[0] = *reinterpret_cast<const unsigned *>(wbase + static_cast<size_t>(row) * wrb + (k0 + 8 * q) / 2);
        scale = __uint_as_float(static_cast<unsigned>(sbase[static_cast<size_t>(row) * srb + k0 / 32]) << 23);
      } else {
        constexpr int bytes = FMT == L2C_Q_FP8 ? 1 : 2;
        const unsigned *src =
            reinterpret_cast<const unsigned *>(wbase + static_cast<size_t>(row) * wrb + bytes * (k0 + 8 * q));
#pragma unroll
        for (int c = 0; c < 2 * bytes; ++c) part[c] = src[c];
      }
      b[j] = convert<FMT>(part, scale);
    }
#pragma unroll
    for (int i = 0; i < MF; ++i) {
      const u32x4 x = *reinterpret_cast<const u32x4 *>(
          X + static_cast<size_t>(m0 + min(16 * i + r, mrows - 1)) * K + k0 + 8 * q);
#pragma unroll
      for (int j = 0; j < NF; ++j)
        acc[i][j] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), b[j], acc[i][j], 0, 0, 0);
    }
  }

  __syncthreads();
  float *partial = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) partial[wave * S::kTile + ((i * NF + j) * 4 + v) * L2C_WAVE + lane] = acc[i][j][v];
  __syncthreads();
  for (int e = tid; e < S::kTile; e += WAVES * L2C_WAVE) {
    float sum = partial[e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += partial[w * S::kTile + e];
    const int block = e / 256, v = e / L2C_WAVE % 4;
    const int m = block / NF * 16 + 4 * q + v, n = block % NF * 16 + r;
    float f = factor[0];
#pragma unroll
    for (int j = 1; j < NF; ++j) f = block % NF == j ? factor[j] : f;
    if (m < mrows && n < nrows) {
      __builtin_nontemporal_store(sum * f, &out[static_cast<size_t>(m0 + m) * N + n0 + n]);
    }
  }
}

// ---------------------------------------------------------------------------
// Choice of the tile.

using Kernel = void (*)(float *, const uint16_t *, const uint8_t *, const void *, int, int, int);

struct Config {
  Kernel fn;
  l2c::KsplitTile tile;
};

template <int FMT, int MF, int NF, int WAVES>
constexpr Config config() {
  return {qgemm_ksplit_kernel<FMT, MF, NF, WAVES>, {MF, NF, WAVES, Shape<FMT, MF, NF>::lds(WAVES)}};
}

// Of tiles that cost the same the first is taken. (Four waves of a 64 x 64 MXFP4
// tile need more than the CU's LDS.)
template <int FMT>
const Config kConfigs[] = {config<FMT, 1, 1, 8>(), config<FMT, 1, 1, 4>(), config<FMT, 1, 2, 4>(),
                           config<FMT, 1, 4, 4>(), config<FMT, 2, 2, 4>(), config<FMT, 3, 2, 4>(),
                           config<FMT, 2, 4, 4>(), config<FMT, 3, 4, 4>(),
                           config<FMT, 4, 4, FMT == L2C_Q_MXFP4 ? 2 : 4>(),
                           config<FMT, 1, 2, 2>(), config<FMT, 2, 2, 2>(), config<FMT, 3, 4, 2>()};

template <int FMT>
double cost(const Config &c, int batch, int cols, int rows) {
  constexpr double w = FMT == L2C_Q_MXFP4 ? 17.0 / 32.0 : FMT == L2C_Q_FP8 ? 1.0 : 2.0;
  return l2c::ksplit_cost(c.tile, 2.0, w, Shape<FMT, 1, 1>::KS, batch, cols, rows);
}

// The tile of least cost that HIP launches, and that cost; null if there is none.
template <int FMT>
const Config *choose(int batch, int cols, int rows, double *least) {
  const Config *best = nullptr;
  for (const Config &c : kConfigs<FMT>) {
    const double t = cost<FMT>(c, batch, cols, rows);
    if (l2c::ksplit_launchable(c.tile, batch, rows) && (!best || t < *least)) {
      best = &c;
      *least = t;
    }
  }
  return best;
}

const Config *choose(int fmt, int batch, int cols, int rows, double *least) {
  return fmt == L2C_Q_MXFP4 ? choose<L2C_Q_MXFP4>(batch, cols, rows, least)
         : fmt == L2C_Q_FP8 ? choose<L2C_Q_FP8>(batch, cols, rows, least)
                            : choose<kFmtBf16>(batch, cols, rows, least);
}

// One form of the contraction, ready to launch; no kernel where a large one is to
// be preferred.
struct Launch {
  Kernel fn;
  unsigned grid, block;
};

// Of the k-split tile of least cost, the 128 x 128 tiles (where `mid` says that
// they take the operands) and a large kernel of `large_tiles` tiles, the one of
// least estimated time. Fitted to the three kernels' GPU times on 96 shapes of 64
// to 1024 x 128 to 16384 x 288 to 11008, each CU taking its tiles in turn: a k-split
// tile's cost at 1 / 73 (MXFP4), 1 / 104 (fp8) or 1 / 119 (bf16) ns a byte, 0.67, 0.48
// or 0.56 ns an output value of a CU and 2.4 to 2.6 us; a 128 x 128 tile 7.1, 5.9 or
// 5.7 ns a k and 5.8, 6.1 or 5.5 us for its first slices and its output, a large one
// 8.4, 7.2 or 7.3 ns a k and 9.9, 10.4 or 10 us; and 1 us. The choice is 0 to 0.3%
// slower than the best of the three in the mean, and never slower than the large
// kernel there. Measured, us, k-split / 128 x 128 / large: 256 x 4096 x 11008 MXFP4
// 65 / 40 / 48, fp8 42 / 35 / 44, bf16 45 / 32 / 42; 797 x 128 x 2467 MXFP4 13 / 9 /
// 13; 545 x 512 x 9893 fp8 25 / 23 / 22, bf16 27 / 21 / 22; 691 x 3840 x 7680
// 93 / 71 / 51, 75 / 69 / 54, 74 / 63 / 49.
// K % 64 == 32 has another large kernel (l2c_qgemm.hip), faster at short K, and the
// k-split tiles take the rest of K straight from memory: 13 to 16% on their estimate.
// Fitted on 660 shapes of 48 to 1100 x 32 to 4128 x 200 to 11008: 1.2 (MXFP4) and 0.2%
// (bf16) slower than the better of the two in the mean, and by more than 3% slower than
// the large kernel on nine of the 1320 (on 92 with the estimates above: 161 x 32 x
// 10576 MXFP4 11.7 us against 6.4, 969 x 96 x 2221 bf16 11.7 against 9.0). fp8, whose large
// kernel is slower there, is on none with the estimates above (398 x 608 x 8821 21 / 19).
Launch choose_form(int fmt, int batch, int cols, int rows, long long large_tiles, bool mid) {
  struct Rate {
    double split, split_out, split_more, mid, mid_tile, large, large_tile;
  };
  constexpr Rate kRates[] = {{73.0, 0.67, 2400.0, 7.1, 5800.0, 8.4, 9900.0},
                             {104.0, 0.48, 2600.0, 5.9, 6100.0, 7.2, 10400.0},
                             {119.0, 0.56, 2400.0, 5.7, 5500.0, 7.3, 10000.0}};
  constexpr double kLaunch = 1000.0;
  const Rate &rate = kRates[fmt];
  double least = 0.0;
  const Config *c = choose(fmt, batch, cols, rows, &least);
  const long long split_tiles = c ? l2c::ksplit_tiles(c->tile, batch, rows) : 0;
  const long long mid_tiles = static_cast<long long>((batch + 127) / 128) * ((rows + 127) / 128);
  auto rounds = [](long long tiles) { return static_cast<double>((tiles + 255) / 256); };
  double split_ns = c ? least / rate.split +
                            rate.split_out * (256.0 * c->tile.mf * c->tile.nf) * rounds(split_tiles) +
                            rate.split_more
                      : HUGE_VAL;
  const double mid_ns = (rate.mid * cols + rate.mid_tile) * rounds(mid_tiles) + kLaunch;
  double large_ns = (rate.large * cols + rate.large_tile) * rounds(large_tiles) + kLaunch;
  if (mid && cols % 64 == 0 && mid_ns < split_ns && mid_ns < large_ns && l2c::launchable(mid_tiles, 512))
    return {l2c_qgemm_mid_kernel(fmt), static_cast<unsigned>(mid_tiles), 512};
  if (cols % 64 != 0 && fmt != L2C_Q_FP8) {
    const bool mx = fmt == L2C_Q_MXFP4;
    split_ns *= mx ? 1.16 : 1.13;
    large_ns = ((mx ? 11.8 : 12.7) * cols + (mx ? 3600.0 : 4000.0)) * rounds(large_tiles) +
               (mx ? 0.00084 : 0.00078) * batch * static_cast<double>(rows) + 2200.0;
  }
  if (split_ns < large_ns)
    return {c->fn, static_cast<unsigned>(split_tiles), static_cast<unsigned>(c->tile.waves * L2C_WAVE)};
  return {nullptr, 0, 0};
}

}  // namespace

bool l2c_qgemm_ksplit(float *out, const uint16_t *X, const uint8_t *Wq, const void *scales, int fmt, int batch,
                      int cols, int rows, long long large_tiles, hipStream_t stream) {
  // The 128 x 128 tiles' scale DMAs read 2 bytes: an odd address takes one of the
  // other two, which read single bytes.
  const bool mid = fmt != L2C_Q_MXFP4 || (reinterpret_cast<uintptr_t>(scales) & 1u) == 0;
  const Launch l = choose_form(fmt, batch, cols, rows, large_tiles, mid);
  if (!l.fn) return false;
  hipLaunchKernelGGL(l.fn, dim3(l.grid), dim3(l.block), 0, stream, out, X, Wq, scales, batch, rows, cols);
  return true;
}

bool l2c_qgemm_ksplit_launch_shape(int fmt, int batch, int cols, int rows, long long large_tiles, int *grid, int *block,
                                   const void **fn) {
  const Launch l = choose_form(fmt, batch, cols, rows, large_tiles, true);
  if (!l.fn) return false;
  *grid = static_cast<int>(l.grid);
  *block = static_cast<int>(l.block);
  *fn = reinterpret_cast<const void *>(l.fn);
  return true;
}
