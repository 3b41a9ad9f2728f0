// Block-scaled contractions for shapes that do not fill the CUs with the large
// tiles of l2c_scgemm.hip and l2c_mxgemm.hip: out[b][r] = sum_k deq(X)[b][k] *
// deq(W)[r][k] with MXFP8 activations and MXFP4 or per-row-scaled fp8 weights,
// or with both operands MXFP6, in the layouts those kernels take.
//
//  * The k-split tiles of l2c_gemm_ksplit.hip on
//    v_mfma_scale_f32_16x16x128_f8f6f4: every wave computes the whole 16 MF x
//    16 NF tile over its own 128-deep k-steps (step s on wave s % WAVES) from its
//    own two LDS stages, waiting for nothing but its own DMA; the waves' partial
//    tiles are added in wave order at the end.
//  * MFMA operands: lane (r, q) = (l % 16, l / 16) supplies row r, and the scale
//    byte of block q (k 32 q .. 32 q + 31). Its codes are, for E2M1 and E3M2,
//    block q in order, and for E4M3 k 16 q .. 16 q + 15 in VGPRs 0-3 and k
//    64 + 16 q .. 64 + 16 q + 15 in VGPRs 4-7 (measured on MI355X: operands and
//    outputs fitted; only this placement fits). Accumulator value v of lane l is
//    C[4 * (l / 16) + v][l % 16].
//  * Staging by LDS DMA: row-major codes in 16-byte chunks XOR-swizzled by row
//    bits on the source side; the tiled E3M2 codes as the four 384-byte block
//    pieces of 16 rows, one and a half instructions; scales as one-byte DMAs, a
//    byte landing zero-extended in its lane's own LDS word, which is the MFMA's
//    scale operand.
//  * Rows past the operands are clamped to the last row (the last 16 padded rows
//    of a tiled operand) and not stored. K % 128 == 0.
//  * Bounds: staging from L2 while tiles are small, HBM for W at decode batches.
//    The product alone, one box, before against now, us (MXFP4 / fp8 / MXFP6):
//    16 x 4096 x 11008 26 / 29 / 24.5, now 9.3 / 9.1 / 8.0; 64 x 4096 x 8192
//    28 / 33 / 25, now 10.2 / 9.4 / 8.5; 11 x 12032 x 2048 61 / 66 / 57, now
//    6.8 / 6.5 / 7.1; 629 x 13056 x 1024 80 / 85 / 65, now 26 / 21.5 / 21.
#include "l2c_common.h"
#include "l2c_ksplit.h"
#include "../../include/l2c.h"

namespace {

using l2c::f32x4;
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_ptr;

constexpr int kMxfp6 = 2;  // both operands MXFP6 in the tiled layout
constexpr int kKS = 128;   // k per step: one 16 x 16 x 128 MFMA a pair of fragments
constexpr int kStages = 2;
constexpr int kE4M3 = 0, kE3M2 = 3, kE2M1 = 4;  // MFMA operand formats

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

// One operand's form. E4M3 and E2M1 rows are row-major; E3M2 fragments are
// pieces of the tiled layout.
template <int CODES, int FRAGS, bool SCALED>
struct Operand {
  static constexpr bool kTiled = CODES == kE3M2;
  static constexpr int kRow = CODES == kE4M3 ? 128 : 64;                     // code bytes of a row and step
  static constexpr int kFrag = kTiled ? 2048 : 16 * kRow;                    // LDS bytes of a fragment
  static constexpr int kDma = FRAGS * kFrag / 1024;
  static constexpr int kScales = FRAGS * kFrag;
  static constexpr int kBytes = kScales + (SCALED ? 256 * FRAGS : 0);
  static constexpr int kIssued = kDma + (SCALED ? FRAGS : 0);
  static __device__ __forceinline__ int swizzle(int row) { return CODES == kE4M3 ? (row >> 1) & 7 : (row >> 2) & 3; }

  int src[kDma];
  int ssrc[FRAGS];

  // Row-major codes of `rows` rows, `pitch` bytes apart.
  __device__ __forceinline__ void init_rows(int lane, int rows, int pitch) {
    constexpr int slots = kRow / 16, per = 64 / slots;
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const int row = per * i + lane / slots;
      src[i] = min(row, rows - 1) * pitch + 16 * ((lane % slots) ^ swizzle(row));
    }
  }
  // Tiled codes from row `first` of an operand padded to `padded` rows: block b
  // of 16 rows is 384 contiguous bytes.
  __device__ __forceinline__ void init_tiled(int lane, int first, int padded) {
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const int row = min(first + 16 * (i / 2), padded - 16);
      const int piece = min(64 * (i % 2) + lane, 95);  // the upper half of the second instruction is padding
      src[i] = row / 32 * 3072 + row % 32 * 24 + piece / 24 * 768 + 16 * (piece % 24);
    }
  }
  // Scale bytes of 4 blocks a row, rows `pitch` bytes apart, the last one `last`.
  __device__ __forceinline__ void init_scales(int lane, int last, int pitch) {
#pragma unroll
    for (int f = 0; f < FRAGS; ++f) ssrc[f] = min(16 * f + lane % 16, last) * pitch + lane / 16;
  }
  __device__ __forceinline__ void load(unsigned char *d, __amdgpu_buffer_rsrc_t codes, int coff,
                                       __amdgpu_buffer_rsrc_t scales, int soff) const {
#pragma unroll
    for (int i = 0; i < kDma; ++i) dma16(codes, d + 1024 * i, src[i], coff);
    if constexpr (SCALED) {
#pragma unroll
      for (int f = 0; f < FRAGS; ++f) dma1(scales, d + kScales + 256 * f, ssrc[f], soff);
    }
  }
  __device__ __forceinline__ void read(const unsigned char *d, int lane, i32x8 (&v)[FRAGS], int (&s)[FRAGS]) const {
    const int r = lane % 16, q = lane / 16;
#pragma unroll
    for (int f = 0; f < FRAGS; ++f) {
      v[f] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
      if constexpr (kTiled) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const u32x2 w = *reinterpret_cast<const u32x2 *>(d + f * kFrag + q * 384 + 24 * r + 8 * c);
          v[f][2 * c] = static_cast<int>(w[0]), v[f][2 * c + 1] = static_cast<int>(w[1]);
        }
      } else {
        const unsigned char *row = d + f * kFrag + r * kRow;
#pragma unroll
        for (int c = 0; c < (CODES == kE4M3 ? 2 : 1); ++c) {
          const u32x4 w = *reinterpret_cast<const u32x4 *>(row + 16 * ((4 * c + q) ^ swizzle(r)));
#pragma unroll
          for (int e = 0; e < 4; ++e) v[f][4 * c + e] = static_cast<int>(w[e]);
        }
      }
      s[f] = 127;
      if constexpr (SCALED) s[f] = *reinterpret_cast<const int *>(d + kScales + 256 * f + 4 * lane);
    }
  }
};

template <int FMT, int MF, int NF>
struct Shape {
  static constexpr bool kTiled = FMT == kMxfp6;
  static constexpr int kXCodes = kTiled ? kE3M2 : kE4M3;
  static constexpr int kWCodes = kTiled ? kE3M2 : FMT == L2C_Q_MXFP4 ? kE2M1 : kE4M3;
  static constexpr bool kWScaled = FMT != L2C_Q_FP8;
  using XOp = Operand<kXCodes, MF, true>;
  using WOp = Operand<kWCodes, NF, kWScaled>;
  static constexpr int kBM = 16 * MF, kBN = 16 * NF, kTile = kBM * kBN;
  static constexpr int kStage = XOp::kBytes + WOp::kBytes, kIssued = XOp::kIssued + WOp::kIssued;
  // The waves' stages, which their partial sums take over at the end.
  static constexpr int lds(int waves) { return waves * (kStages * kStage > kTile * 4 ? kStages * kStage : kTile * 4); }
};

// Mp: rows of the X scale tiles (batch rounded up to 4, or to 32 for MXFP6).
template <int FMT, int MF, int NF, int WAVES>
__global__ __launch_bounds__(WAVES *L2C_WAVE) void scgemm_ksplit_kernel(float *__restrict__ out,
                                                                        const uint8_t *__restrict__ X,
                                                                        const uint8_t *__restrict__ Xs,
                                                                        const uint8_t *__restrict__ Wq,
                                                                        const void *__restrict__ wscales, int M,
                                                                        int N, int K, int Mp) {
  using S = Shape<FMT, MF, NF>;
  using XOp = typename S::XOp;
  using WOp = typename S::WOp;
  constexpr bool kTiled = S::kTiled;
  constexpr int kBM = S::kBM, kBN = S::kBN, kTile = S::kTile, kStage = S::kStage;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S::lds(WAVES)];
  const int tile = l2c::xcd_tile(blockIdx.x, gridDim.x);
  const int mtiles = (M + kBM - 1) / kBM;
  const int m0 = (tile % mtiles) * kBM, n0 = (tile / mtiles) * kBN;
  const int mrows = min(kBM, M - m0), nrows = min(kBN, N - n0);
  const int tid = threadIdx.x, lane = tid % L2C_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / L2C_WAVE);
  // What the sums of the lane's columns are multiplied by, loaded ahead of the DMAs:
  // loads and stores complete in order, and a load between the epilogue's stores
  // waits for them.
  float factor[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) factor[j] = 1.0f;
  if constexpr (FMT == L2C_Q_FP8) {
#pragma unroll
    for (int j = 0; j < NF; ++j)
      factor[j] = static_cast<const float *>(wscales)[n0 + min(16 * j + lane % 16, nrows - 1)];
  }
  const int steps = K / kKS;

  XOp xo;
  WOp wo;
  __amdgpu_buffer_rsrc_t rx, rxs, rw, rws;
  int xstep, wstep, xsstep, wsstep;
  rxs = l2c::buffer_rsrc(Xs, static_cast<uint32_t>(Mp) * 4 * steps);
  xsstep = 4 * Mp;
  xo.init_scales(lane, Mp - m0 - 1, 4);
  if constexpr (kTiled) {
    const int Np = (N + 31) / 32 * 32;
    xstep = Mp / 32 * 3072, wstep = Np / 32 * 3072, wsstep = 4 * Np;
    rx = l2c::buffer_rsrc(X, static_cast<uint32_t>(xstep) * steps);
    rw = l2c::buffer_rsrc(Wq, static_cast<uint32_t>(wstep) * steps);
    rws = l2c::buffer_rsrc(wscales, static_cast<uint32_t>(wsstep) * steps);
    xo.init_tiled(lane, m0, Mp);
    wo.init_tiled(lane, n0, Np);
    wo.init_scales(lane, Np - n0 - 1, 4);
  } else {
    const int wrb = FMT == L2C_Q_MXFP4 ? K / 2 : K, srb = K / 32;
    xstep = kKS, wstep = WOp::kRow, wsstep = 4;
    rx = l2c::buffer_rsrc(X + static_cast<size_t>(m0) * K, static_cast<uint32_t>(mrows) * K);
    rw = l2c::buffer_rsrc(Wq + static_cast<size_t>(n0) * wrb, static_cast<uint32_t>(nrows) * wrb);
    rws = rw;
    xo.init_rows(lane, mrows, K);
    wo.init_rows(lane, nrows, wrb);
    if constexpr (S::kWScaled) {
      rws = l2c::buffer_rsrc(static_cast<const uint8_t *>(wscales) + static_cast<size_t>(n0) * srb,
                             static_cast<uint32_t>(nrows) * srb);
      wo.init_scales(lane, nrows - 1, srb);
    }
  }
  unsigned char *const base = lds + wave * (kStages * kStage);
  auto dma = [&](int stage, int s) __attribute__((always_inline)) {
    unsigned char *d = base + stage * kStage;
    wo.load(d + XOp::kBytes, rw, wstep * s, rws, wsstep * s + (kTiled ? 4 * n0 : 0));
    xo.load(d, rx, xstep * s, rxs, xsstep * s + 4 * m0);
  };
  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  if (wave < steps) {
    const int last = wave + (steps - 1 - wave) / WAVES * WAVES;
    dma(0, wave);
    int cur = 0;
    for (int s = wave; s <= last; s += WAVES) {
      __builtin_amdgcn_sched_barrier(0);
      dma(cur ^ 1, min(s + WAVES, last));
      wait_vmcnt<S::kIssued>();
      const unsigned char *d = base + cur * kStage;
      i32x8 a[MF], b[NF];
      int sa[MF], sb[NF];
      wo.read(d + XOp::kBytes, lane, b, sb);
      xo.read(d, lane, a, sa);
#pragma unroll
      for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NF; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b[j], acc[i][j], S::kXCodes, S::kWCodes, 0,
                                                                       sa[i], 0, sb[j]);
      cur ^= 1;
    }
    wait_vmcnt<0>();
  }

  __syncthreads();
  float *partial = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) partial[wave * kTile + ((i * NF + j) * 4 + v) * L2C_WAVE + lane] = acc[i][j][v];
  __syncthreads();
  for (int e = tid; e < kTile; e += WAVES * L2C_WAVE) {
    float sum = partial[e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += partial[w * kTile + e];
    const int block = e / 256, v = e / L2C_WAVE % 4;
    const int m = block / NF * 16 + 4 * (lane / 16) + v, n = block % NF * 16 + lane % 16;
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

using Kernel = void (*)(float *, const uint8_t *, const uint8_t *, const uint8_t *, const void *, int, int, int, int);

struct Config {
  Kernel fn;
  l2c::KsplitTile tile;
};

template <int FMT, int MF, int NF, int WAVES>
constexpr Config config() {
  return {scgemm_ksplit_kernel<FMT, MF, NF, WAVES>, {MF, NF, WAVES, Shape<FMT, MF, NF>::lds(WAVES)}};
}

// Of tiles that cost the same the first is taken.
template <int FMT>
const Config kConfigs[] = {config<FMT, 1, 1, 8>(), config<FMT, 1, 1, 4>(), config<FMT, 1, 2, 4>(),
                           config<FMT, 1, 4, 4>(), config<FMT, 2, 2, 4>(), config<FMT, 3, 2, 4>(),
                           config<FMT, 2, 4, 4>(), config<FMT, 3, 4, 4>(), config<FMT, 4, 4, 4>(),
                           config<FMT, 1, 2, 2>(), config<FMT, 2, 2, 2>(), config<FMT, 3, 4, 2>()};

// An MXFP4 row (64 bytes a step, half a line) counts as 3/4 of an fp8 row.
template <int FMT>
double cost(const Config &c, int batch, int cols, int rows) {
  constexpr double x = FMT == kMxfp6 ? 25.0 / 32.0 : 1.0;
  constexpr double w = FMT == L2C_Q_MXFP4 ? 0.75 : FMT == L2C_Q_FP8 ? 1.0 : 25.0 / 32.0;
  return l2c::ksplit_cost(c.tile, x, w, kKS, batch, cols, rows);
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
                            : choose<kMxfp6>(batch, cols, rows, least);
}

// The tile of least cost where it is to be preferred to the large tiles, or null.
// Fitted to both kernels' GPU times on 96 shapes of 64 to 1024 x 128 to 16384 x 288
// to 11008, each CU taking its tiles in turn: a k-split tile's cost at 1 / 84
// (MXFP4), 1 / 114 (fp8) or 1 / 93 (MXFP6) ns a byte, 0.33, 0.79 or 0.60 ns an output
// value of a CU and 2.5 to 2.7 us; a large tile 4.9, 4.5 or 4.2 ns a k and 7.3, 10.1 or
// 9.2 us for its first stages and its output, and 1 us. The choice is 0 to 0.3%
// slower than the better of the two in the mean. Where the estimates are within 8%, about
// their error, the large tiles stay, and within 12% for MXFP6, whose k-split tiles are 4
// to 7% slower there (754 x 5376 x 2765: 36 us against 34; 393 x 1280 x 4150, which stays
// too, 15.4 against 16.5). Measured on either side,
// us: 256 x 4096 x 11008 36 / 33 / 33 here, 30 / 31 / 29 there; 934 x 2560 x 1280
// 15 / 15 / 15 here, 24 / 33 / 21 there; 1024 x 4096 x 4096 49 / 45 / 44 here,
// 30 / 34 / 30 there; 693 x 256 x 3128 MXFP6 12 both.
// Products of MXFP8 activations with more than 256 vectors and at most 1152 k
// keep the large tiles whatever the estimates (300 x 1024 x 600: about 10 us against
// 4.5): the tests of the 128 x 256 and 256 x 128 tiles run there and assert their grids.
const Config *preferred(int fmt, int batch, int cols, int rows) {
  if (fmt != kMxfp6 && batch > 256 && cols <= 1152) return nullptr;
  double least = 0.0;
  const Config *c = choose(fmt, batch, cols, rows, &least);
  if (!c) return nullptr;
  struct Rate {
    double split, split_out, split_more, large, large_tile;
  };
  constexpr Rate kRates[] = {
      {84.0, 0.33, 2700.0, 4.9, 7300.0}, {114.0, 0.79, 2500.0, 4.5, 10100.0}, {93.0, 0.60, 2600.0, 4.2, 9200.0}};
  constexpr double kLaunch = 1000.0;
  const Rate &rate = kRates[fmt];
  auto rounds = [](long long tiles) { return static_cast<double>((tiles + 255) / 256); };
  const double split_ns = least / rate.split + rate.split_more +
                          rate.split_out * (256.0 * c->tile.mf * c->tile.nf) *
                              rounds(l2c::ksplit_tiles(c->tile, batch, rows));
  const double large_ns = (rate.large * cols + rate.large_tile) *
                              rounds(static_cast<long long>((batch + 255) / 256) * ((rows + 127) / 128)) +
                          kLaunch;
  return split_ns < (fmt == kMxfp6 ? 0.88 : 0.92) * large_ns ? c : nullptr;
}

}  // namespace

bool l2c_scgemm_ksplit(float *out, const uint8_t *X, const uint8_t *Xs, const uint8_t *Wq, const void *wscales,
                       int fmt, int batch, int cols, int rows, hipStream_t stream) {
  const Config *c = preferred(fmt, batch, cols, rows);
  if (!c) return false;
  const int padded = fmt == kMxfp6 ? (batch + 31) / 32 * 32 : (batch + 3) / 4 * 4;
  hipLaunchKernelGGL(c->fn, dim3(static_cast<unsigned>(l2c::ksplit_tiles(c->tile, batch, rows))),
                     dim3(c->tile.waves * L2C_WAVE), 0, stream, out, X, Xs, Wq, wscales, batch, rows, cols, padded);
  return true;
}

bool l2c_scgemm_ksplit_launch_shape(int fmt, int batch, int cols, int rows, int *grid, int *block, const void **fn) {
  const Config *c = preferred(fmt, batch, cols, rows);
  if (!c) return false;
  *grid = static_cast<int>(l2c::ksplit_tiles(c->tile, batch, rows));
  *block = c->tile.waves * L2C_WAVE;
  *fn = reinterpret_cast<const void *>(c->fn);
  return true;
}
