// fp32 contraction for every shape that does not fill the CUs with the 256 x 128
// tiles of l2c_gemm.hip, and for most rows that are not 16-byte aligned:
// out[b][r] = sum_k X[b][k] * W[r][k] on v_mfma_f32_16x16x4_f32, tiles of 16 to
// 64 batch rows by 16 to 64 weight rows, K split over the workgroup's waves.
//
//  * Every wave computes the whole tile over its own 32-deep k-steps (step s on
//    wave s % WAVES) from its own ring of two LDS stages, so the loop has no
//    barrier: a wave waits only for its own DMA. A small tile is what fills 256
//    CUs when batch and rows are small, and what wastes little on a ragged edge;
//    the k-split is what gives each CU enough waves then. The waves' partial
//    tiles meet once at the end in LDS and are added in wave order, so results
//    do not depend on scheduling; the chains are 1 / WAVES as long as the large
//    kernel's, and the error against 64 bits lower (8.1e-7 against 1.1e-6 at
//    K = 4096).
//  * Staging by LDS DMA, 8 rows x 128 bytes an instruction, with the 16-byte
//    chunks XOR-swizzled by row bits on the source side, as in the other
//    contractions. Loading MFMA operands straight from global memory (16
//    neighbouring lanes in 16 rows) kept the loads at about 11 B a cycle and CU
//    and measured 1.3-2.5 times slower (1024 x 4096 x 8192: 836-1068 us against
//    517-566; 16 x 16384 x 512: 57.9 against 22.4).
//  * The 16-byte DMAs read rows at any 4-byte address (cols % 4 != 0 or an odd
//    base); only their LDS side is aligned. 130 x 5003 x 1501 took 774 us with
//    scalar loads on 256 x 128 tiles and 30 us here with 4-byte DMAs, a quarter of
//    the data an instruction; now 28.8. 142 x 3197 x 2210: 36.5 and 26.5;
//    15 x 2597 x 1109: 9.2 and 6.6; 18% in the mean of 50 unaligned shapes.
//  * MFMA operands: lane (r, q) = (l % 16, l / 16) reads chunk 4 c + q of row r
//    for half-step c; MFMA e of a half takes element e of each lane for both
//    operands (k is summed over, so its order is free). Accumulator value v of
//    lane l is C[4 * (l / 16) + v][l % 16].
//  * Every access is in bounds by construction: operand rows past the end are
//    clamped to the last one and not stored; a partial last step (cols % 32)
//    loads element by element with k clamped and zeros selected past the end.
//  * Bounds at 2.4 GHz and 157 TFLOP/s: the fp32 matrix cores for 64 batch rows
//    and more (64 x 2048 x 8192: 13.7 us, measured 21.9 against 232 before;
//    781 x 2760 x 7587: 208 us, 285 against 324), HBM below
//    (8 x 4096 x 11008: 33 us, 34.8 against 461), and the launch for the
//    smallest (8 x 768 x 2048: 3.5 us against 89).
#include "l2c_common.h"
#include "../../include/l2c.h"

namespace {

using l2c::f32x4;
typedef __attribute__((address_space(3))) void lds_ptr;

constexpr int kStep = 32;    // k per step: 128 bytes of a row
constexpr int kStages = 2;   // LDS stages of a wave

// At most N of this wave's memory instructions are outstanding after it.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void dma_to_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char *dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr *)dst, 16, voffset, soffset, 0, 0);
}

// Tile 16 MF x 16 NF.
template <int MF, int NF, int WAVES>
__global__ __launch_bounds__(WAVES *L2C_WAVE) void gemm_f32_ksplit_kernel(float *__restrict__ out,
                                                                          const float *__restrict__ X,
                                                                          const float *__restrict__ W, int M, int N,
                                                                          int K) {
  constexpr int kBM = 16 * MF, kBN = 16 * NF, kTile = kBM * kBN;
  constexpr int kRows = kBM + kBN, kStage = kRows * 128;
  constexpr int kRowsPerDma = 8;  // 128-byte rows one instruction moves
  constexpr int kXDma = kBM / kRowsPerDma, kWDma = kBN / kRowsPerDma;
  constexpr int kLds = WAVES * kStages * kStage > WAVES * kTile * 4 ? WAVES * kStages * kStage : WAVES * kTile * 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];
  const int tile = l2c::xcd_tile(blockIdx.x, gridDim.x);
  const int mtiles = (M + kBM - 1) / kBM;
  const int m0 = (tile % mtiles) * kBM, n0 = (tile / mtiles) * kBN;
  const int mrows = min(kBM, M - m0), nrows = min(kBN, N - n0);
  const int tid = threadIdx.x, lane = tid % L2C_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / L2C_WAVE);
  const int r = lane % 16, q = lane / 16;

  const __amdgpu_buffer_rsrc_t rx =
      l2c::buffer_rsrc(X + static_cast<size_t>(m0) * K, static_cast<uint32_t>(mrows) * K * 4u);
  const __amdgpu_buffer_rsrc_t rw =
      l2c::buffer_rsrc(W + static_cast<size_t>(n0) * K, static_cast<uint32_t>(nrows) * K * 4u);
  // DMA sources (the step's k offset is scalar): lane l fills row l / 8 of the
  // instruction's rows, 16-byte slot l % 8, from the chunk that the swizzle puts
  // there.
  auto swizzle = [](int row) { return (row >> 1) & 7; };
  int xsrc[kXDma], wsrc[kWDma];
  const int lrow = lane / 8, lslot = lane % 8;
  auto src = [&](int row, int rows) __attribute__((always_inline)) {
    return min(row, rows - 1) * K * 4 + 16 * (lslot ^ swizzle(row));
  };
#pragma unroll
  for (int i = 0; i < kXDma; ++i) xsrc[i] = src(kRowsPerDma * i + lrow, mrows);
#pragma unroll
  for (int j = 0; j < kWDma; ++j) wsrc[j] = src(kRowsPerDma * j + lrow, nrows);

  unsigned char *const base = lds + wave * (kStages * kStage);
  auto dma = [&](int stage, int s) __attribute__((always_inline)) {
    unsigned char *d = base + stage * kStage;
    const int so = s * 128;
#pragma unroll
    for (int j = 0; j < kWDma; ++j)
      dma_to_lds(rw, d + kBM * 128 + j * kRowsPerDma * 128, wsrc[j], so);
#pragma unroll
    for (int i = 0; i < kXDma; ++i)
      dma_to_lds(rx, d + i * kRowsPerDma * 128, xsrc[i], so);
  };
  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  struct Operands {
    f32x4 a[MF][2], b[NF][2];
  };
  const int c0 = r * 128 + 16 * (q ^ swizzle(r)), c1 = r * 128 + 16 * ((4 + q) ^ swizzle(r));
  auto read = [&](Operands &o, int stage) __attribute__((always_inline)) {
    const unsigned char *d = base + stage * kStage;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int i = 0; i < MF; ++i) o.a[i][c] = *reinterpret_cast<const f32x4 *>(d + 2048 * i + (c ? c1 : c0));
#pragma unroll
      for (int j = 0; j < NF; ++j)
        o.b[j][c] = *reinterpret_cast<const f32x4 *>(d + kBM * 128 + 2048 * j + (c ? c1 : c0));
    }
  };
  auto mma = [&](const Operands &o) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int j = 0; j < NF; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[i][c][e], o.b[j][c][e], acc[i][j], 0, 0, 0);
  };

  const int steps = K / kStep;
  if (wave < steps) {
    const int last = wave + (steps - 1 - wave) / WAVES * WAVES;
    dma(0, wave);
    int cur = 0;
    Operands o;
    for (int s = wave; s <= last; s += WAVES) {
      // The other stage's reads fed the MFMAs of the step before, so they are
      // done; the last step's DMA is repeated into a stage nobody reads. The
      // wait leaves only the newer step's DMA in flight.
      __builtin_amdgcn_sched_barrier(0);
      dma(cur ^ 1, min(s + WAVES, last));
      wait_vmcnt<kXDma + kWDma>();
      read(o, cur);
      mma(o);
      cur ^= 1;
    }
    wait_vmcnt<0>();  // the partial sums below reuse the stages
  }
  if (K % kStep != 0 && wave == steps % WAVES) {
    Operands o;
    const int k0 = steps * kStep + 4 * q;
    const float *xrow[MF], *wrow[NF];
#pragma unroll
    for (int i = 0; i < MF; ++i) xrow[i] = X + static_cast<size_t>(min(m0 + 16 * i + r, M - 1)) * K;
#pragma unroll
    for (int j = 0; j < NF; ++j) wrow[j] = W + static_cast<size_t>(min(n0 + 16 * j + r, N - 1)) * K;
    auto tail = [&](const float *row, int c) __attribute__((always_inline)) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + 16 * c + e;
        const float f = row[min(k, K - 1)];
        v[e] = k < K ? f : 0.0f;
      }
      return v;
    };
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int j = 0; j < NF; ++j) o.b[j][c] = tail(wrow[j], c);
#pragma unroll
      for (int i = 0; i < MF; ++i) o.a[i][c] = tail(xrow[i], c);
    }
    mma(o);
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
    const int block = e / 256, v = e / L2C_WAVE % 4, l = e % L2C_WAVE;
    const int m = m0 + block / NF * 16 + 4 * (l / 16) + v, n = n0 + block % NF * 16 + l % 16;
    if (m < M && n < N) __builtin_nontemporal_store(sum, &out[static_cast<size_t>(m) * N + n]);
  }
}

// ---------------------------------------------------------------------------
// Choice of the tile.

struct Config {
  int mf, nf, waves;
  void (*fn)(float *, const float *, const float *, int, int, int);
};

#define L2C_KSPLIT(MF, NF, WAVES) \
  { MF, NF, WAVES, gemm_f32_ksplit_kernel<MF, NF, WAVES> }
const Config kConfigs[] = {L2C_KSPLIT(1, 1, 8), L2C_KSPLIT(2, 1, 8), L2C_KSPLIT(1, 2, 8), L2C_KSPLIT(2, 2, 4),
                           L2C_KSPLIT(2, 2, 8), L2C_KSPLIT(3, 2, 4), L2C_KSPLIT(2, 3, 4), L2C_KSPLIT(4, 4, 4)};
#undef L2C_KSPLIT

// Cycles of the busiest CU: its tiles, each at the slower of its MFMAs (256
// FLOP a cycle) and its staging (30 B a cycle), and 10% more where the CU's only
// workgroup is one wave a SIMD, which nothing hides the latency of. Of tiles
// that cost the same the first is taken. Fitted to 16 tiles on 66 shapes of 1 to
// 1024 x 288 to 16384 x 288 to 11008: the choice is 1.2% slower than the best of
// them in the mean, and up to 13% (28% for one unaligned shape).
double cost(const Config &c, int batch, int cols, int rows) {
  const int bm = 16 * c.mf, bn = 16 * c.nf;
  const long long tiles = static_cast<long long>((batch + bm - 1) / bm) * ((rows + bn - 1) / bn);
  const long long per_cu = (tiles + 255) / 256;
  const double mfma = bm * bn / 128.0, dma = (bm + bn) * 4 / 30.0;
  return static_cast<double>(cols) * per_cu * (mfma > dma ? mfma : dma) * (per_cu * c.waves <= 4 ? 1.1 : 1.0);
}

// The kernel's per-lane byte offsets, row * cols * 4 of a tile, are ints.
bool fits(const Config &c, int cols) {
  return 16LL * (c.mf > c.nf ? c.mf : c.nf) * cols * 4 <= 0x7fffffffLL;
}

long long tiles_of(const Config &c, int batch, int rows) {
  return static_cast<long long>((batch + 16 * c.mf - 1) / (16 * c.mf)) * ((rows + 16 * c.nf - 1) / (16 * c.nf));
}

const Config *choose(int batch, int cols, int rows, double *least) {
  const Config *best = nullptr;
  for (const Config &c : kConfigs) {
    const double t = cost(c, batch, cols, rows);
    if (fits(c, cols) && l2c::launchable(tiles_of(c, batch, rows), c.waves * L2C_WAVE) && (!best || t < *least)) {
      best = &c;
      *least = t;
    }
  }
  return best;
}

// The tile of least cost where it is to be preferred to the 256 x 128 tiles (null
// where it is not): where its estimated time is 5% below theirs. Fitted to the GPU
// times of all nine kernels on 910 aligned shapes of 32 to 1100 x 32 to 8192 x 200
// to 11008, most of them where the two are close: the choice is 0.2% slower than the
// faster of the two in the mean and slower than the 256 x 128 tiles on two of them
// (971 x 156 x 3272 29 us against 25, 740 x 184 x 4447 33 against 30). The outputs count: the costs
// alone took k-split tiles for 716 x 40 x 5338 at 24.8 us against 16.4, 760 x 176 x
// 8364 at 56 against 36 and 963 x 1040 x 7370 at 158 against 136.
// k-split / 256 x 128 tiles, us: 781 x 2760 x 7587 285 / 324, 359 x 2572 x 5113
// 99 / 289, 631 x 528 x 9585 88 / 78.
// Unaligned rows are compared with the scalar kernel on the same tiles, which is faster
// at short K with many outputs only (1000 x 17 x 7772 20 us, 34 here; fitted on 400 shapes
// of 1 to 600 k, the choice is 0.1% slower than the better of the two in the mean).
// Aligned products of at most one 256 x 128 tile keep
// that tile's single chain over k, on one CU: the lowprec experiment's accuracy record
// states its error (5.7e-7 at 64 x 1024 x 128, the published figure; 2.1e-7 on k-split
// tiles). It costs long rows much (64 x 16384 x 128 1808 us against 23, 256 x 4096 x 128
// 456 against 9).
const Config *preferred(int batch, int cols, int rows, bool aligned) {
  double least = 0.0;
  const Config *c = choose(batch, cols, rows, &least);
  if (!c) return nullptr;
  if (aligned && batch <= 256 && rows <= 128) return nullptr;
  auto rounds = [](long long tiles) { return static_cast<double>((tiles + 255) / 256); };
  const double outputs = static_cast<double>(batch) * rows;
  const double split_ns = 0.51 * least + 0.0042 * outputs + 3900.0;
  const double large = rounds(static_cast<long long>((batch + 255) / 256) * ((rows + 127) / 128));
  if (!aligned) return split_ns < 169.0 * ((cols + 31LL) / 32 * 32) * large + 0.001 * outputs + 3500.0 ? c : nullptr;
  return split_ns < 0.95 * (112.0 * cols * large + 0.002 * outputs + 4800.0) ? c : nullptr;
}

}  // namespace

bool l2c_gemm_ksplit(float *out, const float *X, const float *W, int batch, int cols, int rows, bool aligned,
                     hipStream_t stream) {
  const Config *c = preferred(batch, cols, rows, aligned);
  if (!c) return false;
  hipLaunchKernelGGL(c->fn, dim3(static_cast<unsigned>(tiles_of(*c, batch, rows))),
                     dim3(c->waves * L2C_WAVE), 0, stream, out, X, W, batch, rows, cols);
  return true;
}

bool l2c_gemm_ksplit_launch_shape(int batch, int cols, int rows, bool aligned, int *grid, int *block,
                                  const void **fn) {
  const Config *c = preferred(batch, cols, rows, aligned);
  if (!c) return false;
  *grid = static_cast<int>(tiles_of(*c, batch, rows));
  *block = c->waves * L2C_WAVE;
  *fn = reinterpret_cast<const void *>(c->fn);
  return true;
}
