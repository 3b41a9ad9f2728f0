// Row kernels of the llama2c hot path on gfx950: rmsnorm, softmax, the
// matrix-vector product (naive and coalesced) and the single-launch fused
// iteration.
//
// Design (MI355X: 256 CUs in 8 XCDs, wave64, 160 KiB LDS per CU, HBM3E):
//  * rmsnorm and softmax are one-pass: a workgroup owns one row, loads it once
//    into VGPRs with 16-byte loads (V float4 per lane), reduces it with wave64
//    shuffles plus one LDS slot per wave, and writes the result from the same
//    registers. HBM traffic is the floor: one read and one write per element
//    (the reference's rmsnorm reads twice, its softmax reads 3x and writes 2x;
//    llama2c/llama2c_cuda_graph.cu:58-115). When the lanes cover the row
//    exactly (size 16384: 512 lanes x 8 float4) the loads and stores carry
//    no bounds checks.
//  * softmax needs one block barrier: each wavefront exponentiates against
//    its own maximum (exp on the hardware exp2 with Cody-Waite reduction), and
//    the waves' (max, sum) pairs are combined once (l2c_rows.h).
//  * Rows whose address is not 16-byte aligned (size % 4 != 0) keep the same
//    one-pass structure with 16-byte loads at 4-byte addresses; rows longer than 1024 lanes x 64
//    floats take a two-pass path that re-reads the row.
//  * The coalesced matrix-vector product gives each output row to one
//    wavefront (a pair of wavefronts, each half the row, for aligned rows of
//    >= 8192 floats): 64 lanes x 16 B = 1 KiB contiguous per load instruction,
//    several independent loads in flight per lane, one wave reduction per row.
//    W is read with nontemporal loads (they keep it from evicting x from L2),
//    except when it is 128-256 MiB: then ordinary loads let the 256 MB MALL
//    keep it between launches. Measured at 4096 columns, nontemporal against
//    ordinary loads: 64 MiB 10.1 / 10.8 µs, 96 MiB 15.0 / 15.4, 144 MiB
//    24.0 / 22.3, 172 MiB 27.2 / 25.7, 256 MiB 39.2 / 37.2, 288 MiB
//    43.9 / 44.4, 384 MiB 58.0 / 65.1.
//  * The naive product keeps the reference's one-lane-per-row structure and
//    its sequential column order (one fused multiply-add per column), so its
//    result is bit-reproducible by a CPU fmaf chain.
//  * The fused iteration is one grid of the standalone kernels' workgroups:
//    rmsnorm and softmax rows in the row kernels' configuration, then matrix
//    rows one per wavefront (or pair of wavefronts) with the standalone
//    product's load choice, so its outputs equal the three separate launches'
//    bit for bit. At 1024 x 16384
//    x 8192 (one box, alternating runs) it took 123.3 against 135.3 us for
//    the earlier form that ran every part at 256 lanes (a whole workgroup per
//    matrix row, rows at 16 float4 a lane).
#include "l2c_rows.h"
#include "../../include/l2c.h"

namespace {

using l2c::Row;

constexpr int kMaxRowThreads = 1024;
constexpr int kGenericThreads = 256;
// Aligned matrices with at least kPairCols columns, or at least kPairMinCols
// columns and more than kPairBytes, are multiplied a row per pair of
// wavefronts (l2c::matvec_pair_row); the rest a row per wavefront
// (l2c::matvec_wave_row). Small matrices of 4096-column rows run faster a row
// per wavefront (4096 x 4096: 10.0 against 10.4 us), large ones a row per
// pair (4096 x 11008: 25.2 against 25.6 us).
constexpr int kPairCols = 8192;
constexpr int kPairMinCols = 4096;
constexpr unsigned long long kPairBytes = 128ULL << 20;

// ---------------------------------------------------------------------------
// Kernels. V == 0 selects the two-pass generic path; MAXT is the launch
// bound (256 or 1024 lanes), so rows that fit 256 lanes get the full register
// budget.

template <int V, bool VEC, bool EXACT, int MAXT>
__global__ __launch_bounds__(MAXT) void rmsnorm_kernel(float *out, const float *in,
                                                       const float *weight, int size, float eps) {
  __shared__ float slots[32];
  const size_t off = static_cast<size_t>(blockIdx.x) * size;
  if constexpr (V == 0) {
    l2c::rmsnorm_row_generic(out + off, in + off, weight, size, eps, slots);
  } else {
    Row<V, VEC, EXACT> r;
    r.load(in + off, size, 0.0f);
    l2c::rmsnorm_apply(r, out + off, weight, size, eps, slots);
  }
}

template <int V, bool VEC, bool EXACT, int MAXT>
__global__ __launch_bounds__(MAXT) void softmax_kernel(float *out, const float *logits, int size) {
  __shared__ float slots[32];
  const size_t off = static_cast<size_t>(blockIdx.x) * size;
  if constexpr (V == 0) {
    l2c::softmax_row_generic(out + off, logits + off, size, slots);
  } else {
    Row<V, VEC, EXACT> r;
    r.load(logits + off, size, -FLT_MAX);
    l2c::softmax_apply_1r(r, out + off, size, slots);
  }
}

// One launch for a whole llama2c iteration, in workgroups of the row
// kernels' size T. Block b handles:
//   b < 2*pairs           rmsnorm row b/2 (even b) or softmax row b/2 (odd b)
//   then                  the remaining rmsnorm rows, then remaining softmax rows
//   then                  T / 64 matrix rows, one per wavefront
// so the short matrix-vector blocks fill the tail of the launch.
template <int V, bool VEC, bool EXACT, int MAXT, bool NT>
__global__ __launch_bounds__(MAXT) void fused_kernel(
    float *normalized, const float *input, const float *weight, float *softmax,
    const float *logits, float *product, const float *matrix, int size, int rms_rows,
    int softmax_rows, int matmul_rows, int pair, float eps) {
  __shared__ float slots[32];
  int item = blockIdx.x;
  const int pairs = min(rms_rows, softmax_rows);
  int kind, row;
  if (item < 2 * pairs) {
    kind = item & 1;
    row = item >> 1;
  } else if ((item -= 2 * pairs) < rms_rows - pairs) {
    kind = 0;
    row = pairs + item;
  } else if ((item -= rms_rows - pairs) < softmax_rows - pairs) {
    kind = 1;
    row = pairs + item;
  } else {
    kind = 2;
    row = item - (softmax_rows - pairs);  // the matrix workgroup's index
  }
  if (kind == 2) {
    const int waves = blockDim.x / L2C_WAVE, wave = threadIdx.x / L2C_WAVE, lane = threadIdx.x % L2C_WAVE;
    if constexpr (VEC) {
      if (pair) {
        // waves / 2 rows a workgroup; a wave left over (odd wave counts) only
        // takes part in the barrier.
        const int r = row * (waves / 2) + wave / 2;
        const bool live = wave < waves / 2 * 2 && r < matmul_rows;
        l2c::matvec_pair_row<NT>(product, input, matrix, size, r, wave % 2, lane, live, slots);
        return;
      }
    }
    const int r = row * waves + wave;
    if (r < matmul_rows) l2c::matvec_wave_row<VEC, NT>(product, input, matrix, size, r, lane);
    return;
  }
  const size_t off = static_cast<size_t>(row) * size;
  if constexpr (V == 0) {
    if (kind == 0) l2c::rmsnorm_row_generic(normalized + off, input + off, weight, size, eps, slots);
    else l2c::softmax_row_generic(softmax + off, logits + off, size, slots);
  } else {
    Row<V, VEC, EXACT> r;
    if (kind == 0) {
      r.load(input + off, size, 0.0f);
      l2c::rmsnorm_apply(r, normalized + off, weight, size, eps, slots);
    } else {
      r.load(logits + off, size, -FLT_MAX);
      l2c::softmax_apply_1r(r, softmax + off, size, slots);
    }
  }
}

// Reference structure: one lane per output row, columns in order, one fused
// multiply-add per column.
__global__ __launch_bounds__(256) void matvec_naive_kernel(float *out, const float *x,
                                                           const float *W, int cols, int rows) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  const float *w = W + static_cast<size_t>(row) * cols;
  float acc = 0.0f;
  for (int c = 0; c < cols; ++c) acc = fmaf(x[c], w[c], acc);
  out[row] = acc;
}

// One wavefront per output row; kWavesPerBlock rows per block.
constexpr int kMatvecWaves = 4;

template <bool VEC, bool NT>
__global__ __launch_bounds__(kMatvecWaves * L2C_WAVE) void matvec_wave_kernel(
    float *out, const float *x, const float *W, int cols, int rows) {
  const int row = blockIdx.x * kMatvecWaves + threadIdx.x / L2C_WAVE;
  if (row < rows) l2c::matvec_wave_row<VEC, NT>(out, x, W, cols, row, threadIdx.x % L2C_WAVE);
}

// A row per pair of wavefronts, kMatvecWaves / 2 rows a workgroup.
template <bool NT>
__global__ __launch_bounds__(kMatvecWaves * L2C_WAVE) void matvec_pair_kernel(
    float *out, const float *x, const float *W, int cols, int rows) {
  __shared__ float slots[kMatvecWaves];
  const int wave = threadIdx.x / L2C_WAVE;
  const int row = blockIdx.x * (kMatvecWaves / 2) + wave / 2;
  l2c::matvec_pair_row<NT>(out, x, W, cols, row, wave % 2, threadIdx.x % L2C_WAVE, row < rows, slots);
}

// The coalesced product's form: a pair of wavefronts per row for aligned rows
// of >= kPairCols floats, or of >= kPairMinCols floats in a matrix of more
// than kPairBytes; else one wavefront per row.
bool pair_rows(int cols, int rows, bool vec) {
  const unsigned long long w_bytes = 4ULL * static_cast<unsigned long long>(rows) * cols;
  return vec && (cols >= kPairCols || (cols >= kPairMinCols && w_bytes > kPairBytes));
}

// Nontemporal matrix loads, except for a matrix of 128-256 MiB, which the
// 256 MB MALL keeps between launches when it is read with ordinary loads.
bool matvec_nontemporal(int cols, int rows) {
  const unsigned long long w_bytes = 4ULL * static_cast<unsigned long long>(rows) * cols;
  return !(w_bytes > (128ULL << 20) && w_bytes <= (256ULL << 20));
}

// ---------------------------------------------------------------------------
// Launch configuration for the row kernels: the smallest V (float4 per lane)
// up to 8 whose row fits in <= 256 lanes, else in <= 512 lanes, else the
// smallest V up to 16 in <= max_threads lanes, else the generic two-pass
// path. Lanes are rounded up to whole wavefronts; `exact` when the lanes
// cover the row with no remainder. Measured at 1024 x 16384 (rmsnorm, same
// box): 512 lanes x 8 float4 19.53 us against 256 x 16 20.31 us and
// 1024 x 4 20.26 us; with 16 float4 a lane, a whole row's loads in flight
// per lane leave fewer lanes to overlap them.

struct RowConfig {
  int threads;
  int v;  // 0 = generic
  bool exact;   // of aligned rows
  bool single;  // of the others: no more floats than lanes (with v == 1)
};

RowConfig choose_row_config(int size, int max_threads = kMaxRowThreads) {
  const int chunks = (size + 3) / 4;
  for (int limit : {256, 512, max_threads}) {
    if (limit > max_threads) continue;
    for (int v = 1; v <= (limit == max_threads ? 16 : 8); v *= 2) {
      const int lanes = (chunks + v - 1) / v;
      const int threads = (lanes + L2C_WAVE - 1) / L2C_WAVE * L2C_WAVE;
      if (threads <= limit) return {threads, v, size % 4 == 0 && threads * v * 4 == size, size <= threads};
    }
  }
  return {kGenericThreads, 0, false, false};
}

using RmsFn = void (*)(float *, const float *, const float *, int, float);
using SoftFn = void (*)(float *, const float *, int);
using FusedFn = void (*)(float *, const float *, const float *, float *, const float *, float *,
                         const float *, int, int, int, int, int, float);

// Kernel instance for (V, vector path, exact, launch bound).
template <int V, int MAXT>
struct Pick {
  static RmsFn rms(bool vec, bool exact) {
    if constexpr (V == 1 && MAXT == 256)
      if (!vec && exact) return rmsnorm_kernel<V, false, true, MAXT>;
    if (!vec) return rmsnorm_kernel<V, false, false, MAXT>;
    return exact ? rmsnorm_kernel<V, true, true, MAXT> : rmsnorm_kernel<V, true, false, MAXT>;
  }
  static SoftFn soft(bool vec, bool exact) {
    if constexpr (V == 1 && MAXT == 256)
      if (!vec && exact) return softmax_kernel<V, false, true, MAXT>;
    if (!vec) return softmax_kernel<V, false, false, MAXT>;
    return exact ? softmax_kernel<V, true, true, MAXT> : softmax_kernel<V, true, false, MAXT>;
  }
};

template <int MAXT>
RmsFn rms_for(int v, bool vec, bool exact) {
  switch (v) {
    case 1: return Pick<1, MAXT>::rms(vec, exact);
    case 2: return Pick<2, MAXT>::rms(vec, exact);
    case 4: return Pick<4, MAXT>::rms(vec, exact);
    case 8: return Pick<8, MAXT>::rms(vec, exact);
    case 16: return Pick<16, MAXT>::rms(vec, exact);
    default: return rmsnorm_kernel<0, false, false, MAXT>;
  }
}

template <int MAXT>
SoftFn soft_for(int v, bool vec, bool exact) {
  switch (v) {
    case 1: return Pick<1, MAXT>::soft(vec, exact);
    case 2: return Pick<2, MAXT>::soft(vec, exact);
    case 4: return Pick<4, MAXT>::soft(vec, exact);
    case 8: return Pick<8, MAXT>::soft(vec, exact);
    case 16: return Pick<16, MAXT>::soft(vec, exact);
    default: return softmax_kernel<0, false, false, MAXT>;
  }
}

// Fused kernel instances for the (lanes, V) pairs choose_row_config returns:
// up to 256 lanes with V <= 8, 512 lanes with V = 8, 1024 lanes with V = 8 or
// 16, and the generic path (V = 0) at 256 lanes.
template <int V, int MAXT, bool NT>
FusedFn fused_pick(bool vec, bool exact) {
  if constexpr (V == 1)
    if (!vec && exact) return fused_kernel<V, false, true, MAXT, NT>;
  if (!vec) return fused_kernel<V, false, false, MAXT, NT>;
  return exact ? fused_kernel<V, true, true, MAXT, NT> : fused_kernel<V, true, false, MAXT, NT>;
}

// Any other pair gets no instance (null).
template <bool NT>
FusedFn fused_for(const RowConfig &c, bool vec) {
  const bool exact = vec ? c.exact : c.single;
  if (c.v == 0)
    return c.threads == kGenericThreads ? (vec ? fused_kernel<0, true, false, kGenericThreads, NT>
                                               : fused_kernel<0, false, false, kGenericThreads, NT>)
                                        : nullptr;
  if (c.threads <= 256) {
    switch (c.v) {
      case 1: return fused_pick<1, 256, NT>(vec, exact);
      case 2: return fused_pick<2, 256, NT>(vec, exact);
      case 4: return fused_pick<4, 256, NT>(vec, exact);
      case 8: return fused_pick<8, 256, NT>(vec, exact);
      default: return nullptr;
    }
  }
  if (c.threads <= 512) return c.v == 8 ? fused_pick<8, 512, NT>(vec, exact) : nullptr;
  if (c.v == 8) return fused_pick<8, kMaxRowThreads, NT>(vec, exact);
  return c.v == 16 ? fused_pick<16, kMaxRowThreads, NT>(vec, exact) : nullptr;
}

RmsFn rms_fn(const RowConfig &c, bool vec) {
  const bool exact = vec ? c.exact : c.single;
  if (c.threads <= 256) return rms_for<256>(c.v, vec, exact);
  return c.threads <= 512 ? rms_for<512>(c.v, vec, exact) : rms_for<kMaxRowThreads>(c.v, vec, exact);
}

SoftFn soft_fn(const RowConfig &c, bool vec) {
  const bool exact = vec ? c.exact : c.single;
  if (c.threads <= 256) return soft_for<256>(c.v, vec, exact);
  return c.threads <= 512 ? soft_for<512>(c.v, vec, exact) : soft_for<kMaxRowThreads>(c.v, vec, exact);
}

FusedFn fused_fn(const RowConfig &c, bool vec, bool nt) {
  return nt ? fused_for<true>(c, vec) : fused_for<false>(c, vec);
}

// Workgroups of the fused launch: one per rmsnorm and softmax row, then one
// per lanes / 64 matrix rows (lanes / 128 when a pair of wavefronts takes a row).
long long fused_items(const RowConfig &c, bool pair, int rms_rows, int softmax_rows, int matmul_rows) {
  const int per_block = c.threads / L2C_WAVE / (pair ? 2 : 1);
  return static_cast<long long>(rms_rows) + softmax_rows + (static_cast<long long>(matmul_rows) + per_block - 1) / per_block;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI

extern "C" int l2c_rmsnorm(float *out, const float *in, const float *weight, int size, int batch,
                           float eps, hipStream_t stream) {
  if (size <= 0 || batch < 0) return hipErrorInvalidValue;
  if (batch == 0) return hipSuccess;
  if (!out || !in || !weight) return hipErrorInvalidValue;
  const RowConfig cfg = choose_row_config(size);
  const bool vec = size % 4 == 0 && l2c_aligned16(out) && l2c_aligned16(in) &&
                   l2c_aligned16(weight);
  hipLaunchKernelGGL(rms_fn(cfg, vec), dim3(batch), dim3(cfg.threads), 0, stream, out, in,
                     weight, size, eps);
  L2C_LAUNCH_CHECK();
  return hipSuccess;
}

extern "C" int l2c_softmax(float *out, const float *logits, int size, int batch,
                           hipStream_t stream) {
  if (size <= 0 || batch < 0) return hipErrorInvalidValue;
  if (batch == 0) return hipSuccess;
  if (!out || !logits) return hipErrorInvalidValue;
  const RowConfig cfg = choose_row_config(size);
  const bool vec = size % 4 == 0 && l2c_aligned16(out) && l2c_aligned16(logits);
  hipLaunchKernelGGL(soft_fn(cfg, vec), dim3(batch), dim3(cfg.threads), 0, stream, out, logits,
                     size);
  L2C_LAUNCH_CHECK();
  return hipSuccess;
}

extern "C" int l2c_matvec(float *out, const float *x, const float *W, int cols, int rows,
                          int variant, hipStream_t stream) {
  if (cols <= 0 || rows < 0) return hipErrorInvalidValue;
  if (variant != L2C_MATVEC_NAIVE && variant != L2C_MATVEC_COALESCED) return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
  if (!out || !x || !W) return hipErrorInvalidValue;
  if (variant == L2C_MATVEC_NAIVE) {
    hipLaunchKernelGGL(matvec_naive_kernel, dim3((rows + 63) / 64), dim3(64), 0, stream, out, x,
                       W, cols, rows);
  } else {
    const bool vec = cols % 4 == 0 && l2c_aligned16(x) && l2c_aligned16(W);
    const dim3 grid((rows + kMatvecWaves - 1) / kMatvecWaves), block(kMatvecWaves * L2C_WAVE);
    const dim3 pair_grid((rows + kMatvecWaves / 2 - 1) / (kMatvecWaves / 2));
    if (pair_rows(cols, rows, vec) && !matvec_nontemporal(cols, rows))
      hipLaunchKernelGGL(matvec_pair_kernel<false>, pair_grid, block, 0, stream, out, x, W, cols, rows);
    else if (pair_rows(cols, rows, vec))
      hipLaunchKernelGGL(matvec_pair_kernel<true>, pair_grid, block, 0, stream, out, x, W, cols, rows);
    else if (vec && !matvec_nontemporal(cols, rows))
      hipLaunchKernelGGL((matvec_wave_kernel<true, false>), grid, block, 0, stream, out, x, W, cols, rows);
    else if (vec)
      hipLaunchKernelGGL((matvec_wave_kernel<true, true>), grid, block, 0, stream, out, x, W, cols, rows);
    else
      hipLaunchKernelGGL((matvec_wave_kernel<false, true>), grid, block, 0, stream, out, x, W, cols,
                         rows);
  }
  L2C_LAUNCH_CHECK();
  return hipSuccess;
}

extern "C" int l2c_fused(float *normalized, const float *input, const float *weight,
                         float *softmax, const float *logits, float *product,
                         const float *matrix, int size, int rms_rows, int softmax_rows,
                         int matmul_rows, float eps, hipStream_t stream) {
  // Matrix row indexes (block x rows per block + wave) stay below INT_MAX.
  if (size <= 0 || rms_rows < 0 || softmax_rows < 0 || matmul_rows < 0 || matmul_rows > 0x7fffffff - 64)
    return hipErrorInvalidValue;
  const RowConfig cfg = choose_row_config(size);
  auto ok = [](const void *p) { return p == nullptr || l2c_aligned16(p); };
  const bool vec = size % 4 == 0 && ok(normalized) && ok(input) && ok(weight) && ok(softmax) &&
                   ok(logits) && ok(matrix);
  const bool pair = pair_rows(size, matmul_rows, vec);
  const long long items = fused_items(cfg, pair, rms_rows, softmax_rows, matmul_rows);
  if (items == 0) return hipSuccess;
  if (items > 0x7fffffffLL) return hipErrorInvalidValue;
  if (rms_rows > 0 && (!normalized || !input || !weight)) return hipErrorInvalidValue;
  if (softmax_rows > 0 && (!softmax || !logits)) return hipErrorInvalidValue;
  if (matmul_rows > 0 && (!product || !matrix || !input)) return hipErrorInvalidValue;
  const FusedFn fn = fused_fn(cfg, vec, matvec_nontemporal(size, matmul_rows));
  if (!fn) return hipErrorNotSupported;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(items)), dim3(cfg.threads), 0, stream, normalized, input,
                     weight, softmax, logits, product, matrix, size, rms_rows, softmax_rows, matmul_rows,
                     pair ? 1 : 0, eps);
  L2C_LAUNCH_CHECK();
  return hipSuccess;
}

// Launch shapes of the other translation units' kernels.
int l2c_gemm_launch_shape(int batch, int cols, int rows, int *grid, int *block,
                          int *blocks_per_cu);
int l2c_qgemm_launch_shape(int fmt, int batch, int cols, int rows, int *grid, int *block,
                           int *blocks_per_cu);
int l2c_scgemm_occupancy(int fmt, bool wide, int *blocks_per_cu);

extern "C" int l2c_launch_shape(int op, int batch, int cols, int rows, int variant, int *grid,
                                int *block, int *blocks_per_cu) {
  if (!grid || !block || !blocks_per_cu || cols <= 0 || batch < 0 || rows < 0)
    return hipErrorInvalidValue;
  const void *fn = nullptr;
  switch (op) {
    case L2C_OP_RMSNORM:
    case L2C_OP_SOFTMAX: {
      const RowConfig cfg = choose_row_config(cols);
      const bool vec = cols % 4 == 0;
      fn = op == L2C_OP_RMSNORM ? reinterpret_cast<const void *>(rms_fn(cfg, vec))
                                : reinterpret_cast<const void *>(soft_fn(cfg, vec));
      *grid = batch;
      *block = cfg.threads;
      break;
    }
    case L2C_OP_MATVEC:
      if (variant == L2C_MATVEC_NAIVE) {
        fn = reinterpret_cast<const void *>(matvec_naive_kernel);
        *grid = (rows + 63) / 64;
        *block = 64;
      } else if (variant == L2C_MATVEC_COALESCED && pair_rows(cols, rows, cols % 4 == 0)) {
        fn = reinterpret_cast<const void *>(matvec_pair_kernel<true>);
        *grid = (rows + kMatvecWaves / 2 - 1) / (kMatvecWaves / 2);
        *block = kMatvecWaves * L2C_WAVE;
      } else if (variant == L2C_MATVEC_COALESCED) {
        fn = cols % 4 == 0 ? reinterpret_cast<const void *>(matvec_wave_kernel<true, true>)
                           : reinterpret_cast<const void *>(matvec_wave_kernel<false, true>);
        *grid = (rows + kMatvecWaves - 1) / kMatvecWaves;
        *block = kMatvecWaves * L2C_WAVE;
      } else {
        return hipErrorInvalidValue;
      }
      break;
    case L2C_OP_FUSED: {
      const RowConfig cfg = choose_row_config(cols);
      fn = reinterpret_cast<const void *>(fused_fn(cfg, cols % 4 == 0, matvec_nontemporal(cols, rows)));
      const long long items = fused_items(cfg, pair_rows(cols, rows, cols % 4 == 0), batch, batch, rows);
      if (!fn || items > 0x7fffffffLL) return hipErrorInvalidValue;
      *grid = static_cast<int>(items);
      *block = cfg.threads;
      break;
    }
    case L2C_OP_MATMUL:
      return l2c_gemm_launch_shape(batch, cols, rows, grid, block, blocks_per_cu);
    case L2C_OP_MATMUL_Q:
      return l2c_qgemm_launch_shape(variant, batch, cols, rows, grid, block, blocks_per_cu);
    case L2C_OP_MATMUL_QS: {
      if (variant != L2C_Q_MXFP4 && variant != L2C_Q_FP8) return hipErrorInvalidValue;
      if (batch > 0 && rows > 0 && l2c_scgemm_ksplit_launch_shape(variant, batch, cols, rows, grid, block, &fn)) break;
      // MXFP4 with cols % 512 == 0 runs on 128 x 256 tiles (for a 16-byte
      // aligned scale array, as the harness's is), the rest on 256 x 128.
      const bool wide = variant == L2C_Q_MXFP4 && cols % 512 == 0;
      *grid = wide ? ((batch + 127) / 128) * ((rows + 255) / 256) : ((batch + 255) / 256) * ((rows + 127) / 128);
      *block = 512;
      return l2c_scgemm_occupancy(variant, wide, blocks_per_cu);
    }
    default:
      return hipErrorInvalidValue;
  }
  return static_cast<int>(hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, fn, *block, 0));
}

extern "C" const char *l2c_strerror(int code) {
  if (code == 0) return "success";
  return hipGetErrorString(static_cast<hipError_t>(code));
}

extern "C" const char *l2c_version(void) { return "l2c 0.1 gfx950"; }
