// bf16-activation contractions on 128 x 128 tiles: out[b][r] = sum_k X[b][k] *
// deq(W)[r][k] with MXFP4, per-row-scaled fp8 or bf16 weights, K % 64 == 0, for
// shapes between the k-split tiles (l2c_qgemm_ksplit.hip), which stage a row of X
// or W too often to multiply many of both, and the large ones (l2c_qgemm_ks.hip,
// l2c_bfgemm.hip), of which there are too few to fill the CUs: twice as many tiles
// in little more than half the time each.
//
//  * v_mfma_f32_32x32x16_bf16, codes converted exactly to bf16 in registers, as in
//    the large kernels, whose fragment layout this keeps: 8 wavefronts, waves w
//    and w + 4 on the same 64 x 64 sub-tile (2 x 2 blocks of 32 x 32), wave group
//    g = w / 4 taking k-chunks 2 g and 2 g + 1 of every 64-deep slice; the groups'
//    partial sums are added once at the end through LDS.
//  * A ring of 6 (MXFP4), 5 (fp8) or 4 (bf16) slices filled by LDS DMA, chunks
//    XOR-swizzled on the source side; MXFP4 scales as 2-byte DMAs, one row a lane
//    (waves 4 and 5; waves 6 and 7 repeat the W DMAs of waves 2 and 3, so that
//    every wave issues as many DMAs and waits by the same count).
//  * One barrier a slice: behind it a wave reads the fragments of the next slice
//    into a second register set while it multiplies the present one.
//  * Bounds: LDS traffic (72 KB a slice, about 560 cycles) and the MFMAs (512)
//    next to each other more than on top; 5.7 to 7.1 ns a k of every tile. A form
//    with the large kernels' ping-pong schedule measured the same (35 to 38 us at
//    256 x 4096 x 11008 against 32 to 40 here), and two slices a step 32.5 for fp8
//    and 46 for MXFP4. At 1024 x 1024 x 4096 MXFP4 / fp8 / bf16, us: 14.2 / 14.7 /
//    17.4, k-split tiles 34 / 23 / 19, large tiles 19.3 / 20 / 19; 512 x 8192 x
//    8192: 74 / 71 / 67, large 84 / 79 / 76.
//  * Rows past the operands are clamped to the last row and not stored.
#include "l2c_common.h"
#include "../../include/l2c.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_ptr;

constexpr int kFmtBf16 = 2;  // bf16 weights; `scales` is the device alpha or null
constexpr int kBM = 128, kBN = 128, kThreads = 512;
constexpr int kExchange = 4 * 4 * 16 * L2C_WAVE * 4;  // 4 sub-tiles x 4 blocks x 16 values x 64 lanes

template <int FMT>
struct Layout {
  static constexpr bool kMx = FMT == L2C_Q_MXFP4;
  static constexpr int kWRow = kMx ? 32 : FMT == L2C_Q_FP8 ? 64 : 128;  // code bytes of a W row and slice
  static constexpr int kXBytes = kBM * 128;
  static constexpr int kWInstr = kBN * kWRow / 1024;                    // W DMAs of a slice
  static constexpr int kSOff = kXBytes + kBN * kWRow;
  static constexpr int kSlice = kSOff + (kMx ? kBN * 4 : 0);
  static constexpr int kRing = kMx ? 6 : FMT == L2C_Q_FP8 ? 5 : 4;      // slices in the ring
  static constexpr int kDma = FMT == kFmtBf16 ? 4 : 3;                  // DMAs each wave issues a slice
  static constexpr int kLds = kRing * kSlice > kExchange ? kRing * kSlice : kExchange;
  static __device__ __forceinline__ int wswizzle(int row) {
    return kMx ? (row >> 3) & 1 : FMT == L2C_Q_FP8 ? (row >> 2) & 3 : (row >> 1) & 7;
  }
};

__device__ __forceinline__ int xswizzle(int row) { return (row >> 1) & 7; }

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, unsigned char *dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr *)dst, 16, voffset, soffset, 0, 0);
}
__device__ __forceinline__ void dma2(__amdgpu_buffer_rsrc_t rsrc, unsigned char *dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr *)dst, 2, voffset, soffset, 0, 0);
}

template <int FMT>
__global__ __launch_bounds__(kThreads, 1) void qgemm_mid_kernel(float *__restrict__ out,
                                                                const uint16_t *__restrict__ X,
                                                                const uint8_t *__restrict__ Wq,
                                                                const void *__restrict__ scales, int M, int N,
                                                                int K) {
  using L = Layout<FMT>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[L::kLds];
  const int tile = l2c::xcd_tile(blockIdx.x, gridDim.x);
  const int mtiles = (M + kBM - 1) / kBM;
  const int m0 = (tile % mtiles) * kBM, n0 = (tile / mtiles) * kBN;
  const int mrows = min(kBM, M - m0), nrows = min(kBN, N - n0);
  const int tid = threadIdx.x, lane = tid % L2C_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / L2C_WAVE);
  const int g = wave >> 2, p = wave & 3;
  const int wm = p & 1, wn = p >> 1;
  const int r = lane % 32, h = lane / 32;
  const int xrb = 2 * K, wrb = L::kMx ? K / 2 : FMT == L2C_Q_FP8 ? K : 2 * K, srb = K / 32;
  const __amdgpu_buffer_rsrc_t rx =
      l2c::buffer_rsrc(X + static_cast<size_t>(m0) * K, static_cast<uint32_t>(mrows) * xrb);
  const __amdgpu_buffer_rsrc_t rw =
      l2c::buffer_rsrc(Wq + static_cast<size_t>(n0) * wrb, static_cast<uint32_t>(nrows) * wrb);
  const __amdgpu_buffer_rsrc_t rs =
      L::kMx ? l2c::buffer_rsrc(static_cast<const uint8_t *>(scales) + static_cast<size_t>(n0) * srb,
                                static_cast<uint32_t>(nrows) * srb)
             : rw;

  // DMA sources (per-lane parts; the slice's k offset is scalar): X instruction
  // 8 k + wave fills rows 8 (8 k + wave) + lane / 8, W instruction 8 k + wi rows
  // kRows (8 k + wi) + lane / kSlots.
  int xsrc[2], wsrc[2] = {0, 0};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int row = 8 * (8 * k + wave) + lane / 8;
    xsrc[k] = min(row, mrows - 1) * xrb + 16 * ((lane % 8) ^ xswizzle(row));
  }
  constexpr int kSlots = L::kWRow / 16, kRows = 64 / kSlots;
  const int wi = L::kMx ? wave & 3 : wave;
#pragma unroll
  for (int k = 0; k < (FMT == kFmtBf16 ? 2 : 1); ++k) {
    const int row = kRows * (8 * k + wi) + lane / kSlots;
    wsrc[k] = min(row, nrows - 1) * wrb + 16 * ((lane % kSlots) ^ L::wswizzle(row));
  }
  const int ssrc = min(64 * (wave & 1) + lane, nrows - 1) * srb;
  const bool scale_wave = L::kMx && (wave == 4 || wave == 5);
  auto dma = [&](unsigned char *d, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) dma16(rx, d + (8 * k + wave) * 1024, xsrc[k], 128 * t);
    if (scale_wave) {
      dma2(rs, d + L::kSOff + (wave & 1) * 256, ssrc, 2 * t);
    } else {
#pragma unroll
      for (int k = 0; k < (FMT == kFmtBf16 ? 2 : 1); ++k)
        dma16(rw, d + L::kXBytes + (8 * k + wi) * 1024, wsrc[k], L::kWRow * t);
    }
  };
  // This wave's DMAs of all but the kRing - 2 newest slices have landed and its LDS
  // reads are done; then the workgroup barrier.
  auto wait_barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((L::kRing - 2) * L::kDma) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // Fragments: X rows wm * 64 + 32 i + r, chunks 4 h + 2 g (+ 1); W rows wn * 64 +
  // 32 j + r, the codes of the same k (MXFP4: half a chunk; the row's scale word,
  // byte h the lane's block). The swizzles of rows + 32 equal those of the rows.
  const int xsw = xswizzle(r);
  const int a0 = (wm * 64 + r) * 128;
  const int c0 = 16 * ((4 * h + 2 * g) ^ xsw), c1 = 16 * ((4 * h + 2 * g + 1) ^ xsw);
  const int wr0 = wn * 64 + r, wsw = L::wswizzle(wr0);
  const int w0 = L::kXBytes + wr0 * L::kWRow;
  const int wb0 = L::kMx ? w0 + 16 * (h ^ wsw) + 8 * g
                  : FMT == L2C_Q_FP8 ? w0 + 16 * ((2 * h + g) ^ wsw) : w0 + 16 * ((4 * h + 2 * g) ^ wsw);
  const int wb1 = w0 + 16 * ((4 * h + 2 * g + 1) ^ wsw);  // bf16's second chunk
  const int sb = L::kSOff + 4 * wr0;
  struct Frags {
    u32x4 a[2][2];
    u32x4 w[2][FMT == kFmtBf16 ? 2 : 1];
    uint32_t s[2];
  };
  auto read = [&](Frags &f, const unsigned char *d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (L::kMx) {
        const u32x2 v = *reinterpret_cast<const u32x2 *>(d + wb0 + 32 * L::kWRow * j);
        f.w[j][0][0] = v[0], f.w[j][0][1] = v[1];
        f.s[j] = *reinterpret_cast<const uint32_t *>(d + sb + 128 * j);
      } else {
        f.w[j][0] = *reinterpret_cast<const u32x4 *>(d + wb0 + 32 * L::kWRow * j);
        if constexpr (FMT == kFmtBf16) f.w[j][1] = *reinterpret_cast<const u32x4 *>(d + wb1 + 32 * L::kWRow * j);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f.a[i][0] = *reinterpret_cast<const u32x4 *>(d + a0 + 4096 * i + c0);
      f.a[i][1] = *reinterpret_cast<const u32x4 *>(d + a0 + 4096 * i + c1);
    }
  };
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  auto multiply = [&](const Frags &f) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      bf16x8 b[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint32_t d[4];
        if constexpr (L::kMx) {
          const float scale = __uint_as_float(((f.s[j] >> (8 * h)) & 0xffu) << 23);
          const uint32_t w = f.w[j][0][c];
          d[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 0));
          d[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 1));
          d[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 2));
          d[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 3));
        } else if constexpr (FMT == L2C_Q_FP8) {
          const uint32_t u = f.w[j][0][2 * c], v = f.w[j][0][2 * c + 1];
          d[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, false));
          d[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, true));
          d[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, false));
          d[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, true));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e] = f.w[j][c][e];
        }
        b[j] = __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3]));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f.a[i][c]), b[j], acc[i][j],
                                                              0, 0, 0);
    }
  };

  // What the sums of the lane's two output columns are multiplied by, loaded ahead of
  // the DMAs: loads and stores complete in order, and a load between the epilogue's
  // stores waits for them.
  float factor[2] = {1.0f, 1.0f};
  if constexpr (FMT == kFmtBf16) {
    if (scales) factor[0] = factor[1] = *static_cast<const float *>(scales);
  } else if constexpr (FMT == L2C_Q_FP8) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      factor[j] = static_cast<const float *>(scales)[n0 + min(wn * 64 + 32 * j + r, nrows - 1)];
  }
  const int total = K / 64, last = total - 1;
#pragma unroll
  for (int t = 0; t < L::kRing - 1; ++t) dma(lds + t * L::kSlice, min(t, last));
  wait_barrier();  // slice 0 landed everywhere
  Frags f0, f1;
  read(f0, lds);
  int cur = 0;
  auto step = [&](int t, const Frags &use, Frags &next) __attribute__((always_inline)) {
    // `use` holds slice t, in ring place `cur`. The place before it held slice
    // t - 1, whose fragments had arrived in every wave before the last barrier;
    // behind this one slice t + 1 has landed everywhere. Slices past the last
    // re-read it into places nobody multiplies any more.
    const int before = cur == 0 ? L::kRing - 1 : cur - 1, after = cur == L::kRing - 1 ? 0 : cur + 1;
    dma(lds + before * L::kSlice, min(t + L::kRing - 1, last));
    wait_barrier();
    read(next, lds + after * L::kSlice);
    __builtin_amdgcn_sched_barrier(0);
    multiply(use);
    cur = after;
  };
  int t = 0;
  for (; t + 2 <= total; t += 2) {
    step(t, f0, f1);
    step(t + 1, f1, f0);
  }
  if (t < total) multiply(f0);

  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float *exchange = reinterpret_cast<float *>(lds);
  if (g == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) exchange[((p * 4 + i * 2 + j) * 16 + v) * L2C_WAVE + lane] = acc[i][j][v];
  }
  __syncthreads();
  if (g == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = wn * 64 + 32 * j + r;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = wm * 64 + 32 * i + 8 * (v / 4) + 4 * h + v % 4;
          const float sum = acc[i][j][v] + exchange[((p * 4 + i * 2 + j) * 16 + v) * L2C_WAVE + lane];
          if (m < mrows && n < nrows)
            __builtin_nontemporal_store(sum * factor[j], &out[static_cast<size_t>(m0 + m) * N + n0 + n]);
        }
    }
  }
}

}  // namespace

void (*l2c_qgemm_mid_kernel(int fmt))(float *, const uint16_t *, const uint8_t *, const void *, int, int, int) {
  return fmt == L2C_Q_MXFP4 ? qgemm_mid_kernel<L2C_Q_MXFP4>
         : fmt == L2C_Q_FP8 ? qgemm_mid_kernel<L2C_Q_FP8>
                            : qgemm_mid_kernel<kFmtBf16>;
}
