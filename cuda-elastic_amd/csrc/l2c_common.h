// Device-side helpers shared by the l2c kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <cfloat>
#include <cstdint>

#define L2C_WAVE 64

namespace l2c {

// Butterfly sum over the 64 lanes of a wavefront; every lane gets the total.
// __shfl_xor lowers to ds_swizzle / ds_bpermute, which use the LDS crossbar
// but no LDS allocation.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, L2C_WAVE);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, L2C_WAVE));
  return v;
}

// Block-wide reductions through one LDS slot per wave. Every thread returns
// the result. Each call site passes its own slot array, so two reductions in
// a row need no barrier between them. The cross-wave sum runs in wave order,
// so the result does not depend on scheduling.
__device__ __forceinline__ float block_sum(float v, float *slots) {
  v = wave_sum(v);
  const int waves = blockDim.x / L2C_WAVE;
  if (threadIdx.x % L2C_WAVE == 0) slots[threadIdx.x / L2C_WAVE] = v;
  __syncthreads();
  float total = 0.0f;
  for (int w = 0; w < waves; ++w) total += slots[w];
  return total;
}

__device__ __forceinline__ float block_max(float v, float *slots) {
  v = wave_max(v);
  const int waves = blockDim.x / L2C_WAVE;
  if (threadIdx.x % L2C_WAVE == 0) slots[threadIdx.x / L2C_WAVE] = v;
  __syncthreads();
  float m = -FLT_MAX;
  for (int w = 0; w < waves; ++w) m = fmaxf(m, slots[w]);
  return m;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16-byte loads and stores with the nontemporal hint: data touched once
// streams through the caches without displacing reused operands.
__device__ __forceinline__ float4 ld4_stream(const float4 *p) {
  const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void st4_stream(float4 *p, float4 v) {
  const f32x4 w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, reinterpret_cast<f32x4 *>(p));
}

// The same for rows at any 4-byte address: the memory instructions need only
// that, and a row whose length is no multiple of four floats then costs an extra
// cache line now and then instead of four loads of one float.
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 ld4_any(const float *p) {
  const f32x4_a4 v = *reinterpret_cast<const f32x4_a4 *>(p);
  return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ float4 ld4_any_stream(const float *p) {
  const f32x4_a4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4 *>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void st4_any(float *p, float4 v) {
  const f32x4_a4 w = {v.x, v.y, v.z, v.w};
  *reinterpret_cast<f32x4_a4 *>(p) = w;
}
// The last, partial chunk of a row: `rest` of 1 to 3 floats, `fill` after them.
__device__ __forceinline__ float4 ld_rest(const float *p, int rest, float fill) {
  return make_float4(p[0], rest > 1 ? p[1] : fill, rest > 2 ? p[2] : fill, fill);
}
// For short rows, which such loads of their own cost a second latency: the chunk of a
// row of n floats that starts at float j < n. The partial one (j + 4 > n) comes as the
// row's last four floats, to be moved into place by whole_chunk once all loads are
// under way (rows of less than four floats one by one). Long rows lose more by an
// address for every chunk than by the second latency (rmsnorm of 59 x 7713: 5.13 us so,
// 4.75 with a load of its own; of 600 to 1200 floats 4% less so).
__device__ __forceinline__ float4 ld_chunk(const float *row, int j, int n) {
  if (n < 4) return make_float4(0.0f, n > 2 ? row[n - 3] : 0.0f, n > 1 ? row[n - 2] : 0.0f, row[n - 1]);
  return ld4_any(row + min(j, n - 4));
}
__device__ __forceinline__ float4 whole_chunk(float4 q, int j, int n, float fill) {
  const int rest = n - j;
  if (rest >= 4) return q;
  return rest == 3 ? make_float4(q.y, q.z, q.w, fill)
         : rest == 2 ? make_float4(q.z, q.w, fill, fill) : make_float4(q.w, fill, fill, fill);
}
// Stores the first `rest` (1 to 3) floats of the last, partial chunk.
__device__ __forceinline__ void st_rest(float *p, int rest, float4 v) {
  p[0] = v.x;
  if (rest > 1) p[1] = v.y;
  if (rest > 2) p[2] = v.z;
}

// Raw buffer resource over [p, p + bytes). Loads through it take a 32-bit
// per-lane byte offset plus a wave-uniform byte offset held in a scalar
// register, so a loop that walks along K advances one SGPR per step and
// spends no vector instructions on addresses. Word 3 selects the 32-bit data
// format that untyped (raw) buffer loads require on gfx9-family parts.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), static_cast<short>(0),
                                           static_cast<int>(bytes), 0x00020000);
}

// Workgroup i is dispatched to XCD i % 8. The tile order gives each XCD a
// contiguous band of the `tiles` tiles, for any number of them (the first
// tiles % 8 bands are one tile longer).
__device__ __forceinline__ int xcd_tile(int block, int tiles) {
  constexpr int kXcds = 8;
  const int xcd = block % kXcds;
  return xcd * (tiles / kXcds) + min(xcd, tiles % kXcds) + block / kXcds;
}

// Whether HIP takes a launch of this many workgroups: their lanes together stay
// below 2^32.
inline bool launchable(long long blocks, int lanes) { return blocks <= 0xffffffffLL / lanes; }

}  // namespace l2c

// Return code plumbing shared by the extern "C" entry points.
#define L2C_LAUNCH_CHECK()                      \
  do {                                          \
    hipError_t e__ = hipGetLastError();         \
    if (e__ != hipSuccess) return (int)e__;     \
  } while (0)

static inline bool l2c_aligned16(const void *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// The quantized-weight kernel's bf16 form (l2c_qgemm.hip), for contractions
// whose K is not a multiple of 64.
int l2c_matmul_bf16_split(float *out, const uint16_t *X, const uint16_t *W, const float *alpha, int batch, int cols,
                          int rows, hipStream_t stream);
// The quantized-weight contraction for cols % 64 == 0 (l2c_qgemm_ks.hip),
// called by l2c_matmul_q after its argument checks.
int l2c_matmul_q_ks(float *out, const uint16_t *X, const uint8_t *Wq, const void *scales, int fmt, int batch,
                    int cols, int rows, hipStream_t stream);
// Workgroups of that kernel resident per CU (512-lane workgroups, one per
// tile: 256 x 128 for MXFP4, 128 x 256 for fp8).
int l2c_qgemm_ks_occupancy(int fmt, int *blocks_per_cu);
// Workgroups l2c_matmul_q_ks launches for this shape (its tile depends on fmt).
long long l2c_qgemm_ks_tiles(int fmt, int batch, int rows);
// The contractions on small k-split tiles (l2c_gemm_ksplit.hip,
// l2c_qgemm_ksplit.hip, l2c_scgemm_ksplit.hip), called by the entry points after
// their argument checks (batch and rows above 0). Each launches and returns true
// where its shape's small tiles are to be preferred to the large ones, and
// returns false otherwise; the caller reads the launch's error. The
// launch_shape forms return the same choice.
//  * fp32; `aligned`: both operands' rows start at 16-byte addresses.
bool l2c_gemm_ksplit(float *out, const float *X, const float *W, int batch, int cols, int rows, bool aligned,
                     hipStream_t stream);
bool l2c_gemm_ksplit_launch_shape(int batch, int cols, int rows, bool aligned, int *grid, int *block,
                                  const void **fn);
//  * bf16 activations: fmt is an l2c_qformat, or 2 for bf16 weights with the
//    device alpha in `scales`; `large_tiles` tiles of the large kernel. Also
//    takes the shapes of the 128 x 128 tiles (l2c_qgemm_mid.hip).
bool l2c_qgemm_ksplit(float *out, const uint16_t *X, const uint8_t *Wq, const void *scales, int fmt, int batch,
                      int cols, int rows, long long large_tiles, hipStream_t stream);
bool l2c_qgemm_ksplit_launch_shape(int fmt, int batch, int cols, int rows, long long large_tiles, int *grid, int *block,
                                   const void **fn);
//  * block-scaled: fmt is an l2c_qformat with MXFP8 activations as
//    l2c_quantize_mxfp8 leaves them, or 2 for MXFP6 operands.
bool l2c_scgemm_ksplit(float *out, const uint8_t *X, const uint8_t *Xs, const uint8_t *Wq, const void *wscales,
                       int fmt, int batch, int cols, int rows, hipStream_t stream);
bool l2c_scgemm_ksplit_launch_shape(int fmt, int batch, int cols, int rows, int *grid, int *block, const void **fn);
void (*l2c_qgemm_mid_kernel(int fmt))(float *, const uint16_t *, const uint8_t *, const void *, int, int, int);
