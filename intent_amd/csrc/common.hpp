// Shared helpers of libintent_hip.so (gfx950 / CDNA4, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "intent_hip.h"

namespace intent_hip {

// ---------------------------------------------------------------- host-side status handling
// Records `message` as the calling thread's last error and returns `status`.
int fail(int status, const char *format, ...) __attribute__((format(printf, 2, 3)));
// Turns the HIP runtime's launch status into an ABI status.
int launch_status(const char *kernel);

inline hipStream_t as_stream(void *stream) { return reinterpret_cast<hipStream_t>(stream); }

inline bool aligned(const void *p, unsigned bytes) {
  return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
}

// Workgroups of `kernel` (with `block` threads) the current device holds at once: CUs x resident
// workgroups per CU, queried once per device and kernel.
int resident_blocks(const void *kernel, int block);

// Compute units of the current device, queried once per device.
int device_cus();

// Fills `out` from hipFuncGetAttributes of `kernel`.
int describe_kernel(const void *kernel, const char *name, int block_threads,
                    IntentHipKernelResources *out);

// Kernel selection facts exported by each operator file for intent_hip_kernel_resources() and
// intent_hip_call_resources().
int softmax_fwd_resources(int dtype, const void *x, const void *y, int64_t rows, int64_t cols, int64_t xs, int64_t ys,
                          IntentHipKernelResources *out);
int softmax_bwd_resources(int dtype, const void *p, const void *dy, const void *dx, int64_t rows, int64_t cols, int64_t ps,
                          int64_t dys, int64_t dxs, IntentHipKernelResources *out);
int gemm_resources(int dtype, int activation, const void *a, const void *b, const void *c, int64_t m, int64_t n, int64_t k,
                   int64_t lda, int64_t ldb, int64_t ldc, IntentHipKernelResources *out);
int gemm_f32_resources(const void *a, const void *b, const void *c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                       int64_t ldc, int transpose_b, IntentHipKernelResources *out);
int gemm_i8_resources(int64_t m, int64_t n, IntentHipKernelResources *out);
int quantized_gemm_resources(const void *a, const void *b, const void *residual, const void *out, int64_t m, int64_t n,
                             int64_t k, int64_t lda, int64_t ldb, int64_t ldr, int64_t ldo, IntentHipKernelResources *to);
int attention_resources(int dtype, int64_t sq, int64_t d, int64_t dv, int mode, IntentHipKernelResources *out);
int spmv_resources(int64_t rows, int64_t nnz, IntentHipKernelResources *out);
int attention_bwd_resources(int64_t which, int64_t rows, int64_t d, IntentHipKernelResources *out);
int attention_bwd_dkdv_resources(int64_t batch, int64_t q_heads, int64_t head_group, int64_t sq, int64_t sk, int64_t d,
                                 bool causal, bool workspace, IntentHipKernelResources *out);
int decode_resources(int64_t which, int64_t d, int64_t group, IntentHipKernelResources *out);
int paged_decode_resources(int64_t batch, int64_t kv_heads, int64_t group, int64_t d, int64_t positions, int64_t ps,
                           int64_t splits, IntentHipKernelResources *out);
int spmm_resources(int64_t features, IntentHipKernelResources *out);

// f32 products of few output tiles (gemm_f32_few.hip); `workspace` may be null (one workgroup per tile).
bool gemm_f32_few_applies(int64_t m, int64_t n, int64_t k);
size_t gemm_f32_few_bytes(int64_t m, int64_t n, int64_t k);
int gemm_f32_few_resources(int64_t m, int64_t n, int64_t k, int transpose_b, IntentHipKernelResources *out);
int launch_gemm_f32_few(const float *a, const float *b, float *c, int M, int N, int K, int64_t lda, int64_t ldb,
                        int64_t ldc, int transpose_b, void *workspace, size_t workspace_bytes, hipStream_t s);

constexpr int kWave = 64;

// A launch has fewer than 2^32 threads along each axis. Grids of one workgroup per tile go on along z past kGridX
// workgroups in x (a multiple of 8, below the limit for workgroups of up to 512 threads).
constexpr int64_t kGridX = int64_t{1} << 22;
inline dim3 tile_grid(int64_t tiles, int splits) {
  const int64_t blocks = (tiles + 7) / 8 * 8, z = (blocks + kGridX - 1) / kGridX;
  return dim3(static_cast<unsigned>(z > 1 ? kGridX : blocks), static_cast<unsigned>(splits), static_cast<unsigned>(z));
}
__device__ __forceinline__ int grid_block() { return static_cast<int>(blockIdx.x + blockIdx.z * static_cast<unsigned>(kGridX)); }

// Tile of workgroup `block` of a tile_grid (grid_block(), or blockIdx.x where there are few tiles), or -1 for none, when
// each XCD shall take one run of consecutive tiles (neighbouring tiles share an operand through its L2): workgroups go
// to the 8 XCDs in turn. The runs differ by one tile at most.
__device__ __forceinline__ int xcd_tile(int block, int tiles) {
  const int xcd = block & 7;
  const int first = static_cast<int>(static_cast<int64_t>(tiles) * xcd / 8);
  const int last = static_cast<int>(static_cast<int64_t>(tiles) * (xcd + 1) / 8);
  const int tile = first + (block >> 3);
  return tile < last ? tile : -1;
}

// ---------------------------------------------------------------- wave-wide reductions
// Cross-lane moves use DPP within each 16-lane row (quad permutes, half-row and
// row mirrors), then v_readlane of the four row results: no LDS traffic and no
// barrier. Every lane of the wave must be active.
template <int kCtrl>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, false));
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// maximum_num semantics: fmaxf returns the non-NaN operand when one side is NaN.
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_move<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_move<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_move<0x141>(v));  // row_half_mirror
  v = fmaxf(v, dpp_move<0x140>(v));  // row_mirror
  return fmaxf(fmaxf(lane_value(v, 0), lane_value(v, 16)), fmaxf(lane_value(v, 32), lane_value(v, 48)));
}

__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_move<0xB1>(v);
  v += dpp_move<0x4E>(v);
  v += dpp_move<0x141>(v);
  v += dpp_move<0x140>(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// ---------------------------------------------------------------- 16-bit float conversions
// Storage types are raw 16-bit patterns; arithmetic is f32.
struct f16_t {
  uint16_t bits;
};
struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(f16_t v) {
  return static_cast<float>(__builtin_bit_cast(_Float16, v.bits));
}
__device__ __forceinline__ float to_f32(bf16_t v) {
  return __uint_as_float(static_cast<uint32_t>(v.bits) << 16);
}

// f32 -> _Float16 or __bf16, rounded to nearest even. The empty asm makes v opaque, so
// instruction selection cannot fuse the conversion with the f32 product or FMA that produced v:
// v_fma_mixlo_f16 would round once, straight to 16 bits, where the definitions round the f32
// result and then cast. It emits no instruction.
template <typename E>
__device__ __forceinline__ E round_to(float v) {
  asm("" : "+v"(v));
  return static_cast<E>(v);
}

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ f16_t from_f32<f16_t>(float v) {
  // v_cvt_f16_f32 rounds to nearest even; finite overflow gives infinity.
  return f16_t{__builtin_bit_cast(uint16_t, round_to<_Float16>(v))};
}
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) {
  // v_cvt_pk_bf16_f32: round to nearest even; NaN stays a (quiet) NaN.
  return bf16_t{__builtin_bit_cast(uint16_t, round_to<__bf16>(v))};
}

}  // namespace intent_hip
