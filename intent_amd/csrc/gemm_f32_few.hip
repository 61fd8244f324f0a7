// f32 GEMM with few output tiles, for gfx950: the products that gemm_f32.hip's 128 x 128 tiles would run on a part of
// the chip (same definitions: gemm_f32 and linear_f32, contraction/gemm.py:15-38, f32 products and sums).
#include "common.hpp"

namespace intent_hip {
namespace {

// ---------------------------------------------------------------- few tiles: the waves of a workgroup split K
// Where 128 x 128 tiles are too few to fill the chip, the bound is still the matrix rate, so the work has to reach
// every CU: a workgroup owns MT * 16 rows and 64 columns, and its four waves take the 32-deep units of K in
// turn, each with the whole tile in its accumulators and its operands loaded straight into
// registers (the next unit in flight while the current one is multiplied; no LDS, no barrier in the loop).
// The waves' sums meet in LDS. With fewer tiles than CUs, K is also divided over workgroups (blockIdx.y): each
// writes its sums to `partials`, and gemm_f32_splits adds them in order.
//   * v_mfma_f32_16x16x4f32; lane (g = l / 16, r = l % 16) loads the 4 consecutive k = 4 g .. 4 g + 3 of a
//     unit for row r of A (and of W): 64 contiguous bytes per row; instruction i multiplies k = 4 g + i of
//     every g, in both operands alike;
//   * natural B: the lane loads rows k = 4 g + i (i = 0..3), columns 4 r .. 4 r + 3: 256 contiguous bytes
//     per row; column tile t is then the columns 4 r + t;
//   * 16-byte loads need only 4-byte alignment, so every row stride takes this path; groups of 4 that
//     reach past K, or past N for natural B, are loaded one element at a time, zeros past K.
// Measured: linear_f32 256 x 1000 x 2048 158 -> 17.6 us (matrix-rate floor 7; the rest is the first loads, the LDS
// sum and the second launch), 1 x 4096 x 4096 310 -> 15, 2048 x 1024 x 4096 316 -> 144 (119 TFLOP/s).
constexpr int kFewCols = 64, kFewUnit = 32, kFewWaves = 4;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));

// 4 consecutive floats at p, `count` of them (0..4) present; zeros for the others.
__device__ __forceinline__ f32x4_t load_4(const float *p, int count) {
  if (count >= 4) return *reinterpret_cast<const f32x4_any_t *>(p);
  f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (count > 0) v[0] = p[0];
  if (count > 1) v[1] = p[1];
  if (count > 2) v[2] = p[2];
  return v;
}

// The first `count` (at least 1) of 4 floats, at any 4-byte boundary.
__device__ __forceinline__ void store_4(float *p, f32x4_t v, int count) {
  if (count >= 4) {
    *reinterpret_cast<f32x4_any_t *>(p) = v;
  } else {
    p[0] = v[0];
    if (count > 1) p[1] = v[1];
    if (count > 2) p[2] = v[2];
  }
}

template <bool kTransB, int MT>
__global__ __launch_bounds__(kFewWaves * 64) void gemm_f32_few(const float *__restrict__ A, const float *__restrict__ B,
                                                               float *__restrict__ C, int M, int N, int K, int64_t lda,
                                                               int64_t ldb, int64_t ldc, int tiles_m,
                                                               int tiles_n, float *__restrict__ partials) {
  constexpr int kRows = MT * 16, kPad = kFewCols + 4, W = kFewWaves;
  __shared__ float4 sums[W * kRows * kPad / 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  // The row blocks of one column block are neighbours on one XCD; with one row block the XCDs take turns.
  const int tile = tiles_m == 1 ? grid_block() : xcd_tile(grid_block(), tiles_m * tiles_n);
  if (tile < 0 || tile >= tiles_m * tiles_n) return;
  const int m0 = (tile % tiles_m) * kRows, n0 = (tile / tiles_m) * kFewCols;

  // Rows past M or N read a valid row; their products are not stored.
  const float *a_row[MT], *b_row[4];
#pragma unroll
  for (int t = 0; t < MT; ++t) a_row[t] = A + static_cast<int64_t>(min(m0 + 16 * t + r, M - 1)) * lda + 4 * g;
  const int n_count = min(N - (n0 + 4 * r), 4);   // natural B: columns of this lane
#pragma unroll
  for (int t = 0; t < 4; ++t)
    b_row[t] = kTransB ? B + static_cast<int64_t>(min(n0 + 16 * t + r, N - 1)) * ldb + 4 * g
                       : B + static_cast<int64_t>(4 * g + t) * ldb + (n_count > 0 ? n0 + 4 * r : 0);

  f32x4_t acc[MT][4];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  auto load_unit = [&](int unit, f32x4_t (&a)[2][MT], f32x4_t (&b)[2][4]) {   // wholly inside K
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t k0 = static_cast<int64_t>(unit) * kFewUnit + 16 * u;
#pragma unroll
      for (int t = 0; t < MT; ++t) a[u][t] = *reinterpret_cast<const f32x4_any_t *>(a_row[t] + k0);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        b[u][t] = kTransB ? *reinterpret_cast<const f32x4_any_t *>(b_row[t] + k0) : load_4(b_row[t] + k0 * ldb, n_count);
    }
  };
  auto multiply = [&](const f32x4_t (&a)[MT], const f32x4_t (&b)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kTransB ? b[j][i] : b[i][j], a[t][i], acc[t][j], 0, 0, 0);
  };

  const int units = K / kFewUnit;
  const int first = static_cast<int>(static_cast<int64_t>(units) * blockIdx.y / gridDim.y);
  const int last = static_cast<int>(static_cast<int64_t>(units) * (blockIdx.y + 1) / gridDim.y);
  auto multiply_unit = [&](const f32x4_t (&a)[2][MT], const f32x4_t (&b)[2][4]) {
    multiply(a[0], b[0]);
    multiply(a[1], b[1]);
  };
  f32x4_t a[2][2][MT], b[2][2][4];
  int unit = first + wave;
  if (unit < last) load_unit(unit, a[0], b[0]);
  for (; unit + W < last; unit += 2 * W) {
    load_unit(unit + W, a[1], b[1]);
    multiply_unit(a[0], b[0]);
    if (unit + 2 * W < last) load_unit(unit + 2 * W, a[0], b[0]);
    multiply_unit(a[1], b[1]);
  }
  if (unit < last) multiply_unit(a[0], b[0]);
  // The last K % 32, by the next wave in turn of the last split. (As one more unit of the loop above, with
  // the masks in load_unit, the branch made the compiler wait for every load: 620 -> 950 us at 2048 x 4095 x 4095.)
  if (K % kFewUnit != 0 && blockIdx.y == gridDim.y - 1 && wave == (last - first) % W) {
    for (int k0 = units * kFewUnit; k0 < K; k0 += 16) {
      const int count = K - (k0 + 4 * g);   // k of this lane's group of 4
#pragma unroll
      for (int t = 0; t < MT; ++t) a[0][0][t] = load_4(a_row[t] + k0, count);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        b[0][0][t] = kTransB ? load_4(b_row[t] + k0, count)
                             : load_4(b_row[t] + static_cast<int64_t>(k0) * ldb, t < count ? n_count : 0);
      multiply(a[0][0], b[0][0]);
    }
  }

  // acc[t][j][q] is row 16 t + r; column 16 j + 4 g + q of a weight's tile, 16 g + 4 q + j of natural B's.
  float *own = reinterpret_cast<float *>(sums) + wave * kRows * kPad;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = kTransB ? make_float4(acc[t][q][0], acc[t][q][1], acc[t][q][2], acc[t][q][3])
                               : make_float4(acc[t][0][q], acc[t][1][q], acc[t][2][q], acc[t][3][q]);
      *reinterpret_cast<float4 *>(own + (16 * t + r) * kPad + (kTransB ? 16 * q + 4 * g : 16 * g + 4 * q)) = v;
    }
  __syncthreads();
  const float *all = reinterpret_cast<const float *>(sums);
  for (int quad = threadIdx.x; quad < kRows * kFewCols / 4; quad += W * 64) {
    const int row = quad / (kFewCols / 4), col = 4 * (quad % (kFewCols / 4));
    const int m = m0 + row, n = n0 + col;
    if (m >= M || n >= N) continue;
    f32x4_t total = *reinterpret_cast<const f32x4_t *>(all + row * kPad + col);
#pragma unroll
    for (int w = 1; w < W; ++w) total += *reinterpret_cast<const f32x4_t *>(all + (w * kRows + row) * kPad + col);
    if (partials != nullptr) {
      const int64_t width = (N + 3) & ~3;
      *reinterpret_cast<f32x4_t *>(partials + (static_cast<int64_t>(blockIdx.y) * M + m) * width + n) = total;
    } else {
      store_4(C + static_cast<int64_t>(m) * ldc + n, total, N - n);
    }
  }
}

// Adds the K splits of a product in order: one thread per 4 columns.
__global__ __launch_bounds__(256) void gemm_f32_splits(const float *__restrict__ partials, float *__restrict__ C, int M,
                                                       int N, int64_t ldc, int splits) {
  const int quads = (N + 3) / 4;
  const int64_t quad = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, total_quads = static_cast<int64_t>(M) * quads;
  if (quad >= total_quads) return;
  const f32x4_t *p = reinterpret_cast<const f32x4_t *>(partials) + quad;
  f32x4_t total = p[0];
#pragma unroll 8
  for (int s = 1; s < splits; ++s) total += p[s * total_quads];
  const int m = static_cast<int>(quad / quads), n = 4 * static_cast<int>(quad % quads);
  store_4(C + static_cast<int64_t>(m) * ldc + n, total, N - n);
}

// Rows of a tile. 64 load two thirds of the operand bytes per product that 32 do, but with at most 128 such tiles
// twice as many of 32 rows still run in one pass and leave fewer K parts to add; in a long K the bytes count for more.
// Measured, 32 against 64 rows, a weight / natural B in us:
//   * K to 1560: 512^3 9.2 / 8.8 against 10.9 / 10.3, 1067 x 312 x 1560 19.7 / 24.0 and 32.3 / 34.0, 128 x 4096 x 1024
//     15.3 / 13.8 and 18.5 / 17.8;
//   * K = 2048: 256 x 1000 17.6 / 17.6 and 18.6 / 18.3, 128 x 4096 25.8 / 25.5 and 26.1 / 27.5, 48 x 8192 25.8 / 25.7 and
//     24.9 / 26.0;
//   * K = 3072: 256 x 1000 23.0 / 24.6 and 22.6 / 23.4, 128 x 4096 36.7 / 38.3 and 34.4 / 36.3, 48 x 8192 36.5 / 38.0 and
//     33.4 / 38.1.
// More tiles pay a second pass: 640 x 832 x 1000 (130 tiles) 28.7 / 30.0 and 21.7 / 23.4, 1024^3 32.2 / 32.9 and 23.7 / 24.7.
constexpr int64_t kFewTallTiles = 128, kFewTallDepth = 2048;
int few_rows(int64_t m, int64_t n, int64_t k) {
  if (m <= 16) return 16;
  const bool pair = (m + 63) / 64 * ((n + kFewCols - 1) / kFewCols) <= kFewTallTiles && k <= kFewTallDepth;
  return m <= 32 || pair ? 32 : 64;
}
int64_t few_tiles(int64_t m, int64_t n, int64_t k) {
  const int64_t rows = few_rows(m, n, k);
  return (m + rows - 1) / rows * ((n + kFewCols - 1) / kFewCols);
}

// Workgroups along K: about one workgroup per CU, at least 128 k each. The second launch costs about 3 us, which the split
// returns from K = 512 on, or is level there (a weight's product, divided against whole in us: 64 x 512 x 512 7.5 and
// 9.2, 256 x 512 x 512 8.3 and 9.2, 512^3 9.4 and 9.3, 16 x 512 x 512 7.3 and 7.1; 512 x 512 x 1024 12.1 and 14.7,
// 16 x 1024 x 1024 7.8 and 11.4, 256 x 1000 x 2048 17.6 and 25.1). Natural B is 0.4 to 1.8 us behind at K = 512 with 16
// rows or 128 tiles and leads from 640 on.
int few_splits(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || n < 1 || k < 512) return 1;
  const int64_t tiles = few_tiles(m, n, k);
  const int64_t splits = 256 / tiles < k / 128 ? 256 / tiles : k / 128;
  return splits < 2 ? 1 : static_cast<int>(splits);
}

template <bool kTransB>
const void *few_kernel(int rows) {
  return rows == 16   ? reinterpret_cast<const void *>(&gemm_f32_few<kTransB, 1>)
         : rows == 32 ? reinterpret_cast<const void *>(&gemm_f32_few<kTransB, 2>)
                      : reinterpret_cast<const void *>(&gemm_f32_few<kTransB, 4>);
}
const void *few_kernel(int rows, int transpose_b) { return transpose_b ? few_kernel<true>(rows) : few_kernel<false>(rows); }

}  // namespace

// The 128 x 128 kernel takes one round of the chip's 256 CUs for up to 256 tiles (k = 4096: 315 us) and runs at 130 TFLOP/s
// with many; this one at about 108 whatever the tile count, in one pass over the chip up to 64 of those tiles, in two up to 128
// and three up to 192, each with first loads and an LDS sum that a short K does not hide. Measured, the 128 x 128
// kernel's time over this one's, natural B / a weight: up to 64 tiles 1.0 to 5 at every K; 65 to 128 tiles K = 32 0.7 / 0.7,
// 64 0.92 / 0.90, 96 1.1 / 1.04, 256 1.5 / 1.4; 129 to 192 tiles K = 64 0.7 / 0.7, 192 0.9 / 0.87, 320 0.98 / 0.92, 384 1.1 /
// 1.0 (6144 x 512 0.94 / 0.93), 512 1.1 / 1.1. Up to 64 rows, half of a 128 x 128 tile: 64 x 16384 (128 tiles) K = 16 0.93 /
// 0.94, 32 1.0 / 1.05, 64 1.4 / 1.4; 33 x 30000 (235) K = 32 0.67 / 0.71, 64 0.92 / 0.91, 96 1.1 / 1.1.
bool gemm_f32_few_applies(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = (m + 127) / 128 * ((n + 127) / 128);
  if (m <= 64) return tiles <= 128 || k >= 96;
  return tiles <= 64 || (tiles <= 128 && k >= 96) || (tiles <= 192 && k >= 384);
}

size_t gemm_f32_few_bytes(int64_t m, int64_t n, int64_t k) {
  const int splits = gemm_f32_few_applies(m, n, k) ? few_splits(m, n, k) : 1;
  return splits > 1 ? static_cast<size_t>(splits) * m * ((n + 3) / 4 * 4) * sizeof(float) : 0;
}

int gemm_f32_few_resources(int64_t m, int64_t n, int64_t k, int transpose_b, IntentHipKernelResources *out) {
  return describe_kernel(few_kernel(few_rows(m, n, k), transpose_b), "gemm_f32_few", kFewWaves * 64, out);
}

int launch_gemm_f32_few(const float *a, const float *b, float *c, int M, int N, int K, int64_t lda, int64_t ldb,
                        int64_t ldc, int transpose_b, void *workspace, size_t workspace_bytes, hipStream_t s) {
  const bool room = workspace != nullptr && aligned(workspace, 16) && workspace_bytes >= gemm_f32_few_bytes(M, N, K);
  const int splits = room ? few_splits(M, N, K) : 1, rows = few_rows(M, N, K);
  float *partials = splits > 1 ? static_cast<float *>(workspace) : nullptr;
  int tiles_m = (M + rows - 1) / rows, tiles_n = (N + kFewCols - 1) / kFewCols;
  void *args[] = {&a, &b, &c, &M, &N, &K, &lda, &ldb, &ldc, &tiles_m, &tiles_n, &partials};
  if (hipLaunchKernel(few_kernel(rows, transpose_b), tile_grid(static_cast<int64_t>(tiles_m) * tiles_n, splits),
                      dim3(kFewWaves * 64), args, 0, s) != hipSuccess)
    return launch_status("gemm_f32_few");
  if (splits > 1) {
    const int64_t quads = static_cast<int64_t>(M) * ((N + 3) / 4);
    gemm_f32_splits<<<dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, s>>>(partials, c, M, N, ldc, splits);
    if (hipPeekAtLastError() != hipSuccess) return launch_status("gemm_f32_splits");
  }
  return INTENT_HIP_OK;
}

}  // namespace intent_hip
