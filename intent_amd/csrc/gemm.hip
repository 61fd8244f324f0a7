// bf16 GEMM, C = bf16(A @ B) with f32 accumulation, for gfx950 (CDNA4).
//
// Semantics: bf16_gemm (python/intent/examples/kernels/contraction/gemm.py:76-92):
// accumulator = matmul(a, b, acc_dtype=f32); c = cast(accumulator, bf16) (round to
// nearest even). A [M,K], B [K,N], C [M,N], row-major with row strides lda/ldb/ldc.
//
// Design: three MFMA kernels, chosen by the shape and layout (choose).
//   * 256 x 256 tiles (gemm_mfma) for many tiles: 8 waves in 2 x 4, each wave 128 x 64 = 4 x 2 tiles of
//     v_mfma_f32_32x32x16_bf16 (128 accumulator registers per lane, so two waves share
//     each SIMD); A and B stream into LDS with global_load_lds (five 32 KB stages) and B fragments are read
//     with transposing LDS reads; the two waves of a SIMD alternate between their MFMA cluster and their
//     LDS reads (ping-pong), so the matrix pipe is fed while the other wave waits on LDS. The tiles are walked in
//     groups of 2 tile rows, column by column, in dispatch order: those resident at one time share A row
//     panels and B column panels, across XCDs through the MALL and within each XCD through its L2;
//   * 128 x 128 and 64 x 64 tiles (gemm_small) where 256 x 256 tiles would leave CUs idle, and for
//     operands that the DMA does not take (odd extents, strides or addresses);
//   * up to 128 rows (gemm_skinny): waves stream B into registers (f16 relu 32 x 14336 x 4096: 221 us in
//     256 x 256 tiles, 28 there).
// Each issues the MFMA as D = Bt_frag x A_frag, i.e. the transposed product, so that a lane ends with
// consecutive output columns of one output row and writes 4 of them as one 8-byte store. Tiles that reach past M
// or N read valid rows and columns in their place and do not store them; past K (a multiple of 8 where the DMA runs)
// they read zeros.
#include <stdio.h>

#include <type_traits>

#include "common.hpp"

namespace intent_hip {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Operand element type: __bf16 (bf16_gemm) or _Float16 (gemm). Fragments of 8 elements feed
// v_mfma_f32_32x32x16_{bf16,f16}; results are stored 4 at a time.
template <typename E> struct Elem;
template <> struct Elem<__bf16> {
  typedef __bf16 x8 __attribute__((ext_vector_type(8)));
  typedef __bf16 x4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16_t mma(x8 a, x8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4_t mma16(x8 a, x8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Elem<_Float16> {
  typedef _Float16 x8 __attribute__((ext_vector_type(8)));
  typedef _Float16 x4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16_t mma(x8 a, x8 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4_t mma16(x8 a, x8 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Epilogue activation on the f32 accumulator: 0 = none, 1 = ReLU as I.maximum(acc, 0.0)
// (NaN propagates; -0 and +0 give +0).
template <int kAct>
__device__ __forceinline__ float activate(float v) {
  if constexpr (kAct == 1) return v != v ? v : (v > 0.0f ? v : 0.0f);
  return v;
}

template <typename E, int kAct>
__device__ __forceinline__ typename Elem<E>::x4 pack4(float a, float b, float c, float d) {
  typename Elem<E>::x4 r;
  r[0] = static_cast<E>(activate<kAct>(a));
  r[1] = static_cast<E>(activate<kAct>(b));
  r[2] = static_cast<E>(activate<kAct>(c));
  r[3] = static_cast<E>(activate<kAct>(d));
  return r;
}

constexpr int kBM = 256, kBN = 256;
constexpr int kThreads = 512;
constexpr int kGroupM = 2;

template <typename E>
__device__ __forceinline__ float element_to_f32(uint16_t bits) { return static_cast<float>(__builtin_bit_cast(E, bits)); }
template <typename E>
__device__ __forceinline__ uint16_t f32_to_element(float v) { return __builtin_bit_cast(uint16_t, static_cast<E>(v)); }

// Epilogues: quad(i, n, a, b, c, d) receives the f32 accumulators of output row i, columns n .. n+3
// (n a multiple of 4); some(i, n, count, v) the first `count` (1 or more) of 4 (layouts that the DMA does not take). kSums: K may be divided over
// workgroups, whose sums gemm_splits adds before the epilogue.
// gemm / bf16_gemm: act(acc) rounded to E.
template <typename E, int kAct>
struct CastStore {
  static constexpr bool kSums = true;
  uint16_t *C;
  int64_t ldc;
  __device__ __forceinline__ void quad(int i, int n, float a, float b, float c, float d) const {
    *reinterpret_cast<typename Elem<E>::x4 *>(C + static_cast<int64_t>(i) * ldc + n) = pack4<E, kAct>(a, b, c, d);
  }
  __device__ __forceinline__ void one(int i, int n, float a) const {
    C[static_cast<int64_t>(i) * ldc + n] = f32_to_element<E>(activate<kAct>(a));
  }
  __device__ __forceinline__ void some(int i, int n, int count, const float (&v)[4]) const {
    if (count >= 4) {   // one 8-byte store at a 2-byte boundary (4000 x 4001 x 8:
                        // 20.7 us, 48.7 with four stores)
      struct __attribute__((packed, aligned(2))) Quad { uint32_t w[2]; };
      const uint2 w = __builtin_bit_cast(uint2, pack4<E, kAct>(v[0], v[1], v[2], v[3]));
      *reinterpret_cast<Quad *>(C + static_cast<int64_t>(i) * ldc + n) = Quad{{w.x, w.y}};
      return;
    }
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (e < count) one(i, n + e, v[e]);
  }
};

// quantized_gemm (contraction/gemm.py:95-121), each step an f32 operation as written there:
// v = maximum(acc + bias[n], 0) (NaN propagates), v = v + residual[i][n], v = v / scale[n] (IEEE
// division), v = minimum(maximum(v, -128), 127), then the cast to i8, which truncates toward
// zero. NaN is an illegal cast input; it gives 0 here.
struct QuantizeStore {
  static constexpr bool kSums = false;
  const float *bias;
  const uint16_t *residual;   // f16 [M, N]
  int64_t ldr;
  const float *scale;
  int8_t *out;
  int64_t ldo;
  __device__ __forceinline__ static int32_t quantize(float acc, float bias, float residual, float scale) {
    float v = acc + bias;
    v = v != v ? v : (v > 0.0f ? v : 0.0f);
    v = v + residual;
    v = __fdiv_rn(v, scale);
    v = v != v ? v : (v < -128.0f ? -128.0f : (v > 127.0f ? 127.0f : v));
    return v != v ? 0 : static_cast<int32_t>(v);
  }
  __device__ __forceinline__ float residual_at(int i, int n) const {
    return element_to_f32<_Float16>(residual[static_cast<int64_t>(i) * ldr + n]);
  }
  __device__ __forceinline__ void quad(int i, int n, float a, float b, float c, float d) const {
    const uint2 r = *reinterpret_cast<const uint2 *>(residual + static_cast<int64_t>(i) * ldr + n);
    const float r0 = element_to_f32<_Float16>(static_cast<uint16_t>(r.x)), r1 = element_to_f32<_Float16>(static_cast<uint16_t>(r.x >> 16));
    const float r2 = element_to_f32<_Float16>(static_cast<uint16_t>(r.y)), r3 = element_to_f32<_Float16>(static_cast<uint16_t>(r.y >> 16));
    const uint32_t q = (static_cast<uint32_t>(quantize(a, bias[n], r0, scale[n])) & 0xffu) |
                       ((static_cast<uint32_t>(quantize(b, bias[n + 1], r1, scale[n + 1])) & 0xffu) << 8) |
                       ((static_cast<uint32_t>(quantize(c, bias[n + 2], r2, scale[n + 2])) & 0xffu) << 16) |
                       (static_cast<uint32_t>(quantize(d, bias[n + 3], r3, scale[n + 3])) << 24);
    *reinterpret_cast<uint32_t *>(out + static_cast<int64_t>(i) * ldo + n) = q;
  }
  // Byte stores may alias every load, so the loads of a group come before its stores (4000 x 4001 x 8 69 us, 80 when
  // each element's loads waited for the store before).
  __device__ __forceinline__ void some(int i, int n, int count, const float (&v)[4]) const {
    int32_t q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int at = n + (e < count ? e : 0);
      q[e] = quantize(v[e], bias[at], residual_at(i, at), scale[at]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < count) out[static_cast<int64_t>(i) * ldo + n + e] = static_cast<int8_t>(q[e]);
  }
};

// Tile order: groups of kGroupM tile rows walked column by column, in dispatch order (the 8 XCDs
// take consecutive workgroups round-robin). At 8192^3 the 256 resident tiles then span 8 tile
// rows and all columns: each XCD holds 4 rows x 8 columns of them, and every A and B panel is
// read by several XCDs at nearly the same time, which the MALL serves once. Measured against
// other orders (interleaved, 8192^3 bf16): 0.899 ms here; 0.943 ms with XCD-contiguous runs of
// 8-row groups; 1.06 / 1.37 ms with 16 / 32-row groups.
__device__ __forceinline__ void tile_of_block(int block, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int t = block;
  const int per_group = kGroupM * tiles_n;
  const int group = t / per_group;
  const int first_m = group * kGroupM;
  const int rows_in_group = min(tiles_m - first_m, kGroupM);
  const int in_group = t - group * per_group;
  tm = first_m + in_group % rows_in_group;
  tn = in_group / rows_in_group;
}

// ---------------------------------------------------------------- 256 x 256 tiles: LDS-DMA pipeline
// K step 32, five LDS stages of 32 KB (160 KB): up to three later tiles are in flight
// (global_load_lds_dwordx4 writes them straight into LDS, no registers) while tile kt is multiplied. A stage holds A [256 m][32 k]
// (rows of 4 16-byte chunks, chunk c of row r at c ^ ((r >> 2) & 3), which spreads the fragment
// reads of 16 consecutive rows over the 64 LDS banks) and B in its natural
// [32 k][256 n] layout (rows of 32 chunks, chunk c of row k at c ^ 4 (k & 3), so the transposing
// reads of 4 consecutive k rows land on 4 disjoint groups of 4 chunks). B fragments are read
// with ds_read_b64_tr_b16: in each 16-lane group, lane i, slot j receives element i % 4 of the
// 8-byte segment addressed by lane 4 j + i / 4, so lane i addressing B[k0 + i/4][n0 + 4 (i % 4)]
// yields B[k0 .. k0+3][n0 + i], the 4 consecutive k of one n the MFMA operand needs.
constexpr int kDmaBK = 32;
constexpr int kDmaStages = 5;
constexpr int kDmaChunksA = kBM * kDmaBK / 8;            // 1024
constexpr int kDmaStageChunks = (kBM + kBN) * kDmaBK / 8; // 2048 (32 KB)

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;
typedef __attribute__((address_space(3))) void lds_void_t;

// s_waitcnt with only the vector-memory counter constrained (vmcnt <= n), and with only the LDS
// counter constrained (lgkmcnt == 0).
#define INTENT_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8)))
#define INTENT_WAIT_LGKMCNT0() __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4))

// Workgroup barrier of the DMA loop: s_barrier with an acquire fence (later LDS reads stay below
// it) and no release fence. A release fence would wait for every DMA in flight (they are LDS
// writes); DMA completion is awaited explicitly with vmcnt before the barrier instead. The
// scheduling barriers keep each MFMA cluster on its side of the s_barrier.
__device__ __forceinline__ void dma_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  __builtin_amdgcn_sched_barrier(0);
}

// What the DMA reads for chunks past K.
__device__ const uint4 kZeroChunk = {0u, 0u, 0u, 0u};

// Rows past M and columns past N read valid ones instead, and their products are not stored; kTail: K is not a
// multiple of 32, and the last tile's chunks past K are zeros (K is a multiple of 8).
template <typename E, typename Epi, bool kTail>
__device__ __forceinline__ void gemm_tile_dma(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                              const Epi &ep, int M, int N, int K, int64_t lda, int64_t ldb, int m0,
                                              int n0, uint4 *lds) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;

  // Each wave issues 2 A and 2 B DMA instructions (1 KB each) per K tile. The global chunk a lane
  // fetches is the one its LDS slot (base + 16 * lane) must hold under the swizzle.
  const uint16_t *a_src[2];
  const uint16_t *b_src[2];
  int a_k[2], b_row[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int pa = (wave * 2 + i) * 64 + lane;      // A chunk slot: row pa / 4, physical chunk pa % 4
    const int ra = pa >> 2, ca = (pa & 3) ^ ((ra >> 2) & 3);
    a_src[i] = A + static_cast<int64_t>(min(m0 + ra, M - 1)) * lda + ca * 8;
    a_k[i] = ca * 8;
    const int pb = (wave * 2 + i) * 64 + lane;      // B chunk slot: row pb / 32, physical chunk pb % 32
    const int kb = pb >> 5, cb = (pb & 31) ^ (4 * (kb & 3));
    b_src[i] = B + static_cast<int64_t>(kb) * ldb + (n0 + cb * 8 < N ? n0 + cb * 8 : 0);
    b_row[i] = kb;
  }
  auto issue = [&](int kt) {
    uint4 *stage = lds + (kt % kDmaStages) * kDmaStageChunks;
    const int k0 = kt * kDmaBK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint16_t *a = a_src[i] + k0, *b = b_src[i] + static_cast<int64_t>(k0) * ldb;
      if (kTail && k0 + kDmaBK > K) {
        const uint16_t *zero = reinterpret_cast<const uint16_t *>(&kZeroChunk);
        if (k0 + a_k[i] >= K) a = zero;
        if (k0 + b_row[i] >= K) b = zero;
      }
      __builtin_amdgcn_global_load_lds(a, (lds_void_t *)(stage + (wave * 2 + i) * 64), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(b, (lds_void_t *)(stage + kDmaChunksA + (wave * 2 + i) * 64), 16, 0, 0);
    }
  };

  f32x16_t acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int frag_row = lane & 31;
  const int half = lane >> 5;
  const int a_swz = (frag_row >> 2) & 3;
  // B transposed-read address of this lane within a 32 x 32 (k x n) block: group g = lane / 16,
  // source role i = lane % 16 -> k = 8 (g / 2) + i / 4 (+4 for the second read), n = 16 (g % 2) + 4 (i % 4).
  const int g16 = lane >> 4, i16 = lane & 15;
  const int b_k = 8 * (g16 >> 1) + (i16 >> 2);
  const int b_n = 16 * (g16 & 1) + 4 * (i16 & 3);

  // Ping-pong schedule. Waves 0-3 and 4-7 share the four SIMDs (one of each per SIMD). Waves 4-7
  // run one barrier behind, so between two barriers one wave of each SIMD issues its MFMA cluster
  // (M) while the other reads its fragments from LDS and issues its DMA (R):
  //   waves 0-3: b0 |   R0 b M0 b R1 b M1 b ... M(last) b | b
  //   waves 4-7: b0 | b R0 b M0 b R1 b ... M(last) b
  // Every wave executes 2 + 2 * k_tiles barriers. Before the barrier that opens the interval in
  // which waves 0-3 read tile t, every wave has waited for its own DMA of tile t. The DMA of tile
  // t + S - 1 overwrites stage (t - 1) % S, whose reads every wave completed (lgkmcnt 0) before an
  // earlier barrier.
  const bool lag = wave >= 4;
  const int k_tiles = kTail ? (K + kDmaBK - 1) / kDmaBK : K / kDmaBK;
#pragma unroll
  for (int kt = 0; kt < kDmaStages - 1; ++kt)
    if (kt < k_tiles) issue(kt);
  auto wait_tile = [&](int t) {   // this wave's DMA of tile t complete; later tiles may stay in flight
    const int later = min(k_tiles - 1 - t, kDmaStages - 2);
    if (later >= 3) INTENT_WAIT_VMCNT(12);
    else if (later == 2) INTENT_WAIT_VMCNT(8);
    else if (later == 1) INTENT_WAIT_VMCNT(4);
    else INTENT_WAIT_VMCNT(0);
  };
  wait_tile(0);
  dma_barrier();
  if (lag) dma_barrier();
  typedef typename Elem<E>::x8 x8;
  x8 af[2][4], bf[2][2];
  for (int kt = 0; kt < k_tiles; ++kt) {
    const uint4 *sa = lds + (kt % kDmaStages) * kDmaStageChunks;
    const uint16_t *sb = reinterpret_cast<const uint16_t *>(sa + kDmaChunksA);
#pragma unroll
    for (int kk = 0; kk < kDmaBK / 16; ++kk) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        af[kk][t] = __builtin_bit_cast(x8, sa[(wm * 128 + t * 32 + frag_row) * 4 + ((kk * 2 + half) ^ a_swz)]);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        i16x4_t parts[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const int k = kk * 16 + b_k + 4 * r;
          const int n = wn * 64 + t * 32 + b_n;
          const int chunk = (n >> 3) ^ (4 * (k & 3));
          parts[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(sb + k * kBN + chunk * 8 + (n & 7)));
        }
        bf[kk][t] = __builtin_bit_cast(x8, parts);
      }
    }
    if (kt + kDmaStages - 1 < k_tiles) issue(kt + kDmaStages - 1);
    if (lag) wait_tile(kt + 1);
    INTENT_WAIT_LGKMCNT0();
    dma_barrier();
#pragma unroll
    for (int kk = 0; kk < kDmaBK / 16; ++kk)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = Elem<E>::mma(bf[kk][nt], af[kk][mt], acc[mt][nt]);
    if (!lag) wait_tile(kt + 1);
    dma_barrier();
  }
  if (!lag) dma_barrier();

  // The tests cost 5 us of 49 at 4096 x 4096 x 1024 where they are not needed.
  const auto store = [&](auto inside) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int i = m0 + wm * 128 + mt * 32 + frag_row;
      if (!inside && i >= M) continue;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = n0 + wn * 64 + nt * 32 + 8 * g + 4 * half;
          if (!inside && n >= N) continue;
          const f32x16_t &v = acc[mt][nt];
          ep.quad(i, n, v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
        }
    }
  };
  if (m0 + kBM <= M && n0 + kBN <= N) store(std::true_type{});
  else store(std::false_type{});
}

template <typename E, typename Epi, bool kTail>
__global__ __launch_bounds__(kThreads, 1) void gemm_mfma(const uint16_t *__restrict__ A,
                                                              const uint16_t *__restrict__ B, Epi ep, int M,
                                                              int N, int K, int64_t lda, int64_t ldb, int tiles_m,
                                                              int tiles_n) {
  __shared__ uint4 lds[kDmaStages * kDmaStageChunks];
  int tm, tn;
  tile_of_block(blockIdx.x, tiles_m, tiles_n, tm, tn);
  gemm_tile_dma<E, Epi, kTail>(A, B, ep, M, N, K, lda, ldb, tm * kBM, tn * kBN, lds);
}

// ---------------------------------------------------------------- few rows: waves stream B, no LDS tiles
// With few rows the time is the time to read B, and 256-row tiles would leave most of the chip idle and multiply
// padding. A workgroup owns MT * 16 rows and 64 columns (128 bytes, one cache line, of each row of B; a CU
// holds a bounded number of lines in flight, so half lines halve its rate). Its waves take
// the 64-deep units of K in turn, loading straight into registers, the next unit in flight while the
// current one is multiplied. Lane (g = l / 16, c = l % 16) loads rows 8 g + j (j = 0..7) of a
// 32-deep step, columns 4 c .. 4 c + 3. Pairing the words of rows 2 p and 2 p + 1 with v_perm_b32
// gives, for each i < 4, the 8 consecutive k of column 4 c + i that the MFMA takes, so MFMA i covers the columns
// 4 c + i and a lane accumulates 16 consecutive columns of one row. The waves' sums meet in LDS and
// are added in wave order.
// One CU reads about 19 GB/s of B at most, so a call with few column blocks also divides K over workgroups
// (blockIdx.y): each then writes its f32 sums to `partials` and gemm_splits adds them in order.
constexpr int kSkinnyCols = 64;
constexpr int kSkinnyUnit = 64;           // k of one unit (two 32-deep steps)
constexpr int kSkinnyWaves = 8;
constexpr int kSkinnyRows = 128;          // most rows a call may have to run here

// 4 columns of one row of B: non-temporal where one row block reads B (nothing reads it again in the call).
template <bool kStream>
__device__ __forceinline__ uint2 load_columns(const uint16_t *p) {
  if constexpr (kStream) return __builtin_bit_cast(uint2, __builtin_nontemporal_load(reinterpret_cast<const uint64_t *>(p)));
  return *reinterpret_cast<const uint2 *>(p);
}

template <typename E, typename Epi, int MT, bool kStream>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_skinny(const uint16_t *__restrict__ A,
                                                                 const uint16_t *__restrict__ B, Epi ep, int M, int N,
                                                                 int K, int64_t lda, int64_t ldb, int tiles_m,
                                                                 int tiles_n, float *__restrict__ partials) {
  typedef typename Elem<E>::x8 x8;
  constexpr int kRows = MT * 16, kPad = kSkinnyCols + 4, W = kSkinnyWaves;
  __shared__ float4 sums[W * kRows * kPad / 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // The row blocks of one column block are neighbours, so they share its B through the L2 of one XCD. With
  // one row block the XCDs take the column blocks in turn (28.9 against 27.9 us at 32 x 14336 x 4096).
  const int tile = kStream ? grid_block() : xcd_tile(grid_block(), tiles_m * tiles_n);
  if (tile < 0 || tile >= tiles_m * tiles_n) return;
  const int m0 = (tile % tiles_m) * kRows, n0 = (tile / tiles_m) * kSkinnyCols;
  // Columns past N and rows past M read valid ones instead; their products are not stored.
  const int n = n0 + 4 * c < N ? n0 + 4 * c : 0;
  const uint32_t b_lane = static_cast<uint32_t>(8 * g) * static_cast<uint32_t>(ldb) + n;
  uint32_t a_lane[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    a_lane[t] = static_cast<uint32_t>(min(m0 + 16 * t + c, M - 1)) * static_cast<uint32_t>(lda) + 8 * g;

  f32x4_t acc[MT][4];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[t][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // One whole 32-deep step starting at k0.
  auto load_step = [&](int k0, uint2 (&b)[8], uint4 (&a)[MT]) {
    const uint16_t *rows = B + static_cast<int64_t>(k0) * ldb;
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = load_columns<kStream>(rows + j * ldb + b_lane);
#pragma unroll
    for (int t = 0; t < MT; ++t) a[t] = *reinterpret_cast<const uint4 *>(A + k0 + a_lane[t]);
  };
  auto multiply = [&](const uint2 (&b)[8], const uint4 (&a)[MT]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint4 bt;
      uint32_t *w = reinterpret_cast<uint32_t *>(&bt);
#pragma unroll
      for (int p = 0; p < 4; ++p)
        w[p] = __builtin_amdgcn_perm(i < 2 ? b[2 * p + 1].x : b[2 * p + 1].y, i < 2 ? b[2 * p].x : b[2 * p].y,
                                     (i & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t][i] = Elem<E>::mma16(__builtin_bit_cast(x8, bt), __builtin_bit_cast(x8, a[t]), acc[t][i]);
    }
  };

  const int units = K / kSkinnyUnit;
  const int first = static_cast<int>(static_cast<int64_t>(units) * blockIdx.y / gridDim.y);
  const int last = static_cast<int>(static_cast<int64_t>(units) * (blockIdx.y + 1) / gridDim.y);
  uint2 b[2][2][8];
  uint4 a[2][2][MT];
  auto load_unit = [&](int unit, int buffer) {
#pragma unroll
    for (int u = 0; u < 2; ++u) load_step(unit * kSkinnyUnit + 32 * u, b[buffer][u], a[buffer][u]);
  };
  auto multiply_unit = [&](int buffer) {
#pragma unroll
    for (int u = 0; u < 2; ++u) multiply(b[buffer][u], a[buffer][u]);
  };
  int unit = first + wave;
  if (unit < last) load_unit(unit, 0);
  for (; unit + W < last; unit += 2 * W) {
    load_unit(unit + W, 1);
    multiply_unit(0);
    if (unit + 2 * W < last) load_unit(unit + 2 * W, 0);
    multiply_unit(1);
  }
  if (unit < last) multiply_unit(0);
  // The last K % 64 (a multiple of 8), by the next wave in turn of the last split: groups of 8 k
  // past K are zero in both operands.
  if (K % kSkinnyUnit != 0 && blockIdx.y == gridDim.y - 1 && wave == (last - first) % W) {
    for (int k0 = units * kSkinnyUnit; k0 < K; k0 += 32) {
      const bool live = k0 + 8 * g < K;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        b[0][0][j] = make_uint2(0u, 0u);
        if (live) b[0][0][j] = *reinterpret_cast<const uint2 *>(B + (static_cast<int64_t>(k0) + j) * ldb + b_lane);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        a[0][0][t] = make_uint4(0u, 0u, 0u, 0u);
        if (live) a[0][0][t] = *reinterpret_cast<const uint4 *>(A + k0 + a_lane[t]);
      }
      multiply(b[0][0], a[0][0]);
    }
  }

  // acc[t][i][r] is row 16 t + c, column 16 g + 4 r + i of this wave's share of the sum.
  float *own = reinterpret_cast<float *>(sums) + wave * kRows * kPad;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<float4 *>(own + (16 * t + c) * kPad + 16 * g + 4 * r) =
          make_float4(acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]);
  __syncthreads();
  const float *all = reinterpret_cast<const float *>(sums);
  for (int quad = threadIdx.x; quad < kRows * kSkinnyCols / 4; quad += W * 64) {
    const int row = quad / (kSkinnyCols / 4), col = 4 * (quad % (kSkinnyCols / 4));
    if (m0 + row >= M || n0 + col >= N) continue;
    float4 total = *reinterpret_cast<const float4 *>(all + row * kPad + col);
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const float4 v = *reinterpret_cast<const float4 *>(all + (w * kRows + row) * kPad + col);
      total.x += v.x;
      total.y += v.y;
      total.z += v.z;
      total.w += v.w;
    }
    if (Epi::kSums && partials != nullptr)
      *reinterpret_cast<float4 *>(partials + (static_cast<int64_t>(blockIdx.y) * M + m0 + row) * N + n0 + col) = total;
    else
      ep.quad(m0 + row, n0 + col, total.x, total.y, total.z, total.w);
  }
}

// Adds the K splits of a product in order and stores the result: one thread per 4 columns (rows of `partials` are
// padded to a multiple of 4). kQuads: 4 columns may be stored together.
template <typename Epi, bool kQuads>
__global__ __launch_bounds__(256) void gemm_splits(const float *__restrict__ partials, Epi ep, int M, int N, int splits) {
  const int quads = (N + 3) / 4;
  const int64_t quad = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, all = static_cast<int64_t>(M) * quads;
  if (quad >= all) return;
  const int row = static_cast<int>(quad / quads), col = 4 * static_cast<int>(quad % quads);
  const f32x4_t *p = reinterpret_cast<const f32x4_t *>(partials) + quad;
  f32x4_t total = p[0];
#pragma unroll 8
  for (int s = 1; s < splits; ++s) total += p[s * all];
  if (kQuads) {
    ep.quad(row, col, total[0], total[1], total[2], total[3]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < N) ep.one(row, col + e, total[e]);
  }
}

// ---------------------------------------------------------------- small tiles
// Workgroups of 2 x WN waves (each BM / 2 x BN / WN in 32 x 32 MFMA tiles) for products of too few
// 256 x 256 tiles. One barrier per K step; S stages of LDS, written by DMA, the next S - 1 steps in flight. A CU
// gets its operands at 20 to 50 GB/s when they come from HBM or the MALL, so such products are bound by the
// bytes of the busiest CU and the latency of its K steps, and the tiles are chosen to reach every CU.
// The layouts are those of the 256 x 256 kernel, for any BM, BN and BK. kDma false, for operands that are
// not 16-byte aligned or whose extents or strides are not multiples of 8: the same tiles through registers (two
// steps ahead), with 16-byte loads and 8-byte stores at 2-byte boundaries, single elements only where a chunk reaches past
// K or N (bf16 2048 x 2049 x 2047: 84 us; 1222 in f32 FMAs).
template <int BM, int BN, int BK, int S, int WN>
struct SmallTile {
  static constexpr int kThreads = 128 * WN;                       // 2 x WN waves
  static constexpr int kRowChunks = BK / 8;                       // 16-byte chunks of an A row
  static constexpr int kChunksA = BM * kRowChunks, kChunksB = BK * BN / 8;
  static constexpr int kStage = kChunksA + kChunksB;              // chunks of one stage
  static constexpr int kLoadsA = kChunksA / kThreads, kLoadsB = kChunksB / kThreads;   // per thread and stage
  // Chunk c of A row r is stored at c ^ swz_a(r): 16 consecutive rows' fragment reads hit every bank once.
  static __device__ __forceinline__ int swz_a(int r) {
    if constexpr (BK == 64) return (r & 7) ^ ((r >> 3) & 1);
    return (r >> 2) & 3;
  }
  // Chunk c of B row k is stored at c ^ swz_b(k): the transposing reads of 4 consecutive rows hit every bank once.
  static __device__ __forceinline__ int swz_b(int k) {
    if constexpr (BN == 64) return 4 * ((k >> 1) & 1);
    return 4 * (k & 3);
  }
};

// 8 elements at p, `count` of them (0..8) present, at any 2-byte boundary; zeros for the others.
__device__ __forceinline__ uint4 load_8(const uint16_t *p, int count) {
  struct __attribute__((packed, aligned(2))) Chunk { uint32_t w[4]; };
  if (count >= 8) {
    const Chunk c = *reinterpret_cast<const Chunk *>(p);
    return make_uint4(c.w[0], c.w[1], c.w[2], c.w[3]);
  }
  uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 7; ++i)
    if (i < count) w[i / 2] |= static_cast<uint32_t>(p[i]) << (16 * (i & 1));
  return make_uint4(w[0], w[1], w[2], w[3]);
}

template <typename E, typename Epi, int BM, int BN, int BK, int S, bool kDma, int WN>
__global__ __launch_bounds__(128 * WN) void gemm_small(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B, Epi ep,
                                                  int M, int N, int K, int64_t lda, int64_t ldb, int tiles_m,
                                                  int tiles_n, float *__restrict__ partials) {
  typedef SmallTile<BM, BN, BK, S, WN> T;
  typedef typename Elem<E>::x8 x8;
  constexpr int MT = BM / 64, NT = BN / (32 * WN), KT = BK / 16, TH = T::kThreads;
  __shared__ uint4 lds[S * T::kStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  // The row blocks of one column block are neighbours. The DMA kernels run few tiles, along x (grid_block() there:
  // 1021 x 2304 x 768 12.1 -> 12.9 us).
  const int tile = xcd_tile(kDma ? static_cast<int>(blockIdx.x) : grid_block(), tiles_m * tiles_n);
  if (tile < 0) return;
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;

  // Slot p = tid + TH i of a stage's A holds chunk (p % kRowChunks) ^ swz of row p / kRowChunks; of its B,
  // chunk (p % (BN / 8)) ^ swz of row p / (BN / 8). Rows past M and columns past N read valid
  // ones instead; their products are not stored.
  const uint16_t *a_src[T::kLoadsA], *b_src[T::kLoadsB];
  int a_k[T::kLoadsA], b_k[T::kLoadsB], b_n[T::kLoadsB];
#pragma unroll
  for (int i = 0; i < T::kLoadsA; ++i) {
    const int p = tid + TH * i, r = p / T::kRowChunks;
    a_k[i] = ((p % T::kRowChunks) ^ T::swz_a(r)) * 8;
    a_src[i] = A + static_cast<int64_t>(min(m0 + r, M - 1)) * lda + a_k[i];
  }
#pragma unroll
  for (int i = 0; i < T::kLoadsB; ++i) {
    const int p = tid + TH * i, n = ((p % (BN / 8)) ^ T::swz_b(p / (BN / 8))) * 8;
    b_k[i] = p / (BN / 8);
    b_n[i] = n0 + n < N ? n0 + n : 0;
    b_src[i] = B + static_cast<int64_t>(b_k[i]) * ldb + b_n[i];
  }

  f32x16_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int frag = lane & 31, half = lane >> 5;
  const int g16 = lane >> 4, i16 = lane & 15;
  const int t_k = 8 * (g16 >> 1) + (i16 >> 2), t_n = 16 * (g16 & 1) + 4 * (i16 & 3);
  x8 af[KT][MT], bf[KT][NT];
  auto read_tile = [&](int stage) {
    const uint4 *sa = lds + stage * T::kStage;
    const uint16_t *sb = reinterpret_cast<const uint16_t *>(sa + T::kChunksA);
#pragma unroll
    for (int kk = 0; kk < KT; ++kk) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = wm * (BM / 2) + t * 32 + frag;
        af[kk][t] = __builtin_bit_cast(x8, sa[r * T::kRowChunks + ((kk * 2 + half) ^ T::swz_a(r))]);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        i16x4_t parts[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = kk * 16 + t_k + 4 * h, n = wn * (BN / WN) + t * 32 + t_n;
          parts[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_i16x4_t *)(sb + k * BN + ((n >> 3) ^ T::swz_b(k)) * 8 + (n & 7)));
        }
        bf[kk][t] = __builtin_bit_cast(x8, parts);
      }
    }
  };
  auto multiply = [&]() {
#pragma unroll
    for (int kk = 0; kk < KT; ++kk)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = Elem<E>::mma(bf[kk][nt], af[kk][mt], acc[mt][nt]);
  };

  const int all_tiles = (K + BK - 1) / BK;
  const int first = static_cast<int>(static_cast<int64_t>(all_tiles) * blockIdx.y / gridDim.y);
  const int k_tiles = static_cast<int>(static_cast<int64_t>(all_tiles) * (blockIdx.y + 1) / gridDim.y) - first;
  if constexpr (kDma) {
    constexpr int kLoads = T::kLoadsA + T::kLoadsB;
    const uint16_t *zero = reinterpret_cast<const uint16_t *>(&kZeroChunk);
    auto issue = [&](int kt) {
      uint4 *stage = lds + (kt % S) * T::kStage;
      const int k0 = (first + kt) * BK;
      const bool tail = k0 + BK > K;   // uniform
#pragma unroll
      for (int i = 0; i < T::kLoadsA; ++i) {
        const uint16_t *src = a_src[i] + k0;
        if (tail && k0 + a_k[i] >= K) src = zero;
        __builtin_amdgcn_global_load_lds(src, (lds_void_t *)(stage + wave * 64 + TH * i), 16, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < T::kLoadsB; ++i) {
        const uint16_t *src = b_src[i] + static_cast<int64_t>(k0) * ldb;
        if (tail && k0 + b_k[i] >= K) src = zero;
        __builtin_amdgcn_global_load_lds(src, (lds_void_t *)(stage + T::kChunksA + wave * 64 + TH * i), 16, 0, 0);
      }
    };
#pragma unroll
    for (int kt = 0; kt < S - 1; ++kt)
      if (kt < k_tiles) issue(kt);
    for (int kt = 0; kt < k_tiles; ++kt) {
      // This wave's loads of tile kt complete; up to S - 2 later tiles stay in flight.
      const int later = min(k_tiles - 1 - kt, S - 2);
      if (S > 4 && later >= 3) INTENT_WAIT_VMCNT(3 * kLoads);
      else if (S > 3 && later == 2) INTENT_WAIT_VMCNT(2 * kLoads);
      else if (later == 1) INTENT_WAIT_VMCNT(kLoads);
      else INTENT_WAIT_VMCNT(0);
      dma_barrier();
      read_tile(kt % S);
      // Overwrites the stage of tile kt - 1, which every wave read before the barrier.
      if (kt + S - 1 < k_tiles) issue(kt + S - 1);
      multiply();
      INTENT_WAIT_LGKMCNT0();
    }
  } else {
    // Two register sets: the loads of tile kt + 2 are in flight while tile kt is multiplied.
    uint4 ra[2][T::kLoadsA], rb[2][T::kLoadsB];
    auto load = [&](int kt, uint4 (&qa)[T::kLoadsA], uint4 (&qb)[T::kLoadsB]) {
      const int k0 = (first + kt) * BK;
#pragma unroll
      for (int i = 0; i < T::kLoadsA; ++i) qa[i] = load_8(a_src[i] + k0, K - (k0 + a_k[i]));
#pragma unroll
      for (int i = 0; i < T::kLoadsB; ++i)
        qb[i] = load_8(b_src[i] + static_cast<int64_t>(k0) * ldb, k0 + b_k[i] < K ? N - b_n[i] : 0);
    };
    auto store = [&](int stage, const uint4 (&qa)[T::kLoadsA], const uint4 (&qb)[T::kLoadsB]) {
#pragma unroll
      for (int i = 0; i < T::kLoadsA; ++i) lds[stage * T::kStage + tid + TH * i] = qa[i];
#pragma unroll
      for (int i = 0; i < T::kLoadsB; ++i) lds[stage * T::kStage + T::kChunksA + tid + TH * i] = qb[i];
    };
    if (k_tiles > 0) load(0, ra[0], rb[0]);
    if (k_tiles > 1) load(1, ra[1], rb[1]);
    if (k_tiles > 0) store(0, ra[0], rb[0]);
    __syncthreads();
    for (int kt = 0; kt < k_tiles; kt += 2) {
      if (kt + 2 < k_tiles) load(kt + 2, ra[0], rb[0]);
      read_tile(0);
      multiply();
      if (kt + 1 >= k_tiles) break;
      store(1, ra[1], rb[1]);
      __syncthreads();
      if (kt + 3 < k_tiles) load(kt + 3, ra[1], rb[1]);
      read_tile(1);
      multiply();
      if (kt + 2 < k_tiles) store(0, ra[0], rb[0]);
      __syncthreads();
    }
  }

  // acc[mt][nt][4 g + e] is row wm BM / 2 + 32 mt + frag, column wn BN / WN + 32 nt + 8 g + 4 half + e.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int i = m0 + wm * (BM / 2) + mt * 32 + frag;
    if (i >= M) continue;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n0 + wn * (BN / WN) + nt * 32 + 8 * g + 4 * half;
        const f32x16_t &v = acc[mt][nt];
        // Tested for every epilogue: without the branch the compiler writes all quantizing quads out in one straight
        // line, whose instructions arrive late (2048^3 quantized 35 us, 31 with it).
        if (partials != nullptr) {
          const int64_t width = (N + 3) & ~3;
          if (n < N)
            *reinterpret_cast<float4 *>(partials + (static_cast<int64_t>(blockIdx.y) * M + i) * width + n) =
                make_float4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
        } else if (kDma) {
          if (n < N) ep.quad(i, n, v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
        } else if (n < N) {
          ep.some(i, n, N - n, {v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]});
        }
      }
  }
}

// ---------------------------------------------------------------- launches
// The tile size follows from how many tiles the chip's 256 CUs hold at once, bf16 measured on both sides of each line:
//   * up to 128 tiles of 128 x 128: 64 x 64 ones, K divided over workgroups where these are few too (1000^3
//     10.5 us against 15.5 in 128 x 128, 512 x 512 x 4096 14 against 45);
//   * up to 256: 128 x 128 with four stages and eight waves, one a CU (1021 x 2304 x 768 12.1 us against 13.3 with
//     four waves, 15.3 in 64 x 64 and 48 in 256 x 256; 2048^3 30.7 against 32.3, 46 and 54);
//   * up to 512: the same with two stages, two a CU (2639 x 2880 x 6912 125 us against 173 with four stages
//     and 155 in 256 x 256; 8192 x 1024 x 4096 90 against 103 in 256 x 256);
//   * more: 256 x 256 (4096 x 4096 x 1024 44 us against 61, 8000 x 2048 x 520 32 against 41).
constexpr int64_t kChip = 256;

bool fast_path(const void *a, const void *b, const void *c, int64_t n, int64_t k, int64_t lda, int64_t ldb,
               int64_t ldc) {
  return k % 8 == 0 && n % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 4 == 0 && aligned(a, 16) &&
         aligned(b, 16) && aligned(c, 8);
}

}  // namespace

namespace {

// Few rows, and strides that keep a lane's offset (24 rows of B, all rows of A) below 2^31 elements.
bool skinny(int64_t m, int64_t lda, int64_t ldb) {
  return m <= kSkinnyRows && lda < (int64_t{1} << 22) && ldb < (int64_t{1} << 25);
}

// The kernel of a product, its threads and its tile.
enum Family { kSkinnyFamily, kSmallFamily, kLargeFamily };
constexpr const char *kFamilyNames[] = {"gemm_skinny", "gemm_small", "gemm_mfma"};
struct Choice {
  const void *kernel;
  Family family;
  int threads, rows, cols;
};

template <typename E, typename Epi, int MT, bool kStream>
Choice skinny_choice() {
  return {reinterpret_cast<const void *>(&gemm_skinny<E, Epi, MT, kStream>), kSkinnyFamily, kSkinnyWaves * 64, 16 * MT,
          kSkinnyCols};
}
template <typename E, typename Epi, int BM, int BN, int BK, int S, bool kDma, int WN = 2>
Choice small_choice() {
  return {reinterpret_cast<const void *>(&gemm_small<E, Epi, BM, BN, BK, S, kDma, WN>), kSmallFamily, 128 * WN, BM, BN};
}

// `fast`: the operand layout that the DMA takes (fast_path); every other one runs in 64 x 64 tiles through registers.
template <typename E, typename Epi>
Choice choose(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, bool fast) {
  if (!fast || k == 0) return small_choice<E, Epi, 64, 64, 64, 2, false>();
  if (skinny(m, lda, ldb))
    return m <= 16   ? skinny_choice<E, Epi, 1, true>()
           : m <= 32 ? skinny_choice<E, Epi, 2, true>()
           : m <= 64 ? skinny_choice<E, Epi, 4, true>()
                     : skinny_choice<E, Epi, 4, false>();
  const int64_t tiles = (m + 127) / 128 * ((n + 127) / 128);
  if (tiles <= kChip / 2) return small_choice<E, Epi, 64, 64, 64, 4, true>();
  if (tiles <= kChip) return small_choice<E, Epi, 128, 128, 64, 4, true, 4>();
  if (tiles <= 2 * kChip) return small_choice<E, Epi, 128, 128, 64, 2, true>();
  const void *kernel = k % kDmaBK == 0 ? reinterpret_cast<const void *>(&gemm_mfma<E, Epi, false>)
                                       : reinterpret_cast<const void *>(&gemm_mfma<E, Epi, true>);
  return {kernel, kLargeFamily, kThreads, kBM, kBN};
}

template <typename E, typename Epi>
int describe(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, bool fast, const char *elements,
             IntentHipKernelResources *out) {
  const Choice choice = choose<E, Epi>(m, n, k, lda, ldb, fast);
  char name[64];
  snprintf(name, sizeof name, "%s<%s>", kFamilyNames[choice.family], elements);
  return describe_kernel(choice.kernel, name, choice.threads, out);
}

// The MFMA kernels' quantizing epilogue reads 4 residuals as 8 bytes and stores 4 outputs as 4 bytes.
bool quantize_fast_path(const void *a, const void *b, const void *residual, const void *out, int64_t n, int64_t k, int64_t lda,
                        int64_t ldb, int64_t ldr, int64_t ldo) {
  return k % 8 == 0 && n % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && aligned(a, 16) && aligned(b, 16) &&
         ldr % 4 == 0 && aligned(residual, 8) && ldo % 4 == 0 && aligned(out, 4);
}

}  // namespace

int quantized_gemm_resources(const void *a, const void *b, const void *residual, const void *out, int64_t m, int64_t n,
                             int64_t k, int64_t lda, int64_t ldb, int64_t ldr, int64_t ldo, IntentHipKernelResources *to) {
  return describe<_Float16, QuantizeStore>(m, n, k, lda, ldb, quantize_fast_path(a, b, residual, out, n, k, lda, ldb, ldr, ldo),
                                           "f16,quantize", to);
}

int gemm_resources(int dtype, int activation, const void *a, const void *b, const void *c, int64_t m, int64_t n, int64_t k,
                   int64_t lda, int64_t ldb, int64_t ldc, IntentHipKernelResources *out) {
  const bool fast = fast_path(a, b, c, n, k, lda, ldb, ldc);
  if (dtype == INTENT_HIP_F16)
    return activation ? describe<_Float16, CastStore<_Float16, 1>>(m, n, k, lda, ldb, fast, "f16", out)
                      : describe<_Float16, CastStore<_Float16, 0>>(m, n, k, lda, ldb, fast, "f16", out);
  return activation ? describe<__bf16, CastStore<__bf16, 1>>(m, n, k, lda, ldb, fast, "bf16", out)
                    : describe<__bf16, CastStore<__bf16, 0>>(m, n, k, lda, ldb, fast, "bf16", out);
}

namespace {

// Workgroups along K of a few-row product: enough that every CU reads a share of B. The second
// launch costs about 3 us, which the split returns from 2048 rows of B on (m 16, n 1024: k 1024 4.5 us
// unsplit against 6.7, k 2048 7.9 against 7.5; n 2048, k 8192: 37.4 against 12.2; m 64, n = k = 4096:
// 33.1 against 15.5).
int skinny_splits(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || n < 1 || m > kSkinnyRows || k < 2048) return 1;
  const int64_t blocks = (n + kSkinnyCols - 1) / kSkinnyCols * (m <= 64 ? 1 : 2);
  const int64_t splits = 256 / blocks < k / 256 ? 256 / blocks : k / 256;
  return splits < 2 ? 1 : static_cast<int>(splits);
}

// The same for 64 x 64 tiles.
int small_splits(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || n < 1 || k < 1024) return 1;
  const int64_t tiles = (m + 63) / 64 * ((n + 63) / 64);
  const int64_t splits = 256 / tiles < k / 256 ? 256 / tiles : k / 256;
  return splits < 2 ? 1 : static_cast<int>(splits);
}

template <typename Epi, bool kQuads>
void launch_splits(const float *partials, const Epi &ep, int m, int n, int splits, hipStream_t s) {
  const int64_t quads = static_cast<int64_t>(m) * ((n + 3) / 4);
  gemm_splits<Epi, kQuads><<<dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, s>>>(partials, ep, m, n, splits);
}

// `partials`: null (always without Epi::kSums), or room for splits_bytes(m, n, k).
template <typename E, typename Epi>
int launch_epilogue(const uint16_t *A, const uint16_t *B, const Epi &ep, int64_t m, int64_t n, int64_t k, int64_t lda,
                    int64_t ldb, bool fast, float *partials, hipStream_t s) {
  const Choice choice = choose<E, Epi>(m, n, k, lda, ldb, fast);
  int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k);
  int tiles_m = (M + choice.rows - 1) / choice.rows, tiles_n = (N + choice.cols - 1) / choice.cols;
  int splits = 1;
  if (partials != nullptr && choice.family == kSkinnyFamily) splits = skinny_splits(m, n, k);
  if (partials != nullptr && choice.family == kSmallFamily && choice.rows == 64) splits = small_splits(m, n, k);
  if (splits == 1) partials = nullptr;
  const int64_t tiles = static_cast<int64_t>(tiles_m) * tiles_n;
  const dim3 grid = choice.family == kLargeFamily ? dim3(static_cast<unsigned>(tiles)) : tile_grid(tiles, splits);
  Epi epilogue = ep;
  void *args[] = {&A, &B, &epilogue, &M, &N, &K, &lda, &ldb, &tiles_m, &tiles_n, &partials};
  if (hipLaunchKernel(choice.kernel, grid, dim3(choice.threads), args, 0, s) != hipSuccess)
    return launch_status(kFamilyNames[choice.family]);
  if constexpr (Epi::kSums) {
    if (splits == 1) return INTENT_HIP_OK;
    if (fast) launch_splits<Epi, true>(partials, ep, M, N, splits, s);
    else launch_splits<Epi, false>(partials, ep, M, N, splits, s);
    if (hipPeekAtLastError() != hipSuccess) return launch_status("gemm_splits");
  }
  return INTENT_HIP_OK;
}

// Bytes of the f32 partial sums of a product's K splits (0: one workgroup per output tile).
size_t splits_bytes(int64_t m, int64_t n, int64_t k) {
  const int few = skinny_splits(m, n, k), small = small_splits(m, n, k), splits = few > small ? few : small;
  return splits > 1 ? static_cast<size_t>(splits) * m * ((n + 3) / 4 * 4) * sizeof(float) : 0;
}

template <typename E, int kAct>
int launch_gemm(const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                int64_t ldc, void *stream, void *workspace = nullptr, size_t workspace_bytes = 0) {
  if (m < 0 || n < 0 || k < 0) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "negative extent");
  if (m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2)
    return fail(INTENT_HIP_ERR_UNSUPPORTED, "GEMM extents must stay below 2^30");
  if (m == 0 || n == 0) return INTENT_HIP_OK;
  if (a == nullptr || b == nullptr || c == nullptr) {
    if (k > 0 || c == nullptr) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "null tensor pointer");
  }
  if (lda < (m > 1 ? k : 0) || ldb < (k > 1 ? n : 0) || ldc < (m > 1 ? n : 0))
    return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "row stride smaller than the row length");
  const hipStream_t s = as_stream(stream);
  const auto *A = static_cast<const uint16_t *>(a);
  const auto *B = static_cast<const uint16_t *>(b);
  const CastStore<E, kAct> ep{static_cast<uint16_t *>(c), ldc};
  const bool room = workspace != nullptr && aligned(workspace, 16) && workspace_bytes >= splits_bytes(m, n, k);
  return launch_epilogue<E>(A, B, ep, m, n, k, lda, ldb, fast_path(a, b, c, n, k, lda, ldb, ldc),
                            room ? static_cast<float *>(workspace) : nullptr, s);
}

}  // namespace
}  // namespace intent_hip

using namespace intent_hip;

extern "C" int intent_hip_gemm_bf16(const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k,
                                    int64_t lda, int64_t ldb, int64_t ldc, void *stream) {
  return launch_gemm<__bf16, 0>(a, b, c, m, n, k, lda, ldb, ldc, stream);
}

extern "C" int intent_hip_gemm_ws(int dtype, int activation, const void *a, const void *b, void *c, int64_t m,
                                  int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc, void *workspace,
                                  size_t workspace_bytes, void *stream) {
  if (activation != 0 && activation != 1)
    return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "activation code %d (0 = none, 1 = relu)", activation);
  const auto launch = [&](auto run) {
    return run(a, b, c, m, n, k, lda, ldb, ldc, stream, workspace, workspace_bytes);
  };
  if (dtype == INTENT_HIP_F16) return activation ? launch(launch_gemm<_Float16, 1>) : launch(launch_gemm<_Float16, 0>);
  if (dtype == INTENT_HIP_BF16) return activation ? launch(launch_gemm<__bf16, 1>) : launch(launch_gemm<__bf16, 0>);
  return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "16-bit GEMM dtype code %d (1 = f16, 2 = bf16)", dtype);
}

extern "C" int intent_hip_gemm(int dtype, int activation, const void *a, const void *b, void *c, int64_t m, int64_t n,
                               int64_t k, int64_t lda, int64_t ldb, int64_t ldc, void *stream) {
  return intent_hip_gemm_ws(dtype, activation, a, b, c, m, n, k, lda, ldb, ldc, nullptr, 0, stream);
}

extern "C" int intent_hip_gemm_workspace_bytes(int64_t m, int64_t n, int64_t k, size_t *bytes) {
  if (bytes == nullptr) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "null output");
  if (m < 0 || n < 0 || k < 0) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "negative extent");
  *bytes = splits_bytes(m, n, k);
  return INTENT_HIP_OK;
}

extern "C" int intent_hip_quantized_gemm(const void *a, const void *b, const float *bias, const void *residual,
                                         const float *output_scale, void *out, int64_t m, int64_t n, int64_t k,
                                         int64_t lda, int64_t ldb, int64_t ldr, int64_t ldo, void *stream) {
  if (m < 0 || n < 0 || k < 0) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "negative extent");
  if (m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2)
    return fail(INTENT_HIP_ERR_UNSUPPORTED, "GEMM extents must stay below 2^30");
  if (m == 0 || n == 0) return INTENT_HIP_OK;
  if (out == nullptr || bias == nullptr || residual == nullptr || output_scale == nullptr ||
      (k > 0 && (a == nullptr || b == nullptr)))
    return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "null tensor pointer");
  if (lda < (m > 1 ? k : 0) || ldb < (k > 1 ? n : 0) || ldr < (m > 1 ? n : 0) || ldo < (m > 1 ? n : 0))
    return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "row stride smaller than the row length");
  const QuantizeStore ep{bias, static_cast<const uint16_t *>(residual), ldr, output_scale, static_cast<int8_t *>(out),
                         ldo};
  return launch_epilogue<_Float16>(static_cast<const uint16_t *>(a), static_cast<const uint16_t *>(b), ep, m, n, k, lda, ldb,
                                   quantize_fast_path(a, b, residual, out, n, k, lda, ldb, ldr, ldo), nullptr,
                                   as_stream(stream));
}
