// Row softmax forward and backward for gfx950.
//
// Forward  (python/intent/examples/kernels/normalization/softmax.py:12-66):
//   m = maximum_num over the row, e = exp(x - m), s = sum(e)
//   f32:        y = e * (1 / s)
//   f16, bf16:  y = cast(e / s)          (f32 math, round-to-nearest-even cast)
// Backward (python/intent/examples/kernels/backward/softmax.py:9-25):
//   proj = sum(p * dy), dx = p * (dy - proj)   (f32 accumulation; f16 storage variant casts)
//
// Design: one wavefront owns one row at a time. The row is loaded once with
// 128-bit loads (lane l of chunk c reads columns [(64c + l) * V, +V)), held in registers,
// reduced with DPP (no LDS, no barrier), and written once: one HBM read and one write per
// element, the minimum. f16 rows are held as their raw 16-bit words where that frees registers
// (x until its exponentials replace it, dy throughout), which raises the waves per SIMD.
// The 16-bit forward of rows up to 64 * 64 * 8 elements is persistent: a grid of as many waves
// as the device holds at once walks the rows with a grid stride, and each wave loads its next row
// before it computes the current one, so the reads of one row overlap the exponentials of the
// previous (16384 x 4096 f16: 46.7 against 52 us, bit-identical; one wave per row and launch
// leaves HBM idle while a whole round of waves computes).
// Longer rows belong to a workgroup (softmax_*_block), which holds them in registers too, up to 131072 16-bit or
// 65536 f32 elements (forward; backward half of that); rows beyond are read again in each pass
// (softmax_*_stream). Rows whose layout rules out aligned 128-bit access do too, except where a wave that reads
// them element by element is faster (in_wave).
#include <math.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.hpp"

namespace intent_hip {
namespace {

constexpr int kRowsPerBlock = 2;
constexpr int kBlock = kRowsPerBlock * kWave;
constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------- vector load / store
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// 16-bit rows are read with non-temporal loads (each element is read once) and 128-bit accesses.
template <typename T, int V>
__device__ __forceinline__ void load_row_chunk(const T *p, float (&out)[V]) {
  if constexpr (V == 1) {
    out[0] = to_f32(p[0]);
  } else if constexpr (sizeof(T) == 4) {
    static_assert(V == 4, "f32 vectors hold 4 elements");
    const float4 raw = *reinterpret_cast<const float4 *>(p);
    out[0] = raw.x; out[1] = raw.y; out[2] = raw.z; out[3] = raw.w;
  } else {
    static_assert(V == 8, "16-bit vectors hold 8 elements");
    const u32x4_t raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[2 * i] = to_f32(T{static_cast<uint16_t>(raw[i] & 0xffffu)});
      out[2 * i + 1] = to_f32(T{static_cast<uint16_t>(raw[i] >> 16)});
    }
  }
}

// kStream selects non-temporal stores. The forward stores normally: in the forward -> backward
// sequence its output is the backward's input and may still be in the MALL when it is read. The
// backward's output is not read again and is streamed. Measured on the 16384 x 4096 f16 step
// (graph replays): 118.9 us with this choice, 126.0 us with both streamed, 136.1 us with
// neither.
template <typename T, int V, bool kStream>
__device__ __forceinline__ void store_row_chunk(T *p, const float (&in)[V]) {
  if constexpr (V == 1) {
    p[0] = from_f32<T>(in[0]);
  } else if constexpr (sizeof(T) == 4) {
    const f32x4_t v = {in[0], in[1], in[2], in[3]};
    if constexpr (kStream) __builtin_nontemporal_store(v, reinterpret_cast<f32x4_t *>(p));
    else *reinterpret_cast<f32x4_t *>(p) = v;
  } else {
    u32x4_t w;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = static_cast<uint32_t>(from_f32<T>(in[2 * i]).bits) |
             (static_cast<uint32_t>(from_f32<T>(in[2 * i + 1]).bits) << 16);
    if constexpr (kStream) __builtin_nontemporal_store(w, reinterpret_cast<u32x4_t *>(p));
    else *reinterpret_cast<u32x4_t *>(p) = w;
  }
}

// ---------------------------------------------------------------- element math
// exp(x - m). The f32 operator uses the library exp (ordinary IEEE f32 exp of
// x - m, ~1 ulp). The 16-bit operators round their result to 11 or 8 significant
// bits, so they use the hardware 2^x on (x - m) * log2(e): relative error below
// 4e-6 for |x - m| <= 60, far inside one f16 ulp.
template <typename T>
__device__ __forceinline__ float shifted_exp(float x, float m) {
  if constexpr (sizeof(T) == 4) {
    return expf(x - m);
  } else {
    return __builtin_amdgcn_exp2f((x - m) * kLog2e);
  }
}

// e / s for the 16-bit outputs: the quotient e * (1/s) corrected by one residual
// step, which gives the correctly rounded f32 quotient for these operand ranges
// (0 <= e <= 1 <= s), followed by the round-to-nearest-even cast.
__device__ __forceinline__ float quotient(float e, float s, float r) {
  const float q = e * r;
  return fmaf(fmaf(-q, s, e), r, q);
}

// ---------------------------------------------------------------- raw 16-bit rows
// The raw 16-bit words of one 16-byte chunk (8 elements), read once, and element i widened.
__device__ __forceinline__ u32x4_t load_words(const void *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
}
template <typename T>
__device__ __forceinline__ float widen(const u32x4_t &w, int i) {
  const uint32_t word = w[i >> 1];
  return to_f32(T{static_cast<uint16_t>((i & 1) ? (word >> 16) : (word & 0xffffu))});
}

// ---------------------------------------------------------------- forward, persistent 16-bit rows
constexpr int kPipeBlock = 256;   // 4 waves, each its own row stream

// The raw words of one row (CHUNKS 16-byte chunks per lane; chunks past the row read column 0).
template <typename T, int CHUNKS>
__device__ __forceinline__ void load_row_words(const T *xr, int cols, int lane, u32x4_t (&w)[CHUNKS]) {
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int col = (c * kWave + lane) * 8;
    w[c] = load_words(xr + (col < cols ? col : 0));
  }
}

template <typename T, int CHUNKS>
__global__ __launch_bounds__(kPipeBlock) void softmax_fwd_pipe(const T *x, T *y, int64_t rows, int cols,
                                                               int64_t xs, int64_t ys) {
  constexpr int V = 8;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * (kPipeBlock / kWave);
  int64_t row = static_cast<int64_t>(blockIdx.x) * (kPipeBlock / kWave) + (threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform
  u32x4_t cur[CHUNKS];
  load_row_words<T, CHUNKS>(x + row * xs, cols, lane, cur);
  for (; row < rows; row += stride) {
    const int64_t next = row + stride;   // wave-uniform
    u32x4_t nxt[CHUNKS];
    if (next < rows) load_row_words<T, CHUNKS>(x + next * xs, cols, lane, nxt);
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const bool live = (c * kWave + lane) * V < cols;
#pragma unroll
      for (int i = 0; i < V; ++i) m = live ? fmaxf(m, widen<T>(cur[c], i)) : m;
    }
    m = wave_max(m);
    float v[CHUNKS][V];
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const bool live = (c * kWave + lane) * V < cols;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        v[c][i] = live ? shifted_exp<T>(widen<T>(cur[c], i), m) : 0.0f;
        s += v[c][i];
      }
    }
    s = wave_sum(s);
    const float r = 1.0f / s;
    T *yr = y + row * ys;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int col = (c * kWave + lane) * V;
      if (col < cols) {
        float o[V];
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = quotient(v[c][i], s, r);
        store_row_chunk<T, V, false>(yr + col, o);
      }
    }
    if (next < rows) {
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) cur[c] = nxt[c];
    }
  }
}

// ---------------------------------------------------------------- forward, register resident
template <typename T, int V, int CHUNKS>
__global__ __launch_bounds__(kBlock) void softmax_fwd_wave(const T *x, T *y, int64_t rows, int cols,
                                                           int64_t xs, int64_t ys) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform
  const T *xr = x + row * xs;
  float v[CHUNKS][V];
  float m = -INFINITY;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int col = (c * kWave + lane) * V;
    if (col < cols) {
      load_row_chunk<T, V>(xr + col, v[c]);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) v[c][i] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < V; ++i) m = fmaxf(m, v[c][i]);
  }
  m = wave_max(m);
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const bool live = (c * kWave + lane) * V < cols;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      v[c][i] = live ? shifted_exp<T>(v[c][i], m) : 0.0f;
      s += v[c][i];
    }
  }
  s = wave_sum(s);
  const float r = 1.0f / s;
  T *yr = y + row * ys;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int col = (c * kWave + lane) * V;
    if (col < cols) {
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = sizeof(T) == 4 ? v[c][i] * r : quotient(v[c][i], s, r);
      store_row_chunk<T, V, false>(yr + col, o);
    }
  }
}

// ---------------------------------------------------------------- rows of a workgroup
// A row as its 16-byte chunks: chunk q holds columns [q V - shift, q V - shift + V), where shift (0 when
// the row starts at a 16-byte boundary) makes every chunk of x (of p) a 16-byte aligned address. Chunks
// that reach past an end of the row are written one element at a time, and read so where they would leave
// the operand; so is every chunk of another operand whose rows are aligned differently.
template <typename T>
constexpr int kChunk = 16 / sizeof(T);

template <typename T>
__device__ __forceinline__ int row_shift(const T *row) {
  return static_cast<int>((reinterpret_cast<uintptr_t>(row) & 15) / sizeof(T));
}

template <typename T>
__device__ __forceinline__ uint32_t element_bits(T v) {
  if constexpr (sizeof(T) == 4) return __float_as_uint(v);
  else return v.bits;
}

// Element i of a chunk, widened.
template <typename T>
__device__ __forceinline__ float element(const u32x4_t &w, int i) {
  if constexpr (sizeof(T) == 4) {
    const uint32_t word = w[i];
    return __uint_as_float(word);
  } else {
    return widen<T>(w, i);
  }
}

// Two 16-bit or one 32-bit -infinity: what the forward puts for elements outside the row (the maximum
// and the sum are those of the row alone: exp(-inf - m) is 0, and where m is -inf the row's own sum is NaN).
template <typename T>
constexpr uint32_t kMinusInf = sizeof(T) == 4                   ? 0xff800000u
                               : std::is_same<T, f16_t>::value ? 0xfc00fc00u
                                                               : 0xff80ff80u;

// The bytes from an operand's first element to its last: what a row's edge chunks may read (the neighbouring rows'
// elements there, or the gap between rows, are replaced after the load).
struct Span {
  uintptr_t begin, end;
};
template <typename T>
__device__ __forceinline__ Span span_of(const T *base, int64_t rows, int cols, int64_t stride) {
  return {reinterpret_cast<uintptr_t>(base), reinterpret_cast<uintptr_t>(base + (rows - 1) * stride + cols)};
}

// The chunk at `start`, elements outside the row as in `outside`. kRagged false: chunks lie wholly
// inside or wholly outside the row and are aligned. Index: int, or int64_t where a row may end within a
// chunk of 2^31 (start + V).
template <typename T, bool kRagged, typename Index>
__device__ __forceinline__ u32x4_t load_chunk(const T *row, Index start, int cols, bool whole, uint32_t outside,
                                              const Span &span) {
  constexpr int V = kChunk<T>;
  u32x4_t w;
  if constexpr (!kRagged) {
    const bool live = start < cols;
    w = load_words(row + (live ? start : 0));
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = live ? w[k] : outside;
  } else {
    w = u32x4_t{outside, outside, outside, outside};
    const uintptr_t at = reinterpret_cast<uintptr_t>(row) + static_cast<int64_t>(start) * sizeof(T);
    if (start >= cols) return w;
    if (whole && at >= span.begin && at + 16 <= span.end) {
      w = load_words(row + start);
      if (start < 0 || start + V > cols) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const bool keep = start + i >= 0 && start + i < cols;
          if constexpr (sizeof(T) == 4) w[i] = keep ? w[i] : outside;
          else w[i / 2] = keep ? w[i / 2] : (i & 1) ? (w[i / 2] & 0xffffu) | (outside & 0xffff0000u)
                                                    : (w[i / 2] & 0xffff0000u) | (outside & 0xffffu);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) {
        if (start + i < 0 || start + i >= cols) continue;
        const uint32_t bits = element_bits<T>(row[start + i]);
        if constexpr (sizeof(T) == 4) w[i] = bits;
        else w[i / 2] = (i & 1) ? (w[i / 2] & 0xffffu) | (bits << 16) : (w[i / 2] & 0xffff0000u) | bits;
      }
    }
  }
  return w;
}

// Keeps a chunk's raw words: without it the compiler keeps the widened elements of one pass for the
// next, twice the registers (and spills at 1024 threads).
__device__ __forceinline__ void keep_raw(u32x4_t &w) { asm("" : "+v"(w)); }

template <typename T, bool kRagged, bool kStream, typename Index>
__device__ __forceinline__ void store_chunk(T *row, Index start, int cols, bool whole, const float (&in)[kChunk<T>]) {
  constexpr int V = kChunk<T>;
  if (!kRagged ? start < cols : whole && start >= 0 && start + V <= cols) {
    store_row_chunk<T, V, kStream>(row + start, in);
  } else if (kRagged) {
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (start + i >= 0 && start + i < cols) row[start + i] = from_f32<T>(in[i]);
  }
}

// Maximum / sum over a workgroup, in wave order. `parts` holds one value per wave; two calls in a row
// take different arrays, so one barrier each is enough.
template <int THREADS, bool kMax>
__device__ __forceinline__ float block_reduce(float v, float *parts) {
  v = kMax ? wave_max(v) : wave_sum(v);
  if constexpr (THREADS > kWave) {
    if ((threadIdx.x & (kWave - 1)) == 0) parts[threadIdx.x >> 6] = v;
    __syncthreads();
    v = parts[0];
#pragma unroll
    for (int w = 1; w < THREADS / kWave; ++w) v = kMax ? fmaxf(v, parts[w]) : v + parts[w];
  }
  return v;
}

// One workgroup per row (grid stride), the row in registers as raw words until its exponentials
// replace them; from 16 chunks of 16-bit elements on, the exponentials are computed again for the output instead
// (they would take the registers of half the waves). Bound by HBM: bf16 2048 x 32000 in 46 us,
// 5.7 TB/s (548 us with a wave per row, 2-byte accesses and three passes over the row; 4096 x 9001 33
// against 165; backward f16 1024 x 32000 34 against 403).
// THREADS threads per row; rows of one wave go four to a workgroup (16384 x 129 f16: 12.9 us with
// one each).
template <int THREADS>
constexpr int kBlockRows = THREADS == kWave ? 4 : 1;

// The row of workgroup `slot`: rows 16 g + 2 x and 16 g + 2 x + 1 on XCD x, where softmax_bwd_wave, of two rows a workgroup,
// has them. Aligned f32 rows of 2049 to 4096 columns meet both kernels in one step, and what one wrote is then in
// the L2 that the other reads (forward and backward of 1024 x 3072 10.2 us, 15.7 in plain order; 2048 x 4096 25.6, 29.1). Where
// both kernels have one row a workgroup the plain order is faster (f16 384 x 16384 11.4 us, 13.7 in this one).
__device__ __forceinline__ int64_t paired_row(int64_t slot, int64_t rows) {
  if (slot >= rows / 16 * 16) return slot;
  const int64_t in = slot % 16;
  return slot - in + 2 * (in % 8) + in / 8;
}

template <typename T, int THREADS, int CHUNKS, bool kRagged>
__global__ __launch_bounds__(THREADS * kBlockRows<THREADS>) void softmax_fwd_block(const T *x, T *y, int64_t rows, int cols, int64_t xs,
                                                             int64_t ys) {
  constexpr int V = kChunk<T>;
  constexpr bool kHold = CHUNKS * V <= 64;
  constexpr int kRows = kBlockRows<THREADS>;
  constexpr bool kPaired = sizeof(T) == 4 && !kRagged && THREADS == 256;
  __shared__ float maxima[THREADS / kWave], sums[THREADS / kWave];
  const int thread = kRows > 1 ? threadIdx.x % THREADS : threadIdx.x;
  const Span span = span_of(x, rows, cols, xs);
  for (int64_t slot = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / THREADS; slot < rows;
       slot += static_cast<int64_t>(gridDim.x) * kRows) {
    const int64_t row = kPaired ? paired_row(slot, rows) : slot;
    const T *xr = x + row * xs;
    T *yr = y + row * ys;
    const int shift = kRagged ? row_shift(xr) : 0;
    const bool whole = !kRagged || row_shift(yr) == shift;
    const int at = thread * V - shift;
    u32x4_t w[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) w[c] = load_chunk<T, kRagged>(xr, at + c * THREADS * V, cols, true, kMinusInf<T>, span);
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
      for (int i = 0; i < V; ++i) m = fmaxf(m, element<T>(w[c], i));
    m = block_reduce<THREADS, true>(m, maxima);
    float v[kHold ? CHUNKS : 1][V];
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      keep_raw(w[c]);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float e = shifted_exp<T>(element<T>(w[c], i), m);
        if constexpr (kHold) v[c][i] = e;
        s += e;
      }
    }
    s = block_reduce<THREADS, false>(s, sums);
    const float r = 1.0f / s;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if constexpr (!kHold) keep_raw(w[c]);
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float e = kHold ? v[kHold ? c : 0][i] : shifted_exp<T>(element<T>(w[c], i), m);
        o[i] = sizeof(T) == 4 ? e * r : quotient(e, s, r);
      }
      store_chunk<T, kRagged, false>(yr, at + c * THREADS * V, cols, whole, o);
    }
  }
}

// Rows that no workgroup's registers hold: the row is read once for each of the maximum, the sum and the output.
constexpr int kStreamBlock = 1024;

template <typename T>
__global__ __launch_bounds__(kStreamBlock) void softmax_fwd_stream(const T *x, T *y, int64_t rows, int cols,
                                                                   int64_t xs, int64_t ys) {
  constexpr int V = kChunk<T>;
  __shared__ float maxima[kStreamBlock / kWave], sums[kStreamBlock / kWave];
  const Span span = span_of(x, rows, cols, xs);
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const T *xr = x + row * xs;
    T *yr = y + row * ys;
    const int shift = row_shift(xr);
    const bool whole = row_shift(yr) == shift;
    const int64_t first = static_cast<int64_t>(threadIdx.x) * V - shift;
    float m = -INFINITY;
    for (int64_t at = first; at < cols; at += kStreamBlock * V) {
      const u32x4_t w = load_chunk<T, true>(xr, at, cols, true, kMinusInf<T>, span);
#pragma unroll
      for (int i = 0; i < V; ++i) m = fmaxf(m, element<T>(w, i));
    }
    m = block_reduce<kStreamBlock, true>(m, maxima);
    float s = 0.0f;
    for (int64_t at = first; at < cols; at += kStreamBlock * V) {
      const u32x4_t w = load_chunk<T, true>(xr, at, cols, true, kMinusInf<T>, span);
#pragma unroll
      for (int i = 0; i < V; ++i) s += shifted_exp<T>(element<T>(w, i), m);
    }
    s = block_reduce<kStreamBlock, false>(s, sums);
    const float r = 1.0f / s;
    for (int64_t at = first; at < cols; at += kStreamBlock * V) {
      const u32x4_t w = load_chunk<T, true>(xr, at, cols, true, kMinusInf<T>, span);
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float e = shifted_exp<T>(element<T>(w, i), m);
        o[i] = sizeof(T) == 4 ? e * r : quotient(e, s, r);
      }
      store_chunk<T, true, false>(yr, at, cols, whole, o);
    }
  }
}

// ---------------------------------------------------------------- backward, register resident
template <typename T, int V, int CHUNKS>
__global__ __launch_bounds__(kBlock) void softmax_bwd_wave(const T *p, const T *dy, T *dx, int64_t rows,
                                                           int cols, int64_t ps, int64_t dys,
                                                           int64_t dxs) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *pr = p + row * ps;
  const T *gr = dy + row * dys;
  if constexpr (sizeof(T) == 2 && V == 8) {
    // dy stays in its raw words and is widened where it is used (f16: the FMAs take the operands
    // directly, v_fma_mix_f32): 81 VGPRs instead of 141, five waves per SIMD instead of three.
    // Backward of the 16384 x 4096 step, bit-identical outputs: 62.0 us, against 75.7 with both
    // rows widened at load and 68.0 with both kept raw (77 VGPRs, six waves). Every chunk is
    // loaded; one past the row end re-reads the row start and stays out of the projection
    // (conditional loads make the compiler keep widened copies live).
    float pv[CHUNKS][V];
    u32x4_t gw[CHUNKS];
    float proj = 0.0f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int col = (c * kWave + lane) * V;
      const bool live = col < cols;
      const int at = live ? col : 0;
      load_row_chunk<T, V>(pr + at, pv[c]);
      gw[c] = load_words(gr + at);
#pragma unroll
      for (int i = 0; i < V; ++i) proj = live ? fmaf(pv[c][i], widen<T>(gw[c], i), proj) : proj;
    }
    proj = wave_sum(proj);
    T *dr = dx + row * dxs;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int col = (c * kWave + lane) * V;
      if (col < cols) {
        float o[V];
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = pv[c][i] * (widen<T>(gw[c], i) - proj);
        store_row_chunk<T, V, true>(dr + col, o);
      }
    }
    return;
  }
  float pv[CHUNKS][V], gv[CHUNKS][V];
  float proj = 0.0f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int col = (c * kWave + lane) * V;
    if (col < cols) {
      load_row_chunk<T, V>(pr + col, pv[c]);
      load_row_chunk<T, V>(gr + col, gv[c]);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) pv[c][i] = gv[c][i] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < V; ++i) proj = fmaf(pv[c][i], gv[c][i], proj);
  }
  proj = wave_sum(proj);
  T *dr = dx + row * dxs;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int col = (c * kWave + lane) * V;
    if (col < cols) {
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = pv[c][i] * (gv[c][i] - proj);
      store_row_chunk<T, V, true>(dr + col, o);
    }
  }
}

// One workgroup per row (grid stride), p and dy in registers as raw words.
template <typename T, int THREADS, int CHUNKS, bool kRagged>
__global__ __launch_bounds__(THREADS * kBlockRows<THREADS>) void softmax_bwd_block(const T *p, const T *dy, T *dx, int64_t rows, int cols,
                                                             int64_t ps, int64_t dys, int64_t dxs) {
  constexpr int V = kChunk<T>;
  constexpr int kRows = kBlockRows<THREADS>;
  __shared__ float sums[2][THREADS / kWave];
  const int thread = kRows > 1 ? threadIdx.x % THREADS : threadIdx.x;
  const Span span_p = span_of(p, rows, cols, ps), span_g = span_of(dy, rows, cols, dys);
  int turn = 0;
  for (int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / THREADS; row < rows;
       row += static_cast<int64_t>(gridDim.x) * kRows, turn ^= 1) {
    const T *pr = p + row * ps;
    const T *gr = dy + row * dys;
    T *dr = dx + row * dxs;
    const int shift = kRagged ? row_shift(pr) : 0;
    const bool whole_g = !kRagged || row_shift(gr) == shift, whole_d = !kRagged || row_shift(dr) == shift;
    const int at = thread * V - shift;
    u32x4_t pw[CHUNKS], gw[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      pw[c] = load_chunk<T, kRagged>(pr, at + c * THREADS * V, cols, true, 0, span_p);
      gw[c] = load_chunk<T, kRagged>(gr, at + c * THREADS * V, cols, whole_g, 0, span_g);
    }
    float proj = 0.0f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
      for (int i = 0; i < V; ++i) proj = fmaf(element<T>(pw[c], i), element<T>(gw[c], i), proj);
    proj = block_reduce<THREADS, false>(proj, sums[turn]);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      keep_raw(pw[c]);
      keep_raw(gw[c]);
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = element<T>(pw[c], i) * (element<T>(gw[c], i) - proj);
      store_chunk<T, kRagged, true>(dr, at + c * THREADS * V, cols, whole_d, o);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kStreamBlock) void softmax_bwd_stream(const T *p, const T *dy, T *dx, int64_t rows,
                                                                   int cols, int64_t ps, int64_t dys, int64_t dxs) {
  constexpr int V = kChunk<T>;
  __shared__ float sums[2][kStreamBlock / kWave];
  const Span span_p = span_of(p, rows, cols, ps), span_g = span_of(dy, rows, cols, dys);
  int turn = 0;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x, turn ^= 1) {
    const T *pr = p + row * ps;
    const T *gr = dy + row * dys;
    T *dr = dx + row * dxs;
    const int shift = row_shift(pr);
    const bool whole_g = row_shift(gr) == shift, whole_d = row_shift(dr) == shift;
    const int64_t first = static_cast<int64_t>(threadIdx.x) * V - shift;
    float proj = 0.0f;
    for (int64_t at = first; at < cols; at += kStreamBlock * V) {
      const u32x4_t pw = load_chunk<T, true>(pr, at, cols, true, 0, span_p);
      const u32x4_t gw = load_chunk<T, true>(gr, at, cols, whole_g, 0, span_g);
#pragma unroll
      for (int i = 0; i < V; ++i) proj = fmaf(element<T>(pw, i), element<T>(gw, i), proj);
    }
    proj = block_reduce<kStreamBlock, false>(proj, sums[turn]);
    for (int64_t at = first; at < cols; at += kStreamBlock * V) {
      const u32x4_t pw = load_chunk<T, true>(pr, at, cols, true, 0, span_p);
      const u32x4_t gw = load_chunk<T, true>(gr, at, cols, whole_g, 0, span_g);
      float o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = element<T>(pw, i) * (element<T>(gw, i) - proj);
      store_chunk<T, true, true>(dr, at, cols, whole_d, o);
    }
  }
}

// ---------------------------------------------------------------- variant selection
struct Variant {
  const void *kernel;
  const char *name;
  int block = kBlock;                  // threads per workgroup
  int rows_per_block = kRowsPerBlock;  // rows a workgroup takes at a time
  bool persistent = false;             // grid of resident waves walking the rows (rows per wave: any)
};

template <typename T>
Variant pick_fwd_pipe(int chunks) {
  constexpr int kRows = kPipeBlock / kWave;
  switch (chunks) {
    case 1: return {reinterpret_cast<const void *>(&softmax_fwd_pipe<T, 1>), "softmax_fwd_pipe", kPipeBlock, kRows, true};
    case 2: return {reinterpret_cast<const void *>(&softmax_fwd_pipe<T, 2>), "softmax_fwd_pipe", kPipeBlock, kRows, true};
    case 4: return {reinterpret_cast<const void *>(&softmax_fwd_pipe<T, 4>), "softmax_fwd_pipe", kPipeBlock, kRows, true};
    default: return {reinterpret_cast<const void *>(&softmax_fwd_pipe<T, 8>), "softmax_fwd_pipe", kPipeBlock, kRows, true};
  }
}

// The workgroup of a row: the fewest threads that hold it with the registers of many waves left, from one
// wave per 512 16-bit elements on. A ragged row can reach into one more chunk than its length fills.
#define INTENT_BLOCK(THREADS, CHUNKS)                                                                               \
  if (elements <= static_cast<int64_t>(THREADS) * CHUNKS * kChunk<T>)                                               \
    return {reinterpret_cast<const void *>(&INTENT_ROW_KERNEL<T, THREADS, CHUNKS, kRagged>), INTENT_ROW_NAME,   \
            THREADS * kBlockRows<THREADS>, kBlockRows<THREADS>};

template <typename T, bool kRagged>
Variant pick_fwd_block(int64_t cols) {
  const int64_t elements = kRagged ? cols + kChunk<T> - 1 : cols;
#define INTENT_ROW_KERNEL softmax_fwd_block
#define INTENT_ROW_NAME "softmax_fwd_block"
  if constexpr (kRagged && sizeof(T) == 2) {   // shorter f32 rows belong to a wave
    INTENT_BLOCK(64, 1)
    INTENT_BLOCK(64, 2)
  }
  if constexpr (kRagged) {
    INTENT_BLOCK(64, 4)
    INTENT_BLOCK(64, 8)
  }
  INTENT_BLOCK(256, 4)
  INTENT_BLOCK(512, 4)
  INTENT_BLOCK(512, 8)
  INTENT_BLOCK(1024, 8)
  if constexpr (!kRagged) return pick_fwd_block<T, true>(cols);   // its edge selects spill at 16 chunks
  INTENT_BLOCK(1024, 16)
#undef INTENT_ROW_KERNEL
#undef INTENT_ROW_NAME
  return {reinterpret_cast<const void *>(&softmax_fwd_stream<T>), "softmax_fwd_stream", kStreamBlock, 1};
}

template <typename T, bool kRagged>
Variant pick_bwd_block(int64_t cols) {
  const int64_t elements = kRagged ? cols + kChunk<T> - 1 : cols;
#define INTENT_ROW_KERNEL softmax_bwd_block
#define INTENT_ROW_NAME "softmax_bwd_block"
  if constexpr (kRagged && sizeof(T) == 2) {   // shorter f32 rows belong to a wave
    INTENT_BLOCK(64, 1)
    INTENT_BLOCK(64, 2)
  }
  if constexpr (kRagged) {
    INTENT_BLOCK(64, 4)
    INTENT_BLOCK(64, 8)
  }
  INTENT_BLOCK(256, 4)
  INTENT_BLOCK(512, 4)
  INTENT_BLOCK(1024, 4)
  INTENT_BLOCK(1024, 8)
#undef INTENT_ROW_KERNEL
#undef INTENT_ROW_NAME
  return {reinterpret_cast<const void *>(&softmax_bwd_stream<T>), "softmax_bwd_stream", kStreamBlock, 1};
}
#undef INTENT_BLOCK

// Most chunks a wave holds: of single elements 1024 16-bit or 4096 f32 columns, of 16 bytes 4096 columns.
template <typename T, int V>
constexpr int kMostChunks = V == 1 ? (sizeof(T) == 4 ? 64 : 16) : sizeof(T) == 4 ? 16 : 8;

template <typename T, int V, int CHUNKS = 1>
Variant pick_fwd(int chunks) {
  if constexpr (CHUNKS < kMostChunks<T, V>)
    if (chunks > CHUNKS) return pick_fwd<T, V, 2 * CHUNKS>(chunks);
  return {reinterpret_cast<const void *>(&softmax_fwd_wave<T, V, CHUNKS>), "softmax_fwd_wave"};
}

template <typename T, int V, int CHUNKS = 1>
Variant pick_bwd(int chunks) {
  if constexpr (CHUNKS < kMostChunks<T, V>)
    if (chunks > CHUNKS) return pick_bwd<T, V, 2 * CHUNKS>(chunks);
  return {reinterpret_cast<const void *>(&softmax_bwd_wave<T, V, CHUNKS>), "softmax_bwd_wave"};
}

int round_chunks(int64_t cols, int per_chunk) {
  const int64_t needed = (cols + per_chunk - 1) / per_chunk;
  int chunks = 1;
  while (chunks < needed) chunks <<= 1;
  return chunks;
}

// Rows that 16-byte access does not fit: in a wave, one element per lane and chunk (whose time follows the power of two
// that the chunks round up to), or in a workgroup, which reads 16 bytes a lane and selects at the row's ends. While the
// operands lie in the 256 MB of the MALL a wave's reads cost it less; past that HBM bounds both and whole lines
// lead. Measured, workgroup over wave time:
//   * f32 forward: 1.0 to 1.4 up to 2048 columns in the MALL, 0.77 to 0.95 past it (64M elements); from 2049 columns on
//     0.5 (2^19 elements in all) to 1.0 (2^25);
//   * f32 backward: 1.1 to 1.4 up to 2048 columns in the MALL, 0.88 to 0.97 past it; from 2049 on 0.6 to 1.07;
//   * 16 bits, one rule for both directions, by the time of a forward and a backward in turn (where one takes the wave and
//     the other the workgroup, a step loses up to 5 us below 2^23 elements and a quarter past it): up to 384
//     columns 0.97 to 1.2 in the MALL, 0.94 to 1.06 past it; to 505 0.96 to 1.1 below 3M elements, 0.83 to 1.0 from there; to
//     640, just past a step of the workgroup's registers, 0.94 to 1.2 in the MALL; to 1017 0.83 to 1.1; to 1024, the next
//     step, 1.01 to 1.17 below 6M, 0.86 to 1.04 from there; then 0.7 to 0.97;
//   * f32 from 4094 to 4096 columns, a step as well, with 2048 rows or more 1.05 to 1.19 in the MALL.
template <typename T>
bool in_mall(int operands, int64_t rows, int64_t cols) {
  return operands * static_cast<int64_t>(sizeof(T)) * rows * cols <= int64_t{256} << 20;
}

// `operands`: how many of the call's arrays lie in the MALL.
template <typename T>
bool in_wave(int operands, int64_t rows, int64_t cols) {
  if (cols > 4096) return false;
  if constexpr (sizeof(T) == 4)
    return cols <= 512 || (in_mall<T>(operands, rows, cols) && (cols <= 2048 || (cols > 4093 && rows >= 2048)));
  if (cols <= 256) return true;
  if (cols <= 384 || (cols > 505 && cols <= 640)) return in_mall<T>(3, rows, cols);
  return (cols <= 505 && rows * cols < int64_t{3} << 20) || (cols > 1017 && cols <= 1024 && rows * cols < int64_t{6} << 20);
}

// Aligned rows belong to a wave up to kMostChunks (f32 4096 x 4096 backward: 29.5 us, 31.7 in a workgroup). The f32 forward of
// 2049 to 4096 columns does from 10M elements on that lie in the MALL (workgroup over wave time 0.97 to 1.13, 0.65 to 1.0
// below, 0.76 to 0.85 past it).
template <typename T>
Variant select_fwd(const void *x, const void *y, int64_t rows, int64_t cols, int64_t xs, int64_t ys) {
  constexpr int kVec = kChunk<T>;
  const bool vector = cols % kVec == 0 && xs % kVec == 0 && ys % kVec == 0 && aligned(x, 16) && aligned(y, 16);
  if (!vector)
    return in_wave<T>(2, rows, cols) ? pick_fwd<T, 1>(round_chunks(cols, kWave)) : pick_fwd_block<T, true>(cols);
  const int chunks = round_chunks(cols, kWave * kVec);
  const bool wave = chunks <= 8 || (chunks <= kMostChunks<T, kVec> && rows * cols >= int64_t{10} << 20 && in_mall<T>(2, rows, cols));
  if (!wave) return pick_fwd_block<T, false>(cols);
  if constexpr (sizeof(T) == 2) return pick_fwd_pipe<T>(chunks);
  else return pick_fwd<T, kVec>(chunks);
}

template <typename T>
Variant select_bwd(const void *p, const void *dy, const void *dx, int64_t rows, int64_t cols, int64_t ps, int64_t dys,
                   int64_t dxs) {
  constexpr int kVec = kChunk<T>;
  const bool vector = cols % kVec == 0 && ps % kVec == 0 && dys % kVec == 0 && dxs % kVec == 0 &&
                      aligned(p, 16) && aligned(dy, 16) && aligned(dx, 16);
  if (!vector)
    return in_wave<T>(3, rows, cols) ? pick_bwd<T, 1>(round_chunks(cols, kWave)) : pick_bwd_block<T, true>(cols);
  const int chunks = round_chunks(cols, kWave * kVec);
  return chunks > kMostChunks<T, kVec> ? pick_bwd_block<T, false>(cols) : pick_bwd<T, kVec>(chunks);
}

// Input rows may overlap (any non-negative stride, e.g. a broadcast row); output
// rows may not.
int check_extents(int64_t rows, int64_t cols, int64_t in0, int64_t in1, int64_t out) {
  if (rows < 0 || cols < 0) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "negative extent");
  if (cols > INT32_MAX) return fail(INTENT_HIP_ERR_UNSUPPORTED, "softmax rows longer than 2^31-1 columns");
  if (rows > static_cast<int64_t>(UINT32_MAX) * kRowsPerBlock)
    return fail(INTENT_HIP_ERR_UNSUPPORTED, "too many softmax rows for one launch");
  if (in0 < 0 || in1 < 0) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "negative row stride");
  if (rows > 1 && out < cols)
    return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "output row stride smaller than the row length (overlapping rows)");
  return INTENT_HIP_OK;
}

// Workgroups of a launch over `rows`: at most as many as the device holds at once for a persistent
// kernel, and for the softmax_*_block and _stream kernels as many as a launch may have (fewer than 2^32 threads in
// all), which walk the rest with a grid stride.
int64_t grid_blocks(const Variant &v, int64_t rows) {
  const int64_t blocks = (rows + v.rows_per_block - 1) / v.rows_per_block;
  if (v.persistent) return std::min<int64_t>(blocks, resident_blocks(v.kernel, v.block));
  return v.rows_per_block == kRowsPerBlock ? blocks : std::min<int64_t>(blocks, UINT32_MAX / v.block);
}

template <typename T>
int launch_fwd(const void *x, void *y, int64_t rows, int64_t cols, int64_t xs, int64_t ys, hipStream_t stream) {
  const Variant v = select_fwd<T>(x, y, rows, cols, xs, ys);
  const dim3 grid(static_cast<unsigned>(grid_blocks(v, rows)));
  int icols = static_cast<int>(cols);
  void *args[] = {const_cast<void **>(&x), &y, &rows, &icols, &xs, &ys};
  if (hipLaunchKernel(v.kernel, grid, dim3(v.block), args, 0, stream) != hipSuccess) return launch_status(v.name);
  return INTENT_HIP_OK;
}

template <typename T>
int launch_bwd(const void *p, const void *dy, void *dx, int64_t rows, int64_t cols, int64_t ps, int64_t dys,
               int64_t dxs, hipStream_t stream) {
  const Variant v = select_bwd<T>(p, dy, dx, rows, cols, ps, dys, dxs);
  const dim3 grid(static_cast<unsigned>(grid_blocks(v, rows)));
  int icols = static_cast<int>(cols);
  void *args[] = {const_cast<void **>(&p), const_cast<void **>(&dy), &dx, &rows, &icols, &ps, &dys, &dxs};
  if (hipLaunchKernel(v.kernel, grid, dim3(v.block), args, 0, stream) != hipSuccess) return launch_status(v.name);
  return INTENT_HIP_OK;
}

}  // namespace

int softmax_fwd_resources(int dtype, const void *x, const void *y, int64_t rows, int64_t cols, int64_t xs, int64_t ys,
                          IntentHipKernelResources *out) {
  Variant v;
  switch (dtype) {
    case INTENT_HIP_F32: v = select_fwd<float>(x, y, rows, cols, xs, ys); break;
    case INTENT_HIP_F16: v = select_fwd<f16_t>(x, y, rows, cols, xs, ys); break;
    case INTENT_HIP_BF16: v = select_fwd<bf16_t>(x, y, rows, cols, xs, ys); break;
    default: return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "unknown dtype code %d", dtype);
  }
  return describe_kernel(v.kernel, v.name, v.block, out);
}

int softmax_bwd_resources(int dtype, const void *p, const void *dy, const void *dx, int64_t rows, int64_t cols, int64_t ps,
                          int64_t dys, int64_t dxs, IntentHipKernelResources *out) {
  Variant v;
  switch (dtype) {
    case INTENT_HIP_F32: v = select_bwd<float>(p, dy, dx, rows, cols, ps, dys, dxs); break;
    case INTENT_HIP_F16: v = select_bwd<f16_t>(p, dy, dx, rows, cols, ps, dys, dxs); break;
    case INTENT_HIP_BF16: v = select_bwd<bf16_t>(p, dy, dx, rows, cols, ps, dys, dxs); break;
    default: return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "unknown dtype code %d", dtype);
  }
  return describe_kernel(v.kernel, v.name, v.block, out);
}

}  // namespace intent_hip

using namespace intent_hip;

extern "C" int intent_hip_softmax_fwd(int dtype, const void *x, void *y, int64_t rows, int64_t cols,
                                      int64_t x_row_stride, int64_t y_row_stride, void *stream) {
  if (int status = check_extents(rows, cols, x_row_stride, x_row_stride, y_row_stride)) return status;
  if (rows == 0 || cols == 0) return INTENT_HIP_OK;
  if (x == nullptr || y == nullptr) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "null tensor pointer");
  switch (dtype) {
    case INTENT_HIP_F32: return launch_fwd<float>(x, y, rows, cols, x_row_stride, y_row_stride, as_stream(stream));
    case INTENT_HIP_F16: return launch_fwd<f16_t>(x, y, rows, cols, x_row_stride, y_row_stride, as_stream(stream));
    case INTENT_HIP_BF16: return launch_fwd<bf16_t>(x, y, rows, cols, x_row_stride, y_row_stride, as_stream(stream));
  }
  return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "unknown dtype code %d", dtype);
}

extern "C" int intent_hip_softmax_bwd(int dtype, const void *p, const void *dy, void *dx, int64_t rows,
                                      int64_t cols, int64_t p_row_stride, int64_t dy_row_stride,
                                      int64_t dx_row_stride, void *stream) {
  if (int status = check_extents(rows, cols, p_row_stride, dy_row_stride, dx_row_stride)) return status;
  if (rows == 0 || cols == 0) return INTENT_HIP_OK;
  if (p == nullptr || dy == nullptr || dx == nullptr) return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "null tensor pointer");
  switch (dtype) {
    case INTENT_HIP_F32:
      return launch_bwd<float>(p, dy, dx, rows, cols, p_row_stride, dy_row_stride, dx_row_stride, as_stream(stream));
    case INTENT_HIP_F16:
      return launch_bwd<f16_t>(p, dy, dx, rows, cols, p_row_stride, dy_row_stride, dx_row_stride, as_stream(stream));
    case INTENT_HIP_BF16:
      return launch_bwd<bf16_t>(p, dy, dx, rows, cols, p_row_stride, dy_row_stride, dx_row_stride, as_stream(stream));
  }
  return fail(INTENT_HIP_ERR_INVALID_ARGUMENT, "unknown dtype code %d", dtype);
}
