// The other ops of one decode step on the rocm device: rms_norm and softmax
// along the last axis and index_select along either axis of a contiguous
// rank-two tensor (test/parity/catalogs/cuda-apertus-decode-ops.json:1-26;
// ops src/js/ops.ts:97,99,119).
//
// rms_norm(x)[r, c] = x[r, c] / sqrt(mean_c(x[r, :]^2) + epsilon) and
// softmax(x)[r, c] = exp(x[r, c] - max_r) / sum_c exp(x[r, c] - max_r), both
// computed in f32 (bf16 inputs widened exactly, bf16 outputs rounded to
// nearest even). index_select copies whole rows (axis 0) or gathers columns
// (axis 1); an index outside [0, size) selects zeros (the reference's and
// PyTorch's behaviour, test/parity/reference/probe-capabilities.py:150-153).
// All of them are HBM-bound, and latency-bound where the rows are few; a
// softmax of few long rows by its exponentials. A row takes as many threads as
// hold it in a few loads each, up to a workgroup, against one wave per row with
// one element per lane and load before. Device us, before -> now: softmax f32
// 32 x 128256 944 -> 12, 512 x 128256 2485 -> 145 (3.6 TB/s), 512 x 4096 33 ->
// 4.5; rms_norm f32 32 x 4096 19 -> 2.8, bf16 512 x 4096 22 -> 4.1. The sums
// of many short partial sums are also nearer: softmax over 128256 values 3.3e-6
// -> 7.5e-8 off 64 bits.

#include <algorithm>
#include <type_traits>

#include "device.h"
#include "internal.h"

namespace affon {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_word_t __attribute__((aligned(4)));  // 16 bytes at an f32
typedef u32x4_t u32x4_half_t __attribute__((aligned(2)));  // 16 bytes at a bf16

// W values of a row, one or 16 bytes: rows start at any element, the memory
// takes vectors there.
template <typename T, int W>
struct Vec {
  static constexpr int kValues = W;
  static_assert(W == 1 || W * T::bytes == 16, "a value or 16 bytes");
  using unaligned_t = typename std::conditional<T::bytes == 2, u32x4_half_t, u32x4_word_t>::type;
  float v[kValues];
  // Values i*kValues .. of a row of cols; those past its end are `fill`.
  __device__ __forceinline__ void load(const uint8_t* row, int64_t i, int64_t cols, float fill) {
    const int64_t at = i * kValues;
    if constexpr (W == 1) {
      v[0] = at < cols ? T::load(row, at) : fill;
    } else if (at + kValues <= cols) {
      const u32x4_t raw = *reinterpret_cast<const unaligned_t*>(row + at * T::bytes);
#pragma unroll
      for (int e = 0; e < kValues; ++e) {
        if constexpr (T::bytes == 2)
          v[e] = __uint_as_float(e % 2 ? raw[e / 2] & 0xffff0000u : raw[e / 2] << 16);
        else
          v[e] = __uint_as_float(raw[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < kValues; ++e) v[e] = at + e < cols ? T::load(row, at + e) : fill;
    }
  }
  __device__ __forceinline__ void store(uint8_t* row, int64_t i, int64_t cols) const {
    const int64_t at = i * kValues;
    if (W > 1 && at + kValues <= cols) {
      u32x4_t raw;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (W == 1)
          raw[e] = 0;
        else if constexpr (T::bytes == 2)
          raw[e] = f32_to_bf16_bits(v[2 * e]) | static_cast<uint32_t>(f32_to_bf16_bits(v[2 * e + 1])) << 16;
        else
          raw[e] = __float_as_uint(v[e]);
      }
      *reinterpret_cast<unaligned_t*>(row + at * T::bytes) = raw;
    } else {
#pragma unroll
      for (int e = 0; e < kValues; ++e)
        if (at + e < cols) {
          if constexpr (T::bytes == 2)
            reinterpret_cast<uint16_t*>(row)[at + e] = f32_to_bf16_bits(v[e]);
          else
            reinterpret_cast<float*>(row)[at + e] = v[e];
        }
    }
  }
};

template <typename T>
constexpr int kWide = 16 / T::bytes;
constexpr int kAhead = 4;  // vectors a thread of a long row has in flight

// f(index, vector) over a thread's vectors of a row, kAhead loads at a time.
template <typename T, typename F>
__device__ __forceinline__ void for_vectors(const uint8_t* row, int64_t cols, int64_t first, int64_t end, int step,
                                            float fill, F&& f) {
  for (int64_t i = first; i < end; i += static_cast<int64_t>(kAhead) * step) {
    Vec<T, kWide<T>> vec[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (i + j * step < end) vec[j].load(row, i + j * step, cols, fill);
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (i + j * step < end) f(i + j * step, vec[j]);
  }
}

// Combines one value per thread of the THREADS that hold a row (64: a wave;
// fewer: consecutive lanes; more: the workgroup), the same result in every thread.
template <int THREADS, typename V, typename F>
__device__ __forceinline__ V row_reduce(V v, F&& combine) {
#pragma unroll
  for (int offset = THREADS < 64 ? THREADS / 2 : 32; offset > 0; offset >>= 1) v = combine(v, v.from(offset));
  if constexpr (THREADS > 64) {
    __shared__ V part[THREADS / 64];
    __syncthreads();  // an earlier row's values are read
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = part[0];
    for (int i = 1; i < THREADS / 64; ++i) v = combine(v, part[i]);
  }
  return v;
}

struct Sum {
  float s;
  __device__ __forceinline__ Sum from(int offset) const { return Sum{__shfl_xor(s, offset)}; }
};
__device__ __forceinline__ Sum add(Sum a, Sum b) { return Sum{a.s + b.s}; }

struct Max {
  float m;
  __device__ __forceinline__ Max from(int offset) const { return Max{__shfl_xor(m, offset)}; }
};

// The largest value m seen, NaNs skipped (-inf: none), and sum of exp(x - m).
struct Peak {
  float m, s;
};
// exp(x - m) where m may be -inf, the peak of nothing or of -inf alone: 0.
__device__ __forceinline__ float exp_below(float x, float m) { return expf(x - (m == -INFINITY ? 0.0f : m)); }
__device__ __forceinline__ Peak add(Peak a, Peak b) {
  const float m = fmaxf(a.m, b.m);
  return Peak{m, a.s * exp_below(a.m, m) + b.s * exp_below(b.m, m)};
}
// The peak of a row's THREADS peaks: one exponential per thread, where adding
// them pair by pair would take two per level.
template <int THREADS>
__device__ __forceinline__ Peak row_peak(Peak p) {
  const float m = row_reduce<THREADS>(Max{p.m}, [](Max a, Max b) { return Max{fmaxf(a.m, b.m)}; }).m;
  return Peak{m, row_reduce<THREADS>(Sum{p.s * exp_below(p.m, m)}, [](Sum a, Sum b) { return add(a, b); }).s};
}
// The peak of vectors first, first + step, .. below end.
template <typename T>
__device__ __forceinline__ Peak peak_of(const uint8_t* row, int64_t cols, int64_t first, int64_t end, int step) {
  Peak p{-INFINITY, 0.0f};
  for_vectors<T>(row, cols, first, end, step, -INFINITY, [&](int64_t, const Vec<T, kWide<T>>& x) {
    float m = p.m;
#pragma unroll
    for (int e = 0; e < kWide<T>; ++e) m = fmaxf(m, x.v[e]);
    if (m != p.m && p.m != -INFINITY) p.s *= exp_below(p.m, m);
    p.m = m;
#pragma unroll
    for (int e = 0; e < kWide<T>; ++e) p.s += exp_below(x.v[e], m);
  });
  return p;
}
// e / s from inv = 1 / s: the product takes one correction by its exact
// remainder (the final step of division by Newton's method), which rounds it
// as the division does: s lies in [1, cols] and e in [0, 1], so nothing
// overflows, or both are NaN.
__device__ __forceinline__ float quotient(float e, float s, float inv) {
  const float q = e * inv;
  return fmaf(fmaf(-s, q, e), inv, q);
}
// Writes exp(x - p.m) / p.s.
template <typename T>
__device__ __forceinline__ void write_softmax(const uint8_t* row, uint8_t* out, int64_t cols, int64_t first,
                                              int64_t end, int step, Peak p) {
  const float inv = 1.0f / p.s;
  for_vectors<T>(row, cols, first, end, step, -INFINITY, [&](int64_t i, Vec<T, kWide<T>>& x) {
#pragma unroll
    for (int e = 0; e < kWide<T>; ++e) {
      x.v[e] = quotient(expf(x.v[e] - p.m), p.s, inv);
    }
    x.store(out, i, cols);
  });
}

// f(row) for this workgroup's rows with THREADS threads to a row: rows of at
// most a wave several to a workgroup, else one row at a time; workgroups stride
// over what is left (all of a workgroup's threads together where they share
// a row).
constexpr int64_t kMaxGrid = int64_t(1) << 20;
template <int THREADS, typename F>
__device__ __forceinline__ void for_rows(int64_t rows, F&& f) {
  constexpr int kPer = THREADS < 256 ? 256 / THREADS : 1;
  for (int64_t row = static_cast<int64_t>(blockIdx.x) * kPer + (kPer > 1 ? threadIdx.x / THREADS : 0); row < rows;
       row += static_cast<int64_t>(gridDim.x) * kPer)
    f(row);
}

// A row is read twice, the second time from the caches.
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void rms_norm_kernel(const uint8_t* x, uint8_t* out,
                                                                                 int64_t rows, int64_t cols,
                                                                                 float epsilon) {
  const int t = threadIdx.x % THREADS;
  const int64_t n = (cols + kWide<T> - 1) / kWide<T>;
  for_rows<THREADS>(rows, [&](int64_t row) {
    const uint8_t* in = x + row * cols * T::bytes;
    Sum ss{0.0f};
    for_vectors<T>(in, cols, t, n, THREADS, 0.0f, [&](int64_t, const Vec<T, kWide<T>>& v) {
#pragma unroll
      for (int e = 0; e < kWide<T>; ++e) ss.s = fmaf(v.v[e], v.v[e], ss.s);
    });
    ss = row_reduce<THREADS>(ss, [](Sum a, Sum b) { return add(a, b); });
    const float denominator = sqrtf(ss.s / static_cast<float>(cols) + epsilon);
    uint8_t* to = out + row * cols * T::bytes;
    for_vectors<T>(in, cols, t, n, THREADS, 0.0f, [&](int64_t i, Vec<T, kWide<T>>& v) {
#pragma unroll
      for (int e = 0; e < kWide<T>; ++e) v.v[e] = v.v[e] / denominator;
      v.store(to, i, cols);
    });
  });
}

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void softmax_kernel(const uint8_t* x, uint8_t* out,
                                                                                int64_t rows, int64_t cols) {
  const int t = threadIdx.x % THREADS;
  const int64_t n = (cols + kWide<T> - 1) / kWide<T>;
  for_rows<THREADS>(rows, [&](int64_t row) {
    const uint8_t* in = x + row * cols * T::bytes;
    const Peak p = row_peak<THREADS>(peak_of<T>(in, cols, t, n, THREADS));
    write_softmax<T>(in, out + row * cols * T::bytes, cols, t, n, THREADS, p);
  });
}

// Short rows: a thread holds its HELD vectors of W values, so that a row is read
// once and each exponential taken once.
template <typename T, int W, int HELD, int THREADS>
__global__ __launch_bounds__(256) void rms_norm_held_kernel(const uint8_t* x, uint8_t* out, int64_t rows, int64_t cols,
                                                            float epsilon) {
  const int t = threadIdx.x % THREADS;
  for_rows<THREADS>(rows, [&](int64_t row) {
    Vec<T, W> v[HELD];
    Sum ss{0.0f};
#pragma unroll
    for (int j = 0; j < HELD; ++j) v[j].load(x + row * cols * T::bytes, t + j * THREADS, cols, 0.0f);
#pragma unroll
    for (int j = 0; j < HELD; ++j)
#pragma unroll
      for (int e = 0; e < W; ++e) ss.s = fmaf(v[j].v[e], v[j].v[e], ss.s);
    ss = row_reduce<THREADS>(ss, [](Sum a, Sum b) { return add(a, b); });
    const float denominator = sqrtf(ss.s / static_cast<float>(cols) + epsilon);
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
#pragma unroll
      for (int e = 0; e < W; ++e) v[j].v[e] = v[j].v[e] / denominator;
      v[j].store(out + row * cols * T::bytes, t + j * THREADS, cols);
    }
  });
}

template <typename T, int W, int HELD, int THREADS>
__global__ __launch_bounds__(256) void softmax_held_kernel(const uint8_t* x, uint8_t* out, int64_t rows, int64_t cols) {
  const int t = threadIdx.x % THREADS;
  for_rows<THREADS>(rows, [&](int64_t row) {
    Vec<T, W> v[HELD];
#pragma unroll
    for (int j = 0; j < HELD; ++j) v[j].load(x + row * cols * T::bytes, t + j * THREADS, cols, -INFINITY);
    Max peak{-INFINITY};
#pragma unroll
    for (int j = 0; j < HELD; ++j)
#pragma unroll
      for (int e = 0; e < W; ++e) peak.m = fmaxf(peak.m, v[j].v[e]);
    const float m = row_reduce<THREADS>(peak, [](Max a, Max b) { return Max{fmaxf(a.m, b.m)}; }).m;
    Sum sum{0.0f};
#pragma unroll
    for (int j = 0; j < HELD; ++j)
#pragma unroll
      for (int e = 0; e < W; ++e) sum.s += v[j].v[e] = expf(v[j].v[e] - m);
    const float s = row_reduce<THREADS>(sum, [](Sum a, Sum b) { return add(a, b); }).s;
    const float inv = 1.0f / s;
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
#pragma unroll
      for (int e = 0; e < W; ++e) v[j].v[e] = quotient(v[j].v[e], s, inv);
      v[j].store(out + row * cols * T::bytes, t + j * THREADS, cols);
    }
  });
}

// Few long rows: each is cut into parts of kPartVectors, a workgroup each,
// so that the exponentials (about 20 instructions per value, twice; on 32 CUs
// alone some 20 us of issue for 32 x 128256) spread over the GPU. The first launch leaves every part's peak in `parts`
// [rows][count], the second combines a row's and writes.
constexpr int kPartVectors = 1024;

template <typename T>
__global__ __launch_bounds__(256) void softmax_parts_kernel(const uint8_t* x, int64_t cols, int count, Peak* parts) {
  const int64_t row = blockIdx.x / count, part = blockIdx.x % count;
  const int64_t n = (cols + kWide<T> - 1) / kWide<T>;
  const int64_t first = part * kPartVectors, end = min(n, first + kPartVectors);
  const Peak p = row_peak<256>(peak_of<T>(x + row * cols * T::bytes, cols, first + threadIdx.x, end, 256));
  if (threadIdx.x == 0) parts[blockIdx.x] = p;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_write_kernel(const uint8_t* x, uint8_t* out, int64_t cols, int count,
                                                            const Peak* parts) {
  const int64_t row = blockIdx.x / count, part = blockIdx.x % count;
  Peak p{-INFINITY, 0.0f};
  for (int i = threadIdx.x; i < count; i += 256) p = add(p, parts[row * count + i]);
  p = row_peak<256>(p);
  const int64_t n = (cols + kWide<T> - 1) / kWide<T>;
  const int64_t first = part * kPartVectors, end = min(n, first + kPartVectors);
  write_softmax<T>(x + row * cols * T::bytes, out + row * cols * T::bytes, cols, first + threadIdx.x, end, 256, p);
}

// out[i, :] = x[index[i], :]: raw copies of U-sized pieces, `pieces` to a row,
// 256 consecutive ones of the output per workgroup, whichever rows they are of
// (one division for the workgroup's first row; where it is of one or two rows,
// a comparison finds a thread's). Workgroups of one row idle past its end: f32,
// device us, 1000000 rows of 4 148 against 5.3, 20000 of 257 20 and 14, 20000
// of 1024 24 and 25; a thread per element of 4 bytes 8.4, 14 and 44.
template <typename U>
__global__ __launch_bounds__(256) void select_rows_kernel(const U* x, U* out, int64_t rows, int64_t pieces,
                                                          const int64_t* index, int64_t count) {
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256;
  int64_t i = first / pieces;
  int64_t p = first - i * pieces + threadIdx.x;
  if (pieces < 256) {
    const uint32_t at = static_cast<uint32_t>(p), n = static_cast<uint32_t>(pieces);
    i += at / n;
    p = at % n;
  } else if (p >= pieces) {
    ++i;
    p -= pieces;
  }
  if (i >= count) return;
  const int64_t sel = index[i];
  U v{};
  if (sel >= 0 && sel < rows) v = x[sel * pieces + p];
  out[first + threadIdx.x] = v;
}

// out[r, i] = x[r, index[i]], one thread per output element.
template <int BYTES>
__global__ __launch_bounds__(256) void select_columns_kernel(const uint8_t* x, uint8_t* out, int64_t rows, int64_t cols,
                                                             const int64_t* index, int64_t count) {
  const int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (o >= rows * count) return;
  const int64_t r = o / count, sel = index[o - r * count];
  using U = typename std::conditional<BYTES == 2, uint16_t, uint32_t>::type;
  U v = 0;
  if (sel >= 0 && sel < cols) v = reinterpret_cast<const U*>(x)[r * cols + sel];
  reinterpret_cast<U*>(out)[o] = v;
}

}  // namespace

namespace {

template <int N>
using Int = std::integral_constant<int, N>;

// held(values per load, loads per thread, threads per row) for a row that its
// threads hold, or more(threads per row) for a longer one, whose threads take
// about four vectors each. Softmax, device us:
// Many short rows are bound by what their waves issue, and share a wave: f32
// 100000 x 64 24 with a value per lane, 59 with a wave to a row's vectors, 9.5
// now; bf16 100000 x 200 59, 87 and 21.
// Few of them are bound by latency, and bf16 rows of 33 to 40 vectors by the
// pieces at their ends; a value per lane is then ahead of 16 bytes: bf16 300 x
// 128 2.4 against 2.6, 4096 x 100 2.8 against 3.3, 10000 x 300 6.9 against 8.1.
// A workgroup that holds a row is ahead of one that reads it again: f32 20000 x
// 1025 58 a wave a row, 70 and 45 in vectors read twice, 33 held.
template <typename T, typename H, typename M>
void with_row_shape(int64_t rows, int64_t cols, H&& held, M&& more) {
  constexpr int W = kWide<T>;
  const int64_t n = (cols + W - 1) / W;
  if (n <= 40 && (rows <= 8192 || n > 32)) {
    if (cols <= 64) return held(Int<1>{}, Int<1>{}, Int<64>{});
    if (cols <= 128) return held(Int<1>{}, Int<2>{}, Int<64>{});
    return held(Int<1>{}, Int<5>{}, Int<64>{});
  }
  if (n <= 4) return held(Int<W>{}, Int<1>{}, Int<4>{});
  if (n <= 8) return held(Int<W>{}, Int<2>{}, Int<4>{});
  if (n <= 16) return held(Int<W>{}, Int<1>{}, Int<16>{});
  if (n <= 32) return held(Int<W>{}, Int<2>{}, Int<16>{});
  if (n <= 64) return held(Int<W>{}, Int<1>{}, Int<64>{});
  if (n <= 128) return held(Int<W>{}, Int<2>{}, Int<64>{});
  if (n <= 256) return held(Int<W>{}, Int<4>{}, Int<64>{});
  if (n <= 512) return held(Int<W>{}, Int<2>{}, Int<256>{});
  if (n <= 1024) return held(Int<W>{}, Int<4>{}, Int<256>{});
  if (n <= 512 * kAhead) return more(Int<256>{});
  more(Int<1024>{});
}

template <int THREADS>
dim3 row_grid(int64_t rows) {
  constexpr int kPer = THREADS < 256 ? 256 / THREADS : 1;
  return dim3(static_cast<unsigned>(std::min(kMaxGrid, (rows + kPer - 1) / kPer)));
}

template <typename T>
hipError_t rms_norm_typed(const uint8_t* x, int64_t rows, int64_t cols, float epsilon, uint8_t* out,
                          hipStream_t stream) {
  with_row_shape<T>(
      rows, cols,
      [&](auto width, auto held, auto threads) {
        hipLaunchKernelGGL((rms_norm_held_kernel<T, width, held, threads>), row_grid<threads>(rows), dim3(256), 0, stream,
                           x, out, rows, cols, epsilon);
      },
      [&](auto threads) {
        hipLaunchKernelGGL((rms_norm_kernel<T, threads>), row_grid<threads>(rows), dim3(threads), 0, stream, x, out, rows,
                           cols, epsilon);
      });
  return hipGetLastError();
}

// Rows below which a long row is cut into parts: from about half the CUs on,
// a workgroup per row fills the GPU and the second launch costs more than it
// gives.
constexpr int64_t kFewRows = 128;

template <typename T>
hipError_t softmax_typed(const uint8_t* x, int64_t rows, int64_t cols, uint8_t* out, const Launch& l) {
  const int64_t n = (cols + kWide<T> - 1) / kWide<T>;
  const int64_t count = (n + kPartVectors - 1) / kPartVectors;
  if (rows < kFewRows && count > 1 && count <= (int64_t(1) << 16)) {
    // Without scratch (a captured stream whose workspace cannot grow): one workgroup per row.
    if (auto* parts = static_cast<Peak*>(l.scratch(static_cast<size_t>(rows * count) * sizeof(Peak)))) {
      const dim3 grid(static_cast<unsigned>(rows * count));
      hipLaunchKernelGGL(softmax_parts_kernel<T>, grid, dim3(256), 0, l.stream, x, cols, static_cast<int>(count), parts);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL(softmax_write_kernel<T>, grid, dim3(256), 0, l.stream, x, out, cols, static_cast<int>(count),
                         parts);
      return hipGetLastError();
    }
  }
  with_row_shape<T>(
      rows, cols,
      [&](auto width, auto held, auto threads) {
        hipLaunchKernelGGL((softmax_held_kernel<T, width, held, threads>), row_grid<threads>(rows), dim3(256), 0,
                           l.stream, x, out, rows, cols);
      },
      [&](auto threads) {
        hipLaunchKernelGGL((softmax_kernel<T, threads>), row_grid<threads>(rows), dim3(threads), 0, l.stream, x, out, rows,
                           cols);
      });
  return hipGetLastError();
}

}  // namespace

hipError_t rms_norm_launch(const void* x, int dtype, int64_t rows, int64_t cols, float epsilon, void* out,
                           hipStream_t stream) {
  const auto* xi = static_cast<const uint8_t*>(x);
  auto* o = static_cast<uint8_t*>(out);
  return dtype == AFFON_ROCM_BF16 ? rms_norm_typed<BF16>(xi, rows, cols, epsilon, o, stream)
                                  : rms_norm_typed<F32>(xi, rows, cols, epsilon, o, stream);
}

hipError_t softmax_launch(const void* x, int dtype, int64_t rows, int64_t cols, void* out, const Launch& l) {
  const auto* xi = static_cast<const uint8_t*>(x);
  auto* o = static_cast<uint8_t*>(out);
  return dtype == AFFON_ROCM_BF16 ? softmax_typed<BF16>(xi, rows, cols, o, l) : softmax_typed<F32>(xi, rows, cols, o, l);
}

namespace {
template <typename U>
hipError_t select_rows(const void* x, int64_t rows, int64_t row_bytes, const int64_t* index, int64_t count, void* out,
                       hipStream_t stream) {
  const int64_t pieces = row_bytes / static_cast<int64_t>(sizeof(U));
  hipLaunchKernelGGL(select_rows_kernel<U>, dim3(static_cast<unsigned>((count * pieces + 255) / 256)), dim3(256), 0, stream,
                     static_cast<const U*>(x), static_cast<U*>(out), rows, pieces, index, count);
  return hipGetLastError();
}
}  // namespace

hipError_t index_select_launch(const void* x, int dtype, int64_t rows, int64_t cols, int axis, const int64_t* index,
                               int64_t count, void* out, hipStream_t stream) {
  const bool half = dtype == AFFON_ROCM_BF16;
  if (axis == 0) {
    // Rows in the largest pieces of 16, 4 or 2 bytes that every row starts at.
    const int64_t row_bytes = cols * (half ? 2 : 4);
    const uint64_t starts = static_cast<uint64_t>(row_bytes) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out);
    if (starts % 16 == 0) return select_rows<u32x4_t>(x, rows, row_bytes, index, count, out, stream);
    if (starts % 4 == 0) return select_rows<uint32_t>(x, rows, row_bytes, index, count, out, stream);
    return select_rows<uint16_t>(x, rows, row_bytes, index, count, out, stream);
  }
  const dim3 grid(static_cast<unsigned>((rows * count + 255) / 256));
  const auto* xi = static_cast<const uint8_t*>(x);
  auto* o = static_cast<uint8_t*>(out);
  if (half)
    hipLaunchKernelGGL(select_columns_kernel<2>, grid, dim3(256), 0, stream, xi, o, rows, cols, index, count);
  else
    hipLaunchKernelGGL(select_columns_kernel<4>, grid, dim3(256), 0, stream, xi, o, rows, cols, index, count);
  return hipGetLastError();
}

}  // namespace affon
