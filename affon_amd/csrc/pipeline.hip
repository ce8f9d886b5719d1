// Host-side pieces shared by the tiled kernels, and the ordered reduction of
// split-K partial sums.
#include "lds_pipeline.h"

namespace affon {
namespace pipeline {
namespace {

// Values at a multiple of 4 bytes (a K range of an odd number of outputs
// starts at any of them); the memory takes vectors there.
typedef f32x4_t f32x4_word_t __attribute__((aligned(4)));

// Entry i (of `count`) of every K range, added in an order that depends on
// `splits` and on whether the outputs are few for the GPU (FEW, launch_reduce):
// the values V that start there. Few outputs wait for their loads, so that
// those of eight ranges are in flight together, and their ranges may be many,
// so that eight are added as a tree (38 x 276 x 8320, 32 ranges: 1.28e-7 off 64
// bits one after another). Many outputs are bound by HBM and read one range
// after another (512 x 4096, four ranges: eight in flight cost 1.5 us of 76).
template <bool FEW, typename V>
__device__ __forceinline__ V sum_ranges(const float* partial, int64_t i, int64_t count, int splits) {
  auto load = [&](int r) { return __builtin_nontemporal_load(reinterpret_cast<const V*>(partial + r * count + i)); };
  if constexpr (FEW) {
    V sum{};
    for (int r0 = 0; r0 < splits; r0 += 8) {
      V v[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        v[r] = V{};
        if (r0 + r < splits) v[r] = load(r0 + r);
      }
      const V batch = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      sum = r0 == 0 ? batch : sum + batch;
    }
    return sum;
  } else {
    V sum = load(0);
    for (int r = 1; r < splits; ++r) sum += load(r);
    return sum;
  }
}

// out[i] = sum of the K ranges' partial sums (the same result on every run),
// then the output epilogue. Four outputs per thread;
// `count` = M*N, `n` = N. A grouped launch's partials span all its segments'
// columns (row stride n = total columns); each sum goes to its segment's
// output. Bound by latency where the ranges are many and small: per output
// and range a load of its own, as counts that are no multiple of four had it,
// took 2 x 1569 x 13728 (10 ranges) from 15 to 19 us a call.
template <bool FEW>
__global__ __launch_bounds__(256) void reduce_partials_kernel(const float* partial, float* out, int64_t count,
                                                              int64_t n, int splits, Epilogue epi, Segments seg) {
  const int64_t own = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (own >= count) return;
  // The last thread of a count that is no multiple of four sums the last four
  // outputs and stores its own, [first, 4) of them; below four outputs it
  // sums the [0, end) there are.
  const int64_t i = max(min(own, count - 4), int64_t{0});
  const int first = static_cast<int>(own - i), end = static_cast<int>(min(count, int64_t{4}));
  f32x4_t sum{};
  if (end == 4) {
    sum = sum_ranges<FEW, f32x4_word_t>(partial, i, count, splits);
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < end) sum[k] = sum_ranges<FEW, float>(partial, k, count, splits);
  }
  if (seg.count > 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k < first || k >= end) continue;
      const int64_t row = (i + k) / n;
      const int c = static_cast<int>(i + k - row * n);
      const int s = seg_of(seg, seg.col_base, c);
      const int col = c - seg_pick(seg.col_base, s);
      Epilogue e = epi;
      e.bias = seg_pick(seg.bias, s);
      e.kind = e.bias != nullptr ? kEpiBias : kEpiNone;
      store_output(e, seg_pick(seg.out, s), row * seg_pick(seg.n, s) + col, col, sum[k]);
    }
  } else if (epi.kind == kEpiNone && first == 0 && end == 4) {
    *reinterpret_cast<f32x4_word_t*>(out + i) = sum;
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k >= first && k < end) store_output(epi, out, i + k, (i + k) % n, sum[k]);
  }
}

}  // namespace

int device_cus() {
  static std::mutex mutex;
  static int cached[64] = {0};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
  std::lock_guard<std::mutex> lock(mutex);
  if (cached[device] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
    cached[device] = cus;
  }
  return cached[device];
}

int choose_splits(int tiles, int steps) {
  const int target = device_cus() * 3 / 4;
  int splits = 1;
  if (tiles >= target) return 1;
  for (int s = 2; s <= 8; ++s) {
    if ((steps / 4) % s != 0) continue;
    if (steps / s < 8) break;
    splits = s;
    if (tiles * s >= target) break;
  }
  return splits;
}


hipError_t launch_reduce(const TileArgs& args, hipStream_t stream) {
  const int64_t n = args.seg.count > 0 ? args.seg.total_n : args.N;
  const int64_t count = static_cast<int64_t>(args.M) * n;
  const int64_t blocks = (count + 1023) / 1024;
  const dim3 grid(static_cast<unsigned>(blocks));
  if (blocks < 2 * device_cus())
    hipLaunchKernelGGL(reduce_partials_kernel<true>, grid, dim3(256), 0, stream, args.partial, args.out, count, n,
                       args.splits, args.epi, args.seg);
  else
    hipLaunchKernelGGL(reduce_partials_kernel<false>, grid, dim3(256), 0, stream, args.partial, args.out, count, n,
                       args.splits, args.epi, args.seg);
  return hipGetLastError();
}

}  // namespace pipeline
}  // namespace affon
