// Shapes and plans of the general matrix-core kernels (xgemm.h), which
// gemv_launch runs for the problems they take.
#include <algorithm>

#include "xgemm.h"

namespace affon {
namespace xgemm {

hipError_t launch_b2(const Args& args, Shape shape, bool g32, int x_dtype, int p_dtype, hipStream_t stream);
hipError_t launch_b4(const Args& args, Shape shape, bool g32, int x_dtype, int p_dtype, hipStream_t stream);
hipError_t launch_b8(const Args& args, Shape shape, bool g32, int x_dtype, int p_dtype, hipStream_t stream);

namespace {

constexpr int64_t kMaxPartialBytes = int64_t(32) << 20;  // what the no-allocation entry point holds
// Few columns and a long K: with eight ranges 48 x 256 x 14336 takes 38 us a
// call, with 16 24.2 and with 32 18.1; the reduction reads eight at a time.
constexpr int kMaxSplits = 32;

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The most K ranges (at most kMaxSplits) that keep `least` of K's `units` each
// and partial sums within kMaxPartialBytes.
int most_splits(const QmmProblem& p, int64_t units, int least) {
  const int64_t s = std::min<int64_t>(units / least, kMaxPartialBytes / (p.M * p.N * 4));
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(s, kMaxSplits)));
}

// Whether the VALU kernel (gemv.hip) is ahead of one K range here. A range's
// time is that of its steps one after another, the VALU kernel's grows with the
// columns of all its passes. f32, us, VALU kernel first: 8 x 1024 x 14336 at 4
// bits 19 and 52, 4096 columns 72 and 53; 8 x 4096 x 4096 at 8 bits 20 and 18;
// 64-row tiles take longer, 33 x 256 x 4096 at 4 bits 19 and 70, 2048 columns
// 81 and 71; 64 x 1024 x 4096 at 8 bits 33 and 77, 4096 columns 114 and 77.
bool one_range_is_behind(const QmmProblem& p) {
  const int64_t columns = (p.M + 3) / 4 * p.N;
  if (p.M <= 32) return p.K >= 2048 && columns <= p.K;
  const int64_t per_k = p.bits == 4 ? 4 : p.bits == 2 && p.group % 64 == 0 ? 2 : 8;
  return p.K >= 1024 && columns <= per_k * p.K;
}

}  // namespace
}  // namespace xgemm

bool xgemm_supports(const QmmProblem& p) {
  using pipeline::kBK;
  if (p.xs1 != 1 || p.ws1 != 1 || p.ss1 != 1 || p.bs1 != 1) return false;
  if (p.group % 32 != 0) return false;
  const int64_t xbytes = p.x_dtype == AFFON_ROCM_BF16 ? 2 : 4, pbytes = p.p_dtype == AFFON_ROCM_BF16 ? 2 : 4;
  if (reinterpret_cast<uintptr_t>(p.x) % 16 != 0 || (p.xs0 * xbytes) % 16 != 0) return false;
  // 16 codes at a time: 4, 8 or 16 bytes.
  const int64_t run = 2 * p.bits;
  if (reinterpret_cast<uintptr_t>(p.w) % run != 0 || (p.ws0 * 4) % run != 0) return false;
  if (reinterpret_cast<uintptr_t>(p.s) % pbytes != 0 || reinterpret_cast<uintptr_t>(p.b) % pbytes != 0) return false;
  if (p.K * p.bits < 128) return false;  // packed rows of at least 16 bytes
  // 32-bit byte offsets from a uniform base, 32-bit grids, and a group index
  // by multiplication (Args::group_of), exact for blocks * blocks per group < 2^32.
  const int64_t limit = int64_t(1) << 31;
  if (p.M >= limit || p.N >= limit || p.K >= limit - kBK || p.group >= limit) return false;
  if (p.M * p.xs0 * xbytes >= limit || p.N * p.ws0 * 4 >= limit) return false;
  if (p.N * p.ss0 * pbytes >= limit || p.N * p.bs0 * pbytes >= limit) return false;
  if ((p.K / 32) * (p.group / 32) >= (int64_t(1) << 32)) return false;
  return xgemm::ceil_div(p.M, 64) * xgemm::ceil_div(p.N, 64) <= (int64_t(1) << 27);
}

bool xgemm_launch(const QmmProblem& p, const Launch& l, hipError_t* status) {
  using namespace xgemm;
  Args args;
  TileArgs& a = args.t;
  a.x = reinterpret_cast<const uint16_t*>(p.x);
  a.xs0 = p.xs0;
  a.w = p.w;
  a.ws0 = p.ws0;
  a.s = p.s;
  a.ss0 = p.ss0;
  a.b = p.b;
  a.bs0 = p.bs0;
  a.out = p.out;
  a.epi = p.epi;
  a.M = static_cast<int>(p.M);
  a.N = static_cast<int>(p.N);
  a.K = static_cast<int>(p.K);
  a.group_shift = 0;
  a.split_steps = 0;
  a.partial = nullptr;
  args.groups = static_cast<uint32_t>(p.K / p.group);
  const uint64_t gblocks = static_cast<uint64_t>(p.group / 32);
  args.magic = gblocks == 1 ? 0 : static_cast<uint32_t>(((uint64_t(1) << 32) + gblocks - 1) / gblocks);

  // Shapes and K ranges, measured on MI355X in us over whole calls (4096
  // columns unless said). The eight waves of 32 x 32 on 64 x 128 are ahead
  // while the product is small (f32 100 x 4096 at 8 bits: 28.6 against 31.8
  // with 128 x 256 tiles; groups of 32, 512 x 1376: 25.6 against 30.1 with
  // four waves); then four waves of 64 x 32 (groups of 32, 512 x 4096: 60
  // against 72); with f32 activations the 128 x 256 tile, which decodes half
  // as often, where its K ranges fill the GPU (512 x 14336: 176 against 213).
  // Groups of 32 and the running totals of bf16 activations do not fit that
  // tile's registers.
  const int64_t cus = device_cus();
  const bool g32 = p.group % kBK != 0;
  Shape shape;
  int64_t units = ceil_div(p.K, kBK), parts = 1;
  int splits;
  if (p.M <= 32) {
    shape = p.M <= 16 ? kSkinny16 : kSkinny32;
    parts = kWaves;
    units = ceil_div(p.K * p.bits, 512);
    const int64_t tiles = ceil_div(p.N, kSkinnyCols);
    // A K range more costs a reduction, about as much as three steps of a
    // wave (8-bit f32 8 x 2048 x 1024: 10.9 in one range, 13.5 in two), and
    // pays while the CUs have less than a workgroup each (8 x 14336 x 4096:
    // 20.2 in one, 21.6 in two; 16 x 4096 x 14336: 62 in one, 24 in four).
    const int64_t steps = units * (8 / p.bits);
    splits = 1;
    for (int s = most_splits(p, units, kWaves); s > 1; --s)
      if (tiles * s <= cus && steps / kWaves - steps / (kWaves * s) > 3) {
        splits = s;
        break;
      }
  } else {
    const int most = most_splits(p, units, 4);
    int64_t bm = 64, bn = 128, want = cus;
    if (!g32 && p.x_dtype == AFFON_ROCM_F32 && p.M > 64 && ceil_div(p.M, 128) * ceil_div(p.N, 256) * most >= cus * 3 / 4) {
      shape = kTile128x256;
      bm = 128;
      bn = 256;
    } else if (p.M > 64 && static_cast<double>(p.M) * p.N * p.K >= 0x1p32) {
      shape = kTile64x128;
      want = 2 * cus;  // two of its workgroups fit a CU
    } else {
      shape = kTile64x128Wide;
    }
    splits = static_cast<int>(std::min<int64_t>(most, ceil_div(want, ceil_div(p.M, bm) * ceil_div(p.N, bn))));
  }
  if (splits > 1) {
    // Without scratch (a captured stream whose workspace cannot grow): one
    // range, or the VALU kernel where that fills the GPU better.
    a.partial = static_cast<float*>(l.can_split() ? l.scratch(static_cast<size_t>(splits) * p.M * p.N * 4) : nullptr);
    if (a.partial == nullptr) {
      if (one_range_is_behind(p)) return false;
      splits = 1;
    }
  }
  a.splits = splits;
  args.unit = static_cast<int>(units / (parts * splits));
  args.extra = static_cast<int>(units % (parts * splits));
  switch (p.bits) {
    case 2: *status = launch_b2(args, shape, g32, p.x_dtype, p.p_dtype, l.stream); break;
    case 4: *status = launch_b4(args, shape, g32, p.x_dtype, p.p_dtype, l.stream); break;
    default: *status = launch_b8(args, shape, g32, p.x_dtype, p.p_dtype, l.stream); break;
  }
  return true;
}

}  // namespace affon
