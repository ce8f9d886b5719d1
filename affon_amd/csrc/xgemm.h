// Matrix-core kernels for the batches the specialised kernels decline: f32
// activations with more than one row, and bf16 activations whose groups or
// K the direct-transfer kernels do not take (groups of 32 at 2 and 8 bits or
// with f32 parameters, K not a multiple of 256). Groups are any multiple of
// 32, K any whole number of groups.
//
// Numerical class "reassociated": the packed codes q are exact integers in
// bf16 MFMA operands and an f32 activation x enters as three bf16 planes,
//   x = x1 + x2 + x3,  x1 = top 16 bits of x, x2 = top 16 bits of x - x1,
// whose 8 + 8 + 8 significant bits hold all 24 of x (truncation, so that no
// finite x overflows; below 2^-110 what of x lies above 2^-133, the smallest
// bf16 value); bf16 activations are one plane. Every product is
// exact in f32, and each run of 64 k (32 where groups are not multiples of
// 64) adds s * sum(x*q) + b * sum(x) in f32, as the VALU decode kernel does
// per 16 bytes of codes: the run's term is formed first and added
// to the output's sum once, and with bf16 activations, whose products carry next
// to no rounding, a sum of kRunSteps steps is then added to its total and the
// codes count from the middle of their range (centred_start). 100 x 4096 x 1376
// at groups of 32, off 64 bits: 7.3e-8 on the VALU kernel, 1.0e-7 in one chain
// with two roundings per run, 8.2e-8 with runs alone, 7.0e-8 with both. f32
// activations: 2.8e-7 before, 2.0e-7 here, most of it the terms' own; the
// small planes accumulate first.
//
// Two kernels:
//   xskinny  up to 32 rows: each wave of a 64-column workgroup walks a K part
//            of its own, no barrier in the loop. Bound by instruction issue
//            (about 300 vector instructions and 30 MFMAs per 64 k of 64
//            columns, most of them splitting f32 activations and widening
//            8-bit codes): f32 16 x 4096 x 14336 at 8 bits 79.7 us on the
//            VALU kernel, 24 here with its reduction.
//   xtile    more rows: activations are split into planes once per workgroup
//            while they move through registers into LDS (two stages, one
//            barrier per step), words are decoded in registers. With f32
//            activations bound by the matrix cores (three MFMAs per product):
//            512 x 4096 x 14336 at 4 bits 4435 -> 180 us (334 TFLOP/s, 1.0
//            PFLOP/s of MFMA); with bf16 by the vector instructions of decode
//            and group scaling: 2048 x 4096 x 4160 8720 -> 146 us (479
//            TFLOP/s), 100 x 4096 x 1376 at groups of 32 408 -> 17 us.
#pragma once

#include "codes.h"
#include "lds_pipeline.h"

namespace affon {
namespace xgemm {

using namespace pipeline;

// The kernel and tile that run a problem.
enum Shape { kSkinny16, kSkinny32, kTile64x128, kTile64x128Wide, kTile128x256 };

struct Args {
  TileArgs t;         // x as bytes of the activation type; group_shift and split_steps unused
  uint32_t groups;    // groups of a row
  // Group of 32-value block i: i itself where magic is 0 (groups of 32), else
  // the high half of i * magic, magic = 2^32 / (blocks per group) rounded up.
  uint32_t magic;
  // K parts (xskinny: waves; xtile: workgroups): part i has units [i * unit +
  // min(i, extra), ..) of the launch's K units, one more in the first `extra`.
  int unit, extra;
  __device__ __forceinline__ uint32_t group_of(uint32_t block) const {
    const uint32_t g = magic == 0 ? block : __umulhi(block, magic);
    return g < groups ? g : groups - 1;
  }
  __device__ __forceinline__ int part_begin(int i) const { return i * unit + (i < extra ? i : extra); }
};

// K steps of 64; the last one may hold 32 values.
__host__ __device__ constexpr int steps_of(int K) { return (K + kBK - 1) / kBK; }

template <typename XT>
constexpr int kPlanes = XT::bytes == 4 ? 3 : 1;

constexpr int kRunSteps = 8;  // a power of two

// bf16 activations: codes count from the middle of their range, c = 2^(BITS-1),
//   s * sum(x*q) + b * sum(x) = s * (sum(x*q) - c * sum(x)) + (b + c*s) * sum(x).
// The bias of a group lies near its least value, so that the two terms on the
// left are each two to three times their sum, and their roundings most of the
// error; on the right the second is small. The products start from
// -c * sum(x) instead of zero, which costs no instruction per output. (With
// f32 activations the chain starts with the small planes, which that start
// would round.)
// The right side overflows sooner (in c * sum(x) and c * s), and an infinite x
// meets its own negative in it. What has overflowed is never finite again, so
// that finite outputs are right; the others are computed again as on the left
// (plain_sum). That is after the loop, for no registers or instructions in it.
template <typename XT>
constexpr bool kCentred = XT::bytes == 2;
template <int BITS>
constexpr float kCentre = static_cast<float>(1 << (BITS - 1));
// What a run's products start from.
template <int BITS>
__device__ __forceinline__ float centred_start(float sum) {
  return -kCentre<BITS> * sum;
}
template <int BITS, typename XT>
__device__ __forceinline__ float centred_bias(float s, float b) {
  return kCentred<XT> ? fmaf(kCentre<BITS>, s, b) : b;
}

// f32 activations at groups of 32 on 32 x 32 products: those round down, which
// the exact products of bf16 activations do not meet, and every step's sum came
// out low (600 x 1024 x 12800 at 2 bits: 3.4e-7 off 64 bits, a mean of 0.83 of
// that; VALU kernel 2.3e-7). Every other step takes -x and is subtracted, so
// that the errors cancel: 1.9e-7. Other groups, a parameter pair per 64 values,
// stay below the VALU kernel's error without (4.3e-7 and 2.5e-7), and the sign
// costs them 1 % (feed-forward of 512 rows).
template <typename XT, bool G32>
constexpr bool kAlternate = XT::bytes == 4 && G32;

// Eight consecutive activations as loaded.
template <typename XT>
struct Raw8 {
  u32x4_t v[XT::bytes == 4 ? 2 : 1];
  __device__ __forceinline__ void load(const uint8_t* p) {
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(v) / 16); ++i) v[i] = reinterpret_cast<const u32x4_t*>(p)[i];
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(v) / 16); ++i) v[i] = u32x4_t{0u, 0u, 0u, 0u};
  }
  // Signs changed (sign 0x80000000) or kept (0), f32.
  __device__ __forceinline__ void flip(uint32_t sign) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[XT::bytes == 4 ? i / 4 : 0][i % 4] ^= sign;
  }
  // f32 values.
  __device__ __forceinline__ float at(int i) const {
    if constexpr (XT::bytes == 4)
      return __uint_as_float(v[i / 4][i % 4]);
    else
      return __uint_as_float(i % 2 ? v[0][i / 2] & 0xffff0000u : v[0][i / 2] << 16);
  }
};

__device__ __forceinline__ float top16(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// High halves of a (low) and b (high).
__device__ __forceinline__ uint32_t high_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// The planes of eight activations, largest first. An infinite value is its
// own first plane and has zeros below (inf - inf would make it a NaN);
// any_inf says that one may be among them.
template <typename XT>
__device__ __forceinline__ void planes8(const Raw8<XT>& raw, bool any_inf, u32x4_t* out) {
  if constexpr (XT::bytes == 2) {
    out[0] = raw.v[0];
  } else {
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = raw.at(i) - top16(raw.at(i));
    if (any_inf) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (fabsf(raw.at(i)) == INFINITY) r[i] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[0][i] = high_halves(raw.at(2 * i), raw.at(2 * i + 1));
      out[1][i] = high_halves(r[2 * i], r[2 * i + 1]);
      out[2][i] = high_halves(r[2 * i] - top16(r[2 * i]), r[2 * i + 1] - top16(r[2 * i + 1]));
    }
  }
}

typedef u32x4_t u32x4_word_t __attribute__((aligned(4)));  // 16 bytes at a word
typedef u32x2_t u32x2_word_t __attribute__((aligned(4)));
typedef u32x4_t u32x4_half_t __attribute__((aligned(2)));  // at a bf16 value

// One parameter, as raw bits.
template <typename PT>
__device__ __forceinline__ uint32_t load_raw(const uint8_t* p) {
  if constexpr (PT::bytes == 2)
    return *reinterpret_cast<const uint16_t*>(p);
  else
    return *reinterpret_cast<const uint32_t*>(p);
}

// A window of kWindow consecutive groups of one column's scales or biases.
// Reading them one group per step fetches a cache line per column, step and
// parameter of which a few bytes are used. Windows advance by kWindow - 1
// groups: a step's two blocks lie in groups at most one apart, so some window
// holds both.
constexpr int kWindow = 8;
template <typename PT>
struct ParamRun {
  static constexpr int kWords = kWindow * PT::bytes / 4;
  using unaligned_t = typename std::conditional<PT::bytes == 2, u32x4_half_t, u32x4_word_t>::type;
  u32x4_t v[kWords / 4];
  // The first group a window from group `first` holds: rows are read inside
  // their bounds, so the last windows of a row start earlier.
  __device__ __forceinline__ static uint32_t start(uint32_t first, uint32_t groups) {
    return groups < kWindow ? 0 : (first < groups - kWindow ? first : groups - kWindow);
  }
  __device__ __forceinline__ void load(const uint8_t* row, uint32_t first, uint32_t groups) {
    if (groups >= kWindow) {
      const uint8_t* p = row + start(first, groups) * PT::bytes;
#pragma unroll
      for (int i = 0; i < kWords / 4; ++i) v[i] = reinterpret_cast<const unaligned_t*>(p)[i];
    } else {
      // A short row: its groups one by one, the last one repeated.
#pragma unroll
      for (int i = 0; i < kWords; ++i) {
        if constexpr (PT::bytes == 2) {
          const uint16_t* e = reinterpret_cast<const uint16_t*>(row);
          const uint32_t lo = e[min(2u * i, groups - 1)], hi = e[min(2u * i + 1, groups - 1)];
          v[i / 4][i % 4] = lo | (hi << 16);
        } else {
          v[i / 4][i % 4] = reinterpret_cast<const uint32_t*>(row)[min(static_cast<uint32_t>(i), groups - 1)];
        }
      }
    }
  }
  __device__ __forceinline__ void store(uint8_t* p) const {
#pragma unroll
    for (int i = 0; i < kWords / 4; ++i) reinterpret_cast<u32x4_t*>(p)[i] = v[i];
  }
};
// Bytes of a window in LDS: 16 more than it holds, so that reads of
// consecutive columns spread over the banks.
template <typename PT>
constexpr int kWindowBytes = kWindow * PT::bytes + 16;

template <typename PT>
__device__ __forceinline__ float param_at(const uint8_t* window, uint32_t index) {
  if constexpr (PT::bytes == 2)
    return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(window)[index]);
  else
    return reinterpret_cast<const float*>(window)[index];
}

// Sum over the 4 (or 8) consecutive lanes that hold one 32-value (64-value) run.
template <bool G32>
__device__ __forceinline__ float run_sum(float v) {
  auto dpp = [](float x, auto ctrl) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v += dpp(v, std::integral_constant<int, 0xb1>{});                       // quad_perm [1,0,3,2]
  v += dpp(v, std::integral_constant<int, 0x4e>{});                       // quad_perm [2,3,0,1]
  if constexpr (!G32) v += dpp(v, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other quad
  return v;
}

template <typename XT>
__device__ __forceinline__ float sum8(const Raw8<XT>& v) {
  return ((v.at(0) + v.at(1)) + (v.at(2) + v.at(3))) + ((v.at(4) + v.at(5)) + (v.at(6) + v.at(7)));
}

// One output's sum over K steps [step, end) as s * sum(x*q) + b * sum(x) per 32
// values, until it is a NaN: one thread to an output, for those that the
// centred form overflows in. 4-bit groups of 32, 16 x 4096 x 1376 and 512 rows:
// 9.4 and 32 us a call of ordinary values, 18 and 44 of NaNs alone, 94 and 446
// where every output is infinite and stays so (VALU kernel 66 and 2090).
template <int BITS, typename XT, typename PT>
__device__ __forceinline__ float plain_sum(const Args& args, int row, int col, int step, int end) {
  const TileArgs& a = args.t;
  const uint8_t* x = reinterpret_cast<const uint8_t*>(a.x) + static_cast<int64_t>(row) * a.xs0 * XT::bytes;
  const uint32_t* w = a.w + static_cast<int64_t>(col) * a.ws0;
  const uint8_t* s = a.s + static_cast<int64_t>(col) * a.ss0 * PT::bytes;
  const uint8_t* b = a.b + static_cast<int64_t>(col) * a.bs0 * PT::bytes;
  const int blocks = min(2 * end, a.K / 32);
  float total = 0.0f;
#pragma unroll 1
  for (int i = 2 * step; i < blocks && total == total; ++i) {
    const uint32_t g = args.group_of(i);
    Raw8<XT> v[4];
    uint32_t word[BITS];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j].load(x + (static_cast<int64_t>(i) * 32 + 8 * j) * XT::bytes);
#pragma unroll
    for (int j = 0; j < BITS; ++j) word[j] = w[static_cast<int64_t>(i) * BITS + j];
    float xq = 0.0f, xs = 0.0f;
#pragma unroll
    for (int e = 0; e < 32; ++e) {
      const uint32_t code = word[e * BITS / 32] >> (e * BITS % 32) & ((1u << BITS) - 1);
      xq = fmaf(v[e / 8].at(e % 8), static_cast<float>(code), xq);
      xs += v[e / 8].at(e % 8);
    }
    total += fmaf(PT::load(s, g), xq, PT::load(b, g) * xs);
  }
  return total;
}

// ---- up to 32 rows ---------------------------------------------------------

constexpr int kSkinnyCols = 64;

// A wave takes its packed words in units of 64 bytes per column (64, 128 or
// 256 k), so that every load instruction reads 16 runs of 64 contiguous bytes.
template <int BITS>
constexpr int kUnit = 512 / BITS;

// Workgroup: 64 weight columns, its four waves on K parts of their own (no
// barrier in the loop). MFMA t (0, 1) of lane quarter h covers 8 k of both
// operands, chunk 4t + h of the step's 8, so that MFMA t holds one 32-value
// block. In that order a wave's activation loads cover whole lines of 16
// rows and go straight into operand layout. Packed words, 64 bytes per
// column and unit, take theirs through the wave's own LDS: as operand
// loads they touch 16 columns, a power of two apart, for 16 bytes each, and
// fight for the same cache sets (8-bit 16 x 4096 x 14336, f32: 32.8 us).
// Everything is loaded one unit or step ahead, without a branch around a load
// that a wait would then have to cover.
template <int BITS, typename XT, typename PT, int RB, bool G32>
__global__ __launch_bounds__(kThreads, 2) void xskinny_kernel(Args args) {
  const TileArgs& a = args.t;
  constexpr int P = kPlanes<XT>;
  constexpr int kRows = 16 * RB;
  constexpr int kBlocks = G32 ? 2 : 1;      // parameter pairs per step
  constexpr int kSub = kUnit<BITS> / kBK;   // steps per unit
  constexpr int kWCol = 64 + 16;            // LDS bytes per column: 16 more than it holds, to spread over the banks
  constexpr int kPBytes = kSkinnyCols * kWindowBytes<PT>;
  constexpr int kWBytes = kSkinnyCols * kWCol;
  // A wave's words and parameter windows, at the end its sums.
  constexpr int kWaveBytes = kWBytes + 2 * kPBytes > 4 * kRows * kSkinnyCols ? kWBytes + 2 * kPBytes
                                                                             : 4 * kRows * kSkinnyCols;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kWaves][kWaveBytes];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r = lane & 15;
  const int h = lane >> 4;
  uint8_t* own = lds[wave];
  uint8_t *own_s = own + kWBytes, *own_b = own_s + kPBytes;

  int tile, split;
  work_unit((a.N + kSkinnyCols - 1) / kSkinnyCols, a.splits, &tile, &split);
  const int n0 = tile * kSkinnyCols;
  const int part = split * kWaves + wave;
  const int u0 = args.part_begin(part), u1 = args.part_begin(part + 1);

  // Words: load i, lane L reads 16 bytes at 16 (L % 4) of the unit's run of
  // column 16i + L/4. Columns past N feed unstored outputs.
  uint32_t w_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w_off[i] = static_cast<uint32_t>(min(n0 + 16 * i + (lane >> 2), a.N - 1)) * static_cast<uint32_t>(a.ws0 * 4) +
               16 * (lane & 3);
  u32x4_t words[4];
  int w_back = 0;  // bytes the lane's runs in `words` were moved back
  auto load_w = [&](int unit) {
    const uint8_t* base = reinterpret_cast<const uint8_t*>(a.w) + static_cast<int64_t>(unit) * 64;
    // A row that ends inside the unit: runs past the end move back to the
    // row's last 16 bytes (their codes meet cleared activations; a run that
    // is half inside is put right below). No branch: the waits for earlier
    // loads count these as still in flight.
    const int left = (a.K - unit * kUnit<BITS>) * BITS / 8;
    const int back = max(0, 16 * (lane & 3) + 16 - left);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      words[i] = *reinterpret_cast<const u32x4_word_t*>(base + static_cast<int64_t>(static_cast<int32_t>(w_off[i]) - back));
    }
    w_back = back;
  };
  // Activations: row 16rb + r, chunk 4t + h. Rows past M repeat row M-1.
  uint32_t x_off[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
    x_off[rb] = (static_cast<uint32_t>(min(16 * rb + r, a.M - 1)) * static_cast<uint32_t>(a.xs0) + 8 * h) * XT::bytes;
  Raw8<XT> xr[RB][2];
  const int last = (a.K + kBK - 1) / kBK - 1;  // K's last step
  auto load_x = [&](int step) {
    // Blocks past the end of K (the last step's second, or a whole step of
    // the last unit) read an earlier one's places and are cleared.
    const int at = min(step, last);
    const bool no_first = kSub > 1 && step > last, no_second = no_first || (G32 && step * kBK + 32 >= a.K);
    const uint8_t* base = reinterpret_cast<const uint8_t*>(a.x) + static_cast<int64_t>(at) * (kBK * XT::bytes);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      xr[rb][0].load(base + x_off[rb]);
      xr[rb][1].load(base + (G32 && no_second ? 0 : 32 * XT::bytes) + x_off[rb]);
      if (no_first) xr[rb][0].clear();
      if (no_second) xr[rb][1].clear();
    }
  };
  // Parameters: lane L holds column L's next window.
  const uint32_t p_col = static_cast<uint32_t>(min(n0 + lane, a.N - 1));
  const uint8_t* s_row = a.s + p_col * static_cast<uint32_t>(a.ss0 * PT::bytes);
  const uint8_t* b_row = a.b + p_col * static_cast<uint32_t>(a.bs0 * PT::bytes);
  ParamRun<PT> s_run, b_run;
  uint32_t next = 0;  // first group of the window in s_run, b_run
  auto load_p = [&](uint32_t first) {
    next = first;
    s_run.load(s_row, first, args.groups);
    b_run.load(b_row, first, args.groups);
  };
  // Orders the wave's LDS writes before its later reads (the LDS itself
  // works in order) and the other way round.
  auto wave_order = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4_t{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  f32x4_t y[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) y[rb][ct] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // bf16: y holds at most kRunSteps steps and moves to its total then.
  constexpr bool kRuns = P == 1;
  f32x4_t total_y[kRuns ? RB : 1][4];
  auto flush = [&] {
    if constexpr (kRuns) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          total_y[rb][ct] += y[rb][ct];
          y[rb][ct] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
  };
  if constexpr (kRuns) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) total_y[rb][ct] = y[rb][ct];
  }
  if (u0 < u1) {
    load_w(u0);
    load_p(args.group_of(2 * u0 * kSub));
    load_x(u0 * kSub);
  }
  uint32_t window = 0, window_end = 0;  // groups in LDS: [window, window_end)
  for (int u = u0; u < u1; ++u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BITS == 2) {  // 32 codes of a 64-code run
        words[i].x = w_back == 8 ? words[i].z : words[i].x;
        words[i].y = w_back == 8 ? words[i].w : words[i].y;
      }
      *reinterpret_cast<u32x4_t*>(&own[(16 * i + (lane >> 2)) * kWCol + 16 * (lane & 3)]) = words[i];
    }
    load_w(min(u + 1, u1 - 1));
    wave_order();
    // Not unrolled: the operands of a whole unit do not fit the registers together.
#pragma unroll 1
    for (int sub = 0; sub < kSub; ++sub) {
      const int step = u * kSub + sub;
      u32x4_t xp[RB][2][P];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float peak = 0.0f;
          if constexpr (P == 3) {
#pragma unroll
            for (int i = 0; i < 8; ++i) peak = fmaxf(peak, fabsf(xr[rb][t].at(i)));
          }
          planes8<XT>(xr[rb][t], peak == INFINITY, xp[rb][t]);
        }
      uint32_t g[kBlocks];
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) g[i] = args.group_of(2 * step + i);
      if (g[kBlocks - 1] >= window_end) {
        wave_order();
        s_run.store(own_s + lane * kWindowBytes<PT>);
        b_run.store(own_b + lane * kWindowBytes<PT>);
        window = ParamRun<PT>::start(next, args.groups);
        window_end = next + kWindow;
        load_p(next + kWindow - 1);
        wave_order();
      }
      load_x(min(step + 1, u1 * kSub - 1));
      // Each block's sum(x), as the product with ones.
      f32x4_t xs[RB][kBlocks];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) {
          xs[rb][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int p = P - 1; p >= 0; --p)
#pragma unroll
            for (int t = G32 ? i : 0; t < (G32 ? i + 1 : 2); ++t)
              xs[rb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xp[rb][t][p]), ones,
                                                                  xs[rb][i], 0, 0, 0);
        }
      f32x4_t start[RB][kBlocks];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            start[rb][i][v] = kCentred<XT> ? centred_start<BITS>(xs[rb][i][v]) : 0.0f;
      // Two column tiles at a time: their product chains are independent.
#pragma unroll
      for (int c0 = 0; c0 < 4; c0 += 2) {
        u32x4_t op[2][2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const uint8_t* col = &own[(16 * (c0 + c) + r) * kWCol + sub * kBK * BITS / 8];
          uint32_t codes[BITS / 2];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const uint8_t* p = col + (32 * t + 8 * h) * BITS / 8;
            if constexpr (BITS == 8) {
              const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p);
              codes[2 * t] = v.x;
              codes[2 * t + 1] = v.y;
            } else if constexpr (BITS == 4) {
              codes[t] = *reinterpret_cast<const uint32_t*>(p);
            } else {
              const uint32_t v = *reinterpret_cast<const uint16_t*>(p);
              codes[0] = t == 0 ? v : codes[0] | (v << 16);
            }
          }
          codes_bf16<BITS, 512>(codes, op[c]);
        }
        f32x4_t term[RB][2];
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) {
          f32x4_t q[RB][2];
#pragma unroll
          for (int p = P - 1; p >= 0; --p)
#pragma unroll
            for (int t = G32 ? i : 0; t < (G32 ? i + 1 : 2); ++t)
#pragma unroll
              for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                  q[rb][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                      __builtin_bit_cast(bf16x8_t, xp[rb][t][p]), __builtin_bit_cast(bf16x8_t, op[c][t]),
                      p == P - 1 && t == (G32 ? i : 0) ? start[rb][i] : q[rb][c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const int at = (16 * (c0 + c) + r) * kWindowBytes<PT>;
            float sv = param_at<PT>(own_s + at, g[i] - window);
            float bv = centred_bias<BITS, XT>(sv, param_at<PT>(own_b + at, g[i] - window));
            if (step * kBK + 32 * i >= a.K) sv = bv = 0.0f;  // past the end of K
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                term[rb][c][v] =
                    fmaf(sv, q[rb][c][v], i == 0 ? bv * xs[rb][i][v] : fmaf(bv, xs[rb][i][v], term[rb][c][v]));
          }
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int c = 0; c < 2; ++c) y[rb][c0 + c] += term[rb][c];
      }
      if constexpr (kRuns) {
        if (((step - u0 * kSub) & (kRunSteps - 1)) == kRunSteps - 1) flush();
      }
    }
    wave_order();
  }

  // Output element v of row block rb and column tile ct is row 16rb + 4h + v,
  // column 16ct + r. The four K parts are added in order, through each wave's
  // own LDS. Column col of row row sits at col ^ (16 * (row/4 % 2)): the two
  // lane quarters of a 32-lane LDS phase write rows four apart, which then
  // land on different banks.
  auto ysum = [&](int w) { return reinterpret_cast<float*>(lds[w]); };
  auto ypos = [](int row, int col) { return row * kSkinnyCols + (col ^ (16 * ((row >> 2) & 1))); };
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if constexpr (kRuns) y[rb][ct][v] += total_y[rb][ct][v];
        ysum(wave)[ypos(16 * rb + 4 * h + v, 16 * ct + r)] = y[rb][ct][v];
      }
  if constexpr (kCentred<XT>) {
    bool overflow = false;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) overflow |= !(fabsf(y[rb][ct][v]) < INFINITY);
    if (__any(overflow)) {
      wave_order();
#pragma unroll 1
      for (int row = 0; row < min(kRows, a.M); ++row) {
        float* sum = &ysum(wave)[ypos(row, lane)];
        if (n0 + lane < a.N && !(fabsf(*sum) < INFINITY))
          *sum = plain_sum<BITS, XT, PT>(args, row, n0 + lane, u0 * kSub, u1 * kSub);
      }
    }
  }
  __syncthreads();
  float* dst = a.splits == 1 ? a.out : a.partial + split * static_cast<int64_t>(a.M) * a.N;
  with_store_kind(a.splits == 1 ? a.epi.kind : kEpiNone, [&](auto kind) {
    constexpr int KIND = decltype(kind)::value;
#pragma unroll
    for (int e = 0; e < kRows * kSkinnyCols / kThreads; ++e) {
      const int o = e * kThreads + tid;
      const int row = o / kSkinnyCols, col = n0 + o % kSkinnyCols;
      if (row < a.M && col < a.N) {
        const int q = ypos(o / kSkinnyCols, o % kSkinnyCols);
        const float v = (ysum(0)[q] + ysum(1)[q]) + (ysum(2)[q] + ysum(3)[q]);
        store_as<KIND>(a.epi, dst + static_cast<int64_t>(row) * a.N + col, col, v);
      }
    }
  });
}

// ---- more rows -------------------------------------------------------------

// Workgroup tile 32*RT*WM rows x 32*CT*WN columns; wave (mi, ni) of WM x WN
// holds RT x CT accumulator tiles of 32 x 32. MFMA kk (0..3) of lane half lh
// covers 8 k: chunk 4lh + kk of the step's 8, or with G32 chunk
// 4(kk/2) + 2lh + kk%2, so that MFMAs 0, 1 hold the first 32-value block and
// 2, 3 the second. Chunk c of activation row r sits in 16-byte slot
// c ^ (r%8) ^ ((r/8)%2) of the row's 128 bytes (conflict-free fragment reads).
template <int BITS, typename XT, typename PT, int WM, int WN, int RT, int CT, bool G32>
__global__ __launch_bounds__(64 * WM * WN, 2) void xtile_kernel(Args args) {
  const TileArgs& a = args.t;
  constexpr int P = kPlanes<XT>;
  constexpr int kTileThreads = 64 * WM * WN;
  constexpr int BM = 32 * RT * WM, BN = 32 * CT * WN;
  constexpr int kPer = BM * 8 / kTileThreads;   // 8-value chunks a thread stages per step
  constexpr int kBlocks = G32 ? 2 : 1;          // parameter pairs per step
  static_assert(BM * 8 % kTileThreads == 0, "whole chunks per thread");
  __shared__ __attribute__((aligned(16))) uint8_t lds_x[2][P][BM * 128];
  __shared__ __attribute__((aligned(16))) float lds_sum[2][kBlocks][BM];
  __shared__ __attribute__((aligned(16))) float lds_start[kCentred<XT> ? 2 : 1][kBlocks][kCentred<XT> ? BM : 1];
  __shared__ __attribute__((aligned(16))) uint8_t lds_p[2][2][BN * kWindowBytes<PT>];  // [window][scale, bias]
  static_assert(kTileThreads >= 2 * BN, "a thread per column and parameter");

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 31;
  const int lh = lane >> 5;
  const int mi = wave / WN, ni = wave % WN;

  const int nb_n = (a.N + BN - 1) / BN;
  int tile, split;
  work_unit(nb_n * ((a.M + BM - 1) / BM), a.splits, &tile, &split);
  const int m0 = (tile / nb_n) * BM;
  const int n0 = (tile % nb_n) * BN;
  const int t0 = args.part_begin(split), t1 = args.part_begin(split + 1);

  auto slot = [](int row, int chunk) { return row * 128 + 16 * (chunk ^ (row & 7) ^ ((row >> 3) & 1)); };
  // Staging: chunk tid % 8 of local rows tid / 8 + i * (threads / 8). Rows
  // past M repeat row M-1 (unstored outputs).
  const int sq = tid & 7, srow = tid >> 3;
  uint32_t x_off[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    x_off[i] = (static_cast<uint32_t>(min(m0 + srow + i * (kTileThreads / 8), a.M - 1)) * static_cast<uint32_t>(a.xs0) +
                8 * sq) * XT::bytes;
  Raw8<XT> xr[kPer];
  auto load_x = [&](int i, int step) {
    const bool half = G32 && step * kBK + 32 >= a.K;  // the missing half of the last step
    const uint32_t back = half && (sq & 4) ? 32 * XT::bytes : 0;
    const uint8_t* base = reinterpret_cast<const uint8_t*>(a.x) + static_cast<int64_t>(step) * (kBK * XT::bytes);
    xr[i].load(base + (x_off[i] - back));
    if (G32 && half && (sq & 4)) xr[i].clear();
  };
  // f32: the second stage holds -x (see kAlternate).
  auto write_x = [&](int i, int stage) {
    if constexpr (kAlternate<XT, G32>) xr[i].flip(stage == 0 ? 0u : 0x80000000u);
    const float part_sum = sum8(xr[i]);
    u32x4_t pl[P];
    planes8<XT>(xr[i], P == 3 && !(fabsf(part_sum) < INFINITY), pl);
    const int row = srow + i * (kTileThreads / 8);
#pragma unroll
    for (int p = 0; p < P; ++p) *reinterpret_cast<u32x4_t*>(&lds_x[stage][p][slot(row, sq)]) = pl[p];
    const float sum = run_sum<G32>(part_sum);
    if ((sq & (G32 ? 3 : 7)) == 0) {
      lds_sum[stage][G32 ? sq >> 2 : 0][row] = sum;
      if constexpr (kCentred<XT>) lds_start[stage][G32 ? sq >> 2 : 0][row] = centred_start<BITS>(sum);
    }
  };

  // Packed words of a step: two runs of 16 codes per column, run j holding
  // MFMAs 2j, 2j+1. Columns past N feed unstored outputs.
  uint32_t w_off[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const uint32_t n = static_cast<uint32_t>(min(n0 + 32 * (CT * ni + ct) + li, a.N - 1));
    w_off[ct] = n * static_cast<uint32_t>(a.ws0 * 4) + (G32 ? 16 : 32) * lh * BITS / 8;
  }
  uint32_t words[CT][2][BITS / 2];
  auto load_w = [&](int step) {
    const bool half = G32 && step * kBK + 32 >= a.K;  // words past the end of K: the first block's again, times zero
    const uint8_t* base = reinterpret_cast<const uint8_t*>(a.w) + static_cast<int64_t>(step) * (kBK * BITS / 8);
    const uint32_t second = G32 ? (half ? 0 : 32 * BITS / 8) : 16 * BITS / 8;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint8_t* p = base + (j == 0 ? 0 : second) + w_off[ct];
        if constexpr (BITS == 8) {
          const u32x4_t v = *reinterpret_cast<const u32x4_word_t*>(p);
#pragma unroll
          for (int i = 0; i < 4; ++i) words[ct][j][i] = v[i];
        } else if constexpr (BITS == 4) {
          const u32x2_t v = *reinterpret_cast<const u32x2_word_t*>(p);
          words[ct][j][0] = v.x;
          words[ct][j][1] = v.y;
        } else {
          words[ct][j][0] = *reinterpret_cast<const uint32_t*>(p);
        }
      }
  };
  // Parameters: the first BN threads hold the next window of one column's
  // scales, the following BN threads its biases.
  const int p_kind = tid >= BN ? 1 : 0;
  const bool p_on = tid < 2 * BN;
  const uint32_t p_col = static_cast<uint32_t>(min(n0 + (p_kind ? tid - BN : tid), a.N - 1));
  const uint8_t* p_row = p_kind ? a.b + p_col * static_cast<uint32_t>(a.bs0 * PT::bytes)
                                : a.s + p_col * static_cast<uint32_t>(a.ss0 * PT::bytes);
  ParamRun<PT> run;
  uint32_t next = 0;  // first group of the window in `run`
  auto load_p = [&](uint32_t first) {
    next = first;
    if (p_on) run.load(p_row, first, args.groups);
  };

  f32x16_t y[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int v = 0; v < 16; ++v) y[rt][ct][v] = 0.0f;
  const f32x16_t zero = {};
  // bf16: y holds at most kRunSteps steps and moves to its total then.
  constexpr bool kRuns = P == 1;
  f32x16_t total_y[kRuns ? RT : 1][kRuns ? CT : 1];
  auto flush = [&] {
    if constexpr (kRuns) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            total_y[rt][ct][v] += y[rt][ct][v];
            y[rt][ct][v] = 0.0f;
          }
    }
  };
  if constexpr (kRuns) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) total_y[rt][ct] = zero;
  }

  if (t0 < t1) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) load_x(i, t0);
    load_w(t0);
    load_p(args.group_of(2 * t0));
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      write_x(i, 0);
      load_x(i, min(t0 + 1, t1 - 1));
    }
  }
  uint32_t window[2] = {0, 0}, window_end = 0;  // first group of each window in LDS; end of the latest
  int latest = 0;
  // Called before the barrier of step t: the windows in LDS then hold its groups.
  auto window_for = [&](int t) {
    if (args.group_of(2 * t + kBlocks - 1) >= window_end) {
      latest ^= 1;
      if (p_on) run.store(&lds_p[latest][p_kind][(p_kind ? tid - BN : tid) * kWindowBytes<PT>]);
      window[latest] = ParamRun<PT>::start(next, args.groups);
      window_end = next + kWindow;
      load_p(next + kWindow - 1);
    }
  };
  if (t0 < t1) window_for(t0);
  for (int t = t0; t < t1; ++t) {
    const int stage = (t - t0) & 1;
    // The stage of this step is written and the other one read to the end.
    // Loads from memory stay in flight across the barrier.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // Words move on at the last block: the registers they leave take the
    // next step's.
    uint32_t now[CT][2][BITS / 2];
    float sv[CT][kBlocks], bv[CT][kBlocks];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < BITS / 2; ++i) now[ct][j][i] = words[ct][j][i];
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        const int col = (32 * (CT * ni + ct) + li) * kWindowBytes<PT>;
        const uint32_t g = args.group_of(2 * t + i) - (latest ? window[1] : window[0]);
        sv[ct][i] = param_at<PT>(&lds_p[latest][0][col], g);
        bv[ct][i] = centred_bias<BITS, XT>(sv[ct][i], param_at<PT>(&lds_p[latest][1][col], g));
        if (i == 1 && t * kBK + 32 >= a.K) sv[ct][i] = bv[ct][i] = 0.0f;  // past the end of K
      }
    }
    load_w(min(t + 1, t1 - 1));
    u32x4_t op[CT][4];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int j = 0; j < 2; ++j) codes_bf16<BITS, 512>(now[ct][j], &op[ct][2 * j]);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int row0 = 32 * (RT * mi + rt);
      constexpr int kPart = 4 / kBlocks;  // MFMAs per block and plane
      f32x16_t term[CT];
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        f32x16_t acc[CT], start = zero;
        if constexpr (kCentred<XT>) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&lds_start[stage][i][row0 + 8 * u + 4 * lh]);
#pragma unroll
            for (int e = 0; e < 4; ++e) start[4 * u + e] = v[e];
          }
        }
#pragma unroll
        for (int p = P - 1; p >= 0; --p)
#pragma unroll
          for (int kk = 0; kk < kPart; ++kk) {
            const int chunk = G32 ? 4 * i + 2 * lh + kk : 4 * lh + kk;
            const bf16x8_t xf = *reinterpret_cast<const bf16x8_t*>(&lds_x[stage][p][slot(row0 + li, chunk)]);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
              acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf, __builtin_bit_cast(bf16x8_t, op[ct][kPart * i + kk]),
                                                                p == P - 1 && kk == 0 ? (kCentred<XT> ? start : zero) : acc[ct], 0, 0, 0);
          }
        // Accumulator element v of lane l: row 8*(v/4) + 4*(l/32) + v%4, column l%32.
        f32x4_t xs[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          xs[u] = *reinterpret_cast<const f32x4_t*>(&lds_sum[stage][i][row0 + 8 * u + 4 * lh]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const float x = xs[v / 4][v % 4];
            term[ct][v] = fmaf(sv[ct][i], acc[ct][v], i == 0 ? bv[ct][i] * x : fmaf(bv[ct][i], x, term[ct][v]));
          }
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          y[rt][ct][v] = kAlternate<XT, G32> ? fmaf(stage == 0 ? 1.0f : -1.0f, term[ct][v], y[rt][ct][v])
                                        : y[rt][ct][v] + term[ct][v];
      __builtin_amdgcn_sched_barrier(0);
      // The next step's activations, a share after each row tile.
#pragma unroll
      for (int c = rt * kPer / RT; c < (rt + 1) * kPer / RT; ++c) {
        write_x(c, stage ^ 1);
        load_x(c, min(t + 2, t1 - 1));
      }
    }
    if constexpr (kRuns) {
      if (((t - t0) & (kRunSteps - 1)) == kRunSteps - 1) flush();
    }
    if (t + 1 < t1) window_for(t + 1);
  }

  // Element v of accumulator tile (rt, ct) is row row_of(rt, v) and column col_of(ct).
  auto row_of = [&](int rt, int v) { return m0 + 32 * (RT * mi + rt) + 8 * (v / 4) + 4 * lh + v % 4; };
  auto col_of = [&](int ct) { return n0 + 32 * (CT * ni + ct) + li; };
  if constexpr (kCentred<XT>) {
    static_assert(RT * CT * 16 <= 32, "a bit per output");
    uint32_t overflow = 0;
#pragma unroll
    for (int i = 0; i < RT * CT * 16; ++i) {
      y[i / 16 / CT][i / 16 % CT][i % 16] += total_y[i / 16 / CT][i / 16 % CT][i % 16];
      overflow |= fabsf(y[i / 16 / CT][i / 16 % CT][i % 16]) < INFINITY ? 0u : 1u << i;
    }
    if (__any(overflow != 0)) {
#pragma unroll 1
      for (int i = 0; i < RT * CT * 16; ++i) {
        const int row = row_of(i / 16 / CT, i % 16), col = col_of(i / 16 % CT);
        if ((overflow >> i & 1) == 0 || row >= a.M || col >= a.N) continue;
        const float sum = plain_sum<BITS, XT, PT>(args, row, col, t0, t1);
#pragma unroll
        for (int j = 0; j < RT * CT * 16; ++j)
          y[j / 16 / CT][j / 16 % CT][j % 16] = j == i ? sum : y[j / 16 / CT][j / 16 % CT][j % 16];
      }
    }
  }

  float* dst = a.splits == 1 ? a.out : a.partial + split * static_cast<int64_t>(a.M) * a.N;
  with_store_kind(a.splits == 1 ? a.epi.kind : kEpiNone, [&](auto kind) {
    constexpr int KIND = decltype(kind)::value;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int col = col_of(ct);
      if (col < a.N) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int row = row_of(rt, v);
            if (row < a.M) store_as<KIND>(a.epi, dst + static_cast<int64_t>(row) * a.N + col, col, y[rt][ct][v]);
          }
      }
    }
  });
}

// ---- launching -------------------------------------------------------------

template <int BITS, typename XT, typename PT, bool G32>
hipError_t launch_typed(const Args& args, Shape shape, hipStream_t stream) {
  const TileArgs& a = args.t;
  auto grid = [&](int bm, int bn) {
    return dim3(static_cast<unsigned>(((a.N + bn - 1) / bn) * ((a.M + bm - 1) / bm) * a.splits));
  };
  switch (shape) {
    case kSkinny16:
      hipLaunchKernelGGL((xskinny_kernel<BITS, XT, PT, 1, G32>), grid(16, kSkinnyCols), dim3(kThreads), 0, stream, args);
      break;
    case kSkinny32:
      hipLaunchKernelGGL((xskinny_kernel<BITS, XT, PT, 2, G32>), grid(32, kSkinnyCols), dim3(kThreads), 0, stream, args);
      break;
    case kTile64x128:
      hipLaunchKernelGGL((xtile_kernel<BITS, XT, PT, 1, 4, 2, 1, G32>), grid(64, 128), dim3(256), 0, stream, args);
      break;
    case kTile64x128Wide:
      hipLaunchKernelGGL((xtile_kernel<BITS, XT, PT, 2, 4, 1, 1, G32>), grid(64, 128), dim3(512), 0, stream, args);
      break;
    default:
      if constexpr (G32 || XT::bytes == 2) {
        return hipErrorInvalidValue;  // never planned
      } else {
        hipLaunchKernelGGL((xtile_kernel<BITS, XT, PT, 2, 4, 2, 2, false>), grid(128, 256), dim3(512), 0, stream, args);
      }
      break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1) return e;
  return launch_reduce(a, stream);
}

template <int BITS>
hipError_t launch(const Args& args, Shape shape, bool g32, int x_dtype, int p_dtype, hipStream_t stream) {
  auto typed = [&](auto x, auto p) {
    using XT = decltype(x);
    using PT = decltype(p);
    return g32 ? launch_typed<BITS, XT, PT, true>(args, shape, stream)
               : launch_typed<BITS, XT, PT, false>(args, shape, stream);
  };
  if (x_dtype == AFFON_ROCM_BF16)
    return p_dtype == AFFON_ROCM_BF16 ? typed(BF16{}, BF16{}) : typed(BF16{}, F32{});
  return p_dtype == AFFON_ROCM_BF16 ? typed(F32{}, BF16{}) : typed(F32{}, F32{});
}

}  // namespace xgemm
}  // namespace affon
