// MXFP4 mixture-of-experts products for a decoding step (std.quant::mxfp4_experts,
// the reference's `mxfp4_experts` Triton kernel, python/linnet/src/linnet/torch/
// kernels.py:94-209): y[r, k, o] = sum_i x[r, k, i] * W[experts[r, k], o, i], the
// weights MXFP4 as gpt-oss checkpoints store them -- blocks [E, Out, G, 16] bytes
// (32 FP4 E2M1 values a block, element 2j in the low nibble of byte j) and scales
// [E, Out, G] E8M0 bytes (2^(s - 127)) -- read once, as they are.
//
// gfx950 converts a byte of two E2M1 values to two bf16 / f16 values in one
// instruction (v_cvt_scalef32_pk_{bf16,f16}_fp4, exact: E2M1 needs two significant
// bits), which then meet the matching pair of x in one v_dot2_f32_{bf16,f16}; a
// block's sum times its scale (v_ldexp_f32, exact) is added to the row's sum in
// f32, as the reference applies the scale after the block's products.
//
// Layout of the work (the pair kernel; calls whose pairs share experts take the grouped
// one, mxfp4_pass): one workgroup per (row, chosen slot) pair and 16 output
// rows of its expert, 4 waves of 4 rows. Lane l owns blocks l, l + 64, ... of
// every row it visits, so its 32 inputs of x per block stay in registers across
// the rows and a wave's weight loads read 64 consecutive blocks (1 KB) of a row.
// All of a wave's loads are issued before any is used, x and the scales first
// (buffer loads: rows past Out, blocks past G and the rows of an out-of-range
// expert read zeros through the range check). A row's sum is the lanes' partial
// sums added across the wave (fixed order).
#include <cmath>

#include "stream.hpp"

namespace lnq {

namespace mx {
constexpr int WAVES = 4;
constexpr int MAX_SLOTS = 4;  // blocks of a lane per row: G <= 256 (In <= 8192)
// Output rows of a wave (gpt-oss's 2880 -> 5760 at one token: 11.3 us with 4,
// 11.9 with 2, 12.4 with 8; 32 tokens: 55, 63, 55 us).
constexpr int ROWS = 4;
}  // namespace mx

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// sum over byte j of w (two E2M1 codes, elements 2j and 2j + 1) of the codes'
// values times x's pair j (packed 16-bit values, element order), plus c.
template <int DT>
__device__ inline float fp4_dot_byte(uint32_t w, int j, uint32_t xpair, float c) {
  if constexpr (DT == LNQ_BF16) {
    bf16x2_t v;
    switch (j) {
      case 0: v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0); break;
      case 1: v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1); break;
      case 2: v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2); break;
      default: v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3); break;
    }
    return __builtin_amdgcn_fdot2_f32_bf16(v, __builtin_bit_cast(bf16x2_t, xpair), c, false);
  } else {
    f16x2_t v;
    switch (j) {
      case 0: v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0); break;
      case 1: v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1); break;
      case 2: v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2); break;
      default: v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3); break;
    }
    return __builtin_amdgcn_fdot2(v, __builtin_bit_cast(f16x2_t, xpair), c, false);
  }
}

template <int DT, int SLOTS>
__global__ __launch_bounds__(64 * mx::WAVES) void mxfp4_experts_kernel(
    const uint16_t* __restrict__ x, int64_t x_row_stride, int64_t x_slot_stride, int chosen,
    const uint8_t* __restrict__ blocks, const uint8_t* __restrict__ scales,
    const int64_t* __restrict__ experts, int num_experts, uint16_t* __restrict__ y, int out_features,
    int groups) {
  using E = Elem<DT>;
  const int pair = blockIdx.x;
  const int r = pair / chosen, k = pair % chosen;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  constexpr int ROWS = mx::ROWS;
  const int o0 = (blockIdx.y * mx::WAVES + wave) * ROWS;
  const int64_t expert = experts[pair];
  // An expert index outside 0 .. E-1 reads nothing (a 0-byte range) and gives
  // zero rows; rows past Out and blocks past G read zeros through the range.
  const bool valid = expert >= 0 && expert < num_experts;
  const size_t expert_blocks = static_cast<size_t>(out_features) * groups;
  const size_t e0 = valid ? static_cast<size_t>(expert) * expert_blocks : 0;
  const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(blocks + e0 * 16, valid ? static_cast<uint32_t>(expert_blocks * 16) : 0);
  const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(scales + e0, valid ? static_cast<uint32_t>(expert_blocks) : 0);
  const uint16_t* xp = x + r * x_row_stride + k * x_slot_stride;

  // x of this lane's blocks first (32 values, 16 dwords in element order, a
  // block), then the scales, then the weights: the memory pipeline serves a CU's
  // loads in the order they arrive, so the small loads issued first land first
  // and the multiply starts as soon as the weights do (one round trip in all).
  u32x4 xv[SLOTS][4];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int g = lane + 64 * s;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      xv[s][q] = g < groups ? *reinterpret_cast<const u32x4*>(xp + g * 32 + 8 * q) : u32x4{0u, 0u, 0u, 0u};
  }
  // Blocks of rows past Out, or past G within a row, land outside the range.
  uint32_t blk[ROWS][SLOTS];
  int sc[ROWS][SLOTS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const int g = lane + 64 * s;
      const int o = o0 + i;
      blk[i][s] = o < out_features && g < groups ? static_cast<uint32_t>(o * groups + g) : 0xffffffffu >> 4;
      sc[i][s] = __builtin_amdgcn_raw_buffer_load_b8(rs, blk[i][s], 0, 0);
    }
  u32x4 w[ROWS][SLOTS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      w[i][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, blk[i][s] * 16, 0, 2 /* non-temporal */));

  float acc[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    acc[i] = 0.0f;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      float part = 0.0f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) part = fp4_dot_byte<DT>(w[i][s][d], j, xv[s][d][j], part);
      acc[i] += ldexpf(part, sc[i][s] - 127);
    }
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const float v = wave_sum(acc[i]);
    const int o = o0 + i;
    if (lane == 0 && o < out_features) y[static_cast<size_t>(pair) * out_features + o] = E::from_f32(v);
  }
}

// Many pairs: the pairs of one expert together, so that its weights are read and widened
// once for all of them (the kernel above reads an expert's bytes again for each of its
// pairs: 32 tokens, top 4 of 32 experts, 2880 -> 5760 took 213 us, four times the bytes'
// time). Workgroup (n block, expert): the pairs that chose the expert, in order, are
// listed in LDS, then the streaming product (stream.hpp) runs over them 4 XI (16 MT) at a
// time, x rows gathered and output rows scattered by pair. One expert more lists the pairs
// whose choice is out of range and clears their rows.
namespace mx {
constexpr int MAX_PAIRS = 2048;  // pairs of a launch (the list's LDS)
constexpr int GROUP_WAVES = 4;
}

struct ExpertArgs {
  stream::Args a;  // w, scale: every expert's; M unused
  const int64_t* experts;
  int num_experts, pairs, chosen, x_row_stride, x_slot_stride;
  uint32_t x_bytes;
};

template <int DT, int MT, int XI>
__global__ __launch_bounds__(64 * mx::GROUP_WAVES, MT == 1 ? 4 : 2) void mxfp4_grouped_kernel(ExpertArgs g) {
  using E = Elem<DT>;
  constexpr int NT = 4, THREADS = 64 * mx::GROUP_WAVES;
  LNQ_STREAM_STAGES(mx::GROUP_WAVES, XI, MT, NT);
  __shared__ uint16_t list[mx::MAX_PAIRS];
  __shared__ int found[mx::GROUP_WAVES];
  extern __shared__ __attribute__((aligned(16))) uint8_t SC[];
  const int e = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int count = 0;
  for (int p0 = 0; p0 < g.pairs; p0 += THREADS) {
    const int p = p0 + threadIdx.x;
    const int64_t id = p < g.pairs ? g.experts[p] : -1;
    const bool known = id >= 0 && id < g.num_experts;
    const bool mine = p < g.pairs && (known ? id == e : e == g.num_experts);
    const uint64_t mask = __ballot(mine);
    if (lane == 0) found[wave] = __popcll(mask);
    __syncthreads();
    int at = count;
#pragma unroll
    for (int w = 0; w < mx::GROUP_WAVES; ++w) {
      if (w < wave) at += found[w];
      count += found[w];
    }
    if (mine) list[at + __popcll(mask & ((uint64_t{1} << lane) - 1))] = static_cast<uint16_t>(p);
    __syncthreads();
  }
  if (count == 0) return;
  stream::Args a = g.a;
  a.w += static_cast<int64_t>(e) * a.N * a.row_bytes;
  a.scale = static_cast<const uint8_t*>(a.scale) + static_cast<int64_t>(e) * a.N * a.cols;
  const int n0 = blockIdx.x * a.R, n_end = min(a.N, n0 + a.R);
  if (e == g.num_experts) {
    const int width = n_end - n0;
    for (int i = threadIdx.x; i < count * width; i += THREADS)
      a.y[static_cast<int64_t>(list[i / width]) * a.N + n0 + i % width] = 0;
    return;
  }
  constexpr int ROWS = MT == 1 ? 4 * XI : 16 * MT;
  for (int m0 = 0; m0 < count; m0 += ROWS) {
    const int live = min(count - m0, ROWS);
    stream::product<mx::GROUP_WAVES, DT, stream::FP4, 4, MT, XI, NT, stream::ONE_STEP>(
        a, n0, n_end, a.x, g.x_bytes, X0, X1, SC,
        [&](int i) -> int {
          if (i >= live) return -1;
          const int p = list[m0 + i], r = p / g.chosen;
          return r * g.x_row_stride + (p - r * g.chosen) * g.x_slot_stride;
        },
        [&](int m, int n, float v) {
          if (m < live) a.y[static_cast<int64_t>(list[m0 + m]) * a.N + n] = E::from_f32(v);
        });
    __syncthreads();  // the stages and scales are read before the next rows' loads
  }
}

template <int DT, int MT, int XI>
static void launch_grouped(const ExpertArgs& g, hipStream_t stream) {
  const int lds = stream::scale_lds(stream::FP4, false, false, g.a.R, g.a.cols, 1);
  hipLaunchKernelGGL((mxfp4_grouped_kernel<DT, MT, XI>),
                     dim3(static_cast<unsigned>((g.a.N + g.a.R - 1) / g.a.R), static_cast<unsigned>(g.num_experts + 1)),
                     dim3(64 * mx::GROUP_WAVES), static_cast<size_t>(lds), stream, g);
}

template <int DT>
static void launch_grouped_dt(const ExpertArgs& g, int pass, hipStream_t stream) {
  if (pass == 8) launch_grouped<DT, 1, 2>(g, stream);
  else if (pass == 16) launch_grouped<DT, 1, 4>(g, stream);
  else launch_grouped<DT, 2, 8>(g, stream);
}

// The pairs of an expert that the grouped kernel multiplies a pass (8, 16 or 32, by the pairs an
// expert has on average), or 0 for a workgroup a pair. Estimates of both in us, for routers that
// spread their choices, fitted to 1 to 1024 tokens of 1 to 8 choices over 4 to 128 experts in eight
// layers from 1024 -> 1024 to 4096 -> 14336. A pair costs its expert's bytes again, from the caches
// past the first, and each wave's lane slots. The grouped kernel costs a pass of an expert its units
// of 256 inputs, whatever the pairs in it, their longest chain first, and the listing in every
// workgroup.
// us, pair / grouped: 2880 -> 5760, 32 experts, top 4: 4 tokens 32.4 / 38.8, 8 59.4 / 54.9, 32 227 / 80,
// 256 1590 / 190; top 1: 16 tokens 32.9 / 43.3; 4096 -> 1536, 128 experts, top 1: 64 tokens 40.2 / 66.0,
// 256 145 / 101; 1024 -> 1024, 32 experts, top 4: 2 tokens 4.6 / 7.6, 16 14.4 / 8.5. Routers that
// send every token to the same experts are not what is estimated: over a narrow layer the pair
// kernel's reads of one expert then come from the caches, and the grouped kernel has few workgroups
// (4096 -> 1536, 128 experts, top 1, 1024 tokens to one expert 366 / 793; of wide layers the grouped
// kernel is ahead there too, 2880 -> 5760, 32 tokens of top 1 to one of 32 experts 55 / 44).
static int mxfp4_pass(int64_t rows, int64_t chosen, int64_t num_experts, int64_t out_features, int64_t in_features) {
  const double pairs = static_cast<double>(rows) * chosen, experts = static_cast<double>(num_experts);
  const int pass = pairs > 12 * experts ? 32 : pairs > 3 * experts ? 16 : 8;
  const double named = experts * (1 - std::pow(1 - std::fmin(1.0, chosen / experts), static_cast<double>(rows)));
  const int64_t groups = in_features / 32, slots = (groups + 63) / 64;
  const double mb = static_cast<double>(out_features) * groups * 17e-6;
  const double pair = 3.5 + mb * (0.05 * pairs + 0.018 * named) +
                      1.74e-3 * pairs * ((out_features + 15) / 16) * slots + 0.33 * slots;
  const double units = 0.5 * ((in_features + 127) / 128);
  const double blocks = static_cast<double>((out_features + stream::MAX_R - 1) / stream::MAX_R) / compute_units();
  const double passes = named + 1.5 * std::fmax(0.0, pairs / pass - 0.5 * named);
  const double grouped = 4.04 + 1.58 * std::ceil(std::ceil(units) / mx::GROUP_WAVES) + blocks * (0.49 * passes * units + 0.19 * (experts + 1));
  return grouped < pair ? pass : 0;
}

}  // namespace lnq

using namespace lnq;

extern "C" {

LNQ_API LnqStatus lnq_mxfp4_experts(const void* x, int64_t x_row_stride, int64_t x_slot_stride,
                                    const uint8_t* blocks, const uint8_t* scales, const int64_t* experts,
                                    void* y, int64_t rows, int64_t chosen, int64_t num_experts,
                                    int64_t out_features, int64_t in_features, int32_t dtype, void* stream) {
  LNQ_REQUIRE(dtype == LNQ_BF16 || dtype == LNQ_F16, "lnq_mxfp4_experts: x is bf16 or f16, not dtype %d", dtype);
  LNQ_REQUIRE(rows >= 0 && chosen >= 0 && num_experts > 0 && out_features >= 0 && in_features >= 0,
              "lnq_mxfp4_experts: negative size");
  LNQ_REQUIRE(in_features % 32 == 0 && in_features <= 32 * 64 * mx::MAX_SLOTS,
              "lnq_mxfp4_experts: in %lld is not a multiple of 32 up to %d", static_cast<long long>(in_features),
              32 * 64 * mx::MAX_SLOTS);
  LNQ_REQUIRE(rows * chosen <= INT32_MAX && out_features * (in_features / 32) * 16 < (int64_t{1} << 32) - 16,
              "lnq_mxfp4_experts: too large (one expert's blocks past 4 GiB)");
  if (rows == 0 || chosen == 0 || out_features == 0) {
    clear_error();
    return LNQ_OK;
  }
  LNQ_REQUIRE((x || in_features == 0) && blocks && scales && experts && y, "lnq_mxfp4_experts: null pointer");
  LNQ_REQUIRE(aligned(x, 16) && aligned(blocks, 16) && x_row_stride % 8 == 0 && x_slot_stride % 8 == 0,
              "lnq_mxfp4_experts: x (with its row and slot strides) and blocks must be 16-byte aligned");
  const int groups = static_cast<int>(in_features / 32);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* xs = static_cast<const uint16_t*>(x);
  auto* ys = static_cast<uint16_t*>(y);
  // x as the range-checked buffers need it: below 1 GiB, rows and slots forward.
  const int64_t x_span = (rows - 1) * x_row_stride + (chosen - 1) * x_slot_stride + in_features;
  const int pass = in_features >= 32 && x_row_stride >= 0 && x_slot_stride >= 0 && x_span < (int64_t{1} << 29) &&
                           num_experts < 65535 && out_features <= (1 << 24) && chosen <= mx::MAX_PAIRS
                       ? mxfp4_pass(rows, chosen, num_experts, out_features, in_features)
                       : 0;
  if (pass) {
    ExpertArgs g{};
    g.a.w = blocks;
    g.a.scale = scales;
    g.a.row_bytes = groups * 16;
    g.a.N = static_cast<int>(out_features);
    g.a.K = static_cast<int>(in_features);
    g.a.R = stream::MAX_R;
    g.a.span = 1;
    g.a.cols = groups;
    g.a.row_block = 1;
    g.num_experts = static_cast<int>(num_experts);
    g.chosen = static_cast<int>(chosen);
    g.x_row_stride = static_cast<int>(x_row_stride);
    g.x_slot_stride = static_cast<int>(x_slot_stride);
    const int64_t part = mx::MAX_PAIRS / chosen;
    for (int64_t r0 = 0; r0 < rows; r0 += part) {
      const int64_t rc = rows - r0 < part ? rows - r0 : part;
      g.a.x = xs + r0 * x_row_stride;
      g.x_bytes = static_cast<uint32_t>(((rc - 1) * x_row_stride + (chosen - 1) * x_slot_stride + in_features) * 2);
      g.a.y = ys + r0 * chosen * out_features;
      g.experts = experts + r0 * chosen;
      g.pairs = static_cast<int>(rc * chosen);
      if (dtype == LNQ_BF16) launch_grouped_dt<LNQ_BF16>(g, pass, s);
      else launch_grouped_dt<LNQ_F16>(g, pass, s);
      const LnqStatus st = launched("mxfp4_grouped");
      if (st != LNQ_OK) return st;
    }
    return LNQ_OK;
  }
  const int slots = (groups + 63) / 64;
  const int per_wg = mx::WAVES * mx::ROWS;
  const dim3 grid(static_cast<unsigned>(rows * chosen), static_cast<unsigned>((out_features + per_wg - 1) / per_wg));
  LNQ_REQUIRE(grid.y <= 65535, "lnq_mxfp4_experts: too many output features");
  const int C = static_cast<int>(chosen), NE = static_cast<int>(num_experts), O = static_cast<int>(out_features);
#define LNQ_MX(DT, S)                                                                                                 \
  hipLaunchKernelGGL((mxfp4_experts_kernel<DT, S>), grid, dim3(64 * mx::WAVES), 0, s, xs, x_row_stride, x_slot_stride, \
                     C, blocks, scales, experts, NE, ys, O, groups)
#define LNQ_MX_S(DT)                 \
  switch (slots) {                   \
    case 0:                          \
    case 1: LNQ_MX(DT, 1); break;    \
    case 2: LNQ_MX(DT, 2); break;    \
    case 3: LNQ_MX(DT, 3); break;    \
    default: LNQ_MX(DT, 4); break;   \
  }
  if (dtype == LNQ_BF16) {
    LNQ_MX_S(LNQ_BF16);
  } else {
    LNQ_MX_S(LNQ_F16);
  }
#undef LNQ_MX_S
#undef LNQ_MX
  return launched("mxfp4_experts");
}

LNQ_API LnqStatus lnq_mxfp4_experts_plan(int64_t rows, int64_t chosen, int64_t num_experts, int64_t out_features,
                                         int64_t in_features, int32_t* pass) {
  LNQ_REQUIRE(pass != nullptr, "lnq_mxfp4_experts_plan: null pointer");
  LNQ_REQUIRE(rows > 0 && chosen > 0 && num_experts > 0 && out_features > 0 && in_features > 0 && in_features % 32 == 0,
              "lnq_mxfp4_experts_plan: bad shape rows=%lld chosen=%lld experts=%lld in=%lld out=%lld",
              static_cast<long long>(rows), static_cast<long long>(chosen), static_cast<long long>(num_experts),
              static_cast<long long>(in_features), static_cast<long long>(out_features));
  *pass = mxfp4_pass(rows, chosen, num_experts, out_features, in_features);
  clear_error();
  return LNQ_OK;
}

}  // extern "C"
