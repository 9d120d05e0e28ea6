// The 8-bit x 8-bit product in small tiles, for calls whose 256-row tiles would leave the
// chip idle: 33 to a few hundred rows, or narrow outputs (128 rows, 4096 -> 14336: 112 tiles
// of 256 x 128, each half empty).
//
// A workgroup owns BM rows by 64 columns; its waves own 32 x 32 MFMA tiles (FA each). 128
// input bytes a step: both operands move HBM / L2 -> LDS (buffer_load ... lds, 8 rows x 128
// contiguous bytes an instruction) into one of S stages, S - 1 steps ahead, one barrier a
// step. Two or more workgroups share a CU: one's products cover another's waits. Bound
// where the chip is full: the LDS reads plus the MFMAs of a step (with the loads taken out a
// step costs the same sum, one workgroup or two), which is what a larger tile does less of
// and why the 256-row forms stay where they fill the chip. Reading the next depth's
// operands during this one's MFMAs was tried: 5 to 10 percent slower. The MFMAs are
// mm8_kernel's (eight_bit.hpp) in the same k order, so the result has its bits; BLK is its
// block-scaled form (a partial tile a step, folded with x_scale[step, m] * scale[n / 128,
// step]).
//
// Whole calls, rounding of the rows included, us, 256-row tiles -> these, int8 / FP8 /
// block-scaled FP8:
//    48 rows,  4096 -> 14336   28.2 -> 16.8    28.0 -> 16.9    32.7 -> 16.0
//   128 rows,  4096 -> 14336   33.2 -> 24.5    29.4 -> 20.5    37.2 -> 21.9
//   256 rows,  4096 -> 14336   35.0 -> 28.4    33.6 -> 28.6    45.0 -> 31.8
//   128 rows, 14336 ->  4096   82.6 -> 36.4    69.8 -> 36.9   125.7 -> 43.9
//   256 rows, 14336 ->  4096  106.3 -> 48.2   100.8 -> 50.0   133.4 -> 50.7
//   512 rows, 14336 ->  4096   80.8 -> 56.3    79.0 -> 56.3   132.0 -> 68.4
//   128 rows,  2048 ->  2048   19.7 ->  9.7    19.3 ->  9.7    20.1 ->  9.2
#include <algorithm>
#include <cmath>

#include "eight_bit.hpp"

namespace lnq {

namespace mm8s {
constexpr int BK = 128;

template <int BM, int BN>
struct Tile {
  static constexpr int WAVES = BM * BN <= 2048 ? 2 : 4;
  static constexpr int WN = 2;  // waves along the columns
  static constexpr int WM = WAVES / WN;
  static constexpr int FA = BM / 32 / WM, FB = BN / 32 / WN;
  static constexpr int STAGES = BM == 128 ? 3 : 4;  // two workgroups' worth fits a CU
  static constexpr int LA = BM / 8 / WAVES, LB = BN / 8 / WAVES;  // loads of a wave a step
};
}  // namespace mm8s

template <int DT, int FP8, int BM, int BN, bool BLK>
__global__ __launch_bounds__((64 * mm8s::Tile<BM, BN>::WAVES), 2) void mm8_small_kernel(
    const uint8_t* __restrict__ qx, const uint8_t* __restrict__ weight, const float* __restrict__ x_scale,
    const float* __restrict__ scale, uint16_t* __restrict__ y, int M, int N, int K, int xs_stride) {
  using namespace mm8s;
  using E = Elem<DT>;
  using T = Tile<BM, BN>;
  static_assert(!BLK || FP8, "block scales: FP8");
  constexpr int FA = T::FA, FB = T::FB, S = T::STAGES, LA = T::LA, LB = T::LB, NW = T::WAVES;
  constexpr int KPM = FP8 ? 64 : 32;  // inputs per MFMA
  constexpr int KK = BK / KPM;
  constexpr int CPL = KPM / 32;  // 16-byte columns of an operand per lane
  using Op = typename std::conditional<FP8, i32x8, i32x4>::type;
  using Acc = typename std::conditional<FP8, f32x16, i32x16>::type;
  // A stage array each (the compiler tracks loads into LDS by variable).
  constexpr int OPERANDS = (BM + BN) * BK;
  constexpr int STAGE = OPERANDS + (BLK ? NW * 512 : 0);  // then each wave's scales
  __shared__ __attribute__((aligned(16))) uint8_t S0[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t S1[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t S2[S > 2 ? STAGE : 16];
  __shared__ __attribute__((aligned(16))) uint8_t S3[S > 3 ? STAGE : 16];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  mm8_tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
  if (tm >= tiles_m || tn >= tiles_n) return;
  const int m0 = tm * BM, n0 = tn * BN;
  const int steps = K / BK;

  // Rows past M (N) read zeros through the range checks (the row offset is in the lane
  // offset); a step past the end reads through a descriptor of no bytes at offset 0.
  const uint32_t a_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(K);
  const uint32_t b_bytes = static_cast<uint32_t>(N) * static_cast<uint32_t>(K);
  // Load i of this wave: rows 8 (wave + NW i) .. + 7, lane l row l / 8, stored column l % 8
  // holding source column (l % 8) ^ key(row), key = bits 1..3 of the row (the same for
  // every i: NW is even).
  const int lrow8 = 8 * wave + (lane >> 3);
  const int lcol = (lane & 7) ^ ((lrow8 >> 1) & 7);
  const uint32_t aoff_g = static_cast<uint32_t>(m0 + lrow8) * K + lcol * 16;
  const uint32_t boff_g = static_cast<uint32_t>(n0 + lrow8) * K + lcol * 16;
  auto load = [&](int ks, uint8_t* st) {
    const bool in = ks < steps;
    const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(qx, in ? a_bytes : 0u), rb = buffer_rsrc(weight, in ? b_bytes : 0u);
    const int k0 = in ? ks * BK : 0;
#pragma unroll
    for (int i = 0; i < LA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)(st + (wave + NW * i) * 1024), 16,
                                               aoff_g + static_cast<uint32_t>(8 * NW * i) * K, k0, 0, 0);
#pragma unroll
    for (int i = 0; i < LB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)(st + BM * BK + (wave + NW * i) * 1024), 16,
                                               boff_g + static_cast<uint32_t>(8 * NW * i) * K, k0, 0, 0);
  };

  Acc acc[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0;

  const int lrow = lane & 31, lk = lane >> 5;
  uint32_t aoff[KK][CPL], boff[KK][CPL];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int c16 = kk * 2 * CPL + lk * CPL + j;
      const uint32_t col = static_cast<uint32_t>((c16 ^ ((lrow >> 1) & 7)) << 4);
      aoff[kk][j] = static_cast<uint32_t>((wm * FA * 32 + lrow) * BK) + col;
      boff[kk][j] = static_cast<uint32_t>(BM * BK + (wn * FB * 32 + lrow) * BK) + col;
    }
  // The block form's scales of a step ride with its operands, by loads into LDS of the wave's
  // own: its rows' (lane l row l of the wave's; rows past M read row M - 1) and, in every
  // lane, that of its columns' block. (Loads into registers, which nothing ties to their
  // place, were moved past the operands' and broke the count that a step waits by. Products
  // alone, us, so -> now: 256 rows 8192 -> 28672 71 -> 61, 128 rows 45.4 -> 44.5, 4096 -> 14336
  // 16.8 both; 2048 -> 2048 5.9 -> 6.5, two more LDS loads and reads in each short step.)
  const uint32_t sx_off = static_cast<uint32_t>(min(m0 + wm * FA * 32 + lane, M - 1)) * 4u;
  const uint32_t sw_off = static_cast<uint32_t>((n0 + wn * FB * 32) / 128) * static_cast<uint32_t>(steps) * 4u;
  const uint32_t sx_bytes = static_cast<uint32_t>(M) * 4u;
  const uint32_t sw_bytes = static_cast<uint32_t>((N + 127) / 128) * static_cast<uint32_t>(steps) * 4u;
  auto load_scales = [&](int ks, uint8_t* st) {
    if constexpr (BLK) {
      const bool in = ks < steps;
      const int k = in ? ks : 0;
      uint8_t* const to = st + OPERANDS + wave * 512;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          buffer_rsrc(x_scale + static_cast<size_t>(k) * xs_stride, in ? sx_bytes : 0u), (lds_ptr)to, 4, sx_off, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer_rsrc(scale, in ? sw_bytes : 0u), (lds_ptr)(to + 256), 4, sw_off,
                                               k * 4, 0, 0);
    }
  };
  constexpr int LOADS = LA + LB + (BLK ? 2 : 0);  // of a wave a step

  auto step = [&](int ks, const uint8_t* st, uint8_t* next) {
    // This wave's loads of step ks have landed (those of the S - 2 steps after it may be in
    // flight); past the barrier every wave's have, and every wave is done with step
    // ks - 1's stage, which step ks + S - 1 fills.
    wait_vm<(S - 2) * LOADS>();
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    load(ks + S - 1, next);
    load_scales(ks + S - 1, next);
    __builtin_amdgcn_sched_barrier(0);
    Acc part[BLK ? FA : 1][BLK ? FB : 1];
    float sx[FA], sw = 0.f;
    if constexpr (BLK) {
      const float* const from = reinterpret_cast<const float*>(st + OPERANDS + wave * 512);
      sw = from[64];
#pragma unroll
      for (int a = 0; a < FA; ++a) sx[a] = from[32 * a + lrow];
    }
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      Op af[FA], bf[FB];
      auto fetch = [&](Op& o, uint32_t const (&off)[CPL], int f) {
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(st + off[j] + f * 32 * BK);
          if constexpr (FP8) {
            o[4 * j + 0] = (int)v.x;
            o[4 * j + 1] = (int)v.y;
            o[4 * j + 2] = (int)v.z;
            o[4 * j + 3] = (int)v.w;
          } else {
            o = __builtin_bit_cast(i32x4, v);
          }
        }
      };
#pragma unroll
      for (int a = 0; a < FA; ++a) fetch(af[a], aoff[kk], a);
#pragma unroll
      for (int b = 0; b < FB; ++b) fetch(bf[b], boff[kk], b);
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          auto mma = [&](Acc c) -> Acc {
            if constexpr (FP8)
              return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[b], af[a], c, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
            else
              return __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[b], af[a], c, 0, 0, 0);
          };
          if constexpr (BLK) part[a][b] = mma(kk == 0 ? Acc{} : part[a][b]);
          else acc[a][b] = mma(acc[a][b]);
        }
    }
    if constexpr (BLK) {
#pragma unroll
      for (int a = 0; a < FA; ++a) {
        const float f = sx[a] * sw;
#pragma unroll
        for (int b = 0; b < FB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[a][b][r] = fmaf(part[a][b][r], f, acc[a][b][r]);
      }
    }
  };

  uint8_t* const st[4] = {S0, S1, S2, S3};
#pragma unroll
  for (int j = 0; j < S - 1; ++j) {
    load(j, st[j]);
    load_scales(j, st[j]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int ks = 0; ks < steps; ks += S) {
#pragma unroll
    for (int j = 0; j < S; ++j) {
      if (ks + j >= steps) break;
      step(ks + j, st[j], st[(j + S - 1) % S]);
    }
  }
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Lane l, register r of a tile: row m = l % 32, output feature 8 (r / 4) + 4 (l / 32) +
  // r % 4 (the weight is the MFMA's A operand).
  const bool vec_out = (N & 3) == 0;
#pragma unroll
  for (int a = 0; a < FA; ++a) {
    const int m = m0 + (wm * FA + a) * 32 + lrow;
    if (m >= M) continue;
    const float xs = BLK ? 1.0f : x_scale[m];
    uint16_t* yrow = y + static_cast<size_t>(m) * N;
#pragma unroll
    for (int b = 0; b < FB; ++b) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int n = n0 + (wn * FB + b) * 32 + 8 * q4 + 4 * lk;
        uint16_t out[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float ws = BLK ? 1.0f : (n + i < N ? scale[n + i] : 0.f);
          out[i] = E::from_f32(static_cast<float>(acc[a][b][4 * q4 + i]) * xs * ws);
        }
        if (vec_out && n + 3 < N) {
          *reinterpret_cast<u32x2*>(yrow + n) =
              u32x2{static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16),
                    static_cast<uint32_t>(out[2]) | (static_cast<uint32_t>(out[3]) << 16)};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) yrow[n + i] = out[i];
        }
      }
    }
  }
}

template <int DT, int FP8, int BM, int BN, bool BLK>
static LnqStatus launch(const uint8_t* qx, const uint8_t* weight, const float* x_scale, const float* scale, void* y,
                        int M, int N, int K, int xs_stride, hipStream_t s) {
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  hipLaunchKernelGGL((mm8_small_kernel<DT, FP8, BM, BN, BLK>), dim3(tiles), dim3(64 * mm8s::Tile<BM, BN>::WAVES), 0, s,
                     qx, weight, x_scale, scale, static_cast<uint16_t*>(y), M, N, K, xs_stride);
  return launched("mm8_small");
}

template <int DT, int FP8, bool BLK>
static LnqStatus launch_tile(int bm, const uint8_t* qx, const uint8_t* weight, const float* x_scale,
                             const float* scale, void* y, int M, int N, int K, int xs_stride, hipStream_t s) {
  if (bm == 32) return launch<DT, FP8, 32, 64, BLK>(qx, weight, x_scale, scale, y, M, N, K, xs_stride, s);
  if (bm == 64) return launch<DT, FP8, 64, 64, BLK>(qx, weight, x_scale, scale, y, M, N, K, xs_stride, s);
  return launch<DT, FP8, 128, 64, BLK>(qx, weight, x_scale, scale, y, M, N, K, xs_stride, s);
}

// Rows of the tile to take, or 0 for the 256 x 128 tiles: the least of estimates in us, fitted to
// the fastest of the four at 16 to 1500 rows of 35 layers from 1024 -> 1024 to 8192 -> 28672, with the
// weights in memory and in the last-level cache alike (in the mean 0.8 and 0.5 percent off the
// fastest). A large tile costs its steps a round, or the weights' own time from memory (4.87 bytes a
// picosecond). A small tile's step costs its latency or, where several workgroups share a CU, their
// work in turn; a partial second round costs 0.55 of a whole one, further ones all of it. Small tiles
// have to win by 3 percent. us large / 32 / 64 / 128 rows, weights from memory: int8 48 rows 4096 ->
// 14336 27.7 / 18.8 / 17.6 / 20.4, 160 rows 6144 -> 12288 45.1 / 53.8 / 44.8 / 37.0, 777 rows 1024 ->
// 4096 16.7 / 16.4 / 13.9 / 12.1; block-scaled 300 rows 8192 -> 28672 115 / 199 / 154 / 137, 128 rows
// 4096 -> 14336 29.3 / 33.2 / 25.0 / 22.6 (from the cache 28.2 / 26.1 / 17.5 / 19.8). Between 16384 and
// 28672 outputs one row of tiles reads every weight once, and the large tiles have them from memory the
// faster (block-scaled 128 rows 5120 -> 25600 42.0 / 69.4 / 60.0 / 51.5, from the cache 36.7 / 50.0 / 41.4 / 35.8).
int mm8_small_rows(int M, int N, int K, bool blk) {
  const double cus = compute_units(), steps = K / 128;
  const double memory = static_cast<double>(N) * K / 4.87e6;
  const double rounds = std::ceil(std::ceil(M / 256.0) * std::ceil(N / 128.0) / cus);
  double best = 0.97 * ((blk ? 2.96 : 3.77) + std::max(steps * rounds * (blk ? 0.84 : 0.83), 1.16 * memory));
  int rows = 0;
  struct Kind { int bm; double base, latency, work; };
  static constexpr Kind plain[] = {{32, 0.1, 0.21, 0.2}, {64, 0.1, 0.28, 0.27}, {128, 1.56, 0.47, 0.36}};
  static constexpr Kind block[] = {{32, 0.1, 0.24, 0.22}, {64, 0.1, 0.32, 0.3}, {128, 1.56, 0.64, 0.36}};
  for (const Kind& k : blk ? block : plain) {
    double c = std::ceil(static_cast<double>(M) / k.bm) * std::ceil(N / 64.0) / cus;
    if (c > 2) c = std::ceil(c);
    else if (c > 1) c += 0.55 * (2 - c);
    const double t = k.base + steps * std::max(k.latency, c * k.work);
    if (t < best) best = t, rows = k.bm;
  }
  return rows;
}

LnqStatus launch_mm8_small(int bm, const uint8_t* qx, const uint8_t* weight, const float* x_scale,
                           const float* scale, void* y, int M, int N, int K, int fp8, int dtype, hipStream_t s) {
  if (dtype == LNQ_BF16)
    return fp8 ? launch_tile<LNQ_BF16, 1, false>(bm, qx, weight, x_scale, scale, y, M, N, K, 0, s)
               : launch_tile<LNQ_BF16, 0, false>(bm, qx, weight, x_scale, scale, y, M, N, K, 0, s);
  return fp8 ? launch_tile<LNQ_F16, 1, false>(bm, qx, weight, x_scale, scale, y, M, N, K, 0, s)
             : launch_tile<LNQ_F16, 0, false>(bm, qx, weight, x_scale, scale, y, M, N, K, 0, s);
}

LnqStatus launch_mm8_block_small(int bm, const uint8_t* qx, const uint8_t* weight, const float* x_scale,
                                 int xs_stride, const float* scale, void* y, int M, int N, int K, int dtype,
                                 hipStream_t s) {
  return dtype == LNQ_BF16 ? launch_tile<LNQ_BF16, 1, true>(bm, qx, weight, x_scale, scale, y, M, N, K, xs_stride, s)
                           : launch_tile<LNQ_F16, 1, true>(bm, qx, weight, x_scale, scale, y, M, N, K, xs_stride, s);
}

}  // namespace lnq
