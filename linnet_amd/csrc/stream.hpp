// The few-row product over a stored weight in any of the quantized formats, y = x W^T
// for 1..32 rows of x a workgroup: the weight streamed once from HBM in its own bytes,
// widened in registers and multiplied on MFMA (16x16x32). Used by lnq_int4_linear
// (groups and widths the one-workgroup-per-CU GEMVs do not take), lnq_w8a16,
// lnq_nf4_linear and lnq_mxfp4_experts.
//
// Bound: HBM (the weight's bytes), then the CU's memory pipeline, which also moves x (every
// workgroup reads all the x its rows meet), then VALU issue (widening: about 200
// instructions a wave for 4 KB of int4, 480 for NF4). So
// * a workgroup owns up to 64 output rows (R, 16 a tile) and all of K; its waves split
//   K into contiguous ranges of 128-input steps and keep private copies of everything,
//   so nothing but the scales and the last sum has a barrier;
// * a wave's x of a step (4 to 32 rows x 256 bytes) moves by buffer_load ... lds, 256
//   contiguous bytes a row (an instruction of 16 rows x 64 bytes, the operand order, runs
//   at a third of that rate from L2), its 16-byte chunks XOR-swizzled by row so that the
//   operand reads hit distinct banks;
// * weights go straight to registers, 8 rows x 128 contiguous bytes an instruction, and
//   two DPP moves a dword put them in operand order: read in operand order (16 rows x 64
//   bytes) the two halves of a line came far enough apart to be fetched twice (4096 ->
//   28672, groups of 64, 16 rows: 26.4 us so, 21.5 with whole lines). One unit a tile is
//   in flight, asked for again as soon as it is widened; two units were slower (25.5
//   against 23.7 us there: all of a small layer then lands before the first product);
// * scales and zero points, one run of memory for the workgroup's rows, move to LDS in
//   whole kilobytes ahead of everything else (a load a row and step touches as many lines
//   as the weights do: 14.9 us at 4096 -> 14336, groups of 64, 16 rows, 12.5 without them).
// The inputs a lane's 16 bytes hold are dealt to the step's four MFMAs so that none of
// them spans two groups (GPS groups a step); for groups of 64 and 32 that takes a
// transpose among the four lanes of a row (v_permlane32_swap, v_permlane16_swap). The
// fold is f32 per group: acc += s * (C - (MAGIC + z) * sum x) for int4 (the product with
// the exact (q - z) * s), s * C otherwise.
// Measured (us, graphs over rotating copies, before / now): int4 4096 -> 14336 groups of 64
// at 16 rows 37.6 / 12.2, groups of 32 59.1 / 16.7, group 128 at 16 rows 12.4 / 11.0; 14336
// -> 4096 at 8 rows 15.0 / 12.3.
#pragma once

#include "common.hpp"

namespace lnq {
namespace stream {

// How the scales lie: a column a group within a step, columns of several steps (any
// number of STEP / GPS units), the same with a scale row for `row_block` weight rows.
enum Kind { ONE_STEP = 0, SPAN = 1, BLOCK = 2 };

enum Format { INT4 = 0, NF4 = 1, FP4 = 2, INT8 = 3, FP8 = 4 };

constexpr int STEP = 128;   // inputs of a step
constexpr int WAVES = 8;    // waves of a dense workgroup
constexpr int MAX_R = 64;   // output rows of a workgroup
// An offset past every buffer's range (each spans less than 1 GiB): a row that does not exist.
constexpr uint32_t NO_ROW = 0x40000000u;

constexpr bool eight(int f) { return f == INT8 || f == FP8; }
// Formats whose widened codes are offset (int4 by MAGIC + zero, int8 in bf16 by 128; in
// f16 the offset comes off exactly), which sums of x undo.
constexpr bool needs_xsum(int f, int dt) { return f == INT4 || (f == INT8 && dt == LNQ_BF16); }

// Steps whose x a wave has in flight, a stage each.
constexpr int DEPTH = 2;
// x values of a wave's stage of one step: the 4 xi rows that are moved.
// (the stages hold the waves' sums at the end: 512 values a unit of 16 x 16 outputs).
constexpr int stage_values(int xi, int mt, int nt) {
  const int sums = 512 * ((mt * nt + DEPTH - 1) / DEPTH);
  return 4 * xi * STEP > sums ? 4 * xi * STEP : sums;
}

// NF4's 16 values in x's type as byte planes (see nf4.hip).
struct Planes {
  uint32_t lo[4];
  uint32_t hi[4];
};

struct Args {
  const uint16_t* x;
  const uint8_t* w;
  const void* scale;
  const uint8_t* zero;     // INT4
  const uint16_t* bias;
  uint16_t* y;
  int x_stride, y_stride;  // elements
  int row_bytes;           // bytes of a weight row
  int M, N, K;
  int R;           // output rows of a workgroup (a multiple of 8)
  int span;        // scale columns cover `span` units of STEP / GPS inputs each (SPAN, BLOCK)
  int cols;        // scale columns (groups of a row)
  int row_block;   // weight rows that share a scale row (BLOCK)
  Planes planes;
};

// Places of 8-input chunks: lane quarter j, MFMA t of a step holds chunk (of 16).
template <int F, int GPS>
__device__ inline int chunk_of(int j, int t) {
  if constexpr (eight(F)) return 8 * (t >> 1) + 2 * j + (t & 1);
  else if constexpr (GPS == 4) return 4 * t + j;
  else if constexpr (GPS == 2) return 8 * (t >> 1) + 4 * (j & 1) + 2 * (j >> 1) + (t & 1);
  else return 4 * j + t;
}

__device__ inline void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

__device__ inline void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// 8 consecutive 16-bit values reordered 0,2,4,6,1,3,5,7 (the order of nf4_widen).
__device__ inline u32x4 permute_nf4(u32x4 v) {
  u32x4 out;
  out.x = __builtin_amdgcn_perm(v.y, v.x, 0x05040100u);
  out.y = __builtin_amdgcn_perm(v.w, v.z, 0x05040100u);
  out.z = __builtin_amdgcn_perm(v.y, v.x, 0x07060302u);
  out.w = __builtin_amdgcn_perm(v.w, v.z, 0x07060302u);
  return out;
}

// The values of w's eight NF4 codes as pairs (0,2) (4,6) (1,3) (5,7): v_perm_b32 looks
// four codes' bytes up in the 8-entry halves of a plane, and the code's bit 3, spread to
// a byte mask by a v_perm of the shifted word, picks the half.
__device__ inline u32x4 nf4_widen(uint32_t w, const Planes& p) {
  u32x4 v;
  const uint32_t upper[2] = {__builtin_amdgcn_perm(w << 12, w << 4, 0x090B080Au),
                             __builtin_amdgcn_perm(w << 8, w, 0x090B080Au)};
  const uint32_t sel[2] = {w & 0x07070707u, (w >> 4) & 0x07070707u};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t lo = (upper[h] & __builtin_amdgcn_perm(p.lo[3], p.lo[2], sel[h])) |
                        (~upper[h] & __builtin_amdgcn_perm(p.lo[1], p.lo[0], sel[h]));
    const uint32_t hi = (upper[h] & __builtin_amdgcn_perm(p.hi[3], p.hi[2], sel[h])) |
                        (~upper[h] & __builtin_amdgcn_perm(p.hi[1], p.hi[0], sel[h]));
    v[2 * h] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    v[2 * h + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  }
  return v;
}

// w's eight E2M1 codes in element order (exact).
template <int DT>
__device__ inline u32x4 fp4_widen(uint32_t w) {
  u32x4 v;
  if constexpr (DT == LNQ_BF16) {
    v.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0));
    v.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1));
    v.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2));
    v.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3));
  } else {
    v.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0));
    v.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1));
    v.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2));
    v.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3));
  }
  return v;
}

// Four weight bytes as four 16-bit values (two dwords): exactly, but int8 in bf16 plus
// 128 (0..255 are exact in bf16).
template <int DT, int F>
__device__ inline u32x2 byte_widen(uint32_t w) {
  if constexpr (F == FP8) {
    if constexpr (DT == LNQ_BF16)
      return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false)),
                   __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true))};
    else
      return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false)),
                   __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true))};
  } else {
    const uint32_t u = w ^ 0x80808080u;
    if constexpr (DT == LNQ_F16) {
      // (0x6400 | u) read as f16 is 1024 + u; less 1152 it is the signed byte, exactly.
      const f16x2 off = {static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
      const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - off;
      const f16x2 b = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - off;
      return u32x2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
    } else {
      const float f0 = static_cast<float>(u & 0xffu), f1 = static_cast<float>((u >> 8) & 0xffu);
      const float f2 = static_cast<float>((u >> 16) & 0xffu), f3 = static_cast<float>(u >> 24);
      return u32x2{__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f1), __builtin_bit_cast(uint32_t, f0), 0x07060302u),
                   __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f3), __builtin_bit_cast(uint32_t, f2), 0x07060302u)};
    }
  }
}

// Bytes of a scale entry.
constexpr int scale_bytes(int f) { return f == INT4 ? 2 : f == FP4 ? 1 : 4; }

// LDS bytes the scales (and zero points) of `rows` weight rows take, staged as whole
// 16-byte pieces around them.
inline int scale_lds(int f, bool per_row, bool blocks, int rows, int cols, int row_block) {
  if (per_row) return 0;
  const int srows = blocks ? (rows - 1) / row_block + 2 : rows;
  const int s = (srows * cols * scale_bytes(f) + 16 + 1023) / 1024 * 1024;
  return f == INT4 ? s + (rows * cols + 16 + 1023) / 1024 * 1024 : s;
}

// One workgroup's rows n0 .. n0 + R - 1 against the 16 MT rows of x that `row_of` names
// (row_of(i): the element offset of x row i, or a negative number for none; called for
// rows 0 .. 4 XI - 1), and `put(m, n, v)` for every output (m < 16 MT, n < n_end; m may
// lie past the rows that exist). XI: instructions that move a step's x (4 rows each).
// GPS: groups a step (0: one scale a row). NW: the workgroup's waves, which
// all call it.
template <int NW, int DT, int F, int GPS, int MT, int XI, int NT, int KIND, class RowOf, class Put>
__device__ inline void product(const Args& a, int n0, int n_end, const uint16_t* xbase, uint32_t xbytes, uint16_t* X0, uint16_t* X1,
                               uint8_t* SC, RowOf row_of, Put put) {
  using E = Elem<DT>;
  constexpr bool XS = needs_xsum(F, DT);
  constexpr bool MULTI = KIND != ONE_STEP, BLOCKS = KIND == BLOCK;
  constexpr int US = eight(F) ? 1 : 2;         // steps of a weight unit (128 bytes of a row)
  constexpr int GP = GPS == 0 ? 1 : GPS;       // MFMA chains of a step
  constexpr int TPG = 4 / GP;                  // MFMAs of a chain
  constexpr int D = DEPTH;                     // steps in flight
  constexpr int XW = stage_values(XI, MT, NT);         // x values of a wave's stage

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, j = lane >> 4, r7 = lane & 7;
  const int steps = (a.K + STEP - 1) / STEP;
  const int units = (steps + US - 1) / US;
  const int per = (units + NW - 1) / NW;
  const int u0 = min(units, wave * per), u1 = min(units, u0 + per);
  const int s0 = u0 * US, s1 = min(steps, u1 * US);
  uint16_t* const xw[D] = {X0 + wave * XW, X1 + wave * XW};

  // Per-workgroup buffers: the rows' own bytes, so that offsets stay below 1 GiB.
  const int rows = n_end - n0;
  const uint8_t* wbase = a.w + static_cast<int64_t>(n0) * a.row_bytes;
  const uint32_t wbytes = static_cast<uint32_t>(rows * a.row_bytes);
  // A tile's unit is two loads of 8 rows x 128 contiguous bytes: lane l holds row l % 8 and
  // the 16 bytes l / 16 (l % 16 < 8) or 4 + l / 16 of its line.
  uint32_t woff[NT][2];
#pragma unroll
  for (int T = 0; T < NT; ++T)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 16 * T + 8 * h + r7;
      woff[T][h] = row < rows ? static_cast<uint32_t>(row * a.row_bytes + 16 * (j + 4 * (col >> 3))) : NO_ROW;
    }
  uint32_t xoff[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int row = 4 * i + (lane >> 4);
    const int at = row_of(row);
    xoff[i] = at < 0 ? NO_ROW : static_cast<uint32_t>(at + 8 * ((lane & 15) ^ (row & 7))) * 2u;
  }
  // Formats whose K may end inside a step: the lanes past it in the last step.
  constexpr bool TAIL = F == NF4 || F == FP4;
  const int k_last = a.K - (steps - 1) * STEP;
  const uint32_t tail_even = 8 * ((lane & 15) ^ (lane >> 4)) >= k_last ? NO_ROW : 0u;
  const uint32_t tail_odd = 8 * ((lane & 15) ^ ((lane >> 4) + 4)) >= k_last ? NO_ROW : 0u;

  // The rows' scales and zero points are one run of memory each: moved to LDS once, 1 KB
  // an instruction, from the 16 bytes that hold their start to those that hold their end.
  constexpr int SBYTES = scale_bytes(F);
  const int scale_row0 = BLOCKS ? n0 / a.row_block : n0;
  const int scale_rows = BLOCKS ? (n_end - 1) / a.row_block - scale_row0 + 1 : rows;
  auto stage = [&](const uint8_t* p, uint32_t bytes, uint8_t* to) -> uint32_t {
    const uint32_t mis = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 15u);
    const uint32_t total = (bytes + mis + 15u) & ~15u;
    const __amdgpu_buffer_rsrc_t r = buffer_rsrc(p - mis, total);
    for (uint32_t at = wave * 1024u; at < total; at += NW * 1024u)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)(to + at), 16, at + lane * 16, 0, 0, 0);
    return mis;
  };
  uint32_t sat[NT], zat[NT];  // LDS offset of a tile row's first scale / zero point
  if constexpr (GPS > 0) {
    const uint32_t sbytes = static_cast<uint32_t>(scale_rows * a.cols * SBYTES);
    const uint32_t smis = stage(static_cast<const uint8_t*>(a.scale) + static_cast<int64_t>(scale_row0) * a.cols * SBYTES, sbytes, SC);
    uint32_t zbase = 0;
    if constexpr (F == INT4) {
      zbase = (sbytes + 16u + 1023u) / 1024u * 1024u;
      zbase += stage(a.zero + static_cast<int64_t>(n0) * a.cols, static_cast<uint32_t>(rows * a.cols), SC + zbase);
    }
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      const int n = min(16 * T + col, rows - 1);
      sat[T] = smis + static_cast<uint32_t>((BLOCKS ? (n0 + n) / a.row_block - scale_row0 : n) * a.cols * SBYTES);
      zat[T] = zbase + static_cast<uint32_t>(n * a.cols);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // The step rides in the scalar offset; a step past the wave's end reads through a
  // descriptor of no bytes (at offset 0), which returns zeros and moves nothing.
  u32x4 wr[NT][2];
  auto load_w = [&](int u, int T, u32x4 (&dst)[2]) {
    const bool live = u < u1;
    const __amdgpu_buffer_rsrc_t rw = buffer_rsrc(wbase, live ? wbytes : 0u);
    const int at = live ? u * 128 : 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      dst[h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, woff[T][h], at, 2));
  };
  // The two loads of a tile as operands: lane (col, j) of w[0] then holds row col's first
  // half line (16 bytes j of 4), of w[1] its second. The upper eight lanes of a 16-lane
  // row trade places with the lower eight of the other load (row_ror:8).
  auto deal = [&](u32x4 (&w)[2]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int x = static_cast<int>(w[0][e]), y = static_cast<int>(w[1][e]);
      w[0][e] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, y, 0x128, 0xf, 0xc, false));
      w[1][e] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(y, x, 0x128, 0xf, 0x3, false));
    }
  };
  auto load_x = [&](int s, uint16_t* xb) {
    const bool live = s < s1;
    const __amdgpu_buffer_rsrc_t rx = buffer_rsrc(xbase, live ? xbytes : 0u);
    const int at = live ? s * STEP * 2 : 0;
    const bool last = TAIL && s == steps - 1;
    const uint32_t te = last ? tail_even : 0u, to = last ? tail_odd : 0u;
#pragma unroll
    for (int i = 0; i < XI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(xb + i * 4 * STEP), 16,
                                               TAIL ? xoff[i] | ((i & 1) ? to : te) : xoff[i], at, 0, 0);
  };

  // This lane's chunk of A operand t (row `col` of a 16-row block; rows that are not moved
  // repeat the last, their outputs are dropped).
  constexpr int XR = 4 * XI < 16 ? 4 * XI : 16;
  int xa_at[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) xa_at[t] = min(col, XR - 1) * STEP + 8 * (chunk_of<F, GPS>(j, t) ^ (min(col, XR - 1) & 7));

  f32x4 acc[MT][NT], xsum[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    xsum[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int T = 0; T < NT; ++T) acc[mt][T] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  u32x4 ones;
  ones.x = ones.y = ones.z = ones.w = E::ONE2;
  uint32_t nib_mask = 0x000f000fu, nib_magic = E::MAGIC2;
  hide_in_vgpr(nib_mask);
  hide_in_vgpr(nib_magic);

  // Unit u (its steps' x in stages d0, d0 + 1): a tile at a time, each as its own loads
  // land, and its next unit asked for as soon as it is widened.
  auto compute = [&](int u, int d0, u32x4 (&w)[NT][2]) {
    // The unit's stages have landed: all but the loads issued after theirs, the other
    // stages' and the weights' (loads retire in order; the order of issue is held by the
    // scheduling barriers below). The wait is explicit: the compiler's own tracking of
    // loads into LDS let a read of the second stage pass ahead of its loads.
    wait_vm<(D - US) * XI + 2 * NT>();
    u32x4 xa[US][MT][4];
#pragma unroll
    for (int h = 0; h < US; ++h)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          xa[h][mt][t] = *reinterpret_cast<const u32x4*>(xw[(d0 + h) % D] + mt * 16 * STEP + xa_at[t]);
    // The stages are read before the next loads may write them.
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < US; ++h) load_x(u * US + h + D, xw[(d0 + h) % D]);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 cx[US][MT][GP];
    if constexpr (XS) {
#pragma unroll
      for (int h = 0; h < US; ++h)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int g = 0; g < GP; ++g) {
            if constexpr (GPS > 0) cx[h][mt][g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = g * TPG; t < (g + 1) * TPG; ++t) {
              if constexpr (GPS > 0) cx[h][mt][g] = mfma16x16x32<DT>(xa[h][mt][t], ones, cx[h][mt][g]);
              else xsum[mt] = mfma16x16x32<DT>(xa[h][mt][t], ones, xsum[mt]);
            }
          }
    }
#pragma unroll
    for (int h = 0; h < US; ++h)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if constexpr (F == INT4) xa[h][mt][t] = permute_x8(xa[h][mt][t]);
          if constexpr (F == NF4) xa[h][mt][t] = permute_nf4(xa[h][mt][t]);
        }
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      deal(w[T]);
#pragma unroll
      for (int h = 0; h < US; ++h) {
        const int s = u * US + h;
        u32x4 b[4];
        if constexpr (eight(F)) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const u32x4 q = w[T][t >> 1];
            const u32x2 b0 = byte_widen<DT, F>((t & 1) ? q.z : q.x), b1 = byte_widen<DT, F>((t & 1) ? q.w : q.y);
            b[t] = u32x4{b0.x, b0.y, b1.x, b1.y};
          }
        } else {
          uint32_t q[4] = {w[T][h].x, w[T][h].y, w[T][h].z, w[T][h].w};
          if constexpr (GPS == 2 || GPS == 4) {
            swap32(q[0], q[2]);
            swap32(q[1], q[3]);
          }
          if constexpr (GPS == 4) {
            swap16(q[0], q[1]);
            swap16(q[2], q[3]);
          }
          if constexpr (F == INT4) {
            widen_pair<DT>(q[0], q[1], nib_mask, nib_magic, b[0], b[1]);
            widen_pair<DT>(q[2], q[3], nib_mask, nib_magic, b[2], b[3]);
          } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              if constexpr (F == NF4) b[t] = nf4_widen(q[t], a.planes);
              else b[t] = fp4_widen<DT>(q[t]);
            }
          }
        }
        if constexpr (GPS == 0) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[mt][T] = mfma16x16x32<DT>(xa[h][mt][t], b[t], acc[mt][T]);
        } else {
#pragma unroll
          for (int g = 0; g < GP; ++g) {
            // The group's scale column; past the row (K ends inside the unit, whose x is zero
            // from there on) nothing counts.
            const int c = MULTI ? (s * GP + g) / a.span : s * GP + g;
            const bool in = eight(F) || c < a.cols;
            const int cc = eight(F) ? c : min(c, a.cols - 1);
            float sf = 0.f, off = 128.0f;
            int e = 0;
            if constexpr (F == INT4) {
              const uint32_t v = *reinterpret_cast<const uint16_t*>(SC + sat[T] + 2 * cc);
              sf = E::to_f32(static_cast<uint16_t>(in ? v : 0u));
              off = E::MAGIC_VALUE + static_cast<float>(SC[zat[T] + cc]);
            } else if constexpr (F == FP4) {
              e = static_cast<int>(SC[sat[T] + cc]) - 127;
            } else {
              const uint32_t v = *reinterpret_cast<const uint32_t*>(SC + sat[T] + 4 * cc);
              sf = __builtin_bit_cast(float, in ? v : 0u);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              f32x4 p = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int t = g * TPG; t < (g + 1) * TPG; ++t) p = mfma16x16x32<DT>(xa[h][mt][t], b[t], p);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                if constexpr (F == FP4) acc[mt][T][r] += ldexpf(p[r], e);
                else if constexpr (XS) acc[mt][T][r] = fmaf(sf, fmaf(-off, cx[h][mt][g][r], p[r]), acc[mt][T][r]);
                else acc[mt][T][r] = fmaf(sf, p[r], acc[mt][T][r]);
              }
            }
          }
        }
      }
      load_w(u + 1, T, w[T]);
    }
  };

#pragma unroll
  for (int d = 0; d < D; ++d) load_x(s0 + d, xw[d]);
  __builtin_amdgcn_sched_barrier(0);
  // Every wave's small loads go out before any wave's weights: the CU's memory pipeline
  // serves them in the order they arrive, and the last wave's x would wait behind the
  // first waves' weights (a bare barrier: nothing has to land).
  __asm__ volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int T = 0; T < NT; ++T) {
    load_w(u0, T, wr[T]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (GPS > 0) {
    // The scales, issued before everything else, have landed; again a bare barrier (a fence
    // would wait for the x stages too).
    wait_vm<D * XI + 2 * NT>();
    __asm__ volatile("s_barrier" ::: "memory");
  }
  constexpr int TURN = D / US;  // units until the stages come round
  for (int u = u0; u < u1; u += TURN) {
#pragma unroll
    for (int d = 0; d < TURN; ++d) {
      if (u + d >= u1) break;
      compute(u + d, d * US, wr);
    }
  }

  // The waves' sums through LDS (the x stages: the loads still in flight there are of
  // steps past the end, and must have landed), added in wave order.
  __asm__ volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  // Wave w's sums of unit q (an x block and a tile) are 1 KB; the stages hold a whole
  // number of units each, unit by unit over the stage arrays.
  constexpr int UNITS = MT * NT;
  constexpr int PER_ARRAY = XW * 2 / 1024;  // units of a wave an array holds
  static_assert(PER_ARRAY * D >= UNITS, "the sums fit the stages");
  auto unit = [&](int q, int wv) -> f32x4* {
    uint16_t* const base = q / PER_ARRAY == 0 ? X0 : X1;
    return reinterpret_cast<f32x4*>(base + wv * XW + (q % PER_ARRAY) * 512);
  };
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      f32x4 v = acc[mt][T];
      if constexpr (GPS == 0 && XS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaf(-128.0f, xsum[mt][r], v[r]);
      }
      unit(mt * NT + T, wave)[lane] = v;
    }
  __syncthreads();
  for (int q = wave; q < UNITS; q += NW) {
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int wv = 0; wv < NW; ++wv)
      v += unit(q, wv)[lane];
    const int mt = q / NT, T = q % NT;
    const int n = 16 * T + col;
    if (n < rows) {
      float sf = 1.0f;
      if constexpr (GPS == 0) sf = static_cast<const float*>(a.scale)[n0 + n];
#pragma unroll
      for (int r = 0; r < 4; ++r) put(16 * mt + 4 * j + r, n0 + n, GPS == 0 ? v[r] * sf : v[r]);
    }
  }
}

// The x stages, an LDS array each: the compiler tracks the loads into LDS by variable, so
// a stage's reads wait for that stage's loads alone. They are all of a dense workgroup's LDS
// beside its scales: fitting_rows fills what they leave to the last byte.
#define LNQ_STREAM_STAGES(NW, XI, MT, NT)                                                       \
  __shared__ __attribute__((aligned(16))) uint16_t X0[NW * stream::stage_values(XI, MT, NT)];   \
  __shared__ __attribute__((aligned(16))) uint16_t X1[NW * stream::stage_values(XI, MT, NT)]

// x [M, K] row-major, outputs [M, N]; blocks of R output rows and chunks of 16 MT rows of
// x. The chunks of one block sit 8 workgroups apart, on one XCD (workgroups go to the 8
// XCDs in turn), so the block's weights come from HBM once: grid x = 8 chunks, y = blocks / 8.
template <int DT, int F, int GPS, int MT, int XI, int NT, int KIND>
__global__ __launch_bounds__(64 * WAVES) void dense_kernel(Args a) {
  using E = Elem<DT>;
  LNQ_STREAM_STAGES(WAVES, XI, MT, NT);
  extern __shared__ __attribute__((aligned(16))) uint8_t SC[];
  // Every argument at once (left alone, the loads spread over the start, each waited for).
  __asm__ volatile("" ::"s"(a.x), "s"(a.w), "s"(a.scale), "s"(a.zero), "s"(a.x_stride), "s"(a.row_bytes), "s"(a.M),
                   "s"(a.N), "s"(a.K), "s"(a.R), "s"(a.span), "s"(a.cols), "s"(a.row_block));
  const int block = blockIdx.y * 8 + (blockIdx.x & 7);
  const int m0 = (blockIdx.x >> 3) * 16 * MT;
  if (block * a.R >= a.N) return;
  const int n0 = block * a.R, n_end = min(a.N, n0 + a.R);
  const int live = min(a.M - m0, 16 * MT);
  const uint16_t* x = a.x + static_cast<int64_t>(m0) * a.x_stride;
  const uint32_t xbytes = static_cast<uint32_t>(((live - 1) * a.x_stride + a.K) * 2);
  product<WAVES, DT, F, GPS, MT, XI, NT, KIND>(
      a, n0, n_end, x, xbytes, X0, X1, SC, [&](int i) -> int { return i < live ? i * a.x_stride : -1; },
      [&](int m, int n, float v) {
        if (m < live) {
          if constexpr (F == INT4) {
            // The rounded product plus the bias, rounded again (the reference's order).
            uint16_t out = E::from_f32(v);
            if (a.bias != nullptr) out = E::from_f32(E::to_f32(out) + E::to_f32(a.bias[n]));
            a.y[static_cast<int64_t>(m0 + m) * a.y_stride + n] = out;
          } else {
            if (a.bias != nullptr) v += E::to_f32(a.bias[n]);
            a.y[static_cast<int64_t>(m0 + m) * a.y_stride + n] = E::from_f32(v);
          }
        }
      });
}

// Output rows a workgroup takes: whole rounds of one workgroup a CU, at most 64 rows each
// (14336 rows: 256 workgroups of 56; 28672: 512 of 56; 4096: 256 of 16).
inline int rows_per_block(int N, int most) {
  const int cus = compute_units();
  const int rounds = (N + cus * most - 1) / (cus * most);
  const int r = (N + cus * rounds - 1) / (cus * rounds);
  return ((r + 7) / 8) * 8;
}

constexpr int LDS_BYTES = 160 * 1024;

template <int DT, int F, int GPS, int MT, int XI, int NT, int KIND>
inline void launch_one(const Args& a, int chunks, hipStream_t stream) {
  const int blocks = (a.N + a.R - 1) / a.R;
  const int lds = scale_lds(F, GPS == 0, KIND == BLOCK, a.R, a.cols, a.row_block);
  hipLaunchKernelGGL((dense_kernel<DT, F, GPS, MT, XI, NT, KIND>),
                     dim3(8u * static_cast<unsigned>(chunks), static_cast<unsigned>((blocks + 7) / 8)), dim3(64 * WAVES),
                     static_cast<size_t>(lds), stream, a);
}

// The output rows whose scales fit LDS beside the x stages (0: not even 8).
template <int F, int GPS, int MT, int XI, int KIND>
inline int fitting_rows(const Args& a) {
  int most = MAX_R;
  while (most > 0 && scale_lds(F, GPS == 0, KIND == BLOCK, most, a.cols, a.row_block) +
                             DEPTH * WAVES * stage_values(XI, MT, most <= 16 ? 1 : most <= 32 ? 2 : 4) * 2 > LDS_BYTES)
    most -= 8;
  return most;
}

template <int DT, int F, int GPS, int MT, int XI, int KIND>
inline void launch_nt(Args& a, int chunks, hipStream_t stream) {
  a.R = rows_per_block(a.N, fitting_rows<F, GPS, MT, XI, KIND>(a));
  switch ((a.R + 15) / 16) {
    case 1: launch_one<DT, F, GPS, MT, XI, 1, KIND>(a, chunks, stream); break;
    case 2: launch_one<DT, F, GPS, MT, XI, 2, KIND>(a, chunks, stream); break;
    default: launch_one<DT, F, GPS, MT, XI, 4, KIND>(a, chunks, stream); break;
  }
}

// In up to which the kernel takes any call: 32 rows of x and 64 of the weight stay below
// 1 GiB, and the scales of 8 rows (groups of 32) fit beside the stages of 16 rows of x.
constexpr int MAX_K = 65536;
// Out up to which the grid's y holds the blocks of 8 or more outputs, eight a step.
constexpr int MAX_N = 65535 * 64;

// Whole rounds of workgroups, one a CU, over `rows` > 16 rows of x (32 each, 16 where the scales
// leave no room for more); r: the output rows of a workgroup.
template <int F, int GPS, int KIND>
inline int rounds(const Args& a, int64_t rows, int64_t out_features, int& r) {
  int most = fitting_rows<F, GPS, 2, 8, KIND>(a), x_rows = 32;
  if (most < 16) most = fitting_rows<F, GPS, 1, 4, KIND>(a), x_rows = 16;
  r = rows_per_block(static_cast<int>(out_features), most);
  const int64_t groups = (out_features + r - 1) / r * ((rows + x_rows - 1) / x_rows);
  return static_cast<int>((groups + compute_units() - 1) / compute_units());
}

// Past about 4 MB of x the rows that every workgroup reads leave the L2s: calls of 16 outputs a
// workgroup took 1.1 to 1.5 times the estimate by rounds at 8 MB, 1.3 to 1.7 at 15, 1.9 to 2.1 at 29;
// of r outputs, 16 / r of the excess (14336 -> 14336 2048 rows, 56 a workgroup, 59 MB: 1.3).
inline double x_past_l2(int64_t rows, int64_t in_features, int r) {
  const double mb = static_cast<double>(rows) * in_features * 2e-6;
  return mb > 4 ? 1 + (mb - 4) / 24 * 16 / (r > 16 ? r : 16) : 1.0;
}

// The dense product of M rows (a.R is set here): 4, 8, 16 or 32 rows of x a workgroup, 16
// where the scales of very wide layers leave no room for more.
template <int DT, int F, int GPS, int KIND = ONE_STEP>
inline void launch(Args a, hipStream_t stream) {
  if (a.M <= 4) launch_nt<DT, F, GPS, 1, 1, KIND>(a, 1, stream);
  else if (a.M <= 8) launch_nt<DT, F, GPS, 1, 2, KIND>(a, 1, stream);
  else if (a.M <= 16 || fitting_rows<F, GPS, 2, 8, KIND>(a) < 16) launch_nt<DT, F, GPS, 1, 4, KIND>(a, (a.M + 15) / 16, stream);
  else launch_nt<DT, F, GPS, 2, 8, KIND>(a, (a.M + 31) / 32, stream);
}

}  // namespace stream
}  // namespace lnq
