// The int4 dequant-GEMM above 64 rows where 64 x 128 tiles give no CU a second one: there the
// prefill kernels' tiles (int4_gemm.hip) leave CUs idle and hold one wave a SIMD.
//
// A workgroup of 8 waves, two a SIMD, owns 64 rows of x by 128 columns of W and walks K 256
// inputs a step. Wave (cw, kw) owns 64 of the columns and 64 of a step's inputs: with K split
// over four waves a small product has four times the waves, no column is dequantized twice in
// a workgroup, and an x operand read from LDS feeds two MFMAs. The four partial tiles are
// added through LDS at the end (f32, kw ascending).
//   * x and packed W: HBM / L2 -> LDS by buffer_load ... lds (8 rows x 128 contiguous bytes an
//     instruction) into a ring of three 48 KB stages, two steps ahead, 16-byte columns
//     XOR-swizzled by bits 1..3 of the row. W through LDS because a load that takes 16 bytes
//     of 64 different columns costs about 64 clocks: with W, scales and zero points loaded
//     that way a step took 1.9 us.
//   * scales and zero points: a column a lane, 8 groups at once where rows allow (see Scales).
//   * a lane holds column l % 32 of a 32-column block, half h = l / 32 inputs 32 h .. + 31 of
//     the wave's 64, dequantized as the prefill kernels do ((q - z) * s in f32, exact, one
//     rounding) into the MFMA's A operand; MFMA kk sums input blocks kk and kk + 4 of 8.
//   * one barrier a step.
// Bound: a step takes 1.0 us (1.3 with every CU at it); its loads alone take 0.6 and its
// dequantization and MFMAs alone 0.85 (in their order of dependence, without the halves
// pinned behind the MFMAs, 5 percent more in all).
//
// bf16, group 128, us, prefill kernels -> this (matrix-core or memory floor):
//   200 rows  4096 -> 6144    36.1 -> 22.9  (6.8)     96 rows  2048 -> 2048   18.4 -> 12.8
//   128 rows  4096 -> 14336   37.2 -> 23.8  (10.1)   512 rows  2048 -> 2048   20.1 -> 13.9
//   200 rows 14336 -> 4096   122.9 -> 59.1  (15.8)   512 rows 14336 -> 4096  152.0 -> 79.2
// group 64, 200 rows 8192 -> 8192: 84.3 -> 53.6; group 32, 200 rows 4096 -> 4096: 40.1 -> 30.5.
#include "common.hpp"
#include "stream.hpp"

namespace lnq {

namespace mid {
constexpr int BM = 64, BN = 128, CHUNK = 64, KW = 4, STEP = CHUNK * KW, WAVES = 8, THREADS = 64 * WAVES;
constexpr int S = 3;                     // stages
constexpr int XPART = BM * STEP * 2;     // bytes of a stage: x,
constexpr int STAGE = XPART + BN * 128;  // then the packed weights (128 bytes of a column)
constexpr int LOADS = XPART / 1024 / WAVES + BN * 128 / 1024 / WAVES;  // of a wave a step
constexpr int U = 4;                     // scale register sets
}  // namespace mid

template <int DT>
__device__ inline f32x16 mid_mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (DT == LNQ_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// SC, how a lane gets the scales and zero points of its column (lane l: column l of the wave's
// 64; a swap of the wave's halves hands out the two blocks): 8 groups of 128 at once, one for
// four steps (In % 1024 == 0); one a step (groups of 64 and more); two a step (groups of 32).
// NF4 (lnq_nf4_linear): the codes' values in x's type are the MFMA operand, x the other, so a
// lane holds one column of the product; each 64 inputs' partial tile (a block is 64 or more)
// is folded in f32 with the column's absmax.
enum class Scales { BLOCK, ONE, TWO, NF4 };

struct MidArgs {
  const uint16_t* x;
  const uint8_t* packed;
  const void* scale;  // x's type; NF4: f32 absmax
  const uint8_t* zero;
  const uint16_t* bias;
  uint16_t* y;
  int M, N, K, gshift, x_stride, y_stride;
  stream::Planes planes;
};

template <int DT, Scales SC>
__global__ __launch_bounds__(mid::THREADS, 2) void int4_mid_kernel(MidArgs args) {
  const uint16_t* const x = args.x;
  const uint8_t* const packed = args.packed;
  const uint16_t* const bias = args.bias;
  uint16_t* const y = args.y;
  const int M = args.M, N = args.N, K = args.K, gshift = args.gshift;
  constexpr bool NF = SC == Scales::NF4;
  using namespace mid;
  using E = Elem<DT>;
  constexpr int FA = BM / 32, FB = 2;
  // A stage array each (the compiler tracks loads into LDS by variable).
  __shared__ __attribute__((aligned(16))) uint8_t S0[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t S1[STAGE];
  __shared__ __attribute__((aligned(16))) uint8_t S2[STAGE];
  uint8_t* const st[3] = {S0, S1, S2};

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave & 1, kw = wave >> 1;
  const int lcol = lane & 31, h = lane >> 5;
  const int tiles_m = (M + BM - 1) / BM;
  // Row tiles of one column tile are neighbours on one XCD (workgroup b runs on XCD b % 8).
  const int tiles = tiles_m * ((N + BN - 1) / BN);
  const int per = tiles / 8, more = tiles % 8, xcd = blockIdx.x % 8;
  const int tile = xcd * per + min(xcd, more) + blockIdx.x / 8;
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
  const int groups = K >> gshift;
  const int steps = (K + STEP - 1) / STEP;

  // Rows past M and columns past N read zeros through the range checks, and so does a step past
  // the end (a descriptor of no bytes at offset 0). A chunk past the end of K in the last step
  // has zeros for x (likewise) and a scale of 0; its weights are the next column's.
  const uint32_t x_row = static_cast<uint32_t>(args.x_stride) * 2u;
  const uint32_t x_bytes = static_cast<uint32_t>(M - 1) * x_row + static_cast<uint32_t>(K) * 2u;
  const uint32_t w_bytes = static_cast<uint32_t>(N) * static_cast<uint32_t>(K >> 1);
  const uint32_t z_bytes = static_cast<uint32_t>(N) * static_cast<uint32_t>(groups);

  // x load i of a wave: rows 8 (cw + 2 i) .. + 7 of its chunk, lane l row l / 8, stored column
  // l % 8 holding source column (l % 8) ^ key(row), key = bits 1..3 of the row. Weight load i:
  // columns 8 (wave + 8 i) .. + 7 of the tile, in the same layout.
  const int xrow = 8 * cw + (lane >> 3), wrow = 8 * wave + (lane >> 3);
  const uint32_t xoff = static_cast<uint32_t>(m0 + xrow) * x_row + 128u * kw +
                        static_cast<uint32_t>(((lane & 7) ^ ((xrow >> 1) & 7)) * 16);
  const uint32_t woff = static_cast<uint32_t>(n0 + wrow) * static_cast<uint32_t>(K >> 1) +
                        static_cast<uint32_t>(((lane & 7) ^ ((wrow >> 1) & 7)) * 16);
  auto load = [&](int ks, uint8_t* stage) {
    const bool in = ks < steps, xin = ks * STEP + CHUNK * kw < K;
    const __amdgpu_buffer_rsrc_t rx = buffer_rsrc(x, xin ? x_bytes : 0u), rw = buffer_rsrc(packed, in ? w_bytes : 0u);
#pragma unroll
    for (int i = 0; i < BM / 16; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(stage + kw * (BM * 128) + (cw + 2 * i) * 1024), 16,
                                               xoff + static_cast<uint32_t>(16 * i) * x_row, xin ? ks * STEP * 2 : 0, 0, 0);
#pragma unroll
    for (int i = 0; i < BN / 64; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(stage + XPART + (wave + 8 * i) * 1024), 16,
                                               woff + static_cast<uint32_t>(64 * i) * (K >> 1), in ? ks * STEP / 2 : 0, 0, 0);
  };

  struct G {
    u32x4 s;  // BLOCK: 8 scales; else s.x (and s.y: inputs 32 .. 63 of the chunk)
    u32x2 z;
  };
  constexpr int SLOADS = NF ? 1 : SC == Scales::TWO ? 4 : 2;
  const uint32_t goff = static_cast<uint32_t>(n0 + 64 * cw + lane) * static_cast<uint32_t>(groups);
  auto load_scales = [&](int ks, G& r) {
    const int k0 = ks * STEP + CHUNK * kw;
    const bool in = SC == Scales::BLOCK ? ks < steps : k0 < K;
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(args.scale, in ? (NF ? 4u : 2u) * z_bytes : 0u),
                                 rz = buffer_rsrc(args.zero, in ? z_bytes : 0u);
    const uint32_t at = goff + (in ? static_cast<uint32_t>((SC == Scales::BLOCK ? ks * STEP : k0) >> gshift) : 0u);
    if constexpr (NF) {
      r.s.x = __builtin_amdgcn_raw_buffer_load_b32(rs, 4u * at, 0, 0);
    } else if constexpr (SC == Scales::BLOCK) {
      r.s = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, 2u * at, 0, 0));
      r.z = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rz, at, 0, 0));
    } else {
      r.s.x = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rs, 2u * at, 0, 0));
      r.z.x = __builtin_amdgcn_raw_buffer_load_b8(rz, at, 0, 0);
      if constexpr (SC == Scales::TWO) {
        r.s.y = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rs, 2u * at + 2u, 0, 0));
        r.z.y = __builtin_amdgcn_raw_buffer_load_b8(rz, at + 1u, 0, 0);
      }
    }
  };
  // This lane's scale and zero point of column block b, packed (zero << 16 | scale); NF4: absmax.
  auto hand_out = [&](const G& r, int j, uint32_t (&o)[FB]) {
    uint32_t v;
    if constexpr (SC == Scales::BLOCK) {  // group 2 j + kw / 2 of the eight
      const uint32_t gs = r.s[j] >> (16 * (kw >> 1)), gz = r.z[j >> 1] >> (16 * (j & 1) + 8 * (kw >> 1));
      v = (gs & 0xffffu) | (gz << 16);
    } else if constexpr (NF) {
      v = r.s.x;
    } else {
      v = r.s.x | (r.z.x << 16);
    }
    if constexpr (SC == Scales::TWO) {
      // Lane l needs group h of columns l % 32 and 32 + l % 32.
      const uint32_t v1 = r.s.y | (r.z.y << 16);
      const auto p = __builtin_amdgcn_permlane32_swap(v, v1, false, false);
      o[0] = p[0];
      o[1] = p[1];
    } else {
      const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      o[0] = p[0];
      o[1] = p[1];
    }
  };

  // Codes as f16 halves without a conversion (see int4_narrow_kernel): (0x6400 | q) = 1024 + q,
  // (0x6400 | 16 q) = 1024 + 16 q, and (1024 + q) s - (1024 + z) s, (1024 + 16 q) (s / 16) -
  // (64 + z) s are exactly (q - z) s in one f32 fma.
  uint32_t mlo = 0x000f000fu, mhi = 0x00f000f0u, magic = 0x64006400u;
  hide_in_vgpr(mlo);
  hide_in_vgpr(mhi);
  hide_in_vgpr(magic);
  auto half_of = [](uint32_t m, int i) -> float { return static_cast<float>(__builtin_bit_cast(f16x2, m)[i]); };
  auto pack = [](float a, float b) -> uint32_t {
    if constexpr (DT == LNQ_BF16) return pack_bf16x2(a, b);
    else return pack_f16x2(a, b);
  };
  // A dword's 8 codes into one operand, in two halves of 9 and 8 instructions.
  struct Deq {
    uint32_t m0, m1, m2, m3;
    float v0, v1, v2, v3;
  };
  auto dequant_first = [&](uint32_t w, float s, float c, float s16, float c16) -> Deq {
    const uint32_t t = w >> 8;
    Deq d;
    d.m0 = and_or(w, mlo, magic);
    d.m1 = and_or(w, mhi, magic);
    d.m2 = and_or(t, mlo, magic);
    d.m3 = and_or(t, mhi, magic);
    d.v0 = fmaf(half_of(d.m0, 0), s, c);
    d.v1 = fmaf(half_of(d.m1, 0), s16, c16);
    d.v2 = fmaf(half_of(d.m2, 0), s, c);
    d.v3 = fmaf(half_of(d.m3, 0), s16, c16);
    return d;
  };
  auto dequant_rest = [&](const Deq& d, float s, float c, float s16, float c16) -> u32x4 {
    return u32x4{pack(d.v0, d.v1), pack(d.v2, d.v3), pack(fmaf(half_of(d.m0, 1), s, c), fmaf(half_of(d.m1, 1), s16, c16)),
                 pack(fmaf(half_of(d.m2, 1), s, c), fmaf(half_of(d.m3, 1), s16, c16))};
  };

  f32x16 acc[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  uint32_t aoff[4], boff[FB];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    aoff[kk] = static_cast<uint32_t>(kw * (BM * 128) + lcol * 128 + (((kk + 4 * h) ^ ((lcol >> 1) & 7)) << 4));
#pragma unroll
  for (int b = 0; b < FB; ++b)
    boff[b] = static_cast<uint32_t>(XPART + (64 * cw + 32 * b + lcol) * 128 + (((2 * kw + h) ^ ((lcol >> 1) & 7)) << 4));

  // Step ks = 4 q + j. Scales: BLOCK's are requested at j = 0 for the next four steps, the
  // others' three steps ahead.
  auto step = [&](int ks, int j, const uint8_t* stage, uint8_t* next, const G& g, G& req) {
    // This wave's loads of step ks have landed (issued two steps ago; behind them a step's
    // loads and scales); past the barrier every wave's have, and nobody reads step ks - 1's
    // stage, which step ks + 2 fills.
    if (SC == Scales::BLOCK && j != 1) wait_vm<LOADS>();
    else wait_vm<LOADS + SLOADS>();
    lds_barrier();
    load(ks + S - 1, next);
    __builtin_amdgcn_sched_barrier(0);
    if (SC != Scales::BLOCK) load_scales(ks + U - 1, req);
    else if (j == 0) load_scales(ks + U, req);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 wq[FB];
#pragma unroll
    for (int b = 0; b < FB; ++b) wq[b] = *reinterpret_cast<const u32x4*>(stage + boff[b]);
    uint32_t sz[FB];
    hand_out(g, j, sz);
    float s[FB], c[FB], s16[FB], c16[FB];
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      if constexpr (NF) continue;
      s[b] = E::to_f32(static_cast<uint16_t>(sz[b]));
      const float z = static_cast<float>((sz[b] >> 16) & 0xffu);
      c[b] = -(1024.f + z) * s[b];
      s16[b] = s[b] * 0.0625f;
      c16[b] = -(64.f + z) * s[b];
    }
    // Operand i = 2 kk + b: its MFMAs run over operand i + 1's dequantization, half of it
    // behind each (a scheduling region a MFMA pins that).
    u32x4 xa[2][FA], wb[2];
    f32x16 part[NF ? FA : 1][NF ? FB : 1];
    auto read_x = [&](int kk, int a) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(stage + aoff[kk] + a * 4096);
      xa[kk & 1][a] = NF ? stream::permute_nf4(v) : v;
    };
#pragma unroll
    for (int a = 0; a < FA; ++a) read_x(0, a);
    if constexpr (NF) wb[0] = stream::nf4_widen(wq[0][0], args.planes);
    else wb[0] = dequant_rest(dequant_first(wq[0][0], s[0], c[0], s16[0], c16[0]), s[0], c[0], s16[0], c16[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int kk = i / FB, b = i % FB, nb = (i + 1) % FB, nk = (i + 1) / FB;
      Deq d;
      auto multiply = [&](int a) {
        if constexpr (NF) part[a][b] = mid_mfma<DT>(xa[kk & 1][a], wb[i & 1], kk == 0 ? f32x16{} : part[a][b]);
        else acc[a][b] = mid_mfma<DT>(wb[i & 1], xa[kk & 1][a], acc[a][b]);
      };
      multiply(0);
      if constexpr (!NF)
        if (i < 7) d = dequant_first(wq[nb][nk], s[nb], c[nb], s16[nb], c16[nb]);
      if (b == 0 && kk < 3) read_x(kk + 1, 0);
      if constexpr (!NF) __builtin_amdgcn_sched_barrier(0);
      multiply(1);
      if (i < 7) {
        if constexpr (NF) wb[(i + 1) & 1] = stream::nf4_widen(wq[nb][nk], args.planes);
        else wb[(i + 1) & 1] = dequant_rest(d, s[nb], c[nb], s16[nb], c16[nb]);
      }
      if (b == 0 && kk < 3) read_x(kk + 1, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NF) {
#pragma unroll
      for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < FA; ++a)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[a][b][r] = fmaf(part[a][b][r], __builtin_bit_cast(float, sz[b]), acc[a][b][r]);
    }
  };

  G g[U];
  if constexpr (SC == Scales::BLOCK) {
    load_scales(0, g[0]);
  } else {
#pragma unroll
    for (int j = 0; j < U - 1; ++j) load_scales(j, g[j]);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < S - 1; ++j) {
    load(j, st[j]);
    __builtin_amdgcn_sched_barrier(0);
  }
  wait_vm<LOADS>();  // step 0's: no scales behind it
  for (int ks = 0; ks < steps; ks += 12) {
#pragma unroll
    for (int j = 0; j < 12; ++j) {
      if (ks + j >= steps) break;
      if constexpr (SC == Scales::BLOCK) step(ks + j, j % 4, st[j % S], st[(j + 2) % S], g[(j / 4) % 2], g[(j / 4 + 1) % 2]);
      else step(ks + j, 0, st[j % S], st[(j + 2) % S], g[j % U], g[(j + U - 1) % U]);
    }
    // Twelve steps are three blocks: the next iteration begins with the other set.
    if constexpr (SC == Scales::BLOCK) {
      const G t = g[0];
      g[0] = g[1];
      g[1] = t;
    }
  }
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Wave kw finishes tile t = kw of the four (two row blocks by two column blocks): all leave
  // their part of it in LDS, lane-linear, 16 KB for a tile and column half.
  const bool vec_out = (N & 3) == 0;
  uint8_t* const area[4] = {S0 + cw * 16384, S1 + cw * 16384, S2 + cw * 16384, (cw ? S1 : S0) + 32768};
  lds_barrier();
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const f32x16& v = acc[t & 1][t >> 1];
    float* const o = reinterpret_cast<float*>(area[t] + kw * 4096) + 4 * lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(o + 256 * q) = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  }
  lds_barrier();
  const float* const from = reinterpret_cast<const float*>(kw == 0 ? area[0] : kw == 1 ? area[1] : kw == 2 ? area[2] : area[3]) + 4 * lane;
  const int mt = m0 + 32 * (kw & 1), nt = n0 + 64 * cw + 32 * (kw >> 1);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 v = *reinterpret_cast<const f32x4*>(from + 256 * q);
#pragma unroll
    for (int k = 1; k < KW; ++k) v += *reinterpret_cast<const f32x4*>(from + 1024 * k + 256 * q);
    // Four features of one row, the rounded product plus the bias rounded again (the
    // reference's order); NF4: four rows of one feature, rounded once, as its other kernels do.
    uint16_t out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = NF ? nt + lcol : nt + 8 * q + 4 * h + i;
      const bool add = bias != nullptr && n < N;
      if constexpr (NF) {
        out[i] = E::from_f32(add ? v[i] + E::to_f32(bias[n]) : v[i]);
      } else {
        out[i] = E::from_f32(v[i]);
        if (add) out[i] = E::from_f32(E::to_f32(out[i]) + E::to_f32(bias[n]));
      }
    }
    if constexpr (NF) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mt + 8 * q + 4 * h + i;
        if (m < M && nt + lcol < N) y[static_cast<size_t>(m) * args.y_stride + nt + lcol] = out[i];
      }
    } else {
      const int m = mt + lcol, n = nt + 8 * q + 4 * h;
      if (m < M) {
        uint16_t* const yrow = y + static_cast<size_t>(m) * args.y_stride;
        if (vec_out && n + 3 < N) {
          *reinterpret_cast<u32x2*>(yrow + n) = u32x2{static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16),
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

// One tile a CU at most. Past that the second round costs what the 128- or 256-row tiles'
// only one does: 256 rows 4096 -> 14336 (448 tiles) 47.1 us here, 43.7 there; 384 rows
// 8192 -> 8192 (384) 101.3 and 86.9.
bool int4_mid_preferred(int M, int N) {
  return static_cast<int64_t>((M + mid::BM - 1) / mid::BM) * ((N + mid::BN - 1) / mid::BN) <= compute_units();
}

template <int DT, Scales SC>
static void launch(const MidArgs& a, hipStream_t stream) {
  const int tiles = ((a.M + mid::BM - 1) / mid::BM) * ((a.N + mid::BN - 1) / mid::BN);
  hipLaunchKernelGGL((int4_mid_kernel<DT, SC>), dim3(tiles), dim3(mid::THREADS), 0, stream, a);
}

template <int DT>
static void launch_scales(const MidArgs& a, int G, hipStream_t stream) {
  const bool whole = (reinterpret_cast<uintptr_t>(a.scale) | reinterpret_cast<uintptr_t>(a.zero)) % 4 == 0;
  if (G == 128 && a.K % 1024 == 0 && whole) launch<DT, Scales::BLOCK>(a, stream);
  else if (G >= 64) launch<DT, Scales::ONE>(a, stream);
  else launch<DT, Scales::TWO>(a, stream);
}

LnqStatus launch_int4_mid(const void* x, const uint8_t* packed, const void* scale, const uint8_t* zero, const void* bias,
                          void* y, int M, int N, int K, int G, int dtype, hipStream_t stream) {
  const MidArgs a{static_cast<const uint16_t*>(x), packed, scale, zero, static_cast<const uint16_t*>(bias),
                  static_cast<uint16_t*>(y), M, N, K, __builtin_ctz(static_cast<unsigned>(G)), K, N, {}};
  if (dtype == LNQ_BF16) launch_scales<LNQ_BF16>(a, G, stream);
  else launch_scales<LNQ_F16>(a, G, stream);
  return launched("int4_mid");
}

LnqStatus launch_nf4_mid(const void* x, int x_stride, const uint8_t* codes, const float* absmax, const void* bias, void* y,
                         int y_stride, int M, int N, int K, int block, const stream::Planes& planes, int dtype,
                         hipStream_t stream) {
  const MidArgs a{static_cast<const uint16_t*>(x), codes, absmax, codes, static_cast<const uint16_t*>(bias),
                  static_cast<uint16_t*>(y), M, N, K, __builtin_ctz(static_cast<unsigned>(block)), x_stride, y_stride, planes};
  if (dtype == LNQ_BF16) launch<LNQ_BF16, Scales::NF4>(a, stream);
  else launch<LNQ_F16, Scales::NF4>(a, stream);
  return launched("nf4_mid");
}

}  // namespace lnq
