// The streaming few-row product (stream.hpp) over group-wise 4-bit weights: groups of 32,
// 64 and multiples of 128, any width.
#include "stream.hpp"

namespace lnq {

bool int4_stream_supports(int N, int K) { return K <= stream::MAX_K && N <= stream::MAX_N; }

// Whether the skinny kernel is faster than the streaming one, for the calls that both take. It
// gives 16 outputs and all the rows (64 of them past 64) a workgroup of four waves: less to do
// before and after the products, more per input. So it keeps short layers of one round of its
// workgroups (two where In is 256). us, group 128, skinny / streaming: 512 -> 4096 8 / 24 rows 3.3
// / 3.5, 4.1 / 4.6; 1024 -> 1024 17 rows 4.3 / 4.9, 32 rows 4.7 / 4.9. From 33 rows on the
// streaming kernel takes a second round past 1024 outputs, 5 us at 1024 inputs: 1024 -> 4096 33 /
// 64 rows 6.6 / 8.4, 7.6 / 8.3; 2048 -> 2048 33 / 64 rows 8.7 / 9.5, 11.1 / 10.0; 2048 -> 6000 16.0 /
// 11.1. Smaller groups cost the skinny kernel a fold each: groups of 64 1024 -> 4096 64 rows 8.4 /
// 8.8, of 32 768 -> 4096 37 / 48 rows 8.4 / 8.7, 8.8 / 8.7.
// Past 64 rows (groups that the prefill kernels do not take, weights past 2 GiB) estimates of
// both, fitted to 65 to 2048 rows of one scale a row: 1536 -> 2048 65 / 512 rows 9.4 / 12.9, 31 /
// 61; 14336 -> 4096 65 / 512 / 1024 rows 79 / 48, 436 / 300, 866 / 1013; 3072 -> 3072 256 / 2048
// rows 41 / 31, 311 / 342.
bool int4_skinny_preferred(int M, int N, int K, int G) {
  const double k = K / 1024.0;
  const int fine = G >= 128 ? 1 : 128 / G, cus = compute_units();
  const bool one_round = N <= 16 * cus * (K <= 256 ? 2 : 1);
  if (M <= 6) return false;  // 512 -> 4096 4 rows 3.7 / 3.3
  if (M <= 32) return one_round && K * fine <= (M > 16 && M <= 28 ? 1024 : 512);
  const double fold = fine == 1 ? 0 : fine == 2 ? 0.4 : 2.0;
  if (M <= 64) return one_round && N > 4 * cus && (0.037 * M - 0.3 + fold) * k < 2.6;
  const int chunks = (M + 63) / 64;
  const int64_t groups = static_cast<int64_t>((N + 15) / 16) * chunks;
  const double skinny = 3.8 + static_cast<double>((groups + cus - 1) / cus) * (1.3 + 0.037 * M / chunks + fold) * k;
  stream::Args a{};
  a.cols = K / G;
  a.row_block = 1;
  int r = 0;
  const int rounds = stream::rounds<stream::INT4, 4, stream::ONE_STEP>(a, M, N, r);
  const double round = r <= 16 ? 2.45 + 0.9 * k : r <= 32 ? 2.95 + 1.15 * k : 3 + 1.85 * k;
  return skinny < 0.97 * (1.75 + round * rounds) * stream::x_past_l2(M, K, r);
}

// Groups of 32 at 17 rows and more (two row tiles beside a step of eight folds) spill 9 VGPRs, 40
// bytes a lane; the form is kept all the same. us, 4096 -> 14336, the skinny kernel / this one:
// 16 rows 59.3 / 19.3 (one row tile, no spill), 17 63.3 / 23.6, 24 68.2 / 23.7, 32 73.4 / 24.3.
template <int DT>
static void launch(const stream::Args& a, int G, hipStream_t s) {
  if (G == 128) stream::launch<DT, stream::INT4, 1>(a, s);
  else if (G % 128 == 0) stream::launch<DT, stream::INT4, 1, stream::SPAN>(a, s);
  else if (G == 64) stream::launch<DT, stream::INT4, 2>(a, s);
  else stream::launch<DT, stream::INT4, 4>(a, s);
}

LnqStatus launch_int4_stream(const void* x, const uint8_t* packed, const void* scale, const uint8_t* zero,
                             const void* bias, void* y, int M, int N, int K, int G, int dtype, hipStream_t stream) {
  stream::Args a{};
  a.x = static_cast<const uint16_t*>(x);
  a.w = packed;
  a.scale = scale;
  a.zero = zero;
  a.bias = static_cast<const uint16_t*>(bias);
  a.y = static_cast<uint16_t*>(y);
  a.x_stride = K;
  a.y_stride = N;
  a.row_bytes = K / 2;
  a.M = M;
  a.N = N;
  a.K = K;
  a.span = G % 128 == 0 ? G / 128 : 1;
  a.cols = K / G;
  a.row_block = 1;
  if (dtype == LNQ_BF16) launch<LNQ_BF16>(a, G, stream);
  else launch<LNQ_F16>(a, G, stream);
  return launched("int4_stream");
}

}  // namespace lnq
