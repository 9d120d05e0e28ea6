// The streaming few-row product (stream.hpp) over group-wise 4-bit weights: groups of 32,
// 64 and multiples of 128, any width.
#include "stream.hpp"

namespace lnq {

bool int4_stream_supports(int K) { return K <= stream::MAX_K; }

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
