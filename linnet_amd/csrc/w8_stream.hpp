// The streaming few-row product (stream.hpp) over 8-bit weights, one format a source file
// (fp8_stream.hip, int8_stream.hip). Scales are f32: one a row (group 0), or one per
// `group` (a multiple of 64) inputs and `row_block` rows.
#pragma once

#include "stream.hpp"

namespace lnq {

template <int DT, int F>
static void launch_w8_stream_dt(stream::Args& a, int group, int row_block, hipStream_t s) {
  using namespace stream;
  if (group == 0) return launch<DT, F, 0>(a, s);
  a.cols = a.K / group;
  a.row_block = row_block;
  if (group % 128 == 0) {
    a.span = group / 128;
    if (a.span == 1 && row_block == 1) launch<DT, F, 1>(a, s);
    else launch<DT, F, 1, BLOCK>(a, s);
  } else {
    a.span = group / 64;
    if (a.span == 1 && row_block == 1) launch<DT, F, 2>(a, s);
    else launch<DT, F, 2, BLOCK>(a, s);
  }
}

template <int F>
static LnqStatus launch_w8_stream(const void* x, const uint8_t* w, const float* scale, void* y, int M, int N, int K,
                                  int group, int row_block, int dtype, hipStream_t stream) {
  stream::Args a{};
  a.x = static_cast<const uint16_t*>(x);
  a.w = w;
  a.scale = scale;
  a.y = static_cast<uint16_t*>(y);
  a.x_stride = K;
  a.y_stride = N;
  a.row_bytes = K;
  a.M = M;
  a.N = N;
  a.K = K;
  a.span = 1;
  a.cols = 1;
  a.row_block = 1;
  if (dtype == LNQ_BF16) launch_w8_stream_dt<LNQ_BF16, F>(a, group, row_block, stream);
  else launch_w8_stream_dt<LNQ_F16, F>(a, group, row_block, stream);
  return launched("w8_stream");
}

}  // namespace lnq
