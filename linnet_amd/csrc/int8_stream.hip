// The weight-only int8 product at few rows (lnq_w8a16): stream.hpp's kernel.
#include "w8_stream.hpp"

namespace lnq {

LnqStatus launch_int8_stream(const void* x, const uint8_t* w, const float* scale, void* y, int M, int N, int K, int group,
                           int row_block, int dtype, hipStream_t stream) {
  return launch_w8_stream<stream::INT8>(x, w, scale, y, M, N, K, group, row_block, dtype, stream);
}

}  // namespace lnq
