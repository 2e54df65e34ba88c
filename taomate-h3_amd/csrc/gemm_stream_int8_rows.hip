// Instances of the weight-streaming GEMM (gemm_stream.hpp): int8 codes, row-major weights.
#include "gemm_stream.hpp"

namespace h3q {

hipError_t launch_stream_int8_rows(int tile, const GemmArgs& a, hipStream_t st) {
    return launch_stream_op<kOpInt8, false>(tile, a, st);
}

}  // namespace h3q
