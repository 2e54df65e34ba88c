// Instances of the weight-streaming GEMM (gemm_stream.hpp): e4m3 codes, row-major weights.
#include "gemm_stream.hpp"

namespace h3q {

hipError_t launch_stream_e4m3_rows(int tile, const GemmArgs& a, hipStream_t st) {
    return launch_stream_op<kOpE4M3, false>(tile, a, st);
}

}  // namespace h3q
