// The pipelined dequant-GEMM (gguf_gemm_pipe.hip) of Q4_1, Q5_0, Q5_1, Q2_K and Q3_K: fp16 activations,
// K within one workgroup.
//   Q4_1 / Q5_0 / Q5_1: a step is two whole blocks, as Q4_0's, with the minimum and the fifth bits.
//   Q2_K / Q3_K: a step is planes 2 (s % 2), 2 (s % 2) + 1 of half h = (s % 4) / 2 of a super-block: the
//     half's 32 quant bytes, four scales and (Q3_K) two bits of each of the 32 third-bit bytes.
#include "gguf_gemm_pipe.h"

namespace tensor_gguf {

template <int TYPE>
static hipError_t launch_more(const GemmGroupArgs& a, int tile, hipStream_t stream) {
  return a.out_half ? launch_tile<TYPE, _Float16, _Float16>(a, tile, 1, nullptr, stream)
                    : launch_tile<TYPE, float, _Float16>(a, tile, 1, nullptr, stream);
}

hipError_t launch_gemm_pipe_more(const GemmGroupArgs& a, int tile, hipStream_t stream) {
  if (a.x_f32) return hipErrorInvalidValue;
  switch (a.type) {
    case kQ4_1: return launch_more<kQ4_1>(a, tile, stream);
    case kQ5_0: return launch_more<kQ5_0>(a, tile, stream);
    case kQ5_1: return launch_more<kQ5_1>(a, tile, stream);
    case kQ2_K: return launch_more<kQ2_K>(a, tile, stream);
    case kQ3_K: return launch_more<kQ3_K>(a, tile, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tensor_gguf
