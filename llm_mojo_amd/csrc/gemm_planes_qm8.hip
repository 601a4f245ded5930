// The activation-plane matmul (gemm_planes.h) of int8 QuantMatrix with float activations.
#include "gemm_planes.h"

namespace planes {

template int launch_tile<kQm8, 1>(hipStream_t, int, const Args &);
template int launch_tile<kQm8, 8>(hipStream_t, int, const Args &);

}  // namespace planes
