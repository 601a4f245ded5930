// The activation-plane matmul (gemm_planes.h) of int8 QuantMatrix with int16 activations.
#include "gemm_planes.h"

namespace planes {

template int launch_tile<kA8, 1>(hipStream_t, int, const Args &);
template int launch_tile<kA8, 2>(hipStream_t, int, const Args &);
template int launch_tile<kA8, 4>(hipStream_t, int, const Args &);
template int launch_tile<kA8, 8>(hipStream_t, int, const Args &);

}  // namespace planes
