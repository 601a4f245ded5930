// The activation-plane matmul (gemm_planes.h) of Q8_0, Q4_0 and Q4_1.
#include "gemm_planes.h"

namespace planes {

template int launch_tile<kQ8_0, 1>(hipStream_t, int, const Args &);
template int launch_tile<kQ4_0, 1>(hipStream_t, int, const Args &);
template int launch_tile<kQ4_1, 1>(hipStream_t, int, const Args &);

}  // namespace planes
