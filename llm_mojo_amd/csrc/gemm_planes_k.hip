// The activation-plane matmul (gemm_planes.h) of the K quants.
#include "gemm_planes.h"

namespace planes {

template int launch_tile<kQ4_K, 8>(hipStream_t, int, const Args &);
template int launch_tile<kQ5_K, 1>(hipStream_t, int, const Args &);
template int launch_tile<kQ6_K, 8>(hipStream_t, int, const Args &);

}  // namespace planes
