#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_tail_gelu(int tile, const void* args, hipStream_t stream) {
  return launch<EPI_TAIL_GELU, false>(tile, *static_cast<const MidArgs*>(args), stream);
}
