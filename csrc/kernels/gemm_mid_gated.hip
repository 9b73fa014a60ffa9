#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_gated(int tile, const void* args, hipStream_t stream) {
  return launch<EPI_SILU_MUL, false>(tile, *static_cast<const MidArgs*>(args), stream);
}
