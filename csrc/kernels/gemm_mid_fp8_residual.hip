#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_fp8_residual(int tile, const void* args, hipStream_t stream) {
  return launch<EPI_RESIDUAL, true>(tile, *static_cast<const MidArgs*>(args), stream);
}
