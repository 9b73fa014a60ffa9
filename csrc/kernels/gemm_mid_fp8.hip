#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_fp8(int tile, const void* args, hipStream_t stream) {
  return launch<EPI_STORE, true>(tile, *static_cast<const MidArgs*>(args), stream);
}
