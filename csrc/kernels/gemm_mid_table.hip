#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_gelu_table(int tile, const void* args, hipStream_t stream) {
  return launch<EPI_GELU_TABLE, false>(tile, *static_cast<const MidArgs*>(args), stream);
}
