// The row-adaptive kernel (gmm_rows_kernel.h) for bf16 operands, and its launch; fp16 in gmm_rows_f16.hip.
#include "gmm_rows_kernel.h"

namespace gmoe {

int launch_gmm_rows_f16(const GmmParams& p, int mode, int out_dtype, int epi, hipStream_t st);

int launch_gmm_rows(const GmmParams& p, int mode, int dtype, int out_dtype, int epi, hipStream_t st) {
  if (dtype == GMOE_BF16) return rows::launch_dt<GMOE_BF16>(p, mode, out_dtype, epi, st);
  if (dtype == GMOE_F16) return launch_gmm_rows_f16(p, mode, out_dtype, epi, st);
  return GMOE_ERR_UNSUPPORTED;
}

}  // namespace gmoe
