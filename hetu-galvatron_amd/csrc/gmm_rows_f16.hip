// The row-adaptive kernel (gmm_rows_kernel.h) for fp16 operands.
#include "gmm_rows_kernel.h"

namespace gmoe {

int launch_gmm_rows_f16(const GmmParams& p, int mode, int out_dtype, int epi, hipStream_t st) {
  return rows::launch_dt<GMOE_F16>(p, mode, out_dtype, epi, st);
}

}  // namespace gmoe
