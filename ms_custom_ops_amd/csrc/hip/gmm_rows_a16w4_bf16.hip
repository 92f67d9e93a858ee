// bf16 x, 4-bit [E,K,N] weights: the kernels of gmm_rows_a16w8_kernel.h, one translation unit per pair of types and layouts (a minute of compilation each)
#include "gmm_rows_a16w8_kernel.h"

namespace msco {

hipError_t rows_a16w4_bf16(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream) {
  return rows_a16w8_pick<true, true, true>(p, strip_cols, sets, grid, stream);
}

}  // namespace msco
