// Persistent four-wave tile kernel, packed weights, the outputs that have 256 x 256 tiles only: see gmm_tile4m_kernel.h.
#include "gmm_tile4m_kernel.h"

namespace msco {
hipError_t tile4m_packed(const GmmParams &p, const T4mPick &pick, hipStream_t s) {
  if (p.out_dtype == DT_I32) return t4m_launch<2, 1, 0, false>(p, pick, s);
  const bool relu = p.act_type == ACT_RELU;
  if (p.out_dtype == DT_BF16) return relu ? t4m_launch<0, 1, 3, false>(p, pick, s) : t4m_launch<0, 1, 1, false>(p, pick, s);
  return relu ? t4m_launch<1, 1, 3, false>(p, pick, s) : t4m_launch<1, 1, 1, false>(p, pick, s);
}
}  // namespace msco
