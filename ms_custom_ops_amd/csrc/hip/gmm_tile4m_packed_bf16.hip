// Persistent four-wave tile kernel, packed weights, bfloat16 output, no activation: see gmm_tile4m_kernel.h.
#include "gmm_tile4m_kernel.h"

namespace msco {
hipError_t tile4m_packed_bf16(const GmmParams &p, const T4mPick &pick, hipStream_t s) { return t4m_launch<0, 1, 0, true>(p, pick, s); }
}  // namespace msco
