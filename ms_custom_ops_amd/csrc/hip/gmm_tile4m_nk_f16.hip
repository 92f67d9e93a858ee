// Persistent four-wave tile kernel, [E,N,K] weights, float16 output, no activation: see gmm_tile4m_kernel.h.
#include "gmm_tile4m_kernel.h"

namespace msco {
hipError_t tile4m_nk_f16(const GmmParams &p, const T4mPick &pick, hipStream_t s) { return t4m_launch<1, 0, 0, true>(p, pick, s); }
}  // namespace msco
