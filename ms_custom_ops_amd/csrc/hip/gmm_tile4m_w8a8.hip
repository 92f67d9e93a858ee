// Persistent four-wave tile kernels (gmm_tile4m_kernel.h): one translation unit per layout, output type and activation.
#include "gmm_kernels.h"
#include "gmm_tile4_common.h"

namespace msco {

#define MSCO_T4M_DECLARE(LAYOUT) \
  hipError_t tile4m_##LAYOUT(const GmmParams &p, const T4mPick &pick, hipStream_t s); \
  hipError_t tile4m_##LAYOUT##_bf16(const GmmParams &p, const T4mPick &pick, hipStream_t s); \
  hipError_t tile4m_##LAYOUT##_f16(const GmmParams &p, const T4mPick &pick, hipStream_t s); \
  hipError_t tile4m_##LAYOUT##_bf16_silu(const GmmParams &p, const T4mPick &pick, hipStream_t s); \
  hipError_t tile4m_##LAYOUT##_f16_silu(const GmmParams &p, const T4mPick &pick, hipStream_t s);
MSCO_T4M_DECLARE(nk)
MSCO_T4M_DECLARE(packed)
MSCO_T4M_DECLARE(kn)
#undef MSCO_T4M_DECLARE

hipError_t launch_tile4m_w8a8(const GmmParams &p, const T4mPick &pick, int layout, hipStream_t s) {
  // layout 0 [E,N,K], 1 packed, 2 [E,K,N] (read in 16-column chunks); the operand stream runs up to four slabs ahead inside
  // one tile; the group table lives in LDS
  if (p.k < 4 * T4_BK || p.e > T4_MAX_E || layout < 0 || layout > 2 || (layout == 2 && p.n % 16 != 0)) return hipErrorInvalidValue;
  const bool silu = p.act_type == ACT_SILU || p.act_type == ACT_FAST_GELU, any = (p.out_dtype == DT_BF16 || p.out_dtype == DT_F16) && (silu || p.act_type == ACT_NONE);
  if (!any && p.out_dtype != DT_BF16 && p.out_dtype != DT_F16 && p.out_dtype != DT_I32) return hipErrorInvalidValue;
  if (pick.shape >= T4M_SHAPES || (pick.shape >= 0 && !t4m_has(pick.shape, layout)) || (!any && pick.shape != 0)) return hipErrorInvalidValue;
#define MSCO_T4M_RUN(LAYOUT) \
  (!any ? tile4m_##LAYOUT(p, pick, s) \
   : p.out_dtype == DT_BF16 ? (silu ? tile4m_##LAYOUT##_bf16_silu(p, pick, s) : tile4m_##LAYOUT##_bf16(p, pick, s)) \
                            : (silu ? tile4m_##LAYOUT##_f16_silu(p, pick, s) : tile4m_##LAYOUT##_f16(p, pick, s)))
  return layout == 1 ? MSCO_T4M_RUN(packed) : layout == 2 ? MSCO_T4M_RUN(kn) : MSCO_T4M_RUN(nk);
#undef MSCO_T4M_RUN
}

}  // namespace msco
