// bf16 x, packed weights: the kernels of gmm_rows_a16w8_kernel.h, one translation unit per pair of types and layouts (a minute of compilation each); and the launcher of all of them
#include "gmm_rows_a16w8_kernel.h"

namespace msco {

hipError_t rows_a16w8_bf16_packed(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream) {
  return rows_a16w8_pick<true, false>(p, strip_cols, sets, grid, stream);
}

hipError_t rows_a16w8_bf16_kn(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream);
hipError_t rows_a16w8_f16_packed(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream);
hipError_t rows_a16w8_f16_kn(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream);
hipError_t rows_a16w4_bf16(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream);
hipError_t rows_a16w4_f16(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream);

size_t rows_a16w8_slice_bytes() { return (size_t)XA_SLICE_WORDS * 256 * 8; }

// packed or [E,K,N] weights, the latter of 8 or 4 bits; K % 16 == 0, N % 16 == 0, K < 2^22 (an out-of-range mark plus the offset of a chunk's last row, 256 K
// bytes, stays a 32-bit offset out of range) and one group's weights below 2^31 bytes; M is not bounded by offsets.
// strip_cols 512, or 256 with one or two wave sets; p.split_k > 1 (strips of 256): a partial tile per (chunk, strip, slice) and a
// counter per (chunk, strip)
hipError_t launch_rows_a16w8(const GmmParams &p_in, bool packed, bool w4, int strip_cols, int sets, hipStream_t stream) {
  if (p_in.m == 0) return hipSuccess;
  if (packed && w4) return hipErrorInvalidValue;
  if (p_in.k % 16 != 0 || p_in.n % 16 != 0 || p_in.k >= (1 << 22) || p_in.split_k < 1 || p_in.split_k > 65535) return hipErrorInvalidValue;
  if ((strip_cols != 512 && strip_cols != 256) || (strip_cols == 512 && p_in.split_k != 1)) return hipErrorInvalidValue;
  if (p_in.split_k > 1 && (p_in.partial == nullptr || p_in.counters == nullptr)) return hipErrorInvalidValue;
  GmmParams p = p_in;
  p.n_strips = (p.n + strip_cols - 1) / strip_cols;
  const long long slots = xcd_slots(p, XA_ROWS);
  if (slots > 0x7FFFFFFFll) return hipErrorInvalidValue;
  const dim3 grid((unsigned)slots, (unsigned)p.split_k);
  if (w4) return p.x_dtype == DT_BF16 ? rows_a16w4_bf16(p, strip_cols, sets, grid, stream) : rows_a16w4_f16(p, strip_cols, sets, grid, stream);
  if (p.x_dtype == DT_BF16) return packed ? rows_a16w8_bf16_packed(p, strip_cols, sets, grid, stream) : rows_a16w8_bf16_kn(p, strip_cols, sets, grid, stream);
  return packed ? rows_a16w8_f16_packed(p, strip_cols, sets, grid, stream) : rows_a16w8_f16_kn(p, strip_cols, sets, grid, stream);
}

}  // namespace msco
