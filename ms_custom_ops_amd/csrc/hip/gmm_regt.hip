// Grouped matmul on row-major weights [E,K,N] that have to be transposed and converted on their way to the matrix cores
// (gfx950): 4-bit ([E,K,N/2]) or 8-bit weights, int8 or 16-bit activations, groups of one to a few dozen rows.
//
// Both jobs are done in registers.  A lane of a wave requests, for every one of its K rows of a step, CPL neighbouring
// columns (16 lanes cover 16 CPL columns of a row in whole lines); lane group h takes K rows KR h .. KR h + KR - 1 of the
// step, which is exactly the K range lane group h supplies to the MFMA.  What is left to do is to gather column j of the
// KR registers of a column word, which a handful of v_perm_b32, masks and conversions do:
//
//   int8 x    v_mfma_i32_16x16x64_i8, KR = 16.  Four rows of a word are transposed as bytes (8 v_perm per 16 bytes).  8-bit
//             weights: that is the operand.  4-bit weights: a byte holds an even and an odd column, and both become int8
//             operands of 16 times their value ((c << 4) & 0xF0.., c & 0xF0..): 20 instructions per 32 weights, nothing to
//             sign-extend, and the int32 sums are exactly 16 times the true ones (K x 2^14 < 2^31 is checked by the plan, for this form alone).
//   16-bit x  v_mfma_f32_16x16x32, KR = 8.  A signed byte of two rows each goes through v_cvt_f32_i32 (byte select) and
//             one pack: exact in bf16 and f16.  4-bit weights enter as a sixteenth of their value (one conversion takes the low half
//             of a byte): every product and every rounding is a sixteenth of the one 8-bit weights of the same value give, so with
//             the same chunks the results are the same bits (16 times the value, which this was, loses sums from 2^124 on; a sixteenth
//             loses nothing: products are multiples of 2^-137).  The antiquant offset is folded into the epilogue with the row sums of x (one MFMA
//             against ones per x fragment):  out = s * (sum_k x w + o sum_k x).
//
// The output column of MFMA column c of word position j is CPL c + j: a permutation that only the epilogue sees.
//
// Workgroup = one chunk of at most 16 R rows of one group x one strip of 16 CPL WN columns x one K slice; WN waves sit side
// by side in columns, WK = CPL / 4 rows of waves take interleaved K steps and meet in LDS at the end, in wave order.  K
// slices of different workgroups meet in the workspace, in slice order: results are reproducible run to run.
//
// The grid runs over strips, K slices, chunk slots, the last slowest: the slots past the last chunk then are the last
// workgroups.  With the slices slowest these empty ones stood between the slices, and CUs that had got one were passed over
// for the next slice while others took two of it (weight-only, 8 x 4 rows, K = 8192, N = 4096, two slices on 256 CUs: 69.3 -> 49.2 us;
// 4-bit weights, 8 x 8 rows, K = N = 4096: 32.0 -> 21.5 us).
//
// SHALLOW (16-bit x, 8-bit weights): one K step in flight per wave and four waves per SIMD in place of three steps and two
// waves.  Where a CU gets several workgroups, one's ends (first requests, reduction, stores) lie under the other's walk: 64
// experts, N = 4096, 8 rows per group, K = 512 / 1024: 38.3 -> 29.2, 55.9 -> 48.9 us; 8 experts, K = 4096, N = 14336, 4 rows: 76.1 -> 74.6
// us.  With one workgroup per CU or less it has too few requests in flight (one row, K = 4096, N = 11008: 16.4 -> 17.8 us).
#include <type_traits>

#include "gmm_common.h"
#include "gmm_kernels.h"

namespace msco {

namespace {
typedef long long i64;
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));

template <int XT, int WB, int R, int CPL, int WN>
struct RtShape {
  static constexpr int kWk = CPL / 4;                   // waves that share a strip's columns and split its K steps
  static constexpr int kThreads = 64 * WN * kWk;
  static constexpr int kStep = XT == DT_I8 ? 64 : 32;    // K per MFMA
  static constexpr int kKr = kStep / 4;                 // K rows per lane and step
  static constexpr int kDw = CPL * WB / 32;             // dwords per lane and K row
  static constexpr int kCols = 16 * CPL * WN;
  static constexpr int kRed = WN * kWk * 8 * 1024;      // 16 rows x 8 word positions of every wave's accumulators
  static constexpr int kEp = kRed + WN * kWk * R * 64 + 16;   // + row sums of x per wave, ticket
  static_assert(kThreads == kCols, "a thread brings the epilogue operands of one column");
  static constexpr size_t kLds = (size_t)kEp + 8 * kCols + 64 * R;   // + the columns' scales and offsets (biases), the rows' scales
  static constexpr size_t kSliceWords = (size_t)R * (16 * kCols / 2 + 8);   // 64-bit words of a K slice's partial tile (+ row sums)
};

template <int DW>
__device__ __forceinline__ void load_words(int *w, __amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff) {
  if constexpr (DW == 1) {
    w[0] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, voff, soff, kStreamAux);
  } else if constexpr (DW == 2) {
    const v2i v = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, kStreamAux));
    w[0] = v[0];
    w[1] = v[1];
  } else {
    const v4i v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, kStreamAux));
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = v[i];
  }
}

// bytes B of two K rows -> two 16-bit floating-point values (exact: integers of at most eight significant bits)
template <bool BF16, int B>
__device__ __forceinline__ int byte_pair(unsigned lo, unsigned hi) {
  const float f0 = (float)(int)(signed char)(lo >> (8 * B)), f1 = (float)(int)(signed char)(hi >> (8 * B));
  if constexpr (BF16) return (int)perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
  else return __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(f0, f1));
}
// the signed 4-bit numbers in the low halves of these bytes -> a sixteenth of each
template <bool BF16, int B>
__device__ __forceinline__ int nibble_pair(unsigned lo, unsigned hi) {
  const float f0 = __builtin_amdgcn_cvt_off_f32_i4((int)(lo >> (8 * B) & 0xFFu)), f1 = __builtin_amdgcn_cvt_off_f32_i4((int)(hi >> (8 * B) & 0xFFu));
  if constexpr (BF16) return (int)perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
  else return __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(f0, f1));
}

template <int XT>
__device__ __forceinline__ void rt_mfma(v4i &acc, const v4i &a, const v4i &b) {
  acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc, 0, 0, 0);
}
template <int XT>
__device__ __forceinline__ void rt_mfma(v4f &acc, const v4i &a, const v4i &b) {
  if constexpr (XT == DT_BF16) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
  else acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), acc, 0, 0, 0);
}
}  // namespace

// L = 16-row blocks of the chunk that hold rows
template <int XT, int WB, int R, int CPL, int WN, bool SHALLOW, int L>
__device__ __forceinline__ void regt_run(const GmmParams &p, unsigned char *smem, int grp, int m0, int chunk_rows) {
  using S = RtShape<XT, WB, R, CPL, WN>;
  using Acc = std::conditional_t<XT == DT_I8, v4i, v4f>;
  using Elem = std::conditional_t<XT == DT_I8, int, float>;
  constexpr int WK = S::kWk, KR = S::kKr, DW = S::kDw, SX = XT == DT_I8 ? 1 : 2;
  constexpr bool FP = XT != DT_I8, BF16 = XT == DT_BF16;
  constexpr int NB = SHALLOW ? 1 : FP ? (R == 1 && WB == 4 ? 4 : 3) : 2;   // steps in flight per wave, the one being multiplied included

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, h = lane >> 4;
  const int wn = wave % WN, wk = wave / WN;
  const int strip = blockIdx.x, ks = blockIdx.y;
  const int n0 = strip * S::kCols;
  const int pitch = p.n * WB / 8;                         // bytes of a K row
  const long long group_bytes = (long long)p.k * pitch;   // planned only below 2^31
  const __amdgpu_buffer_rsrc_t rw = buffer_over(p.w + (long long)grp * group_bytes, group_bytes);
  const __amdgpu_buffer_rsrc_t rx = buffer_over(static_cast<const char *>(p.x) + (long long)m0 * p.k * SX, (long long)chunk_rows * p.k * SX);
  const int steps = (p.k + S::kStep - 1) / S::kStep;
  const int per_split = (steps + p.split_k - 1) / p.split_k;
  const int s_begin = ks * per_split, s_end = min(steps, s_begin + per_split);

  const int n_lane = n0 + 16 * CPL * wn + CPL * c16;      // N % 16 == 0: a lane's columns are all inside or all outside
  const unsigned w_lane = n_lane < p.n ? (unsigned)(h * KR * pitch + n_lane * WB / 8) : kBufferOob;
  unsigned x_lane[L];
#pragma unroll
  for (int t = 0; t < L; ++t) x_lane[t] = (unsigned)((min(16 * t + c16, chunk_rows - 1) * p.k + h * KR) * SX);

  Acc acc[CPL][L];
#pragma unroll
  for (int j = 0; j < CPL; ++j)
#pragma unroll
    for (int t = 0; t < L; ++t) acc[j][t] = Acc{0, 0, 0, 0};
  v4f rs[L];
#pragma unroll
  for (int t = 0; t < L; ++t) rs[t] = v4f{0.f, 0.f, 0.f, 0.f};
  const unsigned ones = BF16 ? 0x3F803F80u : 0x3C003C00u;
  const v4i ones_frag = v4i{(int)ones, (int)ones, (int)ones, (int)ones};

  int wbuf[NB][KR][DW];
  v4i xbuf[NB][L];
  auto issue = [&](auto b_c, int step) {
    constexpr int B = decltype(b_c)::value;
    // (K % 16 == 0: a lane group's K rows are all inside or all outside; only the vector offset is range-checked)
    const bool ok = step < s_end && step * S::kStep + h * KR < p.k;
    const unsigned wo = ok ? w_lane : kBufferOob;
#pragma unroll
    for (int t = 0; t < L; ++t)
      xbuf[B][t] = __builtin_amdgcn_raw_buffer_load_b128(rx, ok ? x_lane[t] : kBufferOob, (unsigned)(step * S::kStep * SX), 0);
#pragma unroll
    for (int i = 0; i < KR; ++i) load_words<DW>(wbuf[B][i], rw, wo, (unsigned)(step * S::kStep + i) * (unsigned)pitch);
  };
  auto multiply = [&](auto b_c) {
    constexpr int B = decltype(b_c)::value;
    static_for<DW>([&](auto d_c) {
      constexpr int D = decltype(d_c)::value;
      if constexpr (!FP) {
        unsigned c[4][4];   // [row quad][byte column]: four K rows of two columns
#pragma unroll
        for (int g = 0; g < 4; ++g)
          transpose4x4((unsigned)wbuf[B][4 * g][D], (unsigned)wbuf[B][4 * g + 1][D], (unsigned)wbuf[B][4 * g + 2][D],
                       (unsigned)wbuf[B][4 * g + 3][D], c[g][0], c[g][1], c[g][2], c[g][3]);
        static_for<4>([&](auto b4_c) {
          constexpr int Q = decltype(b4_c)::value;
          if constexpr (WB == 8) {
            const v4i f = v4i{(int)c[0][Q], (int)c[1][Q], (int)c[2][Q], (int)c[3][Q]};
#pragma unroll
            for (int t = 0; t < L; ++t) rt_mfma<XT>(acc[4 * D + Q][t], xbuf[B][t], f);
          } else {
            v4i even, odd;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              even[g] = (int)((c[g][Q] << 4) & 0xF0F0F0F0u);
              odd[g] = (int)(c[g][Q] & 0xF0F0F0F0u);
            }
#pragma unroll
            for (int t = 0; t < L; ++t) {
              rt_mfma<XT>(acc[8 * D + 2 * Q][t], xbuf[B][t], even);
              rt_mfma<XT>(acc[8 * D + 2 * Q + 1][t], xbuf[B][t], odd);
            }
          }
        });
      } else if constexpr (WB == 8) {
        static_for<4>([&](auto b4_c) {
          constexpr int Q = decltype(b4_c)::value;
          v4i f;
#pragma unroll
          for (int q = 0; q < 4; ++q) f[q] = byte_pair<BF16, Q>((unsigned)wbuf[B][2 * q][D], (unsigned)wbuf[B][2 * q + 1][D]);
#pragma unroll
          for (int t = 0; t < L; ++t) rt_mfma<XT>(acc[4 * D + Q][t], xbuf[B][t], f);
        });
      } else {
        unsigned odd[8];   // columns 1, 3, 5, 7 of the word in the low halves of the bytes, where 0, 2, 4, 6 are in the word itself
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          odd[i] = (unsigned)wbuf[B][i][D] >> 4;
          asm("" : "+v"(odd[i]));   // (or the shift joins the byte select: one more instruction for each weight)
        }
        static_for<4>([&](auto b4_c) {
          constexpr int Q = decltype(b4_c)::value;
          v4i fe, fo;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            fe[q] = nibble_pair<BF16, Q>((unsigned)wbuf[B][2 * q][D], (unsigned)wbuf[B][2 * q + 1][D]);
            fo[q] = nibble_pair<BF16, Q>(odd[2 * q], odd[2 * q + 1]);
          }
#pragma unroll
          for (int t = 0; t < L; ++t) {
            rt_mfma<XT>(acc[8 * D + 2 * Q][t], xbuf[B][t], fe);
            rt_mfma<XT>(acc[8 * D + 2 * Q + 1][t], xbuf[B][t], fo);
          }
        });
      }
    });
    if constexpr (FP) {
#pragma unroll
      for (int t = 0; t < L; ++t) rt_mfma<XT>(rs[t], xbuf[B][t], ones_frag);
    }
  };
  // Epilogue operands, one column (and one row) per thread: requested here and handed over through LDS behind the loop.  Asked for where
  // they are used, they cost a memory round trip of 1 to 2 us behind the last weight (6 rows over 16 experts, 1568 x 2048, two slices:
  // 4700 of 24000 cycles from the last slice's arrival to the end); int8 x looked its scales and biases up one by one.  us, before -> now: 25 rows
  // over 32 experts, 4064 x 1296, int8 x on 4 bits 28.8 -> 25.4; 120 decode shapes: int8 x on 4 bits 0.88 of the time, 16-bit x 0.975.  Nothing is
  // converted here: that would wait.
  unsigned ep_scale = 0x3F800000u, ep_other = 0u;   // scale: 16 or 32 bits as they are; offset or bias
  float ep_pt = 1.0f;
  {
    const bool in = n0 + tid < p.n;
    if constexpr (FP) {
      const unsigned at = in ? (unsigned)(n0 + tid) * 2u : kBufferOob;
      const long long row = (long long)grp * p.n * 2;
      ep_scale = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(buffer_over(static_cast<const char *>(p.aq_scale) + row, 2ll * p.n), at, 0, 0);
      ep_other = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(buffer_over(static_cast<const char *>(p.aq_offset) + (p.aq_offset ? row : 0), p.aq_offset ? 2ll * p.n : 0), at, 0, 0);
    } else if (in) {
      const long long idx = (p.scale_per_group ? (long long)grp * p.n : 0) + n0 + tid, at = p.scale_is_scalar ? 0 : idx;
      if (p.scale_dtype == DT_F32) ep_scale = reinterpret_cast<const unsigned *>(p.scale)[at];
      else if (p.scale_dtype == DT_BF16) ep_scale = reinterpret_cast<const unsigned short *>(p.scale)[at];
      else if (p.scale_dtype != DT_NONE) ep_scale = reinterpret_cast<const unsigned *>(p.scale)[2 * at];
      if (p.bias) ep_other = (unsigned)p.bias[idx];
    }
    if (!FP && p.per_token && tid < chunk_rows) ep_pt = p.per_token[m0 + tid];
  }
  static_for<NB - 1>([&](auto b_c) { issue(b_c, s_begin + wk + WK * decltype(b_c)::value); });
  for (int s = s_begin + wk; s < s_end; s += NB * WK) {
    static_for<NB>([&](auto b_c) {
      constexpr int B = decltype(b_c)::value;
      issue(std::integral_constant<int, (B + NB - 1) % NB>{}, s + (B + NB - 1) * WK);
      // the requests stay in front of the step they overlap with
      __builtin_amdgcn_sched_barrier(0);
      multiply(b_c);
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // ---- the waves' K parts, added in wave order, 16 rows x 8 word positions at a time ------------------------------------
  constexpr int NT = S::kThreads, NJ = CPL / 8, ITEMS = 4 / WK;   // an item is one row of 8 neighbouring columns
  Elem(*red)[8][4][64] = reinterpret_cast<Elem(*)[8][4][64]>(smem);   // [wave][word position][row of the lane's four][lane]
  float *red_rs = reinterpret_cast<float *>(smem + S::kRed);           // [wave][16 R rows]
  unsigned *s_ticket = reinterpret_cast<unsigned *>(smem + S::kRed + WN * WK * R * 64);
  if constexpr (FP) {
    if (c16 == 0) {
#pragma unroll
      for (int t = 0; t < L; ++t) *reinterpret_cast<v4f *>(red_rs + wave * 16 * R + 16 * t + 4 * h) = rs[t];
    }
  }
  float *s_scale = reinterpret_cast<float *>(smem + S::kEp), *s_pt = s_scale + 2 * S::kCols;
  int *s_other = reinterpret_cast<int *>(s_scale + S::kCols);   // offsets as float32, biases as they are
  if constexpr (FP) {
    s_scale[tid] = BF16 ? __uint_as_float(ep_scale << 16) : f16_bits_to_f32((unsigned short)ep_scale);
    s_other[tid] = __float_as_int(BF16 ? __uint_as_float(ep_other << 16) : f16_bits_to_f32((unsigned short)ep_other));
  } else {
    s_scale[tid] = __uint_as_float(p.scale_dtype == DT_BF16 ? ep_scale << 16 : ep_scale);
    s_other[tid] = (int)ep_other;
    if (tid < 16 * R) s_pt[tid] = ep_pt;
  }
  // item u of this thread: lane position `lane` of wave column iwn, row ir of the lane's four
  auto item_wn = [&](int u) { return (tid + NT * u) >> 8; };
  auto item_row = [&](int u) { return 4 * h + (((tid + NT * u) >> 6) & 3); };

  auto finish = [&](int row, int n, const Elem (&v)[8], float xs) {
    if (n >= p.n) return;
    constexpr int shift = WB == 4 ? 4 : 0;   // int8 x: the operands were 16 times the nibbles, 16-bit x: a sixteenth of them; exact
    float f[8];
    const float *sc = s_scale + (n - n0);
    const int *other = s_other + (n - n0);
    if constexpr (FP) {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = fmaf(__int_as_float(other[j]), xs, v[j] * (float)(1 << shift)) * sc[j];
    } else {
      if (p.out_dtype == DT_I32) {
        int *dst = reinterpret_cast<int *>(p.out) + (long long)(m0 + row) * p.n + n;
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[j] = (v[j] >> shift) + other[j];
        return;
      }
      const float pt = s_pt[row];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = dequant((v[j] >> shift) + other[j], sc[j], pt);
    }
    unsigned q[4];
    activate_n(f, p.act_type);
    pack_half_n(f, p.out_dtype, q);
    *reinterpret_cast<uint4 *>(reinterpret_cast<unsigned short *>(p.out) + (long long)(m0 + row) * p.n + n) = make_uint4(q[0], q[1], q[2], q[3]);
  };

  const long long tile = (long long)blockIdx.z * p.n_strips + strip;
  i64 *base = reinterpret_cast<i64 *>(p.partial) + tile * p.split_k * (long long)S::kSliceWords;
  constexpr int kSums = R * 16 * S::kCols / 2;   // where a slice's row sums start, in words; item (T, J, u) has words ((T NJ + J) ITEMS + u) 4 ..
  static_for<L>([&](auto t_c) {
    constexpr int T = decltype(t_c)::value;
    static_for<NJ>([&](auto j_c) {
      constexpr int J = decltype(j_c)::value;
      if constexpr (T > 0 || J > 0) __syncthreads();   // the block before is read
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][j][r][lane] = acc[8 * J + j][T][r];
      __syncthreads();
#pragma unroll
      for (int u = 0; u < ITEMS; ++u) {
        const int iwn = item_wn(u), row = 16 * T + item_row(u);
        if (row >= chunk_rows) continue;   // (few rows: most of the block is padding that no slice needs to exchange)
        Elem v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          v[j] = red[iwn][j][((tid + NT * u) >> 6) & 3][lane];
#pragma unroll
          for (int w = 1; w < WK; ++w) v[j] += red[w * WN + iwn][j][((tid + NT * u) >> 6) & 3][lane];
        }
        float xs = 0.f;
        if constexpr (FP) {
          xs = red_rs[iwn * 16 * R + row];
#pragma unroll
          for (int w = 1; w < WK; ++w) xs += red_rs[(w * WN + iwn) * 16 * R + row];
        }
        if (p.split_k == 1) {
          finish(row, n0 + 16 * CPL * iwn + CPL * c16 + 8 * J, v, xs);
        } else {
          i64 *mine = base + (long long)ks * S::kSliceWords + ((T * NJ + J) * ITEMS + u) * 4 * NT + tid;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __hip_atomic_store(mine + e * NT, (i64)(((unsigned long long)__builtin_bit_cast(unsigned, v[2 * e + 1]) << 32) | __builtin_bit_cast(unsigned, v[2 * e])),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (FP && J == 0 && c16 == 0 && iwn == 0)
            __hip_atomic_store(reinterpret_cast<float *>(base + (long long)ks * S::kSliceWords + kSums) + row, xs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    });
  });
  if (p.split_k == 1) return;

  // ---- K slices of different workgroups: the last one to arrive adds them in slice order --------------------------------
  publish_partials_and_sync();
  if (tid == 0) *s_ticket = __hip_atomic_fetch_add(&p.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*s_ticket != (unsigned)(p.split_k - 1)) return;
  if (tid == 0) __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll 1
  for (int tu = 0; tu < L * ITEMS; ++tu) {
    const int t = tu / ITEMS, u = tu % ITEMS;
    const int iwn = item_wn(u), row = 16 * t + item_row(u);
    if (row >= chunk_rows) continue;
    Elem v[NJ][8];   // (both pieces of a row are requested together)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[j][e] = 0;
    float xs = 0.f;
    for (int s0 = 0; s0 < p.split_k; s0 += 4) {
      i64 part[4][NJ][4];
      float ps[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const i64 *src = base + (long long)min(s0 + q, p.split_k - 1) * S::kSliceWords;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            part[q][j][e] = __hip_atomic_load(src + (((t * NJ + j) * ITEMS + u) * 4 + e) * NT + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ps[q] = FP ? __hip_atomic_load(reinterpret_cast<const float *>(src + kSums) + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (s0 + q < p.split_k) {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[j][2 * e] += __builtin_bit_cast(Elem, (unsigned)(unsigned long long)part[q][j][e]);
              v[j][2 * e + 1] += __builtin_bit_cast(Elem, (unsigned)((unsigned long long)part[q][j][e] >> 32));
            }
          xs += ps[q];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) finish(row, n0 + 16 * CPL * iwn + CPL * c16 + 8 * j, v[j], xs);
  }
}

template <int XT, int WB, int R, int CPL, int WN, bool SHALLOW>
__global__ void __launch_bounds__(64 * WN * CPL / 4, SHALLOW ? 4 : 2) gmm_regt_kernel(const GmmParams p) {
  extern __shared__ __align__(16) unsigned char rt_smem[];
  const int lane = threadIdx.x & 63;
  // (grid.z enumerates the chunks that hold rows, group after group: a slot past the last one has nothing to do)
  int grp, mc, g_start, g_end;
  if (!chunk_of_slot(p, (int)blockIdx.z, 16 * R, lane, grp, mc, g_start, g_end)) return;
  const int m0 = g_start + mc * 16 * R;
  const int chunk_rows = min(16 * R, g_end - m0);
  const int live = (chunk_rows + 15) / 16;
  bool done = false;
  static_for<R>([&](auto i_c) {   // one copy of the loop per number of live row blocks
    constexpr int L = decltype(i_c)::value + 1;
    if (!done && live <= L) {
      regt_run<XT, WB, R, CPL, WN, SHALLOW, L>(p, rt_smem, grp, m0, chunk_rows);
      done = true;
    }
  });
}

namespace {
template <int XT, int WB, int R, int CPL, int WN, bool SHALLOW = false>
hipError_t regt_launch(const GmmParams &p, hipStream_t stream) {
  using S = RtShape<XT, WB, R, CPL, WN>;
  auto kern = gmm_regt_kernel<XT, WB, R, CPL, WN, SHALLOW>;
  static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race between first launches repeats it at worst
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  if (p.n_strips != (p.n + S::kCols - 1) / S::kCols) return hipErrorInvalidValue;
  const dim3 grid((unsigned)p.n_strips, (unsigned)p.split_k, chunk_slots(p, 16 * R));
  if (grid.y > 65535u || grid.z > 65535u) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kern, grid, dim3(S::kThreads), S::kLds, stream, p);
  return hipGetLastError();
}
template <int XT, int WB, int WN>
hipError_t regt_dispatch(const GmmParams &p, int row_blocks, bool shallow, hipStream_t stream) {
  if constexpr (XT != DT_I8 && WB == 8) {
    if (row_blocks == 1 && shallow) return regt_launch<XT, WB, 1, 16, WN, true>(p, stream);
  }
  if (shallow) return hipErrorInvalidValue;
  if constexpr (XT == DT_I8 || WB == 4 || WN == 1) {   // (16-bit x on 8-bit weights: strips of 512 columns are always shallow)
    if (row_blocks == 1) return regt_launch<XT, WB, 1, 16, WN>(p, stream);
  }
  if constexpr (WB == 4) {   // (8-bit weights of more than 16 rows per group have LDS kernels of their own)
    if (row_blocks == 2) return regt_launch<XT, WB, 2, 16, WN>(p, stream);
  }
  return hipErrorInvalidValue;
}
template <int XT, int WB>
hipError_t regt_by_strip(const GmmParams &p, int row_blocks, int strip_cols, bool shallow, hipStream_t stream) {
  if (strip_cols == 256) return regt_dispatch<XT, WB, 1>(p, row_blocks, shallow, stream);
  if (strip_cols == 512) return regt_dispatch<XT, WB, 2>(p, row_blocks, shallow, stream);
  return hipErrorInvalidValue;
}
}  // namespace

size_t regt_slice_bytes(int row_blocks, int strip_cols) { return (size_t)row_blocks * (16 * strip_cols / 2 + 8) * 8; }

// row_blocks = 16-row blocks per chunk (1 or 2), strip_cols = columns per strip (256 or 512), shallow: 16-bit x on 8-bit weights only.
// The plan takes int8 x on 4-bit weights with 16-row chunks only and int8 x on 8-bit weights never: those forms run under
// kernel_override (the tests compare them with the oracle).
hipError_t launch_regt(const GmmParams &p, int weight_bits, int row_blocks, int strip_cols, bool shallow, hipStream_t stream) {
  if (p.m == 0) return hipSuccess;
  if (p.k % 16 != 0 || p.n % 16 != 0) return hipErrorInvalidValue;
  if (weight_bits == 4) {
    if (p.x_dtype == DT_I8) return regt_by_strip<DT_I8, 4>(p, row_blocks, strip_cols, shallow, stream);
    if (p.x_dtype == DT_BF16) return regt_by_strip<DT_BF16, 4>(p, row_blocks, strip_cols, shallow, stream);
    return regt_by_strip<DT_F16, 4>(p, row_blocks, strip_cols, shallow, stream);
  }
  if (p.x_dtype == DT_I8) return regt_by_strip<DT_I8, 8>(p, row_blocks, strip_cols, shallow, stream);
  if (p.x_dtype == DT_BF16) return regt_by_strip<DT_BF16, 8>(p, row_blocks, strip_cols, shallow, stream);
  return regt_by_strip<DT_F16, 8>(p, row_blocks, strip_cols, shallow, stream);
}

}  // namespace msco
