// Grouped weight-only matmul (16-bit x, 8-bit weights) for groups of a few dozen rows and more (gfx950): packed or row-major
// [E,K,N] weights go from memory into registers, are converted there once and meet up to 128 rows of x from LDS.
//
// The matrix pipe wants a 16 x 16 x 32 MFMA every 16 cycles from every SIMD.  What stands in its way is the conversion (one
// and a half vector instructions per weight: a converted weight has to meet as many rows as possible), the x rows (every
// wave needs all of them) and, with one wave per SIMD, the wave's own issue rate.  Hence:
//
//   * workgroup (8 waves, two per SIMD) = one chunk of at most 128 rows of one group x a strip of 512 columns x all of K;
//     wave w owns columns 64 w .. 64 w + 63 and all rows: 8 x 4 blocks of 16 x 16 in 128 registers.  No weight passes
//     through LDS and none is converted twice in a workgroup: 6 vector instructions per 4 MFMAs, behind which the SIMD's other wave multiplies.
//     Per K position 256 bytes of x and 512 of weights for 64 cycles of MFMAs per SIMD: 24 bytes per cycle and CU where
//     256-column strips would need 32 (L2 delivers 28).
//   * packed weights: lane (c, h) of a 1 KiB block holds K bytes 16 h .. 16 h + 15 of column c, the operands of two MFMAs.
//     [E,K,N]: a lane requests four neighbouring columns of its 16 K rows; column j of two rows is converted and packed by
//     the same instructions (byte select), so the turn costs nothing.  The output column of MFMA column c of word position j
//     then is 4 c + j.
//   * the weights are the MFMA's first operand: a lane ends up with neighbouring columns of one row ([E,K,N]: 16; packed: 8,
//     once two lane rows have changed places), stored straight from the accumulators.
//   * x goes straight into a ring of LDS stages of 64 K positions (128 bytes) per row; 16-byte piece q of row r sits at piece
//     q ^ ((r >> 1) & 7): fragment reads meet 16 different bank groups.  One barrier per stage.  Weights and x are requested
//     two K blocks ahead and more (requests complete in order: one K block ahead, x through registers, 480 against 435 us).
//   * 16 x 16 x 32 MFMAs rather than 32 x 32 x 16: alone a tile takes 105 against 94 us with the same loop, on all CUs, where the
//     power limit sets the clock, 118 against 131 us.
//   * a group's rows are cut into equal chunks of whole 16-row blocks, and the K loop exists once per number of blocks: 530
//     rows cost the MFMAs of 544, not of 640 (128-row chunks) or 768.
//   * the antiquant offset needs the row sums of x: every wave sums one block of rows from LDS with v_dot2 against ones.
//       out = s * (sum_k x w + o sum_k x)
//   * dispatch: (group, strip) pairs are dealt to the XCDs in turn and all chunks of a pair run on the same one, one after
//     the other: a weight strip comes into one L2 once.
//
// What bounds it (4096 x 4096 x 11008, three rounds of tiles): 327 us = 1.13 PFLOP/s.  Per 64 K positions and round 1.38 us, of which
// the MFMAs alone 0.94 (2048 cycles), fragment reads 0.05, conversions 0.17, operand requests 0.22; and 21 .. 25 us per round that do not
// depend on K (first requests, epilogue, stores in step on all CUs).  Two workgroups of four waves x 256 columns per CU
// overlap those but request x twice: 349 us.  The barrier in the middle of a block with the fragment reads running on: the same.
#include "gmm_common.h"
#include "gmm_kernels.h"

namespace msco {

namespace {
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr int XA_RB = 8;                       // 16-row blocks per chunk at most
constexpr int XA_ROWS = 16 * XA_RB;
constexpr int XA_WAVES = 8;
constexpr int XA_THREADS = 64 * XA_WAVES;
constexpr int XA_COLS = 64 * XA_WAVES;         // one thread per column (scales and offsets)
constexpr int XA_STAGES = 48 * 1024;           // bytes of x stages: 3 of 128 rows, 4 or 6 of 64

// Signed bytes B0 and B1 of two words -> two 16-bit floating-point values, exact.
//   bf16: a conversion with byte select each and one pack.  (The bytes + 128 as float32 denormals times 2^127, which needs no
//         conversion but the xor and the 128 taken out of the sums again: 8 x 512 rows on [E,K,N] 482 against 456 us.)
//   f16:  0x6400 | (b + 128) is 1152 + b: one byte shuffle, one or and one packed addition for both.
template <bool BF16, int B0, int B1>
__device__ __forceinline__ int xa_pair(unsigned w0, unsigned w1) {
  if constexpr (BF16) {
    const float f0 = (float)(int)(signed char)(w0 >> (8 * B0)), f1 = (float)(int)(signed char)(w1 >> (8 * B1));
    return (int)perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
  } else {
    const unsigned bytes = perm(w1, w0, 0x0C000C00u | ((4u + B1) << 16) | B0) ^ 0x64806480u;
    return __builtin_bit_cast(int, __builtin_bit_cast(v2h, bytes) + v2h{(_Float16)-1152.0f, (_Float16)-1152.0f});
  }
}

// acc += a x b in the registers of acc (left to the compiler, accumulator blocks move between the unrolled K blocks, and the
// 128-row form runs out of registers).  The compiler does not see a matrix instruction here: no vector instruction may write a
// or b in the two cycles in front of it (xa_settle) or read acc behind it before the pipe has drained (xa_drain).
template <bool BF16>
__device__ __forceinline__ void xa_mfma(v4f &acc, const v4i &a, const v4i &b) {
  if constexpr (BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void xa_settle() { asm volatile("s_nop 3" ::: "memory"); }
__device__ __forceinline__ void xa_drain() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

template <bool BF16>
__device__ __forceinline__ float xa_half(unsigned bits) {
  return BF16 ? bf16_bits_to_f32((unsigned short)bits) : f16_bits_to_f32((unsigned short)bits);
}

// c + the two values of a word, products with one in float32
template <bool BF16>
__device__ __forceinline__ float xa_add2(int v, float c) {
  typedef __bf16 v2b __attribute__((ext_vector_type(2)));
  if constexpr (BF16) return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2b, v), __builtin_bit_cast(v2b, 0x3F803F80), c, false);
  else return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, v), __builtin_bit_cast(v2h, 0x3C003C00), c, false);
}

// 16 bytes per lane from a buffer straight into LDS: lane l writes lds + 16 l.  (The address-space cast only exists in the device pass.)
__device__ __forceinline__ void xa_load_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char *lds, unsigned voffset, unsigned soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (void __attribute__((address_space(3))) *)(lds), 16, voffset, soffset, 0, 0);
#else
  (void)rsrc; (void)lds; (void)voffset; (void)soffset;
#endif
}

}  // namespace

// RB = 16-row blocks of the chunk
template <bool BF16, bool KN, int RB>
__device__ __forceinline__ void rows_a16w8_run(const GmmParams &p, unsigned char *smem, int grp, int strip, int m0, int chunk_rows) {
  constexpr int DEPTH = RB <= 2 ? 6 : RB <= 4 ? 4 : 3;   // register sets for the weights of a K block; x stages
  constexpr int XP = (2 * RB + XA_WAVES - 1) / XA_WAVES;   // LDS-direct requests of a stage per wave (8 XA_WAVES rows per pass)
  constexpr int STAGE = XP * XA_WAVES * 1024;                 // bytes of an x stage
  constexpr int AHEAD = RB >= 7 ? 2 : 3;   // x fragments requested from LDS ahead of their MFMAs
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, h = lane >> 4;
  const int k_blocks = (p.k + 63) / 64, col_groups = p.n / 16;
  const int n_wave = strip * XA_COLS + 64 * wave;

  // ---- weights: a wave's four blocks of 16 columns x 64 K bytes, 16 registers per lane and K block.  Packed: one descriptor
  // per column group over exactly its K blocks; [E,K,N]: one over the expert's matrix, a lane outside N x K out of its range.
  // (K % 16 == 0: a lane's 16 K rows are all inside or all outside; only the vector offset is range-checked)
  const long long group_bytes = KN ? (long long)p.k * p.n : (long long)col_groups * k_blocks * 1024;
  __amdgpu_buffer_rsrc_t rw[4];
  if constexpr (KN) {
    rw[0] = buffer_over(p.w + (long long)grp * group_bytes, group_bytes);
  } else {
#pragma unroll
    for (int cg = 0; cg < 4; ++cg) {
      const int g = n_wave / 16 + cg;
      rw[cg] = buffer_over(p.w + (long long)grp * group_bytes + (long long)min(g, col_groups - 1) * k_blocks * 1024, g < col_groups ? (long long)k_blocks * 1024 : 0);
    }
  }
  const unsigned w_lane = KN ? (n_wave + 4 * c16 < p.n ? (unsigned)(16 * h) * (unsigned)p.n + (unsigned)(n_wave + 4 * c16) : kBufferOob) : (unsigned)lane * 16u;
  int raw[DEPTH][4][4];   // packed: [column group][dword]; [E,K,N]: K row 4 i + j in [i][j]
  constexpr int WL = KN ? 16 : 4;   // requests per K block
  auto wload1 = [&](auto set_c, auto i_c, int kb) {
    constexpr int SET = decltype(set_c)::value, I = decltype(i_c)::value;
    if constexpr (KN) {
      const unsigned vo = 64 * kb + 16 * h < p.k ? w_lane : kBufferOob;
      raw[SET][I / 4][I % 4] = (int)__builtin_amdgcn_raw_buffer_load_b32(rw[0], vo, (unsigned)(64 * kb + I) * (unsigned)p.n, 0);
    } else {
      const v4i v = __builtin_amdgcn_raw_buffer_load_b128(rw[I], (unsigned)kb * 1024u + w_lane, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) raw[SET][I][i] = v[i];
    }
  };
  // sixteenth I of the operands of K half HALF (K positions 16 h + 8 HALF .. + 7 of the block): word D for the wave's J-th 16
  // columns, in the order that frees the weights' registers soonest
  auto convert = [&](auto set_c, auto half_c, auto i_c, v4i (&f)[4]) {
    constexpr int SET = decltype(set_c)::value, HALF = decltype(half_c)::value, I = decltype(i_c)::value;
    constexpr int J = KN ? I % 4 : I / 4, D = KN ? I / 4 : I % 4;
    if constexpr (KN) {
      constexpr int R = 8 * HALF + 2 * D;
      f[J][D] = xa_pair<BF16, J, J>((unsigned)raw[SET][R / 4][R % 4], (unsigned)raw[SET][(R + 1) / 4][(R + 1) % 4]);
    } else {
      constexpr int W = 2 * HALF + D / 2;
      f[J][D] = xa_pair<BF16, 2 * (D % 2), 2 * (D % 2) + 1>((unsigned)raw[SET][J][W], (unsigned)raw[SET][J][W]);
    }
  };

  // ---- x: straight into LDS; request u of wave w brings rows 8 (XA_WAVES u + w) .. + 7 of a stage, lane l piece (l % 8) ^ swizzle of row
  // l / 8.  Rows past the chunk and K positions past K arrive as zeros.
  const __amdgpu_buffer_rsrc_t rx = buffer_over(static_cast<const char *>(p.x) + 2ll * m0 * p.k, 2ll * chunk_rows * p.k);
  const int xrow = 8 * wave + (lane >> 3), xpiece = (lane & 7) ^ ((xrow >> 1) & 7);
  const unsigned x_voff = 2u * (unsigned)xrow * (unsigned)p.k + 16u * (unsigned)xpiece;
  auto xload = [&](int stage, int kb) {
    const unsigned vo = 64 * kb + 8 * xpiece < p.k ? x_voff : kBufferOob;
#pragma unroll
    for (int u = 0; u < XP; ++u)   // (128 rows of K: below 2^31 bytes by the plan, so the out-of-range mark survives the addition)
      xa_load_lds(rx, smem + stage * STAGE + (u * XA_WAVES + wave) * 1024, vo + (unsigned)(u * XA_WAVES * 16) * (unsigned)p.k, (unsigned)kb * 128u);
  };
  // fragment reads: lane (c16, h) takes piece 2 h + HALF of row c16; the sums of row blocks wave, wave + XA_WAVES are kept by this wave
  constexpr int SB = (RB + XA_WAVES - 1) / XA_WAVES;
  float x_sum[SB];
#pragma unroll
  for (int i = 0; i < SB; ++i) x_sum[i] = 0.f;
  const int swz = (c16 >> 1) & 7;
  const unsigned char *xr[2] = {smem + c16 * 128 + (((2 * h) ^ swz) << 4), smem + c16 * 128 + (((2 * h + 1) ^ swz) << 4)};

  // antiquant scale and offset of column strip XA_COLS + tid, one half each of a register until the epilogue
  unsigned scale_offset = BF16 ? 0x3F80u : 0x3C00u;
  if (strip * XA_COLS + tid < p.n) {
    const long long idx = (long long)grp * p.n + strip * XA_COLS + tid;
    if (p.aq_scale) scale_offset = reinterpret_cast<const unsigned short *>(p.aq_scale)[idx];
    if (p.aq_offset) scale_offset |= (unsigned)reinterpret_cast<const unsigned short *>(p.aq_offset)[idx] << 16;
  }
  v4f acc[4][RB];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[j][rb] = v4f{0.f, 0.f, 0.f, 0.f};

  v4i wf[2][4];
  // Requests complete in order, and a step makes the same ones in the same order: x of K block kb + DEPTH - 1, weights of
  // kb + DEPTH.  A stage may be read once no more than those issued behind its request are outstanding.
  constexpr int YOUNGER = WL + (DEPTH - 2) * (XP + WL);
  auto stage_barrier = [] { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER < 63 ? YOUNGER : 63) : "memory"); };
  static_for<DEPTH>([&](auto s_c) {
    constexpr int B = decltype(s_c)::value;
    if constexpr (B > 0) xload(B - 1, B - 1);
    __builtin_amdgcn_sched_barrier(0);
    static_for<WL>([&](auto i_c) { wload1(s_c, i_c, B); });
    __builtin_amdgcn_sched_barrier(0);
  });
  static_for<16>([&](auto i_c) { convert(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, i_c, wf[0]); });

  // K block kb: x in stage kb % DEPTH, weights in register set kb % DEPTH
  auto step = [&](auto s_c, int kb) {
    constexpr int J = decltype(s_c)::value;
    stage_barrier();   // block kb is in its stage; every wave is done with block kb - 1's
    xload((J + DEPTH - 1) % DEPTH, kb + DEPTH - 1);
    __builtin_amdgcn_sched_barrier(0);
    auto frag = [&](int i) { return *reinterpret_cast<const v4i *>(xr[i >= RB] + J * STAGE + (i % RB) * 16 * 128); };
    v4i fq[AHEAD + 1];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fq[i] = frag(i < 2 * RB ? i : 0);
    static_for<2>([&](auto half_c) {
      constexpr int HALF = decltype(half_c)::value;
      xa_settle();
      v4i sf[SB];
      static_for<RB>([&](auto r_c) {
        constexpr int R = decltype(r_c)::value, I = HALF * RB + R;
        if constexpr (I + AHEAD < 2 * RB) fq[(I + AHEAD) % (AHEAD + 1)] = frag(I + AHEAD);
        if constexpr (R == RB - 1) {
#pragma unroll
          for (int i = 0; i < SB; ++i) sf[i] = *reinterpret_cast<const v4i *>(xr[HALF] + J * STAGE + min(wave + i * XA_WAVES, RB - 1) * 16 * 128);
        }
        // the operands of the next half (of the next block's first one) are converted while this half is multiplied
        constexpr int C0 = 16 * R / RB, C1 = 16 * (R + 1) / RB;
        static_for<C1 - C0>([&](auto c_c) {
          constexpr int C = C0 + decltype(c_c)::value;
          convert(std::integral_constant<int, HALF == 0 ? J : (J + 1) % DEPTH>{}, std::integral_constant<int, 1 - HALF>{}, std::integral_constant<int, C>{}, wf[1 - HALF]);
        });
        // (block kb is converted by now: its registers take block kb + DEPTH, a few requests at a time)
        constexpr int L0 = HALF * WL * R / RB, L1 = HALF * WL * (R + 1) / RB;
        static_for<L1 - L0>([&](auto l_c) { wload1(std::integral_constant<int, J>{}, std::integral_constant<int, L0 + decltype(l_c)::value>{}, kb + DEPTH); });
#pragma unroll
        for (int j = 0; j < 4; ++j) xa_mfma<BF16>(acc[j][R], wf[HALF][j], fq[I % (AHEAD + 1)]);
        // (one fragment read and the conversions it covers per four MFMAs: moved further forward they need more registers)
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int i = 0; i < SB; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) x_sum[i] = xa_add2<BF16>(sf[i][d], x_sum[i]);
    });
  };
  // (whole rounds: blocks past K multiply zeros)
  for (int kb = 0; kb < k_blocks; kb += DEPTH)
    static_for<DEPTH>([&](auto s_c) { step(s_c, kb + decltype(s_c)::value); });

  // ---- epilogue
  xa_drain();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // nothing lands in the stages or reads them any more
  float *s_sum = reinterpret_cast<float *>(smem), *s_scale = s_sum + XA_ROWS, *s_offset = s_scale + XA_COLS;
  s_scale[tid] = xa_half<BF16>(scale_offset & 0xFFFFu);
  s_offset[tid] = xa_half<BF16>(scale_offset >> 16);
#pragma unroll
  for (int i = 0; i < SB; ++i) {
    float v = x_sum[i];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (wave + i * XA_WAVES < RB && h == 0) s_sum[16 * (wave + i * XA_WAVES) + c16] = v;
  }
  __syncthreads();
  // out = s * (sum_k x w + o sum_k x)
  constexpr int NV = KN ? 16 : 8, NG = KN ? 1 : 2;   // neighbouring columns per lane, and groups of them
  auto finish = [&](auto act_c) {
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    // packed: column groups 2 g and 2 g + 1; once the lane rows have been swapped, h & 1 says which and h >> 1 which half of it
    const int n = KN ? n_wave + 16 * h : n_wave + 16 * (2 * g + (h & 1)) + 8 * (h >> 1);
    const bool live = n < p.n;   // N % 16 == 0: all NV inside or all outside
    float sc[NV], of[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      sc[v] = s_scale[n - strip * XA_COLS + v];
      of[v] = s_offset[n - strip * XA_COLS + v];
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int row = 16 * rb + c16;
      const float xs_row = s_sum[row];
      float a[NV];
      if constexpr (KN) {
#pragma unroll
        for (int v = 0; v < NV; ++v) a[v] = acc[v % 4][rb][v / 4];
      } else {
        // rows 1 and 3 of 16 lanes of the first group change places with rows 0 and 2 of the second one
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[2 * g][rb][v]), __float_as_uint(acc[2 * g + 1][rb][v]), false, false);
          a[v] = __uint_as_float(t[0]);
          a[4 + v] = __uint_as_float(t[1]);
        }
      }
      if (live && row < chunk_rows) {
        unsigned q[NV / 2];
#pragma unroll
        for (int v = 0; v < NV; ++v) a[v] = fmaf(of[v], xs_row, a[v]) * sc[v];
        if constexpr (decltype(act_c)::value) activate_n(a, p.act_type);
        pack_half_n(a, BF16 ? DT_BF16 : DT_F16, q);
        uint4 *dst = reinterpret_cast<uint4 *>(reinterpret_cast<unsigned short *>(p.out) + (long long)(m0 + row) * p.n + n);
#pragma unroll
        for (int i = 0; i < NV / 8; ++i) dst[i] = uint4{q[4 * i], q[4 * i + 1], q[4 * i + 2], q[4 * i + 3]};
      }
    }
  }
  };
  if (p.act_type == ACT_NONE) finish(std::false_type{});
  else finish(std::true_type{});
}

template <bool BF16, bool KN>
__global__ void __launch_bounds__(XA_THREADS, 2) gmm_a16w8_rows128_kernel(const GmmParams p) {
  __shared__ __align__(16) unsigned char smem[XA_STAGES];
  const int lane = threadIdx.x & 63;
  int grp, strip, m0, chunk_rows;
  if (!chunk_of_xcd_slot(p, XA_ROWS, (int)blockIdx.x, lane, grp, strip, m0, chunk_rows)) return;
  const int rb = (chunk_rows + 15) / 16;
  bool done = false;
  static_for<XA_RB>([&](auto i_c) {   // one copy of the K loop per number of 16-row blocks
    constexpr int RB = decltype(i_c)::value + 1;
    if (!done && rb == RB) {
      rows_a16w8_run<BF16, KN, RB>(p, smem, grp, strip, m0, chunk_rows);
      done = true;
    }
  });
}

// packed or [E,K,N] weights; K % 16 == 0, N % 16 == 0, K < 2^22 (an out-of-range mark plus the offset of a chunk's last row, 256 K
// bytes, stays a 32-bit offset out of range) and one group's weights below 2^31 bytes; M is not bounded by offsets
hipError_t launch_rows_a16w8(const GmmParams &p_in, bool packed, hipStream_t stream) {
  if (p_in.m == 0) return hipSuccess;
  if (p_in.k % 16 != 0 || p_in.n % 16 != 0 || p_in.k >= (1 << 22) || p_in.split_k != 1) return hipErrorInvalidValue;
  GmmParams p = p_in;
  p.n_strips = (p.n + XA_COLS - 1) / XA_COLS;
  const long long grid = xcd_slots(p, XA_ROWS);
  if (grid > 0x7FFFFFFFll) return hipErrorInvalidValue;
  const bool bf = p.x_dtype == DT_BF16;
  auto kern = bf ? (packed ? gmm_a16w8_rows128_kernel<true, false> : gmm_a16w8_rows128_kernel<true, true>)
                 : (packed ? gmm_a16w8_rows128_kernel<false, false> : gmm_a16w8_rows128_kernel<false, true>);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(XA_THREADS), 0, stream, p);
  return hipGetLastError();
}

}  // namespace msco
