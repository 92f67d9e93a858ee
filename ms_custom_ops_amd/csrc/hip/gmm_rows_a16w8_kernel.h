// Grouped weight-only matmul (16-bit x, 8-bit weights, or 4-bit ones as [E,K,N]) for groups of a few dozen rows and more (gfx950): packed or row-major
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
//     4-bit [E,K,N]: two bytes hold the lane's four columns of a row; a word holds two rows.  bfloat16 x: one conversion of a
//     signed 4-bit number each, at a sixteenth of its value (products and sums stay exact where they are subnormal, and none is
//     infinite that the numbers themselves keep finite; bytes at 16 times the value lost the sums above 2^124 and took 1.01 of
//     the time, nibbles taken out one by one at their value 1.06).  float16 x: four instructions make signed bytes of two rows,
//     at 16 times their value (exact, and float16 products are far from the end of float32).  The epilogue takes the factor out.
//     Bit for bit what the int8 copy of the weights gives, without the launch that writes it (1.5 bytes per weight) and the
//     second byte of every later read.
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
//   * narrower forms where strips of 512 do not fill N or the chip (the rule is with the plan): strips of 256 columns, either
//     four waves and two workgroups per CU, or two sets of four waves that take turns at the K blocks and add their sums through
//     LDS, each finishing half of the rows.  A wave alone on its SIMD takes 1630 cycles per K block of 96 rows whose MFMAs take
//     768 (it issues an instruction every six cycles or so); two sets hide that under one another's where there is one
//     workgroup per CU.  Both forms can split K over workgroups; the last slice to arrive adds all in slice order.
//   * dispatch: (group, strip) pairs are dealt to the XCDs in turn and all chunks of a pair run on the same one, one after
//     the other: a weight strip comes into one L2 once.
//
// What bounds it (4096 x 4096 x 11008, three rounds of tiles): 327 us = 1.13 PFLOP/s before the epilogue's
// branches went (8 x 512 rows, 4096 x 14336: 456 -> 437 us with them gone).  Per 64 K positions and round 1.38 us, of which
// the MFMAs alone 0.94 (2048 cycles), fragment reads 0.05, conversions 0.17, operand requests 0.22; and 21 .. 25 us per round that do not
// depend on K (first requests, epilogue, stores in step on all CUs).  Two workgroups of four waves x 256 columns per CU
// overlap those but request x twice: 349 us.  The barrier in the middle of a block with the fragment reads running on: the same.
#ifndef MSCO_GMM_ROWS_A16W8_KERNEL_H_
#define MSCO_GMM_ROWS_A16W8_KERNEL_H_

#include "gmm_common.h"
#include "gmm_kernels.h"

namespace msco {

namespace {
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr int XA_RB = 8;                       // 16-row blocks per chunk at most
constexpr int XA_ROWS = 16 * XA_RB;
constexpr int XA_STAGES = 48 * 1024;           // bytes of x stages of a wave set: 3 of 128 rows, 4 or 6 of 64
constexpr int XA_MERGE = 2 * 4 * 4 * 4 * 1024; // two wave sets: the accumulators each parks for the other, 4 waves x 16 blocks of 1 KiB
constexpr int XA_SUMS = XA_MERGE + 4 * 2 * 256;   // ... behind them the row sums of set 1, then the epilogue's vectors
constexpr int xa_lds(int sets) { return sets == 1 ? XA_STAGES : XA_SUMS + (XA_ROWS + 2 * 256) * 4; }
constexpr int XA_SLICE_WORDS = 8 * XA_RB + 1;  // 64-bit words per thread of a K slice's partial tile: accumulators, row sums

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

// Signed 4-bit numbers in the low halves of bytes B0 and B1 -> two bfloat16 values, a sixteenth of the numbers, exact.
template <int B0, int B1>
__device__ __forceinline__ int xa_nibble_pair(unsigned w) {
  const float f0 = __builtin_amdgcn_cvt_off_f32_i4((int)(w >> (8 * B0) & 0xFFu)), f1 = __builtin_amdgcn_cvt_off_f32_i4((int)(w >> (8 * B1) & 0xFFu));
  return (int)perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
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

// RB = 16-row blocks of the chunk; NW = waves side by side, 64 columns each; KS = sets of them that take turns at the K blocks;
// tile = number of the (chunk, strip) pair
template <bool BF16, bool KN, bool W4, int RB, int NW, int KS>
__device__ __forceinline__ void rows_a16w8_run(const GmmParams &p, unsigned char *smem, int grp, int strip, int m0, int chunk_rows, long long tile) {
  static_assert(KN || !W4);
  constexpr bool SPLIT = NW == 4;   // (wide strips are planned where they fill the chip)
  constexpr int XA_WAVES = NW, XA_COLS = 64 * NW;
  constexpr int DEPTH = RB <= 2 ? 6 : RB <= 4 ? 4 : 3;   // register sets for the weights of a K block; x stages
  constexpr int XP = (2 * RB + XA_WAVES - 1) / XA_WAVES;   // LDS-direct requests of a stage per wave (8 XA_WAVES rows per pass)
  constexpr int STAGE = XP * XA_WAVES * 1024;                 // bytes of an x stage
  constexpr int AHEAD = RB >= 7 ? 2 : 3;   // x fragments requested from LDS ahead of their MFMAs
  constexpr int H0 = KS == 1 ? RB : (RB + 1) / 2;          // row blocks that set 0 finishes
  const int set = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / (64 * NW)), tid = (int)threadIdx.x - 64 * NW * set;   // thread of the set: one per column
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char *stages = smem + set * XA_STAGES;
  const int c16 = lane & 15, h = lane >> 4;
  const int k_blocks = (p.k + 63) / 64, col_groups = p.n / 16;
  const int n_wave = strip * XA_COLS + 64 * wave;
  // K slice of this workgroup: whole 64-position blocks, everything past its end reads as zeros
  const int per_slice = (k_blocks + p.split_k - 1) / p.split_k, slice = (int)blockIdx.y;
  const int kb_begin = min(slice * per_slice, k_blocks), kb_end = min(kb_begin + per_slice, k_blocks), k_end = min(p.k, 64 * kb_end);
  const int kb_first = kb_begin + set;   // this set takes blocks kb_first, kb_first + KS, ..

  // ---- weights: a wave's four blocks of 16 columns x 64 K bytes, 16 registers per lane and K block.  Packed: one descriptor
  // per column group over exactly its K blocks; [E,K,N]: one over the expert's matrix, a lane outside N x K out of its range.
  // (K % 16 == 0: a lane's 16 K rows are all inside or all outside; only the vector offset is range-checked)
  const unsigned row_bytes = W4 ? (unsigned)p.n / 2 : (unsigned)p.n;   // [E,K,N]
  const long long group_bytes = KN ? (long long)p.k * row_bytes : (long long)col_groups * k_blocks * 1024;
  __amdgpu_buffer_rsrc_t rw[4];
  if constexpr (KN) {
    rw[0] = buffer_over(p.w + (long long)grp * group_bytes, group_bytes);
  } else {
#pragma unroll
    for (int cg = 0; cg < 4; ++cg) {
      const int g = n_wave / 16 + cg;
      rw[cg] = buffer_over(p.w + (long long)grp * group_bytes + (long long)min(g, col_groups - 1) * k_blocks * 1024, g < col_groups ? (long long)kb_end * 1024 : 0);
    }
  }
  const unsigned w_lane = KN ? (n_wave + 4 * c16 < p.n ? (unsigned)(16 * h) * row_bytes + (unsigned)(n_wave + 4 * c16) / (W4 ? 2 : 1) : kBufferOob) : (unsigned)lane * 16u;
  int raw[DEPTH][4][4];   // packed: [column group][dword]; [E,K,N]: K row 4 i + j in [i][j]
  constexpr int WL = KN ? 16 : 4;   // requests per K block
  auto wload1 = [&](auto set_c, auto i_c, int kb) {
    constexpr int SET = decltype(set_c)::value, I = decltype(i_c)::value;
    if constexpr (KN) {
      const unsigned vo = 64 * kb + 16 * h < k_end ? w_lane : kBufferOob;
      const unsigned so = (unsigned)(64 * kb + I) * row_bytes;
      if constexpr (W4) raw[SET][I / 4][I % 4] = (int)__builtin_amdgcn_raw_buffer_load_b16(rw[0], vo, so, 0);
      else raw[SET][I / 4][I % 4] = (int)__builtin_amdgcn_raw_buffer_load_b32(rw[0], vo, so, 0);
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
      if constexpr (W4) {
        // four columns of two rows in one word: the even columns in the low halves of its bytes, the odd ones in the high halves
        int &even = raw[SET][R / 4][R % 4], &odd = raw[SET][(R + 1) / 4][(R + 1) % 4];
        if constexpr (J == 0) {
          const unsigned both = (unsigned)even | (unsigned)odd << 16;
          if constexpr (BF16) {          // (the conversion looks at the low half of a byte alone)
            even = (int)both;
            odd = (int)(both >> 4);
            asm("" : "+v"(odd));         // (or the shift joins the byte select: one more instruction for each weight)
          } else {                       // 16 times their values as signed bytes
            even = (int)((both << 4) & 0xF0F0F0F0u);
            odd = (int)(both & 0xF0F0F0F0u);
          }
        }
        const unsigned w = (unsigned)(J % 2 == 0 ? even : odd);
        if constexpr (BF16) f[J][D] = xa_nibble_pair<J / 2, 2 + J / 2>(w);
        else f[J][D] = xa_pair<false, J / 2, 2 + J / 2>(w, w);
      } else f[J][D] = xa_pair<BF16, J, J>((unsigned)raw[SET][R / 4][R % 4], (unsigned)raw[SET][(R + 1) / 4][(R + 1) % 4]);
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
    const unsigned vo = 64 * kb + 8 * xpiece < k_end ? x_voff : kBufferOob;
#pragma unroll
    for (int u = 0; u < XP; ++u)   // (128 rows of K: below 2^31 bytes by the plan, so the out-of-range mark survives the addition)
      xa_load_lds(rx, stages + stage * STAGE + (u * XA_WAVES + wave) * 1024, vo + (unsigned)(u * XA_WAVES * 16) * (unsigned)p.k, (unsigned)kb * 128u);
  };
  // fragment reads: lane (c16, h) takes piece 2 h + HALF of row c16; the sums of row blocks wave, wave + XA_WAVES are kept by this wave
  constexpr int SB = (RB + XA_WAVES - 1) / XA_WAVES;
  float x_sum[SB];
#pragma unroll
  for (int i = 0; i < SB; ++i) x_sum[i] = 0.f;
  const int swz = (c16 >> 1) & 7;
  const unsigned char *xr[2] = {stages + c16 * 128 + (((2 * h) ^ swz) << 4), stages + c16 * 128 + (((2 * h + 1) ^ swz) << 4)};

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
    if constexpr (B > 0) xload(B - 1, kb_first + KS * (B - 1));
    __builtin_amdgcn_sched_barrier(0);
    static_for<WL>([&](auto i_c) { wload1(s_c, i_c, kb_first + KS * B); });
    __builtin_amdgcn_sched_barrier(0);
  });
  static_for<16>([&](auto i_c) { convert(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, i_c, wf[0]); });

  // K block kb: x in stage kb % DEPTH, weights in register set kb % DEPTH
  auto step = [&](auto s_c, int kb) {
    constexpr int J = decltype(s_c)::value;
    stage_barrier();   // block kb is in its stage; every wave is done with block kb - 1's
    xload((J + DEPTH - 1) % DEPTH, kb + KS * (DEPTH - 1));
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
        static_for<L1 - L0>([&](auto l_c) { wload1(std::integral_constant<int, J>{}, std::integral_constant<int, L0 + decltype(l_c)::value>{}, kb + KS * DEPTH); });
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
  // (whole rounds, the same number for both sets: blocks past the slice multiply zeros)
  for (int kb = kb_begin; kb < kb_end; kb += KS * DEPTH)
    static_for<DEPTH>([&](auto s_c) { step(s_c, kb + set + KS * decltype(s_c)::value); });

  // ---- epilogue
  xa_drain();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // nothing lands in the stages or reads them any more
  // row block rb is finished by this wave (of two sets, each finishes half of them)
  auto mine = [&](int rb) { return KS == 1 || (rb < H0) == (set == 0); };
  if constexpr (KS == 2) {
    v4f *area = reinterpret_cast<v4f *>(smem);
    float *sums = reinterpret_cast<float *>(smem + XA_MERGE);
    auto parked = [&](int from, int j, int rb) { return area + ((from * NW + wave) * 16 + 4 * (from == 0 ? rb - H0 : rb) + j) * 64 + lane; };
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      if (!mine(rb)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) *parked(rb < H0, j, rb) = acc[j][rb];
        __builtin_amdgcn_sched_barrier(0);
      }
    if (set == 1) {
#pragma unroll
      for (int i = 0; i < SB; ++i) sums[(i * NW + wave) * 64 + lane] = x_sum[i];
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      if (mine(rb)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j][rb] += *parked(rb < H0, j, rb);
        __builtin_amdgcn_sched_barrier(0);   // (all blocks' reads at once would not fit the registers)
      }
    if (set == 0) {
#pragma unroll
      for (int i = 0; i < SB; ++i) x_sum[i] += sums[(i * NW + wave) * 64 + lane];
    }
  }
  if (SPLIT && p.split_k > 1) {
    // Every slice parks its sums, the last one to arrive adds all of them in slice order (the same result whoever that is) and goes
    // on.  Agent-scope accesses; word i of a set's thread t at (i 64 NW + t).
    constexpr int NT = 64 * NW;
    unsigned long long *words = reinterpret_cast<unsigned long long *>(p.partial) + (tile * p.split_k) * (long long)(XA_SLICE_WORDS * NT);   // (wave-uniform: the thread is the 32-bit part of an address)
    const unsigned thread = (unsigned)tid;
    auto put = [&](int i, float lo, float hi) {
      __hip_atomic_store(words + ((long long)slice * XA_SLICE_WORDS + i) * NT + thread, (unsigned long long)__float_as_uint(hi) << 32 | __float_as_uint(lo), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      if (mine(rb)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          put(8 * rb + 2 * j, acc[j][rb][0], acc[j][rb][1]);
          put(8 * rb + 2 * j + 1, acc[j][rb][2], acc[j][rb][3]);
        }
      }
    if (set == 0) put(8 * RB, x_sum[0], SB > 1 ? x_sum[SB - 1] : 0.f);
    publish_partials_and_sync();
    unsigned *s_ticket = reinterpret_cast<unsigned *>(smem);
    if (threadIdx.x == 0) *s_ticket = __hip_atomic_fetch_add(&p.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*s_ticket != (unsigned)(p.split_k - 1)) return;
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    auto get = [&](int s, int i) {
      return __hip_atomic_load(words + ((long long)s * XA_SLICE_WORDS + i) * NT + thread, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // (some row blocks at a time: all accumulators and a slice's words would not fit the registers)
    constexpr int HB = KS == 1 ? (RB + 1) / 2 : 2;
    static_for<(RB + HB - 1) / HB + KS - 1>([&](auto h_c) {
      constexpr int I = decltype(h_c)::value, PER_SET = (H0 + HB - 1) / HB;   // (a piece belongs to one set)
      constexpr int R0 = KS == 1 || I < PER_SET ? I * HB : H0 + (I - PER_SET) * HB, END = KS == 1 || I >= PER_SET ? RB : H0, R1 = R0 + HB < END ? R0 + HB : END;
      if (R1 > R0 && mine(R0)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int rb = R0; rb < R1; ++rb) acc[j][rb] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < p.split_k; ++s) {
          unsigned long long t[8 * HB];
#pragma unroll
          for (int i = 0; i < 8 * (R1 - R0); ++i) t[i] = get(s, 8 * R0 + i);
#pragma unroll
          for (int i = 0; i < 8 * (R1 - R0); ++i) {
            v4f &a = acc[(i / 2) % 4][R0 + i / 8];
            a[2 * (i % 2)] += __uint_as_float((unsigned)t[i]);
            a[2 * (i % 2) + 1] += __uint_as_float((unsigned)(t[i] >> 32));
          }
        }
      }
    });
#pragma unroll
    for (int i = 0; i < SB; ++i) x_sum[i] = 0.f;
    for (int s = 0; s < p.split_k; ++s) {
      const unsigned long long t = get(s, 8 * RB);
      x_sum[0] += __uint_as_float((unsigned)t);
      if constexpr (SB > 1) x_sum[SB - 1] += __uint_as_float((unsigned)(t >> 32));
    }
  }
  float *s_sum = reinterpret_cast<float *>(KS == 1 ? smem : smem + XA_SUMS), *s_scale = s_sum + XA_ROWS, *s_offset = s_scale + XA_COLS;
  s_scale[tid] = xa_half<BF16>(scale_offset & 0xFFFFu);
  s_offset[tid] = xa_half<BF16>(scale_offset >> 16);
#pragma unroll
  for (int i = 0; i < SB; ++i) {
    float v = x_sum[i];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (set == 0 && wave + i * XA_WAVES < RB && h == 0) s_sum[16 * (wave + i * XA_WAVES) + c16] = v;
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
      if (!mine(rb)) continue;
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
        for (int v = 0; v < NV; ++v) a[v] = fmaf(of[v], xs_row, W4 ? a[v] * (BF16 ? 16.0f : 0.0625f) : a[v]) * sc[v];
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

template <bool BF16, bool KN, bool W4, int NW, int KS>
__global__ void __launch_bounds__(64 * NW * KS, 2) gmm_a16w8_rows128_kernel(const GmmParams p) {
  extern __shared__ __align__(16) unsigned char xa_smem[];
  const int lane = threadIdx.x & 63;
  int grp, strip, m0, chunk_rows, chunk;
  if (!chunk_of_xcd_slot(p, XA_ROWS, (int)blockIdx.x, lane, grp, strip, m0, chunk_rows, chunk)) return;
  const int rb = (chunk_rows + 15) / 16;
  bool done = false;
  static_for<XA_RB>([&](auto i_c) {   // one copy of the K loop per number of 16-row blocks
    constexpr int RB = decltype(i_c)::value + 1;
    if (!done && rb == RB) {
      rows_a16w8_run<BF16, KN, W4, RB, NW, KS>(p, xa_smem, grp, strip, m0, chunk_rows, (long long)chunk * p.n_strips + strip);
      done = true;
    }
  });
}

template <bool BF16, bool KN, bool W4, int NW, int KS>
static hipError_t rows_a16w8_form(const GmmParams &p, dim3 grid, hipStream_t stream) {
  auto kern = gmm_a16w8_rows128_kernel<BF16, KN, W4, NW, KS>;
  constexpr int lds = xa_lds(KS);
  if (lds > 64 * 1024) {
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race between first launches repeats it at worst
    if (!attr_set) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return e;
      attr_set = true;
    }
  }
  hipLaunchKernelGGL(kern, grid, dim3(64 * NW * KS), lds, stream, p);
  return hipGetLastError();
}

// wave sets: 1, or 2 with strips of 256 columns
template <bool BF16, bool KN, bool W4 = false>
static hipError_t rows_a16w8_pick(const GmmParams &p, int strip_cols, int sets, dim3 grid, hipStream_t stream) {
  if (strip_cols == 512 && sets == 1) return rows_a16w8_form<BF16, KN, W4, 8, 1>(p, grid, stream);
  if (strip_cols == 256 && sets == 1) return rows_a16w8_form<BF16, KN, W4, 4, 1>(p, grid, stream);
  if (strip_cols == 256 && sets == 2) return rows_a16w8_form<BF16, KN, W4, 4, 2>(p, grid, stream);
  return hipErrorInvalidValue;
}

}  // namespace msco
#endif  // MSCO_GMM_ROWS_A16W8_KERNEL_H_
