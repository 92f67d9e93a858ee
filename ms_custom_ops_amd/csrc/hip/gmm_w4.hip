// Grouped A8W4 matmul for gfx950: int8 activations x int4 weights (two per byte, [E, N, K/2], K contiguous), float32
// scales per (expert, K group, column), per-token activation scales, float16 out.
//
//   out[m, n] = x_scale[m] * sum_g w_scale[e, g, n] * sum_{k in g} x[m, k] * w[e, n, k]        (e = the group of row m)
//
// (tests/st/test_grouped_matmul_w4.py:100-113; ops/c_api/grouped_matmul_w4/grouped_matmul_w4.cc:50-88.)  The
// reference's workloads route 5 .. 32 rows to 256 experts: almost every group is empty or holds one row, so this is a
// batch of matrix-vector products bound by the bytes of the weights of the experts that were hit.  Hence no MFMA:
//   * one workgroup per (group that holds rows, share of the columns): the grid has min(E, M) group slots and a workgroup
//     finds the group of its slot's rank with ballots over group_list; a short K lets several columns share a wavefront's lanes;
//   * the group's rows (a few at a time) sit in LDS, de-interleaved into even-k and odd-k bytes so that they line up
//     with the low and the high nibbles of a weight word;
//   * a wavefront takes blocks of C neighbouring columns per lane segment, lane L holding the 16-byte pieces L, L + 64, ... of a
//     column (32 consecutive k, always inside one K group), and requests the next block while it multiplies this one: the
//     group look-up, the x rows and the first round trip are paid once per workgroup, of which the launch has four
//     per CU and more (launch_a8w4).  nibbles are multiplied as u ^ 8 in [0, 15] with v_dot4_i32_i8 and 8 * sum(x) of the piece is subtracted
//     (u ^ 8 = s + 8 for the signed nibble s); the int32 sum of a piece is exact, is scaled by its K group's float32
//     scale and added up in float32; the lanes' sums of C columns are added in a tree that halves the columns a lane
//     holds with every step.
#include "gmm_common.h"
#include "gmm_kernels.h"
#include "msco_gmm.h"

namespace msco {
namespace {

constexpr int W4_MAX_K = 8192;
constexpr int W4_LDS_BYTES = 32 * 1024;              // x rows in LDS at a time: 32 KiB / K, at most W4_MAX_ROWS
constexpr int W4_MAX_ROWS = 16;
constexpr int W4_TARGET_WGS = 1024;                  // four workgroups per CU (one group; see launch_a8w4)
constexpr int w4_cols(int p) { return p == 1 ? 8 : 4; }   // columns of a block per lane segment: 32 weight registers (64 with the longest K)
inline int w4_rows(int64_t k, int64_t m) {
  int64_t r = W4_LDS_BYTES / k;
  r = r > W4_MAX_ROWS ? W4_MAX_ROWS : r < 1 ? 1 : r;
  return (int)(r < m ? r : m);
}

__device__ __forceinline__ int dot4(int a, int b, int c) { return __builtin_amdgcn_sdot4(a, b, c, false); }

// P = 16-byte pieces of a column per lane (K <= 2048 P); VEC: four scales of a lane's columns are one request (N % 4 == 0)
template <int P, bool VEC>
__global__ void __launch_bounds__(256, VEC ? 3 : 2) gmm_a8w4_kernel(const int8_t *x, const unsigned char *w, const int *group_list,
                                                       const float *x_scale, const float *w_scale, unsigned short *out, int m,
                                                       int k, int n, int e, int group_size, int lds_rows) {
  constexpr int C = w4_cols(P);
  extern __shared__ __align__(16) int xs[];   // lds_rows rows: [row][piece of 32 k]: 4 words of even-k bytes, then 4 of odd-k bytes
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // blockIdx.y counts the groups that hold rows (at most min(e, m) of them): find the one with that rank, 64 groups
  // per round of ballots, and leave if there are fewer
  int grp = -1, g_start = 0, g_end = 0;
  const __amdgpu_buffer_rsrc_t rs_list = buffer_over(group_list, 4ll * e);
  for (int g0 = 0, seen = 0, carry = 0; g0 < e && grp < 0; g0 += 256) {
    // four rounds' worth of boundaries requested together: one memory round trip per 256 groups.  Through a buffer
    // descriptor over the list (entries past its end read as 0): a load under `g < e ? ... : 0` is a branch, and the
    // compiler waits for every such load (vmcnt(0)) where its value meets the 0 of the other path.
    int lo[4], hi[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) hi[u] = __builtin_amdgcn_raw_buffer_load_b32(rs_list, 4u * (unsigned)(g0 + 64 * u + lane), 0, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) hi[u] = min(max(hi[u], 0), m);
    // row end of a group = running maximum of the list clamped into [0, m] (a list that is not monotonic can then
    // never make two groups overlap); `carry` is the end of the last group of the round before
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      hi[u] = max(carry, wave_scan_max(hi[u]));
      lo[u] = wave_from_below(hi[u], carry);
      carry = wave_bcast(hi[u], 63);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      unsigned long long holds = __ballot(hi[u] > lo[u]);
      const int here = __popcll(holds);
      if (grp < 0 && seen + here > (int)blockIdx.y) {
        for (int skip = (int)blockIdx.y - seen; skip > 0; --skip) holds &= holds - 1;
        const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)holds) - 1);
        grp = g0 + 64 * u + src;
        g_start = wave_bcast(lo[u], src);
        g_end = wave_bcast(hi[u], src);
      }
      seen += here;
    }
  }
  if (grp < 0) return;
  const int pieces = k / 32;
  // a short K leaves lanes over: lanes_per_col lanes share a column segment, the wavefront works on 64 / lanes_per_col segments side by side
  int lanes_per_col = 64;
  if constexpr (P == 1) {
    while (lanes_per_col > C && lanes_per_col / 2 >= pieces) lanes_per_col /= 2;
  }
  const int side = 64 / lanes_per_col;
  const int pl = lane & (lanes_per_col - 1), sub = lane / lanes_per_col;
  const int pieces_per_group = group_size / 32, k_groups = k / group_size;
  const int block_cols = 4 * C * side;                       // columns of a workgroup's block
  const int col_lane = C * (wave * side + sub);               // this lane's first column in it
  const int blocks = (n + block_cols - 1) / block_cols;
  const unsigned char *wg = w + (long long)grp * n * (k / 2);
  const float *sg = w_scale + (long long)grp * k_groups * n;

  // A block of this lane's columns: every piece and its scale requested at once.  Branch-free, through buffer descriptors over
  // the block's weights and scales: what a lane has no use for (a piece past K, a column past N) is asked at an offset beyond the
  // descriptor and reads as 0.
  struct Block {
    v4i w[P][C];
    float s[P][C];
  };
  auto request = [&](Block &b, int block) {
    const long long n0 = (long long)block * block_cols;
    const int cols = block < blocks ? min(block_cols, n - (int)n0) : 0;
    const __amdgpu_buffer_rsrc_t rs_w = buffer_over(wg + n0 * (k / 2), (long long)cols * (k / 2));
    const __amdgpu_buffer_rsrc_t rs_s = buffer_over(sg + n0, cols > 0 ? 4ll * ((long long)(k_groups - 1) * n + cols) : 0);
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int p = pl + 64 * i;
      const bool live = p < pieces;
#pragma unroll
      for (int c = 0; c < C; ++c)
        b.w[i][c] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, live && col_lane + c < cols ? (unsigned)(col_lane + c) * (unsigned)(k / 2) + 16u * (unsigned)p : 0xFFFFFFF0u, 0, 0);
      const unsigned at = 4u * ((unsigned)(p / pieces_per_group) * (unsigned)n + (unsigned)col_lane);
      if constexpr (VEC) {
#pragma unroll
        for (int c = 0; c < C; c += 4) {
          const v4i v = __builtin_amdgcn_raw_buffer_load_b128(rs_s, live && col_lane < cols ? at + 4u * c : 0xFFFFFFF0u, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; ++q) b.s[i][c + q] = __uint_as_float((unsigned)v[q]);
        }
      } else {
#pragma unroll
        for (int c = 0; c < C; ++c)
          b.s[i][c] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rs_s, live && col_lane + c < cols ? at + 4u * c : 0xFFFFFFFCu, 0, 0));
      }
    }
  };

  // rows r0 .. r0 + rows of the block in LDS (piece idx is 16 bytes, k0 .. k15 of half a piece: two words of even-k bytes and two of odd-k bytes)
  auto stage_rows = [&](int r0, int rows) {
    const uint4 *src = reinterpret_cast<const uint4 *>(x + (long long)r0 * k);
    const int total = rows * pieces * 2;
    for (int idx = threadIdx.x; idx < total; idx += 256) {
      const uint4 v = src[idx];
      const int r = idx / (pieces * 2), h = idx - r * pieces * 2;
      const unsigned e0 = __builtin_amdgcn_perm(v.y, v.x, 0x06040200u), o0 = __builtin_amdgcn_perm(v.y, v.x, 0x07050301u);
      const unsigned e1 = __builtin_amdgcn_perm(v.w, v.z, 0x06040200u), o1 = __builtin_amdgcn_perm(v.w, v.z, 0x07050301u);
      int *dst = xs + (r * pieces + (h >> 1)) * 8 + (h & 1) * 2;
      dst[0] = (int)e0; dst[1] = (int)e1; dst[4] = (int)o0; dst[5] = (int)o1;
    }
  };

  auto multiply = [&](const Block &b, int block, int r0, int rows) {
    const int c0 = block * block_cols + col_lane;
    for (int r = 0; r < rows; ++r) {
      unsigned low = 0x0F0F0F0Fu;   // (opaque: split once for all rows, the nibbles would take more registers than there are)
      asm volatile("" : "+s"(low));
      float acc[C];
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = 0.f;
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int p = pl + 64 * i;
        if (p < pieces) {
          const int4 xe = *reinterpret_cast<const int4 *>(xs + (r * pieces + p) * 8);
          const int4 xo = *reinterpret_cast<const int4 *>(xs + (r * pieces + p) * 8 + 4);
          const int xev[4] = {xe.x, xe.y, xe.z, xe.w}, xov[4] = {xo.x, xo.y, xo.z, xo.w};
          int sx = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) sx = dot4(xov[j], 0x01010101, dot4(xev[j], 0x01010101, sx));
#pragma unroll
          for (int c = 0; c < C; ++c) {
            int d = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const unsigned t = (unsigned)b.w[i][c][j] ^ 0x88888888u;
              d = dot4(xev[j], (int)(t & low), d);           // k = 8 j + 0, 2, 4, 6
              d = dot4(xov[j], (int)((t >> 4) & low), d);    // k = 8 j + 1, 3, 5, 7
            }
            acc[c] += (float)(d - 8 * sx) * b.s[i][c];
          }
        }
      }
      // lanes pl of a segment: the sums of columns c and c + half change sides, so that a lane is left with the column its low bits name
#pragma unroll
      for (int half = C / 2, bit = 1; half > 0; half /= 2, bit *= 2) {
        const bool up = (lane & bit) != 0;
#pragma unroll
        for (int c = 0; c < half; ++c) {
          const float give = up ? acc[c] : acc[c + half], keep = up ? acc[c + half] : acc[c];
          acc[c] = keep + __shfl_xor(give, bit);
        }
      }
      float v = acc[0];
      for (int o = C; o < lanes_per_col; o *= 2) v += __shfl_xor(v, o);   // wave-uniform
      // bit 0 of the lane chose between halves C / 2 apart, bit 1 between quarters, ..
      int col = 0;
#pragma unroll
      for (int half = C / 2, bit = 1; half > 0; half /= 2, bit *= 2) col += (lane & bit) ? half : 0;
      if (pl < C && c0 + col < n) out[(long long)(r0 + r) * n + c0 + col] = f32_to_f16_rne(v * x_scale[r0 + r]);
    }
  };

  Block even, odd;   // (the longest K has one block in flight: with half as many columns each, or both blocks, slower, 14.5 against 12.4 us)
  const int stride = (int)gridDim.x;
  if constexpr (P == 4) {
    // A block's weights stay in registers for all rows of the group: a group with more rows than LDS holds (four to seven with this K) brings its rows
    // once per block, not its weights once per batch of rows (one group of 16 and more rows 0.80 -> 0.68 of the time of a launch with one block per workgroup)
    int staged = -1;   // the batch of rows in LDS
    for (int block = (int)blockIdx.x; block < blocks; block += stride) {
      request(even, block);
      for (int r0 = g_start; r0 < g_end; r0 += lds_rows) {
        const int rows = min(lds_rows, g_end - r0);
        if (staged != r0) {
          if (staged >= 0) __syncthreads();   // the rows before are no longer read
          stage_rows(r0, rows);
          __syncthreads();
          staged = r0;
        }
        multiply(even, block, r0, rows);
      }
    }
    return;
  }
  for (int r0 = g_start; r0 < g_end; r0 += lds_rows) {
    const int rows = min(lds_rows, g_end - r0);
    int block = (int)blockIdx.x;
    request(even, block);
    if (r0 != g_start) __syncthreads();   // the rows before are no longer read
    stage_rows(r0, rows);
    __syncthreads();
    for (; block < blocks; block += 2 * stride) {
      request(odd, block + stride);
      multiply(even, block, r0, rows);
      if (block + stride >= blocks) break;
      request(even, block + 2 * stride);
      multiply(odd, block + stride, r0, rows);
    }
  }
}

template <int P>
hipError_t launch_a8w4(const int8_t *x, const unsigned char *w, const int *group_list, const float *x_scale, const float *w_scale,
                       unsigned short *out, int m, int k, int n, int e, int group_size, hipStream_t stream) {
  constexpr int C = w4_cols(P);
  int lanes_per_col = 64;
  while (P == 1 && lanes_per_col > C && lanes_per_col / 2 >= k / 32) lanes_per_col /= 2;
  const int block_cols = 4 * C * (64 / lanes_per_col), blocks = (n + block_cols - 1) / block_cols;
  const int slots = e < m ? e : m;
  // (slots past the last group that holds rows leave at once: counting them all makes the shares of the columns larger, not smaller)
  // With several groups the launch ends with the largest one, which does rows x columns of work in its shares: more of them, by twice the average rows of a
  // group, let the others' CUs take part (172 rows over 64 experts, 8064 x 6128 701 -> 372 us; 106 rows, 5312 x 6064 431 -> 246; 12342 random
  // shapes 0.95 of the time; one group is even whatever the shares).  Up to half as many rows as experts, most groups hold one row and are even
  // too: twice the shares are a second round of workgroups there (20 rows over 64 experts, 2816 x 1200 11.25 against 12.4 us; 600 random
  // shapes of 2 to 64 rows, no more than experts: 6 slower by more than 3 % than a launch of 1024 workgroups, 54 with twice the shares everywhere).
  const long long wanted = (W4_TARGET_WGS + slots - 1ll) / slots * (slots > 1 && 2ll * m > e ? (2ll * m + slots - 1) / slots : 1);
  const int shares = wanted < blocks ? (int)wanted : blocks, steps = (blocks + shares - 1) / shares;
  const dim3 grid((unsigned)((blocks + steps - 1) / steps), (unsigned)slots);
  const int rows = w4_rows(k, m);
  const size_t lds = (size_t)rows * (size_t)k;
  auto kern = n % 4 == 0 ? gmm_a8w4_kernel<P, true> : gmm_a8w4_kernel<P, false>;
  hipLaunchKernelGGL(kern, grid, dim3(256), lds, stream, x, w, group_list, x_scale, w_scale, out, m, k, n, e, group_size, rows);
  return hipGetLastError();
}

// 4-bit values widened to int8: 16 source bytes (32 nibbles) -> 32 bytes per thread, low nibble first, sign extended
__global__ void __launch_bounds__(256) unpack_int4_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, long long pieces,
                                                          const unsigned char *src_tail, signed char *dst_tail, int tail_bytes) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  auto widen = [](unsigned w, unsigned &lo, unsigned &hi) {
    // bytes b0 b1 b2 b3 of w -> lo = {b0.lo, b0.hi, b1.lo, b1.hi}, hi = {b2.lo, b2.hi, b3.lo, b3.hi}, each nibble sign extended
    const unsigned even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
    const unsigned l = __builtin_amdgcn_perm(odd, even, 0x05010400u);   // e0 o0 e1 o1
    const unsigned h = __builtin_amdgcn_perm(odd, even, 0x07030602u);   // e2 o2 e3 o3
    // sign extension of a 4-bit value held in a byte: (v ^ 8) - 8, per byte without carries between bytes
    lo = ((l ^ 0x08080808u) | 0x80808080u) - 0x08080808u;
    lo ^= 0x80808080u;
    hi = ((h ^ 0x08080808u) | 0x80808080u) - 0x08080808u;
    hi ^= 0x80808080u;
  };
  if (i < pieces) {
    const uint4 v = src[i];
    uint4 a, b;
    widen(v.x, a.x, a.y); widen(v.y, a.z, a.w); widen(v.z, b.x, b.y); widen(v.w, b.z, b.w);
    dst[2 * i] = a;
    dst[2 * i + 1] = b;
  }
  if (i < tail_bytes) {   // the last bytes of a source whose size is not a multiple of 16
    const unsigned char t = src_tail[i];
    const int lo = t & 15, hi = t >> 4;
    dst_tail[2 * i] = (signed char)(lo >= 8 ? lo - 16 : lo);
    dst_tail[2 * i + 1] = (signed char)(hi >= 8 ? hi - 16 : hi);
  }
}

}  // namespace

hipError_t launch_unpack_int4(const void *src, void *dst, long long src_bytes, hipStream_t stream) {
  const long long pieces = src_bytes / 16;
  const int tail = (int)(src_bytes % 16);
  const long long threads = pieces > tail ? pieces : tail;
  if (threads == 0) return hipSuccess;
  if ((threads + 255) / 256 > 0x7FFFFFFFll) return hipErrorInvalidValue;
  const unsigned char *s8 = static_cast<const unsigned char *>(src);
  hipLaunchKernelGGL(unpack_int4_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream,
                     static_cast<const uint4 *>(src), static_cast<uint4 *>(dst), pieces, s8 + pieces * 16,
                     static_cast<signed char *>(dst) + pieces * 32, tail);
  return hipGetLastError();
}
}  // namespace msco

extern "C" int msco_unpack_int4(const void *src, void *dst, int64_t src_bytes, void *stream) {
  using namespace msco;
  if (src_bytes < 0) return MSCO_ERR_SHAPE;
  if (src_bytes == 0) return MSCO_OK;
  if (src == nullptr || dst == nullptr) return MSCO_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(src) & 15) != 0 || (reinterpret_cast<uintptr_t>(dst) & 15) != 0) return MSCO_ERR_INVALID_ARG;
  if ((src_bytes / 16 + 255) / 256 > 0x7FFFFFFFll) return MSCO_ERR_SHAPE;
  return launch_unpack_int4(src, dst, src_bytes, static_cast<hipStream_t>(stream)) == hipSuccess ? MSCO_OK : MSCO_ERR_DEVICE;
}

extern "C" int msco_gmm_a8w4(const int8_t *x, const void *weight, const int32_t *group_list, const float *x_scale,
                             const float *weight_scale, void *out, int64_t m, int64_t k, int64_t n, int64_t e,
                             int64_t group_size, void *stream) {
  using namespace msco;
  if (m < 0 || k <= 0 || n <= 0 || e <= 0 || group_size <= 0) return MSCO_ERR_SHAPE;
  if (k % 32 != 0 || group_size % 32 != 0 || k % group_size != 0) return MSCO_ERR_SHAPE;
  if (k > W4_MAX_K || e > 65535 || m > INT32_MAX || n > INT32_MAX) return MSCO_ERR_UNSUPPORTED;
  if (m == 0) return MSCO_OK;
  if (x == nullptr || weight == nullptr || group_list == nullptr || x_scale == nullptr || weight_scale == nullptr || out == nullptr)
    return MSCO_ERR_INVALID_ARG;
  auto launch = k <= 2048 ? launch_a8w4<1> : k <= 4096 ? launch_a8w4<2> : launch_a8w4<4>;
  return launch(x, static_cast<const unsigned char *>(weight), group_list, x_scale, weight_scale, static_cast<unsigned short *>(out),
                (int)m, (int)k, (int)n, (int)e, (int)group_size, static_cast<hipStream_t>(stream)) == hipSuccess
           ? MSCO_OK
           : MSCO_ERR_DEVICE;
}
