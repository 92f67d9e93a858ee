// Where the 4-bit tile kernels (gmm_tile_w8a8.hip) find a 16-byte piece of [K, N/2] weights and, in it, its columns.  Plain
// C++, so that a host program can walk every piece of a matrix.
#ifndef MSCO_GMM_W4_PIECE_H_
#define MSCO_GMM_W4_PIECE_H_

#if defined(__HIPCC__)
#define MSCO_PIECE_FN __host__ __device__ __forceinline__ constexpr
#else
#define MSCO_PIECE_FN constexpr
#endif

namespace msco {

// A piece is 32 columns of one K row, from column `col` (a multiple of 32).  N is a multiple of 16 only: where col + 16 == N the
// row has 8 bytes of it left, and 16 bytes from there would end 8 bytes behind the row -- behind the tensor in the last row
// of the last expert.  Such a piece is requested 8 bytes early and its columns are found in the second half.  The one row
// with nothing in front of it (N = 16: K row 0 of the first expert) is requested as it is, it has a row behind it; so are the
// other rows `krow` % 32 == 0 of a slab, which the same lanes read (K is a multiple of 16: their next row exists).
MSCO_PIECE_FN int w4_early(int krow, int col, int n) { return col + 16 == n && (col > 0 || krow % 32 != 0) ? 8 : 0; }

// byte offset of the piece of slab row `krow` from the slab's first K row
MSCO_PIECE_FN unsigned w4_piece_offset(int krow, int col, int n) {
  return (unsigned)krow * (unsigned)(n / 2) + (unsigned)(col / 2 - w4_early(krow, col, n));
}

// where in the piece the 16 columns from col + 16 half are (columns past N: somewhere inside it)
MSCO_PIECE_FN int w4_half_offset(int krow, int col, int n, int half) { return col + 16 == n ? w4_early(krow, col, n) : 8 * half; }

}  // namespace msco
#endif  // MSCO_GMM_W4_PIECE_H_
