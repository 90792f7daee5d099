// Rules of kernels that have to hold for every size and value (indexes that
// stay in range, NaN that is not lost), free of HIP types so they can be
// compiled and checked on the host (constexpr functions are host and device
// functions alike).
#pragma once

// Element of the matrix (column-major, leading dimension lda) that k_lu_panel
// reads for entry (i, k), k < i < 64, of the block at K0 when it stages the
// strictly lower L11 for its inverse.  The block is kb wide: entries past it
// (the upper half of a 32-wide last block) are replaced by zeros after the
// load, so row and column both fall back to the block's corner, as the last
// block ends with the matrix and a column past it is a column past the buffer.
constexpr long long lu_l11_src(int K0, int kb, int i, int k, int lda) {
  return (long long)(K0 + (i < kb ? k : 0)) * lda + K0 + (i < kb ? i : 0);
}

// Row that k_schur moves to position pos (pos < m <= 64) when it orders the
// eigenvalues: the first lane of the ballot `at` of the lanes that hold the
// largest modulus.  A lane outside [pos, m) carries -1 and no eigenvalue; with
// NaN in every lane of the range (the factors of a singular matrix) the
// maximum is that -1 and only such lanes are in the ballot, so they are masked
// and pos stays where it is.
constexpr int schur_pick(unsigned long long at, int pos, int m) {
  at &= (m < 64 ? (1ull << m) - 1 : ~0ull) & ~((1ull << pos) - 1);
  return at ? __builtin_ctzll(at) : pos;
}

// The largest of n residual estimates (none negative), NaN when any is: NaN
// must not pass for the zero that fmax would leave of it.
constexpr double est_max(const double *est, int n) {
  double mx = 0.0;
  for (int i = 0; i < n; ++i) mx = (est[i] > mx || est[i] != est[i]) ? est[i] : mx;
  return mx;
}
