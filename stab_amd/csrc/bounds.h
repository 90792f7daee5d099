// Index rules of kernels that have to stay in range for every size, free of
// HIP types so they can be compiled and checked on the host (constexpr
// functions are host and device functions alike).
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
