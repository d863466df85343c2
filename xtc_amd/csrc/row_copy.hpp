// SPDX-License-Identifier: BSD-3-Clause
// Index arithmetic of row_copy_kernel (runtime.hip): constant pad and crop of
// tensors of fewer than 2^31 elements, four consecutive elements of an output
// row per thread.  Host and device code, so that its limits are checked on the
// CPU: an innermost extent may be any up to 2^31 - 1, and no index or bound
// below is computed by adding to one.
#pragma once
#include <stdint.h>

namespace xtc_hip {

struct RowCopyDims {
  int outer;  // dims before the innermost
  unsigned out_shape[7];
  unsigned in_shape[7], before[7];
  unsigned out_len, in_len;  // innermost
  unsigned shift;            // its `before`
  unsigned groups;           // ceil(out_len / 4)
  unsigned total;            // rows * groups
};

// Whether element c + e exists in a row of `len` elements; c counts modulo
// 2^32 (an element before the row's first is 2^32 - 1 or a little less, and
// len < 2^31).
__host__ __device__ inline bool row_has(unsigned c, unsigned e, unsigned len) { return c + e < len; }
// Whether all of c .. c + 3 do.
__host__ __device__ inline bool row_has4(unsigned c, unsigned len) { return len >= 4 && c <= len - 4; }

// Four elements of one row: output elements col .. col + 3 of row `row`, from
// elements c .. c + 3 (c modulo 2^32) of input row `src_row` where `inside`.
struct RowGroup {
  unsigned row, col;
  unsigned src_row, c;
  bool inside;
};

template <bool PAD>
__host__ __device__ inline RowGroup row_group(const RowCopyDims& d, unsigned i) {
  RowGroup g;
  g.row = i / d.groups;
  g.col = 4u * (i - g.row * d.groups);
  g.src_row = 0;
  g.inside = true;
  unsigned rem = g.row, stride = 1;
  for (int k = d.outer - 1; k >= 0; --k) {
    const unsigned q = k > 0 ? rem / d.out_shape[k] : 0u;
    const unsigned o = rem - q * d.out_shape[k];
    rem = q;
    const unsigned s = PAD ? o - d.before[k] : o + d.before[k];
    g.inside = g.inside && s < d.in_shape[k];
    g.src_row += s * stride;
    stride *= d.in_shape[k];
  }
  g.c = PAD ? g.col - d.shift : g.col + d.shift;
  return g;
}

}  // namespace xtc_hip
