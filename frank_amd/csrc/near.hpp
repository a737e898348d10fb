// Reach of the operands of a low-rank addition (host side, no HIP types).
#pragma once
#include <algorithm>
#include <cstdint>

namespace frk {

// Whether every element of an r x c operand (strides in elements of `size` bytes) is
// addressed by a byte offset below 2^31: what the blocked kernels of the additions take.
inline bool near_operand(int size, int64_t r, int64_t rs, int64_t c, int64_t cs) {
  if (r <= 0 || c <= 0) return true;
  const int64_t lim = (int64_t)0x7fffff00 / size;
  return rs >= 0 && cs >= 0 && rs < lim && cs < lim && (r - 1) * rs + (c - 1) * cs < lim;
}

// The operands of the addition x of elements of type T: C's bases with the columns that
// are there and those that the update may write (up to its capacity or every column of
// the sum), C's core, X's factors.
template <typename T, class Desc>
bool near_addition(const Desc& x) {
  const int s = sizeof(T);
  const int64_t k = std::max<int64_t>(x.kc, std::min<int64_t>(x.cap, (int64_t)x.kc + x.kx2));
  return near_operand(s, x.m, x.cu_rs, k, x.cu_cs) && near_operand(s, k, x.cv_rs, x.n, x.cv_cs) &&
         near_operand(s, k, x.lds, k, 1) && near_operand(s, x.m, x.xu_rs, x.kx1, x.xu_cs) &&
         near_operand(s, x.kx1, x.xs_ld, x.kx2, 1) && near_operand(s, x.kx2, x.xv_rs, x.n, x.xv_cs);
}

}  // namespace frk
