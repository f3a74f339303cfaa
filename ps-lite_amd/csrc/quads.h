// How far the row kernels may read in a request's values. (No GPU code: the host's tests run it for every quad of a request.)
// Rows of k floats are cut into quads of their own, the last one of a row shorter when k is not a multiple of four. That one
// is read whole all the same, since one access costs less than a choice between four, but where the values end nothing says
// that the memory behind them can be read: a row of one float needs three further ones.
#ifndef PSKV_QUADS_H_
#define PSKV_QUADS_H_
#include <stdint.h>

namespace pskv {

// Whether every quad of the first `rows` of n rows may be read whole: the last one of the last of them reaches furthest, up
// to three floats into the rows behind it, which are three rows if they are of one float, and one row if they are longer (the
// rest of a quad behind two floats is two, behind three one).
constexpr bool whole_quads(uint64_t rows, uint64_t k, uint64_t n) {
  return (k & 3) == 0 || rows + (k == 1 ? 2 : 0) < n;
}

}  // namespace pskv
#endif  // PSKV_QUADS_H_
