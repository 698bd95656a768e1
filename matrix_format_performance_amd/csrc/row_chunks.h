// Index arithmetic shared by kernels and host code: constexpr functions, which
// hipcc compiles for both.
#pragma once

#include <cstdint>

namespace mfp {

// body(start, n) for the chunks of at most `chunk` elements that [b, e) is made
// of.  Entries are numbered up to 2^32 - 1, so the position behind the last
// full chunk may not fit in 32 bits: what is left is counted down instead.
template <class F>
constexpr void for_row_chunks(uint32_t b, uint32_t e, uint32_t chunk, F body)
{
  for (uint32_t left = e > b ? e - b : 0u; left;) {
    const uint32_t n = left < chunk ? left : chunk;
    body(b, n);
    b += n;
    left -= n;
  }
}

} // namespace mfp
