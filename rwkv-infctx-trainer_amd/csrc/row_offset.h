// Where a token's elements lie in its sequence, for the accesses that a buffer instruction's range check leaves out past
// the sequence's end.  (Plain C++: the arithmetic is checked on the host.)
#pragma once
#include <stdint.h>

namespace wkv {

// Offset, in elements, of channels c, c+1, .. of token t in a sequence of T tokens and C channels that starts at a head's
// first channel.  T C < 2^30.  A step is 64 tokens whatever T is, so t can lie up to 63 rows past the end, where t C, and
// its bytes all the more, need not fit 32 bits: T 31, C 34 636 800, t 63 would come out inside row 0 again.  All tokens past
// the end therefore count as the first of them, whose offset, T C + c <= 2^30 - 64 + c, still fits as bytes of four-byte elements
// and is beyond every element of the sequence.
constexpr uint32_t row_offset(int t, int T, int C, int c) { return (uint32_t)(t < T ? t : T) * (uint32_t)C + (uint32_t)c; }

}  // namespace wkv
