// rules.h -- the conditions by which launches and epilogues choose a path, as
// plain functions of sizes (no HIP types: the CPU tests compile them alone).
#pragma once

#include <cstdint>

namespace lbt {

// Whether a wavefront block of `tokens` tokens from tok0 and `rows` rows of an
// m x ld matrix of 32-bit values can store through 32-bit byte offsets from
// its first element, with tokens past m dropped by the end of a buffer of
// m ld values.  The block's last token may lie past m: its offset has to stay
// below 2^32 too, or it wraps round to the first tokens' values.
constexpr bool lean_offsets_fit(int64_t m, int64_t ld, int64_t tok0, int64_t tokens, int64_t rows) {
    constexpr int64_t kMax = int64_t{1} << 30;  // 4-byte values
    return m * ld < kMax && (tok0 + tokens) * ld + rows < kMax;
}

}  // namespace lbt
