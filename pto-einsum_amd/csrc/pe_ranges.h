// Extents and launch limits that must hold up to the largest accepted sizes.
// Plain constexpr functions (usable in kernels, on the host and in a host
// compiler's test of them).
#pragma once

#include <cstdint>

namespace pe {

// k of the range that starts at kb, of at most `per`.  K may be any int32:
// the last range's kb + per can pass 2^31 (a dot product of 2^31 - 100000
// float16 values: 1024 ranges of 2^21), so that sum is never formed.
constexpr int32_t k_range(int32_t K, int32_t kb, int32_t per) { return K - kb < per ? K - kb : per; }

// Slabs of bk k that cover len (>= 0): as a signed sum, len + bk - 1 can pass
// 2^31 too.
constexpr int32_t k_slabs(int32_t len, int32_t bk) {
    return int32_t((uint32_t(len) + uint32_t(bk) - 1u) / uint32_t(bk));
}

// Rows (or columns) of a GEMM that run in one launch, the rest in another:
// the kernels form the end of a tile (at most 256 rows) in 32 bits, and an
// axis that ends within a tile of 2^31 would end at 2^31.
constexpr int64_t axis_part(int64_t n) { return n > (int64_t(1) << 31) - 256 ? int64_t(1) << 30 : n; }

// The index after i of a walk over n (i < n) in steps of `stride`, n at its
// end: i + stride can pass 2^32.
constexpr uint32_t next_index(uint32_t i, uint32_t stride, uint32_t n) { return n - i > stride ? i + stride : n; }

}  // namespace pe
