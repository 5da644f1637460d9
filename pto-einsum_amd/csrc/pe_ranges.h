// Extents and launch limits that must hold up to the largest accepted sizes.
// Plain constexpr functions (usable in kernels, on the host and in a host
// compiler's test of them).
#pragma once

#include <cstdint>

namespace pe {

// k of the range that starts at kb, of at most `per`.  K may be any int32:
// the last range's kb + per can pass 2^31 (a dot product of 2^31 - 100000
// float16 values: 1024 ranges of 2^21), so the sum is unsigned.
constexpr int32_t k_range(int32_t K, int32_t kb, int32_t per) {
    const uint32_t end = uint32_t(kb) + uint32_t(per);
    return int32_t((uint32_t(K) < end ? uint32_t(K) : end) - uint32_t(kb));
}

// Slabs of bk k that cover len (>= 0): as a signed sum, len + bk - 1 can pass
// 2^31 too.
constexpr int32_t k_slabs(int32_t len, int32_t bk) {
    return int32_t((uint32_t(len) + uint32_t(bk) - 1u) / uint32_t(bk));
}

// Whether every range of K and every slab of it ends below 2^31, however K is
// split (splits of whole slabs end less than 2^20 past K).  GEMM kernels form
// these ends as plain sums and take such K only, but for one that takes the
// rest: with k_range in all of them, the direct-load float32 64x64 tiles ran up
// to 9 % longer (82 x 152 x 400, K = 1024, 129 -> 141 us), staged ones up to 6.
constexpr bool k_ends_fit(int64_t K) { return K <= INT32_MAX - (1 << 20); }

// Rows (or columns) of a GEMM that run in one launch, the rest in another:
// the kernels form the end of a tile (at most 256 rows) in 32 bits, and an
// axis that ends within a tile of 2^31 would end at 2^31.
constexpr int64_t axis_part(int64_t n) { return n > (int64_t(1) << 31) - 256 ? int64_t(1) << 30 : n; }

// The index after i of a walk over n (i < n) in steps of `stride`, n at its
// end: i + stride can pass 2^32.
constexpr uint32_t next_index(uint32_t i, uint32_t stride, uint32_t n) { return n - i > stride ? i + stride : n; }

// Blocks of 256 threads in a launch: HIP takes fewer than 2^32 threads along an
// axis of the grid.
constexpr int64_t kMaxBlocks = (int64_t(1) << 24) - 1;

// Blocks of the product kernel's 64 x 64 tiles over `batches` matrices of P x
// Q, or 0 where it does not serve: more than a launch holds, or tiles less
// than a sixteenth full (it moves a whole tile's elements whatever part of it
// is there).  One MI355X, one element per lane against tiles, 8.4 million
// outputs: 8 x 8 matrices f16 142 against 297 us, f32 142 / 228, 12 x 12 143 /
// 155 and 169 / 107, 16 x 16 145 / 97 and 144 / 65, 8 x 64 142 / 51 and 145 /
// 34.
constexpr int64_t product_tile_blocks(int64_t P, int64_t Q, int64_t batches) {
    const int64_t tiles = ((P + 63) / 64) * ((Q + 63) / 64);
    return 16 * P * Q >= 64 * 64 * tiles && tiles * batches <= kMaxBlocks ? tiles * batches : 0;
}

}  // namespace pe
