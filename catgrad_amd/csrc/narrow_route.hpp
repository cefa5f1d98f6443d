// Which kernels a product of a narrow dtype runs on: decided from its geometry alone, before any operand's address is asked for
// (an operand that is taken as it lies in memory has no words, and must not reach a kernel that reads words).
#pragma once

#include <cstdint>

namespace cg {

// One operand: rows of k, `pitch` elements apart.  lies: in memory in the kind's patterns, k contiguous, rows on 16-byte boundaries.
struct NarrowSide {
    int64_t rows, pitch;
    bool lies;
};

// kind: 1 bfloat16, 2 binary16, 3 fp8
inline int64_t narrow_bytes(int kind) { return kind == 3 ? 1 : 2; }

// The 128-wide tiles address both operands with byte offsets of 32 bits.
inline bool fits_narrow_tiles(int kind, int64_t x_pitch, int64_t rows, int64_t w_pitch, int64_t n, int64_t k) {
    const int64_t eb = narrow_bytes(kind);
    auto side = [&](int64_t pitch, int64_t r) { return r > 0 && r < (1ll << 31) && pitch >= 0 && pitch < (1ll << 32) && pitch * eb % 16 == 0 && r * pitch * eb < (1ll << 32); };
    return k > 0 && k * eb % 16 == 0 && k * eb < (1ll << 31) && side(x_pitch, rows) && side(w_pitch, n);
}

enum class NarrowRoute {
    words, // 32-bit words, widened first where an operand lies narrow
    low,   // patterns, 128-wide tiles (narrow_tile_kernel)
    wide   // patterns, 256-wide tiles
};

// packable: both operands have buffers, there is no batch, and rows of k are whole 16-byte pieces.  big: there are enough 256-wide
// tiles.  An operand that does not lie narrow is packed first; where neither does, only the 256-wide tiles are worth that.
inline NarrowRoute narrow_route(int kind, const NarrowSide &x, const NarrowSide &y, int64_t k, bool packable, bool big, bool wide_only) {
    if (!packable) return NarrowRoute::words;
    if (big) return NarrowRoute::wide;
    if (wide_only || !(x.lies || y.lies)) return NarrowRoute::words;
    return fits_narrow_tiles(kind, x.lies ? x.pitch : k, x.rows, y.lies ? y.pitch : k, y.rows, k) ? NarrowRoute::low : NarrowRoute::words;
}

// Columns of an [M, N] result that the 256-wide tiles compute.  Their workgroups, one per compute unit, walk the tiles in rounds; where
// the last round leaves three quarters of the units idle, its columns go to the 128-wide tiles instead.  16-bit operands, us with a
// last round and without: 1024 x 2048 x 16484 (4 tiles of 256 left over) 100 and 82, 18432 (32) 102 and 95, 20480 (64) 109 and 103, 24576
// (128) 117 and 121; 2048 x 8192 x 8256 (8) 346 and 236, 10240 (64) 352 and 314, 12288 (128) 380 and 388.
// Whole columns of tiles move, of which a tall result has many in one, so how many tiles that are counts too: 5000 x 1024 x 4000 (64 left
// over, 80 moved) 75 and 69, 20000 x 2048 x 1000 (60, 79) 120 and 107; 7424 x 512 x 2816 (63, 87) 39.5 and 40.9, with 2048 values of k
// 101 and 100.5; 66600 x 1024 x 500 (10, 261) 116 and 127.  (What stays then fills its last round to eleven sixteenths or all of it.)
inline int64_t wide_columns(int64_t units, int kind, int64_t M, int64_t N) {
    const int64_t rows = (M + 255) / 256, tiles = rows * ((N + 255) / 256), over = tiles % units;
    if (kind == 3 || tiles <= units || over == 0 || over * 4 > units) return N;
    const int64_t columns = (tiles - over) / rows; // of tiles
    return columns > 0 && (tiles - columns * rows) * 16 <= 5 * units ? columns * 256 : N;
}

} // namespace cg
