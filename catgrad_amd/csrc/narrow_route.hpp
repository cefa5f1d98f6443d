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

} // namespace cg
