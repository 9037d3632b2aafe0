// Which tiles of `tile` inner rows the outer rows of a workgroup, and of one of its waves, walk in the kernels of plain local
// attention for 2-byte inputs.  The pair (outer o, inner n) is in the band when n - o lies in [-below, above) and n < inner.
// Plain C++, so that the host can check it over all shapes.
#pragma once

namespace flyhip {

struct TileRange { int lo, hi; };                    // tiles lo .. hi - 1

// of the outer rows first .. end - 1
constexpr TileRange band_tiles(int first, int end, int below, int above, int inner, int tile) {
    const int lo = first - below > 0 ? first - below : 0;
    const int hi = end <= first ? 0 : (inner < end - 1 + above ? inner : end - 1 + above);
    return {lo / tile, hi > lo ? (hi + tile - 1) / tile : lo / tile};
}

// of a wave's rows w_first .. w_end - 1 among the workgroup's tiles `all`.  Both ends lie inside `all`, also for rows past the last
// inner row that any of them sees: every wave then passes the barriers of exactly all.hi - all.lo tiles, its own and the others'.
constexpr TileRange wave_tiles(TileRange all, int w_first, int w_end, int below, int above, int inner, int tile) {
    if (w_end <= w_first) return {all.hi, all.hi};
    const TileRange own = band_tiles(w_first, w_end, below, above, inner, tile);
    const int lo = own.lo > all.lo ? own.lo : all.lo;
    return {lo < all.hi ? lo : all.hi, own.hi < all.hi ? own.hi : all.hi};
}

}  // namespace flyhip
