// How the splits of a ragged attention batch are shared out: the part of the rule that needs no device.
#pragma once

namespace dflash {

// The smallest number L of tiles per workgroup, at least `lo`, with fits(L) := sum over the sequences of ceil(tiles / L) <= W, where
// `lo` >= total / W and `hi` fits: total / (W - B) does, as the sum is at most total / L + B, and so does the longest
// sequence's tile count, which leaves every sequence one split (B <= W).  The sum does not grow with L, so the range is halved:
// twelve sums at most for the 3,200 tiles of 102,400 keys, most often the one at `lo`.
template <typename Fits> constexpr int tiles_per_share(int lo, int hi, Fits fits) {
    if (lo >= hi || fits(lo)) return lo;
    while (hi - lo > 1) {
        const int mid = lo + (hi - lo) / 2;
        if (fits(mid)) hi = mid;
        else lo = mid;
    }
    return hi;
}

// ceil(tiles / L) - 1 before it is rounded down, from a reciprocal of L that may be off by a few units in the last place: the
// quotient keeps half a tile's distance from the next whole number, more than its error for any tile count below 2^20.
constexpr float share_quotient(float tiles, float inv_L) { return (tiles - 0.5f) * inv_L; }

}  // namespace dflash
