// Dispatch arithmetic of the persistent GEMM: plain C++, no device code.
#pragma once

namespace pq {

// A persistent product's tiles lie in 8 lists, one per XCD, of tiles / 8 tiles and, the first tiles % 8 of them, one more.
// The tiles of such a list that go out whole; the others, past its last whole round of `wgx` tiles (one per workgroup of
// the XCD), go out as four quarters each.
struct WholeTiles {
  int lo, hi;   // of a list of tiles / 8 tiles, and of one more
};

// Quarters end the product earlier where they are few: a quarter takes a third of a tile's time at K = 3072, and more of
// it the shorter K is (its first stages and its epilogue do not shrink with K), and one wave of quarters waits for the
// slowest workgroup of the round before, where the tiles would have gone to the fastest. GEMMs alone, time in quarters over
// whole, by the tiles past the round of 32 (the longer list's) in an XCD's list:
//   2 to 4 whole rounds   K = 640: 0.97 at 1-3, 1.00 at 5, 1.01-1.04 at 6, 1.04-1.05 at 7, 1.09 at 8
//                         K = 1280: 0.90-0.97 at 1-5, 1.00 at 6, 1.02 at 7, 1.04-1.06 at 8
//                         K = 2048: 0.90-0.98 at 1-4, 0.92-1.00 at 5, 0.94-0.99 at 6, 0.97-0.99 at 7, 1.01 at 8
//                         K = 3072: 0.90-0.99 at 2-6, 0.95-1.00 at 7, 1.00-1.01 at 8
//                         K = 5120: 0.89-0.97 at 1-6, 0.96-0.98 at 8; K = 12288: 0.88-0.94 at 1-7, 0.91 at 8
//   5 and more            K = 640 to 3072: 0.99-1.02 at 1-7 (claims from the XCDs that run behind cover a short round),
//                         1.01-1.06 at 8; K = 4032 to 5120: 0.94-0.99 at 1-6, 1.00 at 7
// Either both kinds of list or neither: a workgroup that has had its quarter takes a tile left in another list as four
// quarters one after the other, a third more than the tile whole, so lists with quarters beside lists of whole tiles ended
// later (lists of 8 and 9 past the round: 95129 x 2752 x 1152 418 us whole, 439 with quarters; 11296 x 3392 x 11904 402 and 433).
constexpr WholeTiles whole_tiles(int tiles, int wgx, int K) {
  const int lo = tiles / 8, rounds = lo / wgx;
  const int past_lo = lo % wgx, past_hi = tiles % 8 ? (lo + 1) % wgx : past_lo;
  const int past = past_lo > past_hi ? past_lo : past_hi;
  const bool quarters = K >= 4096 ? 4 * past <= wgx : rounds <= 4 && (K >= 2048 ? 4 * past < wgx : 6 * past <= wgx);
  if (!quarters) return {lo, lo + 1};
  return {lo - past_lo, lo + 1 - (lo + 1) % wgx};
}

}  // namespace pq
