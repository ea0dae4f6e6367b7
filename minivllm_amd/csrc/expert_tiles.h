// Which tiles a workgroup of the experts' products takes: whole numbers alone, for the device and for programs on the host that look them over.
#pragma once
#include <hip/hip_runtime.h>

#define EXPERT_TILES_FN __host__ __device__ __forceinline__

namespace mvllm {

constexpr int kLargeGroups = 32;                    // workgroups per XCD that go on to another tile: its CUs

// at: a place among an XCD's (row tile, weight tile) pairs, which begin with pair `low` of all and end before `high`
EXPERT_TILES_FN void pair_at(int n, int low, int high, int place, int& tile, int& n_tile) {
  constexpr int kTogether = 4;
  // the last weight tiles of a row tile that the XCD before began, row tiles of its own, the first weight tiles of one more
  const int first_own = (low + n - 1) / n, begun = first_own * n - low, own = high / n - first_own, at = place - begun;
  if (at < 0) {
    tile = first_own - 1;
    n_tile = n + at;
  } else if (at < own * n) {
    const int first = at / (kTogether * n) * kTogether, in = at - first * n, together = min(kTogether, own - first);
    tile = first_own + first + in % together;
    n_tile = in / together;
  } else {
    tile = first_own + own;
    n_tile = at - own * n;
  }
}

struct TilePlace { int tile, n_tile, half; bool shared; };       // half: -1 a whole tile, 0 and 1 its halves of 128 rows

// The large tiles of an XCD and the order in which its workgroups take them: place j of all goes to workgroup j % groups.  The shared expert's tiles come
// first.  One whose K is longer stands for `units` rounds' places of its workgroup, of which the first is it and the others are nothing.  Where the
// experts' tiles leave a last round of no more than half its workgroups, that round's tiles are taken in halves, unless these push the tiles of
// few rows, which come behind them, into one round more.
struct LargeShare {
  int n_tiles, whole, low, high, rest_low, rest, sh_n_tiles, sh_low, sh, sh_rounds, sh_more, units, full, halved;
  bool walks;                                       // (otherwise there is a workgroup for every tile, and units is 1)

  EXPERT_TILES_FN LargeShare(int n_tiles_, int whole_, int rest_tiles, int sh_row_tiles, int sh_n_tiles_, int units_, int xcd, int groups)
      : n_tiles(n_tiles_), whole(whole_), sh_n_tiles(sh_n_tiles_), units(units_), walks(groups == kLargeGroups) {
    const int per = (whole * n_tiles + 7) / 8, rest_per = (rest_tiles * n_tiles + 7) / 8;
    low = min(xcd * per, whole * n_tiles);
    high = min(low + per, whole * n_tiles);
    rest_low = min(xcd * rest_per, rest_tiles * n_tiles);
    rest = min(rest_low + rest_per, rest_tiles * n_tiles) - rest_low;
    const int sh_all = sh_row_tiles * sh_n_tiles, sh_per = (sh_all + 7) / 8;
    sh_low = min(xcd * sh_per, sh_all);
    sh = min(sh_low + sh_per, sh_all) - sh_low;
    sh_rounds = walks ? sh / kLargeGroups * units : 0;
    sh_more = walks ? sh % kLargeGroups : sh;
    // places of a round beside the shared tiles' own, if all of the experts' tiles fit beside them, or the whole round's
    const int own = high - low, beside = walks ? kLargeGroups - sh_more : kLargeGroups;
    const bool fit = own <= units * beside;
    const int width = fit ? beside : kLargeGroups, last = fit ? own % width : (own + sh_more * units) % kLargeGroups, behind = last + rest;
    halved = 2 * last <= width && last <= own && (behind + last - 1) / width == (behind - 1) / width ? last : 0;
    full = own - halved;
  }
  // place j of the XCD's; false: there are no tiles there and behind it
  EXPERT_TILES_FN bool find(int j, TilePlace& t) const {
    t.shared = false;
    t.half = -1;
    if (sh > 0) {
      const int round = walks ? j / kLargeGroups : 0, of = j - round * kLargeGroups, in = round - sh_rounds;
      if (in < 0 || (in < units && of < sh_more)) {
        t.shared = true;
        pair_at(sh_n_tiles, sh_low, sh_low + sh, min(round, sh_rounds) / units * kLargeGroups + of, t.tile, t.n_tile);
        return true;
      }
      j -= sh_rounds * kLargeGroups + sh_more * min(in + 1, units);
    }
    if (j < full + 2 * halved) {
      const int over = j - full;
      if (over >= 0) t.half = over & 1;
      pair_at(n_tiles, low, high, over < 0 ? j : full + (over >> 1), t.tile, t.n_tile);
      return true;
    }
    const int behind = j - full - 2 * halved, at = rest_low + behind;
    t.tile = whole + at / n_tiles;
    t.n_tile = at % n_tiles;
    return behind < rest;
  }
};

}  // namespace mvllm
