// Launch order of a tiled product, over rows that may be sorted by expert.
#pragma once
#include "common.h"

namespace jla {

// launch-order tile index -> (m tile, n tile), M-grouped by gm so that neighbouring workgroups share weight columns
JLA_DEV void row_tile_coords(int pid, int tiles_m, int tiles_n, int gm, int& tm, int& tn) {
  const int in_group = gm * tiles_n;
  const int first_m = (pid / in_group) * gm;
  const int gsz = min(tiles_m - first_m, gm);
  tm = first_m + (pid % in_group) % gsz;
  tn = (pid % in_group) / gsz;
}

// This workgroup's expert e, its rows [r0, rend) and column tile; false: no such tile. offs [E + 1] (or nullptr: R rows of one
// matrix) bounds the experts' rows. Workgroups are dealt round robin to the 8 XCDs, so XCD x takes the x-th eighth of the
// order (expert by expert, groups of 4 m-tiles across every column tile): the tiles that run side by side behind one L2
// share weight columns and activation rows. Every wave computes the same answer: lane l looks at experts l, l + 64, ...
// The grid is a multiple of 8 and at least the number of tiles. With splits, every tile is there that many times, one split after the
// other in the order, so that an XCD's share of all of them is even (81 tiles in three splits: 31 workgroups at most behind an XCD,
// where three launches' eighths of 81 would put 33 on its 32 units).
template <int BM>
JLA_DEV bool row_tile(const int32_t* offs, int experts, int R, int tiles_n, int lane, int& e, int& r0, int& rend, int& tn, int splits,
                      int& split) {
  const int E = offs ? experts : 1;
  auto rows = [&](int x) { return x < E ? (offs ? offs[x + 1] - offs[x] : R) : 0; };
  int total = 0;
  for (int b = 0; b < E; b += 64) {
    int n = (rows(b + lane) + BM - 1) / BM;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    total += n;
  }
  total *= tiles_n;
  const int per = (total * splits + 7) / 8, at = blockIdx.x >> 3;
  int pid = (int)(blockIdx.x & 7) * per + at;
  if (at >= per || pid >= total * splits) return false;
  split = pid / max(total, 1);
  pid -= split * total;
  int before = 0;  // m-tiles of the experts passed
  for (int b = 0; b < E; b += 64) {
    const int n = (rows(b + lane) + BM - 1) / BM;
    int inc = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    const unsigned long long hit = __ballot(pid < (before + inc) * tiles_n);
    if (hit) {
      const int src = (int)__builtin_ctzll(hit);
      e = __builtin_amdgcn_readfirstlane(b + src);
      const int mine = __builtin_amdgcn_readlane(n, src);
      const int start = (before + __builtin_amdgcn_readlane(inc, src) - mine) * tiles_n;
      int tm;
      row_tile_coords(pid - start, mine, tiles_n, 4, tm, tn);
      r0 = (offs ? offs[e] : 0) + tm * BM;
      rend = offs ? offs[e + 1] : R;
      return true;
    }
    before += __builtin_amdgcn_readlane(inc, 63);
  }
  return false;
}
template <int BM>
JLA_DEV bool row_tile(const int32_t* offs, int experts, int R, int tiles_n, int lane, int& e, int& r0, int& rend, int& tn) {
  int split;
  return row_tile<BM>(offs, experts, R, tiles_n, lane, e, r0, rend, tn, 1, split);
}

}  // namespace jla
