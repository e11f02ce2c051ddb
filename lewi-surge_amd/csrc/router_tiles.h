// Tile sizes of the fused router (router_fused_kernel<E, TT, HT, DC>, described there) for t tokens of depth d and e
// experts.  The rule alone, without device code: the tests compile it for the host, to see that their shapes reach
// every instantiation.
#pragma once
#include <stdint.h>

namespace lsurge {

struct RouterTiles {
  int tt, ht, dc;  // token tiles and expert tiles of a wave, depth of x's chunks in LDS
};

inline RouterTiles router_tiles(int64_t t, int64_t d, int64_t e) {
  const int64_t chunks = (t + 63) / 64, per16 = chunks * 4 * (e / 32);  // waves at one token tile and two expert tiles
  // token tiles per wave: the largest of 4, 2, 1 that leaves two waves per SIMD (2048).  Measured alone, at 1 / 2 /
  // 4: T = 4096, E = 64 20 / - / 55 us; T = 16384, E = 64 30 / 32 / 57; T = 16384, E = 128 53 / 49 / 80; T = 65536,
  // E = 256, d = 2048 700 / 629 / 613
  const int tt = per16 / 4 >= 2048 ? 4 : per16 / 2 >= 2048 ? 2 : 1;
  // one expert tile a wave while its waves (E / 16 a workgroup) have a SIMD each: the logits' chain is then half as
  // many matrix steps.  Alone, cold: T = 64 / 1024 / 4096, E = 64 20.5 / 19.8 / 20.4 -> 15.6 / 15.0 / 16.1 us; T = 64,
  // E = 32 18.5 -> 13.9.  With more waves than SIMDs the steps only move between waves (T = 16384, E = 64 34 -> 37
  // us; E = 128, whose eight waves share a CU's four SIMDs, 20.6 -> 20.5)
  const bool narrow = e <= 64 && chunks * 4 * (e / 16) <= 1024;
  return {tt, narrow ? 1 : 2, d % 128 == 0 ? 128 : 64};
}

}  // namespace lsurge
