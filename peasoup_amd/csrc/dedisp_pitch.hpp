// dedisp_pitch.hpp - how much of a channel's row a group of DM trials reads
// (host only, no HIP).
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

namespace psx {

constexpr int kTileSamps = 1024;  // output samples per tile of the dedispersion

// Dwords per shifted copy for groups of `per` DM trials of an ascending list
// (0: does not ascend): delays of one channel differ inside a group by at most
// the DM difference times the largest table entry tmax, plus the roundings of
// both delays: to whole samples, and of the float products dm * table[c], half
// an ulp each (past 2^24 samples of delay more than the whole samples': with 2
// for all of them stretches were too short from 2^28 on).
inline uint32_t staged_pitch(const float* dm, uint32_t ndm, uint32_t per, float tmax) {
  double spread = 0;
  for (uint32_t d = 1; d < ndm; ++d)
    if (!(dm[d] >= dm[d - 1])) return 0;
  for (uint32_t g = 0; g < ndm; g += per) {
    const double lo = dm[g], hi = dm[std::min(g + per, ndm) - 1];
    spread = std::max(spread, (hi - lo) * (double)tmax * (1 + 1e-6) + 2 + hi * (double)tmax * 0x1p-23);
  }
  // the tile, the spread, one dword past them for the shifts, whole 16-byte steps
  const double dwords = std::ceil((kTileSamps + spread) / 4) + 1;
  return dwords > 1e6 ? UINT32_MAX : ((uint32_t)dwords + 3) / 4 * 4;
}

}  // namespace psx
