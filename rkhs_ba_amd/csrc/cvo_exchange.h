// Reading the words of an exchange between resident blocks (cvo_loop.hip): plain
// C++ over a wave given by its caller, so that a CPU build runs the same code.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define CVO_WAVE_FN __device__ __forceinline__
#else
#define CVO_WAVE_FN inline
#endif

namespace cvo {

// The wave's lanes read n_lines lines of NW words, USED of them published: lane
// l's v[u] is word l + 64 u.  Words that do not carry the tag in their upper half
// are loaded again until all do.  The decision is the wave's, not the lane's:
// false when the wait runs out before every lane has its words, whichever line
// is late.
template <int NW, int USED, class Wave, class Load, class Clock>
CVO_WAVE_FN bool read_words(Wave& wave, int n_lines, uint32_t tag, uint64_t wait_ticks, Load load, Clock clock) {
  wave.each([&](int lane, auto& v) {
    const int n = (lane & (NW - 1)) < USED ? n_lines * NW : 0;
#pragma unroll
    for (int u = 0; u < Wave::kWords; ++u) {
      const int i = lane + u * 64;
      v[u] = (uint64_t)tag << 32;
      if (i < n) v[u] = load(i);
    }
  });
  uint64_t t0 = 0;
  for (uint32_t tries = 0;; ++tries) {
    const bool all = wave.every([&](int, auto& v) {
      bool there = true;
#pragma unroll
      for (int u = 0; u < Wave::kWords; ++u) there = there && (uint32_t)(v[u] >> 32) == tag;
      return there;
    });
    if (all) return true;
    // only the words still missing
    wave.each([&](int lane, auto& v) {
#pragma unroll
      for (int u = 0; u < Wave::kWords; ++u)
        if ((uint32_t)(v[u] >> 32) != tag) v[u] = load(lane + u * 64);
    });
    // the clock's own read costs as much as a poll: every 64th (a wait of 0 ends
    // at the first missing word)
    if ((tries & 63) == 63 || wait_ticks == 0) {
      const uint64_t now = clock();
      if (t0 == 0) t0 = now;
      if (now - t0 >= wait_ticks) return false;
    }
  }
}

}  // namespace cvo
