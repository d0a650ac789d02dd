// The resident loop's exchange on the CPU (cvo_exchange.h): one word missing on
// each line in turn must end the wait for the whole wave.  Prints the number of
// cases; exit code 1 and the case when one is missed.
#include <array>
#include <cstdio>
#include <vector>

#include "../../rkhs_ba_amd/csrc/cvo_exchange.h"

namespace {

constexpr uint32_t kTag = 7;

template <int PER>
struct CpuWave {
  static constexpr int kWords = PER;
  uint64_t v[64][PER];
  bool lane_ok[64];
  template <class F>
  void each(F f) {
    for (int l = 0; l < 64; ++l) f(l, v[l]);
  }
  template <class F>
  bool every(F f) {
    bool all = true;
    for (int l = 0; l < 64; ++l) {
      lane_ok[l] = f(l, v[l]);
      all = all && lane_ok[l];
    }
    return all;
  }
};

int g_cases = 0, g_hidden = 0;

// NW, USED: words of a line; LINES: lines a reader covers; n: lines in use.
template <int NW, int USED, int LINES>
bool check(int n) {
  constexpr int PER = (LINES * NW + 63) / 64;
  CpuWave<PER> wave;
  std::vector<uint64_t> words((size_t)LINES * NW, ~0ull);  // not the tag: never to be waited for
  for (int l = 0; l < n; ++l)
    for (int w = 0; w < USED; ++w) words[l * NW + w] = ((uint64_t)kTag << 32) | (uint32_t)(100 * l + w);
  uint64_t ticks = 1;
  auto clock = [&]() { return ticks++; };
  auto load = [&](int i) { return words[i]; };
  for (uint64_t wait : {(uint64_t)0, (uint64_t)5}) {
    ++g_cases;
    if (!cvo::read_words<NW, USED>(wave, n, kTag, wait, load, clock)) {
      std::printf("NW %d lines %d: all words there, wait reported out\n", NW, n);
      return false;
    }
    for (int l = 0; l < 64; ++l)
      for (int u = 0; u < PER; ++u) {
        const int i = l + 64 * u;
        if ((l & (NW - 1)) < USED && i < n * NW && wave.v[l][u] != words[i]) {
          std::printf("NW %d lines %d: word %d read wrong\n", NW, n, i);
          return false;
        }
      }
    for (int line = 0; line < n; ++line) {
      ++g_cases;
      std::vector<uint64_t> full = words;
      // a late block has written none of its words, the last of a line none
      for (int w = line % 2 ? 0 : USED - 1; w < USED; ++w) words[line * NW + w] = ((uint64_t)(kTag - 1) << 32) | 5u;
      const bool ok = cvo::read_words<NW, USED>(wave, n, kTag, wait, load, clock);
      words = full;
      if (ok) {
        std::printf("NW %d lines %d wait %d: line %d missing, wait not reported out\n", NW, n, (int)wait, line);
        return false;
      }
      g_hidden += wave.lane_ok[0];
    }
  }
  // a word that comes while the wave waits
  for (int line = 0; line < n; ++line) {
    ++g_cases;
    int reads = 0;
    auto late = [&](int i) { return i / NW == line && ++reads <= 200 ? 0ull : words[i]; };
    if (!cvo::read_words<NW, USED>(wave, n, kTag, 1000, late, clock)) {
      std::printf("NW %d lines %d: line %d late, wait reported out\n", NW, n, line);
      return false;
    }
  }
  return true;
}

}  // namespace

int main() {
  bool ok = true;
  for (int n : {1, 2, 5, 8, 31, 32}) {
    ok = ok && check<16, 14, 32>(n);  // a registration's association
    ok = ok && check<32, 22, 32>(n);  // with its self problems
    ok = ok && check<8, 8, 32>(n);    // the step
  }
  for (int n : {8}) {  // the groups' lines
    ok = ok && check<16, 14, 8>(n);
    ok = ok && check<32, 22, 8>(n);
    ok = ok && check<8, 8, 8>(n);
  }
  // lines whose absence lane 0 does not see
  if (g_hidden == 0) ok = false;
  std::printf("%d cases, %d unseen by lane 0\n", g_cases, g_hidden);
  return ok ? 0 : 1;
}
