// Graph keys of decode steps (axiomlm_amd/csrc/step_attn.h): for the splits of each attention form over
// all lengths, a key is new only where the launches differ.
#include <cstdio>
#include <map>

#include "step_attn.h"

// Keys over lengths 1..n of a split rule.
template <typename F>
static int keys(F splits, bool parts_form, bool grouped, int n) {
  std::map<int, StepAttn> seen;
  for (int len = 1; len <= n; ++len) {
    const int want = splits(len);
    const StepAttn a = step_attn_of(want, parts_form && want > 1, grouped, 64, len);
    const auto it = seen.emplace(a.key(), a).first;
    if (it->second.splits != a.splits || it->second.parts != a.parts || it->second.short_splits != a.short_splits ||
        it->second.p32 != a.p32)
      return -1;
  }
  return (int)seen.size();
}

int main() {
  // Merged by a reduce launch: 1 split to 256 keys, under 32 with fp16 weights, then 4 to 32 doubling: one graph each.
  const int reduce = keys([](int len) {
    int s = len <= 256 ? 1 : 4;
    while (s > 1 && s < 32 && 128 * s < len) s <<= 1;
    return s;
  }, false, true, 20000);
  // Merged by the O projection: 1, 2, 4, 8 splits, those over one split with a short and a long shape.
  const int parts = keys([](int len) {
    int s = 8;
    while (s > 1 && len < 16 * s) s >>= 1;
    return s;
  }, true, false, 20000);
  std::printf("%d %d\n", reduce, parts);
  return reduce == 6 && parts == 5 ? 0 : 1;  // (2 and 4 splits are always short ones)
}
