// How a one-token decode step runs its attention.  Plain C++, checked on the CPU
// (tests/cpu/step_attn_check.cpp).
#pragma once

// Key splits (bucketed, so that one graph covers a range of lengths), whether the split partials
// stay for the O projection to merge while staging its activations (parts) or a reduce launch
// merges them, and, of the former alone, whether splits of at most 64 keys take the smaller
// launch shape.  key() names the captured graph: steps that enqueue the same launches share it.
struct StepAttn {
  int splits;
  bool short_splits, parts;
  int key() const { return 4 * splits + (parts ? 2 : 0) + (short_splits ? 1 : 0); }
};

inline StepAttn step_attn_of(int want, bool parts, int max_splits, int active_len) {
  int bucket = 1;
  while (bucket < want) bucket <<= 1;
  if (bucket > max_splits) bucket = max_splits;
  return {bucket, parts && active_len <= 64 * bucket, parts};
}
