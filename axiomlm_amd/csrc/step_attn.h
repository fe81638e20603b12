// How a one-token decode step runs its attention.  Plain C++, checked on the CPU
// (tests/cpu/step_attn_check.cpp).
#pragma once

// Key splits (bucketed, so that one graph covers a range of lengths), whether the split partials
// stay for the O projection to merge while staging its activations (parts) or a reduce launch
// merges them, of the former alone, whether splits of at most 64 keys take the smaller
// launch shape, and whether grouped-query heads keep their softmax weights in fp32 (p32).  key()
// names the captured graph: steps that enqueue the same launches share it.
struct StepAttn {
  int splits;
  bool short_splits, parts, p32;
  int key() const { return 8 * splits + (p32 ? 4 : 0) + (parts ? 2 : 0) + (short_splits ? 1 : 0); }
};

// grouped: two to sixteen query heads per KV head, without parts.
inline StepAttn step_attn_of(int want, bool parts, bool grouped, int max_splits, int active_len) {
  int bucket = 1;
  while (bucket < want) bucket <<= 1;
  if (bucket > max_splits) bucket = max_splits;
  // Under 32 keys fp16 weights, as in the batched decode attention (20 keys, per layer: 41.4 us, fp32 42.0).
  return {bucket, parts && active_len <= 64 * bucket, parts, grouped && active_len >= 32};
}
