// Which keys the workgroups of an attention launch take: shared by the kernels of fmha_keys.hip and by the launcher, which plans with the same
// numbers.  A workgroup too few, or one that counts others than there are, would leave a query tile without a result and its counter in the
// stream's workspace short for good.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define CUTILE_KEYS_FN __host__ __device__ inline
#else
#define CUTILE_KEYS_FN inline
#endif

namespace cutile {

// Keys that any of the query rows before `end_row` sees (rows that are not there see none), the first row standing behind `input_pos` keys.
CUTILE_KEYS_FN int32_t keys_seen(int32_t end_row, int32_t q_len, int32_t input_pos, int32_t k_len, int32_t causal) {
  const uint32_t past = (uint32_t)input_pos + (uint32_t)(end_row < q_len ? end_row : q_len);
  return causal && past < (uint32_t)k_len ? (int32_t)past : k_len;
}

// The key steps [first, end) of workgroup `z` of the `launched` that a query tile has, `each` to a workgroup, and how many of them have any.  The last one takes
// what is left, so that every step has its workgroup whatever the launcher counted on.
struct KeySteps {
  int32_t first, end;
  uint32_t shares;
};
CUTILE_KEYS_FN KeySteps key_steps(int32_t keys, int32_t step, int32_t each, uint32_t z, uint32_t launched) {
  const int32_t all = (keys + step - 1) / step, first = (int32_t)z * each;
  const uint32_t wanted = (uint32_t)((all + each - 1) / each);
  return {first, z + 1 < launched && all - first > each ? first + each : all, wanted < launched ? wanted : launched};
}

}  // namespace cutile
