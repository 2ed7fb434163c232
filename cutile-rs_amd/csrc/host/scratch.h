// Size of the device-resident scratch array (scratch.hip) and the one function the
// side library libcutile_hip_scratch.so exports.
#pragma once
#include <stddef.h>

// 8 MiB of partial results per GPU, held from the first call on that GPU until the process ends.
#define CUTILE_SCRATCH_BYTES (8u << 20)
// Behind them, counters that are 0 between launches (the array starts as zeros): CUTILE_SCRATCH_REGIONS sets that launches
// take in turn, a counter per KV head (fmha.hip, merge_if_last).
#define CUTILE_SCRATCH_REGIONS 64u
#define CUTILE_SCRATCH_HEADS 64u
#define CUTILE_SCRATCH_COUNTER_BYTES (CUTILE_SCRATCH_REGIONS * CUTILE_SCRATCH_HEADS * 4u)

#define CUTILE_SCRATCH_LIBRARY "libcutile_hip_scratch.so"
#define CUTILE_SCRATCH_LOOKUP_SYMBOL "cutile_scratch_lookup"

#ifdef __cplusplus
extern "C"
#endif
int cutile_scratch_lookup(void** device_ptr, size_t* bytes, int* device_ordinal);
