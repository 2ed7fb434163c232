// Process-global runtime objects behind the opaque C handles.
#pragma once
#include <atomic>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "common.h"

struct cutile_module {
  struct cutile_device* device = nullptr;
  hipModule_t handle = nullptr;
};

// One per device ordinal, created on first use and kept for the life of the
// process (cuda-core/src/runtime.rs:126-139 keeps one Device per ordinal).
struct cutile_device {
  int ordinal = 0;
  std::mutex mutex;
  std::vector<hipStream_t> idle_streams;  // released streams, reused before creating new ones
  uint64_t streams_created = 0;
  std::atomic<int> compute_units{0};  // filled on first use by compute_units()
  std::map<hipStream_t, void*> split_workspaces;   // workspace.cpp
  uint32_t split_retry_after = 0;                  // launches to go before a refused workspace is asked for again
  // Code objects of the kernel table loaded on this device: image id -> module.
  std::map<int, cutile_module*> table_modules;
  // Resolved functions: symbol -> hipFunction_t.
  std::map<std::string, hipFunction_t> functions;
  // The same by position in the kernel table, readable without the mutex (one slot per table entry, made with the device).
  std::unique_ptr<std::atomic<hipFunction_t>[]> function_slots;
};

namespace cutile {

cutile_status_t ensure_init();
void count_module_load();
void reset_runtime_for_testing();
void reset_async_runtime_for_testing();
// Device the calling thread is bound to (hipGetDevice), as a handle.
cutile_status_t current_device(cutile_device_t* device);
// Where the workgroups of a launch that splits the K axis of one output block leave their partial sums (workspace.cpp).
constexpr size_t kSplitCounters = 4096;                  // output blocks of one launch
constexpr size_t kSplitPartialBytes = 40u << 20;   // beyond it sharing K gains little (1500 x 4096 x 14336 f16 on 48 MiB 161 us, unshared 164)
struct SplitWorkspace {
  float* partials = nullptr;      // nullptr: none to be had, the launch must not split
  uint32_t* counters = nullptr;   // kSplitCounters words, all 0 between launches
};
SplitWorkspace split_workspace(cutile_device_t device, hipStream_t stream);
void release_split_workspace(cutile_device_t device, hipStream_t stream);
// The device of that ordinal if cutile_device_get has handed it out before, else nullptr.
cutile_device_t known_device(int ordinal);
// Compute units of the device (cached).
cutile_status_t compute_units(cutile_device_t device, int* count);

}  // namespace cutile
