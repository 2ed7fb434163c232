// Device memory for launches whose workgroups add up partial sums of one output block (split K).
//
// One workspace per (device, stream), allocated at the first launch that wants one and kept: launches on a stream run one
// after another, so its workspace has one user at a time, from whatever host thread they were enqueued, and different
// streams never share one.  A stream handle names another stream only after the runtime has drained and freed the first.
// At most kMaxWorkspaces per device (40 MiB each); cutile_stream_release gives back the one of its stream.  Where there is
// none to be had, the caller launches its unsplit form: beyond the limit, while the stream is being captured (a graph may
// be replayed on another stream beside eager work on this one), on the per-thread default stream (one handle, many streams),
// and where the runtime refuses the memory (another allocator may hold the card): a product needs none to be computed.
#include "runtime_state.h"

namespace cutile {
namespace {
// More than the 32 streams that torch's pool deals out on a device, its default stream and as many of a program's own: a
// stream made elsewhere keeps its workspace until the process ends (nothing tells this library that it is gone).  2.5 GiB at most.
constexpr size_t kMaxWorkspaces = 64;
// After a refused allocation this many launches of streams without a workspace go ahead unsplit before it is asked for again:
// a request that fails costs more than the launch.
constexpr uint32_t kRetryAfter = 256;

// The runtime's own record of a refusal that is dealt with here: the next call of somebody else would report it.
SplitWorkspace none_to_be_had(const HipApi* api) {
  api->hipGetLastError();
  return {};
}
}  // namespace

SplitWorkspace split_workspace(cutile_device_t device, hipStream_t stream) {
  const HipApi* api = hip();
  if (!api || stream == hipStreamPerThread) return {};
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (api->hipStreamIsCapturing(stream, &capture) != hipSuccess) return none_to_be_had(api);   // the launch itself will say why
  if (capture != hipStreamCaptureStatusNone) return {};
  std::lock_guard<std::mutex> lock(device->mutex);
  auto it = device->split_workspaces.find(stream);
  if (it == device->split_workspaces.end()) {
    if (device->split_workspaces.size() >= kMaxWorkspaces) return {};
    if (device->split_retry_after > 0) {
      --device->split_retry_after;
      return {};
    }
    void* p = nullptr;
    if (api->hipMallocAsync(&p, kSplitCounters * sizeof(uint32_t) + kSplitPartialBytes, stream) != hipSuccess) {
      device->split_retry_after = kRetryAfter;
      return none_to_be_had(api);
    }
    if (api->hipMemsetD8Async((hipDeviceptr_t)p, 0, kSplitCounters * sizeof(uint32_t), stream) != hipSuccess) {
      api->hipFreeAsync(p, stream);
      device->split_retry_after = kRetryAfter;
      return none_to_be_had(api);
    }
    it = device->split_workspaces.emplace(stream, p).first;
  }
  SplitWorkspace ws;
  ws.counters = (uint32_t*)it->second;
  ws.partials = (float*)((unsigned char*)it->second + kSplitCounters * sizeof(uint32_t));
  return ws;
}

void release_split_workspace(cutile_device_t device, hipStream_t stream) {
  const HipApi* api = hip();
  std::lock_guard<std::mutex> lock(device->mutex);
  auto it = device->split_workspaces.find(stream);
  if (it == device->split_workspaces.end()) return;
  if (api) api->hipFreeAsync(it->second, stream);   // after what the stream still has to run
  device->split_workspaces.erase(it);
}

}  // namespace cutile
