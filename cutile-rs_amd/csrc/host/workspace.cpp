// Device memory for launches whose workgroups add up partial sums of one output block (split K).
//
// One workspace per (device, stream), allocated at the first launch that wants one and kept: launches on a stream run one
// after another, so its workspace has one user at a time, from whatever host thread they were enqueued, and different
// streams never share one.  A stream handle names another stream only after the runtime has drained and freed the first.
// At most kMaxWorkspaces per device (16 MiB each); cutile_stream_release gives back the one of its stream.  Where there is
// none to be had, the caller launches its unsplit form: beyond the limit, while the stream is being captured (a graph may
// be replayed on another stream beside eager work on this one), and on the per-thread default stream (one handle, many streams).
#include "runtime_state.h"

namespace cutile {
namespace {
constexpr size_t kMaxWorkspaces = 16;
}

cutile_status_t split_workspace(cutile_device_t device, hipStream_t stream, SplitWorkspace* out) {
  *out = {};
  CUTILE_API_OR_RETURN(api);
  if (stream == hipStreamPerThread) return CUTILE_SUCCESS;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  CUTILE_HIP_OR_RETURN(api, hipStreamIsCapturing(stream, &capture));
  if (capture != hipStreamCaptureStatusNone) return CUTILE_SUCCESS;
  std::lock_guard<std::mutex> lock(device->mutex);
  auto it = device->split_workspaces.find(stream);
  if (it == device->split_workspaces.end()) {
    if (device->split_workspaces.size() >= kMaxWorkspaces) return CUTILE_SUCCESS;
    void* p = nullptr;
    CUTILE_HIP_OR_RETURN(api, hipMallocAsync(&p, kSplitCounters * sizeof(uint32_t) + kSplitPartialBytes, stream));
    const hipError_t e = api->hipMemsetD8Async((hipDeviceptr_t)p, 0, kSplitCounters * sizeof(uint32_t), stream);
    if (e != hipSuccess) {
      api->hipFreeAsync(p, stream);
      return from_hip(e, "hipMemsetD8Async");
    }
    it = device->split_workspaces.emplace(stream, p).first;
  }
  out->counters = (uint32_t*)it->second;
  out->partials = (float*)((unsigned char*)it->second + kSplitCounters * sizeof(uint32_t));
  return CUTILE_SUCCESS;
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
