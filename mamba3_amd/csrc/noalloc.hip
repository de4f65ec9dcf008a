// m3_scan_fwd_noalloc: the chunked scan with the library's own device scratch in place of a
// caller-allocated workspace, for callers that cannot allocate device memory.
//
// The scratch is one file-scope __device__ array of M3_SCRATCH_BYTES per GPU, alive until the
// process ends. Host code never passes the array's name to a kernel (on the host it names a
// stand-in, not device memory): the first call on each device looks up the array's device
// address with hipGetSymbolAddress, with that device current, and keeps it; every later call on
// that device passes the kept address as the scan's workspace.
//
// The scan's workspace needs no clearing between calls: prep writes every region the scan reads
// (the RMSNorm factors or q / k rows, the angle tiles, the scalar blocks), and a split call's segment buffers
// are written by its pass 1 and composition before pass 2 reads them. So nothing is zeroed here,
// and no call allocates, frees or synchronises.
#include <hip/hip_runtime.h>

#include <mutex>

#include "m3_host.hpp"

namespace m3 {
namespace {

__device__ __align__(256) unsigned char scratch[M3_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device (looked up once per device).
int scratch_address(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    return fail(M3_ELAUNCH, "m3_scan_fwd_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  }
  if (dev < 0 || dev >= kMaxDevices) {
    return fail(M3_EUNSUPPORTED, "m3_scan_fwd_noalloc: device %d >= %d", dev, kMaxDevices);
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      return fail(M3_ELAUNCH, "m3_scan_fwd_noalloc: hipGetSymbolAddress: %s",
                  hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return M3_OK;
}

}  // namespace
}  // namespace m3

extern "C" int m3_scan_fwd_noalloc(const m3_scan_args* args, hipStream_t stream) {
  using namespace m3;
  clear_error();
  if (args == nullptr) return fail(M3_EINVAL, "m3_scan_fwd_noalloc: args is NULL");
  // The call as m3_scan_fwd would run it, or, where that outgrows the scratch, the first of these
  // that fits: by the routes that need less (no copies of the q / k rows), still split; unsplit;
  // unsplit by the routes that need less; the recurrent scan, which needs nothing (a d_state that
  // is no power of 2). The split goes last but for the recurrent scan: 1 x 65,536 tokens of 24
  // heads, hook form, split 536 us and unsplit 2,618.
  m3_scan_args a = *args;
  const size_t want = scan_need(a, true);
  struct Try {
    bool rows;
    int segments;
  };
  const Try tries[] = {{true, a.segments}, {false, a.segments}, {true, 1}, {false, 1}};
  const int n = a.segments == 0 ? 4 : 2;
  int pick = -1;
  for (int i = 0; i < n && pick < 0; ++i) {
    a.segments = tries[i].segments;
    const size_t need = scan_need(a, tries[i].rows);
    // (nothing needed where a workspace was asked for: the recurrent scan)
    if (need <= M3_SCRATCH_BYTES && (need > 0 || want == 0 || i == n - 1)) pick = i;
  }
  if (pick < 0) {
    return fail(M3_EWORKSPACE,
                "m3_scan_fwd_noalloc: the call needs %zu bytes of scratch, above the %u-byte "
                "maximum (use m3_scan_fwd with a workspace)",
                want, static_cast<unsigned>(M3_SCRATCH_BYTES));
  }
  a.segments = tries[pick].segments;
  void* ptr = nullptr;
  const int rc = scratch_address(&ptr);
  if (rc != M3_OK) return rc;
  a.workspace = ptr;
  a.workspace_bytes = M3_SCRATCH_BYTES;
  return scan_run(a, tries[pick].rows, stream);
}
