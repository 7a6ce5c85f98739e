// nan_screen.hip -- rejects float point sets that contain NaN coordinates
// before a single-tree build touches them.
//
// The reference's comparator is a plain '<' on coordinates
// (builder_thrust.h:401-404), which is no strict weak order once a NaN is
// present, so its result is undefined there.  cukd_build_tree screens the
// coordinates first and returns CUKD_ERR_INVALID, leaving the array as it
// was.  The result word of each call lives in pinned host memory of the
// library's own (one 256-byte line per slot, allocated once), so no builder,
// the in-place one included, allocates device memory for it, and reading it
// needs no copy: the scan stores to it only where it finds a NaN, and the
// wait for the stream makes that store visible.  The scan and the wait are
// two calls, so that a builder plans and allocates while the scan runs.
#include <condition_variable>
#include <mutex>

#include "cukd_common.h"

namespace cukd_amd {

enum { NAN_SLOTS = 64, NAN_SLOT_WORDS = 64 };


// One thread per element (grid-stride): any NaN coordinate sets the flag.
__global__ __launch_bounds__(256) void k_nan_scan(const uint8_t *points, long long n,
                                                  cukd_layout L, uint32_t *flag)
{
  bool bad = false;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const uint8_t *e = points + i * L.stride;
    for (int d = 0; d < L.num_dims; d++) {
      const uint32_t b = load_coord_bits(e, L, d);
      bad |= (b & 0x7f800000u) == 0x7f800000u && (b & 0x007fffffu) != 0u;
    }
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) flag[0] = 1u;
}

namespace {

std::mutex g_mu;
std::condition_variable g_cv;
uint64_t g_busy = 0;       // slots in use, one bit each
uint32_t *g_slots = nullptr;  // pinned host memory, readable by every device

int slot_base(uint32_t **base)
{
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_slots) {
#ifdef hipHostMallocPortable
    const unsigned flags = hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent;
#else
    const unsigned flags = hipHostMallocDefault;
#endif
    void *p = nullptr;
    CUKD_HIP(hipHostMalloc(&p, NAN_SLOTS * NAN_SLOT_WORDS * 4, flags));
    g_slots = (uint32_t *)p;
  }
  *base = g_slots;
  return CUKD_OK;
}

int take_slot()
{
  std::unique_lock<std::mutex> lk(g_mu);
  g_cv.wait(lk, [] { return g_busy != ~0ull; });
  const int s = __builtin_ctzll(~g_busy);
  g_busy |= 1ull << s;
  return s;
}

void give_slot(int s)
{
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_busy &= ~(1ull << s);
  }
  g_cv.notify_one();
}

}  // namespace

// Launches the scan.  Under stream capture nothing is screened (a capture
// cannot wait for a result), nor for int layouts.
int NanScreen::begin(const void *d_points, int n, const cukd_layout &L, hipStream_t s)
{
  if (L.scalar_type != CUKD_SCALAR_F32 || n < 1) return CUKD_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  CUKD_HIP(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone) return CUKD_OK;
  uint32_t *base = nullptr;
  if (int rc = slot_base(&base)) return rc;
  stream = s;
  slot = take_slot();
  volatile uint32_t *flag = base + slot * NAN_SLOT_WORDS;
  *flag = 0u;
  const long long blocks = ((long long)n + 255) / 256;
  hipLaunchKernelGGL(k_nan_scan, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s,
                     (const uint8_t *)d_points, (long long)n, L, base + slot * NAN_SLOT_WORDS);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return CUKD_OK;
  give_slot(slot);
  slot = -1;
  set_last_error("NaN screen failed: %s", hipGetErrorString(e));
  return CUKD_ERR_HIP;
}

// Waits for the scan: CUKD_OK when no coordinate is NaN, CUKD_ERR_INVALID when
// one is.
int NanScreen::end()
{
  if (slot < 0) return CUKD_OK;
  const hipError_t e = hipStreamSynchronize(stream);
  const uint32_t h = *(volatile uint32_t *)(g_slots + slot * NAN_SLOT_WORDS);
  give_slot(slot);
  slot = -1;
  if (e != hipSuccess) {
    set_last_error("NaN screen failed: %s", hipGetErrorString(e));
    return CUKD_ERR_HIP;
  }
  if (h) {
    set_last_error("points contain NaN coordinates (no strict weak order for the "
                   "builder's '<' comparison); the array is left unchanged");
    return CUKD_ERR_INVALID;
  }
  return CUKD_OK;
}

}  // namespace cukd_amd
