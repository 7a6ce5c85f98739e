// multiround.hip -- final extraction of persistent multi-round kNN lists
// (extractFinalResult, samples/mpiHugeQuery.cu:90-103).
#pragma clang fp contract(off)

#include "cukd_common.h"
#include "query_impl.h"

namespace cukd_amd {

// radius = sqrt(max dist2) unless infinite, as the reference; ids/dist2 (each
// nullable) get the k entries in ascending (dist2, id) order.  One entry per
// lane, as many whole lists as fit a workgroup: an entry's place is the
// number of entries before it, counted over the list in LDS, so the lists
// are read and written coalesced.  (250K lists of 20: 324 -> 28 us; one
// list per lane sorted by insertion in scratch.)
enum { EX_NT = 256 };
__global__ __launch_bounds__(EX_NT) void k_knn_extract(const uint64_t *lists, int nq, int k,
                                                       int32_t *ids, float *dist2, float *radius)
{
  __shared__ uint64_t s_in[EX_NT], s_out[EX_NT];
  const int per = EX_NT / k, tid = (int)threadIdx.x;
  const long long q0 = (long long)blockIdx.x * per;
  const int live = q0 + per <= nq ? per * k : (int)(nq - q0) * k;
  const size_t at = (size_t)q0 * k + tid;
  uint64_t v = 0;
  if (tid < live) s_in[tid] = v = lists[at];
  __syncthreads();
  const int first = tid / k * k, mine = tid - first;
  if (tid < live && (ids || dist2)) {
    int before = 0;
    for (int j = 0; j < k; j++) {
      const uint64_t o = s_in[first + j];
      before += (o < v || (o == v && j < mine)) ? 1 : 0;
    }
    s_out[first + before] = v;
  }
  __syncthreads();
  if (tid >= live) return;
  if (radius && mine == 0) {
    const float m = __uint_as_float((uint32_t)(v >> 32));
    radius[q0 + tid / k] = isinf(m) ? m : sqrtf(m);
  }
  if (!ids && !dist2) return;
  const uint64_t e = s_out[tid];
  if (ids) ids[at] = (int32_t)(uint32_t)e;
  if (dist2) dist2[at] = __uint_as_float((uint32_t)(e >> 32));
}

hipError_t launch_knn_extract(const uint64_t *lists, int nq, int k, int32_t *ids, float *dist2,
                              float *radius, hipStream_t s)
{
  const int per = EX_NT / k;
  hipLaunchKernelGGL(k_knn_extract, dim3((nq + per - 1) / per), dim3(EX_NT), 0, s, lists, nq, k,
                     ids, dist2, radius);
  return hipGetLastError();
}

}  // namespace cukd_amd
