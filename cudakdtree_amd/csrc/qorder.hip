// qorder.hip -- Morton ordering of query batches (CUKD_QUERY_SORT).
//
// Queries are bucketed by a Morton code of their position inside the
// batch's bounding box (MORTON_BITS bits spread evenly over the dims), so
// the lanes of a wave start from nearby points and walk mostly the same
// tree nodes.  Only the launch order changes: every query's result is
// written at its own index, so results are identical with and without
// ordering.  Order inside a cell is whatever the atomics give; it affects
// speed, never results.
//
// A counting sort without returning global atomics: each tile of queries
// counts its cells in LDS (k_qcount), one thread per cell turns the
// per-tile counts into per-tile starts, up to the cells of earlier blocks
// (k_qcolscan), and each tile then places its queries from its starts with
// LDS atomics (k_qplace).
//
// Bound by latency: a few LDS and memory rounds per kernel.  1M float3 queries:
// 78 -> 63 us, 250K: 66 -> 45 us, where every workgroup had read the cell totals
// at a stride of 128 bytes to scan them itself, into LDS columns of one
// bank, and 16K-query tiles left most CUs idle.
#include "cukd_common.h"

namespace cukd_amd {

// 15-bit cells: on a 10M-point tree, kNN-8 over 1M uniform queries took
// 0.789 / 0.764 / 0.747 / 0.737 ms launched in 9 / 12 / 15 / 18-bit cell
// order; 2^15 counters (128 KB) are the most one workgroup's LDS holds.
enum { MORTON_BITS = 15, QB_NT = 256, QB_BLOCKS = 512 };
enum { QO_CELLS = 1 << MORTON_BITS, QO_NT = 1024, QO_SCAN_NT = 256, QO_BLOCKS = QO_CELLS / QO_SCAN_NT };

// Bounds: (lo[CUKD_MAX_DIMS], hi[CUKD_MAX_DIMS]) as ordered keys per workgroup
// of k_qbounds, folded by their readers.
enum { QB_WORDS = QB_BLOCKS * 2 * CUKD_MAX_DIMS };

// Per-dim min / max of the nq*D query coordinates.  The flat array is read
// coalesced with a thread stride T that is a multiple of D, so each thread
// sees one dim only; four loads are in flight per thread.
__global__ __launch_bounds__(QB_NT) void k_qbounds(uint32_t *acc, const float *q, long long E, int D,
                                                  long long T)
{
  __shared__ uint32_t s_lo[CUKD_MAX_DIMS], s_hi[CUKD_MAX_DIMS];
  if (threadIdx.x < CUKD_MAX_DIMS) {
    s_lo[threadIdx.x] = 0xffffffffu;
    s_hi[threadIdx.x] = 0u;
  }
  __syncthreads();
  const long long tid = (long long)blockIdx.x * QB_NT + threadIdx.x;
  if (tid < T) {
    uint32_t lo = 0xffffffffu, hi = 0u;
    for (long long e = tid; e < E; e += 4 * T) {
      uint32_t v[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const long long x = e + j * T;
        v[j] = x < E ? ordered_key(__float_as_uint(q[x]), true) : ordered_key(__float_as_uint(q[e]), true);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        lo = min(lo, v[j]);
        hi = max(hi, v[j]);
      }
    }
    const int d = (int)(tid % D);
    if (tid < E) {
      atomicMin(&s_lo[d], lo);
      atomicMax(&s_hi[d], hi);
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < 2 * CUKD_MAX_DIMS) {
    const int w = (int)threadIdx.x;
    acc[blockIdx.x * 2 * CUKD_MAX_DIMS + w] =
        w < CUKD_MAX_DIMS ? s_lo[w] : s_hi[w - CUKD_MAX_DIMS];
  }
}

// the batch box, folded from the workgroups' bounds by a whole workgroup of
// QO_NT threads; ends with a barrier
__device__ inline void qbox_load(const uint32_t *acc, int nblocks, int D, float *s_lo, float *s_hi)
{
  __shared__ uint32_t s_key[2 * CUKD_MAX_DIMS];
  const int tid = (int)threadIdx.x;
  if (tid < 2 * CUKD_MAX_DIMS) s_key[tid] = tid < CUKD_MAX_DIMS ? 0xffffffffu : 0u;
  __syncthreads();
  // a thread's words are of one dim and side: QO_NT is a multiple of the row
  const int w = tid % (2 * CUKD_MAX_DIMS);
  const bool up = w >= CUKD_MAX_DIMS;
  uint32_t v = up ? 0u : 0xffffffffu;
  for (int i = tid; i < nblocks * 2 * CUKD_MAX_DIMS; i += QO_NT) {
    const uint32_t x = acc[i];
    v = up ? max(v, x) : min(v, x);
  }
  if (up) atomicMax(&s_key[w], v);
  else atomicMin(&s_key[w], v);
  __syncthreads();
  if (tid < D) {
    s_lo[tid] = __uint_as_float(unordered_key(s_key[tid], true));
    s_hi[tid] = __uint_as_float(unordered_key(s_key[CUKD_MAX_DIMS + tid], true));
  }
  __syncthreads();
}

// Morton cell of one query from its coordinates (DC dims)
template <int DC>
__device__ inline uint32_t morton_cell(const float *x, const float *lo_, const float *hi_)
{
  constexpr int b = MORTON_BITS / DC > 0 ? MORTON_BITS / DC : 1;
  uint32_t code = 0;
#pragma unroll
  for (int d = 0; d < DC && d < MORTON_BITS; d++) {
    const float lo = lo_[d];
    const float hi = hi_[d];
    const float w = hi - lo;
    float t = w > 0.f ? (x[d] - lo) / w : 0.f;
    int c = (int)(t * (float)(1 << b));
    c = c < 0 ? 0 : (c >= (1 << b) ? (1 << b) - 1 : c);
#pragma unroll
    for (int j = 0; j < b; j++) code |= (uint32_t)((c >> j) & 1) << (j * DC + d);
  }
  return code & ((1u << MORTON_BITS) - 1);
}

// The cells of a thread's queries in one tile of ITEMS * QO_NT, QO_BATCH at a
// time: every coordinate load of a batch is issued before any is used.
enum { QO_BATCH = 4, QO_NONE = 0xffffffffu };
template <int DC, int ITEMS>
__device__ inline void tile_cells(uint32_t (&cell)[ITEMS], const float *q, int nq,
                                  const float *s_lo, const float *s_hi)
{
  const long long i0 = (long long)blockIdx.x * (ITEMS * QO_NT) + threadIdx.x;
#pragma unroll
  for (int k0 = 0; k0 < ITEMS; k0 += QO_BATCH) {
    float x[QO_BATCH][DC];
#pragma unroll
    for (int k = 0; k < QO_BATCH; k++) {
      const long long i = i0 + (long long)(k0 + k) * QO_NT;
#pragma unroll
      for (int d = 0; d < DC; d++) x[k][d] = i < nq ? q[(size_t)i * DC + d] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < QO_BATCH; k++) {
      const long long i = i0 + (long long)(k0 + k) * QO_NT;
      cell[k0 + k] = i < nq ? morton_cell<DC>(x[k], s_lo, s_hi) : (uint32_t)QO_NONE;
    }
  }
}

// Cell counts of one tile: row 'tile' of th (tile-major, QO_CELLS words a
// row).
template <int DC, int ITEMS>
__global__ __launch_bounds__(QO_NT) void k_qcount(uint32_t *th, const float *q, int nq,
                                                 const uint32_t *acc, int nblocks)
{
  __shared__ uint32_t h[QO_CELLS];
  __shared__ float s_lo[CUKD_MAX_DIMS], s_hi[CUKD_MAX_DIMS];
  for (int c = threadIdx.x; c < QO_CELLS; c += QO_NT) h[c] = 0u;
  qbox_load(acc, nblocks, DC, s_lo, s_hi);  // ends with a barrier
  uint32_t cell[ITEMS];
  tile_cells<DC, ITEMS>(cell, q, nq, s_lo, s_hi);
#pragma unroll
  for (int k = 0; k < ITEMS; k++)
    if (cell[k] != QO_NONE) atomicAdd(&h[cell[k]], 1u);
  __syncthreads();
  uint32_t *row = th + (size_t)blockIdx.x * QO_CELLS;
  for (int c = threadIdx.x; c < QO_CELLS; c += QO_NT) row[c] = h[c];
}

// The counts of the tiles become each tile's start among the cells of this
// workgroup (cell order, then tile order), and tot[block] the workgroup's
// queries.  QO_SPLIT threads per cell, each with a run of the tiles, and eight
// tiles' counts in flight: the kernel is a chain of loads.
enum { QO_SPLIT = 4 };
__global__ __launch_bounds__(QO_SCAN_NT * QO_SPLIT) void k_qcolscan(uint32_t *th, uint32_t *tot,
                                                                    int ntiles)
{
  __shared__ uint32_t part[QO_SPLIT][QO_SCAN_NT], wsum[QO_SCAN_NT / 64];
  const int cl = (int)threadIdx.x % QO_SCAN_NT, g = (int)threadIdx.x / QO_SCAN_NT;
  const int c = blockIdx.x * QO_SCAN_NT + cl;
  const int lane = cl & 63, w = cl >> 6;
  const int per = (ntiles + QO_SPLIT - 1) / QO_SPLIT;
  const int ta = g * per, tz = ta + per < ntiles ? ta + per : ntiles;
  uint32_t sum = 0;
  for (int t0 = ta; t0 < tz; t0 += 8) {
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = t0 + j < tz ? th[(size_t)(t0 + j) * QO_CELLS + c] : 0u;
#pragma unroll
    for (int j = 0; j < 8; j++) sum += v[j];
  }
  part[g][cl] = sum;
  __syncthreads();
  uint32_t all = 0, before = 0;
#pragma unroll
  for (int i = 0; i < QO_SPLIT; i++) {
    all += part[i][cl];
    if (i < g) before += part[i][cl];
  }
  uint32_t incl = all;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = (uint32_t)__shfl_up((int)incl, o);
    if (lane >= o) incl += u;
  }
  if (g == 0 && lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t run = incl - all;
  for (int i = 0; i < w; i++) run += wsum[i];
  if (g == 0 && cl == QO_SCAN_NT - 1) tot[blockIdx.x] = run + all;
  run += before;
  for (int t0 = ta; t0 < tz; t0 += 8) {
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = t0 + j < tz ? th[(size_t)(t0 + j) * QO_CELLS + c] : 0u;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if (t0 + j < tz) th[(size_t)(t0 + j) * QO_CELLS + c] = run;
      run += v[j];
    }
  }
}

// Places one tile's queries: consecutive slots from the tile's start in each
// cell, behind the queries of the earlier blocks' cells.
template <int DC, int ITEMS>
__global__ __launch_bounds__(QO_NT) void k_qplace(int32_t *order, const uint32_t *th,
                                                 const uint32_t *tot, const float *q, int nq,
                                                 const uint32_t *acc, int nblocks)
{
  static_assert(QO_BLOCKS <= 2 * 64 && QO_CELLS % QO_NT == 0, "one wave scans the blocks");
  __shared__ uint32_t base[QO_CELLS];
  __shared__ uint32_t s_blk[QO_BLOCKS];
  __shared__ float s_lo[CUKD_MAX_DIMS], s_hi[CUKD_MAX_DIMS];
  const int tid = (int)threadIdx.x;
  const uint32_t *row = th + (size_t)blockIdx.x * QO_CELLS;
  uint32_t v[QO_CELLS / QO_NT];
#pragma unroll
  for (int j = 0; j < QO_CELLS / QO_NT; j++) v[j] = row[j * QO_NT + tid];
  if (tid < 64) {
    const uint32_t a = 2 * tid < QO_BLOCKS ? tot[2 * tid] : 0u;
    const uint32_t b = 2 * tid + 1 < QO_BLOCKS ? tot[2 * tid + 1] : 0u;
    uint32_t incl = a + b;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t u = (uint32_t)__shfl_up((int)incl, o);
      if (tid >= o) incl += u;
    }
    if (2 * tid < QO_BLOCKS) s_blk[2 * tid] = incl - a - b;
    if (2 * tid + 1 < QO_BLOCKS) s_blk[2 * tid + 1] = incl - b;
  }
  qbox_load(acc, nblocks, DC, s_lo, s_hi);  // ends with a barrier
#pragma unroll
  for (int j = 0; j < QO_CELLS / QO_NT; j++) {
    const int c = j * QO_NT + tid;
    base[c] = v[j] + s_blk[c / QO_SCAN_NT];
  }
  uint32_t cell[ITEMS];
  tile_cells<DC, ITEMS>(cell, q, nq, s_lo, s_hi);
  __syncthreads();
  const long long i0 = (long long)blockIdx.x * (ITEMS * QO_NT) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < ITEMS; k++)
    if (cell[k] != QO_NONE) order[atomicAdd(&base[cell[k]], 1u)] = (int32_t)(i0 + (long long)k * QO_NT);
}

static size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// queries per thread of a tile: the tiles of a small batch are small, so that
// they spread over the CUs (each reads and writes 128 KB of counts, so no
// smaller)
static int order_items(int nq) { return nq <= (1 << 18) ? 4 : nq <= (1 << 20) ? 8 : 16; }
static int order_tiles(int nq)
{
  const int tile = order_items(nq) * QO_NT;
  return (nq + tile - 1) / tile;
}

size_t query_order_temp_bytes(int nq)
{
  // the tile size steps up with nq, so a smaller batch may have more tiles
  int tiles = order_tiles(nq);
  if (nq > (1 << 18)) tiles = tiles > order_tiles(1 << 18) ? tiles : order_tiles(1 << 18);
  if (nq > (1 << 20)) tiles = tiles > order_tiles(1 << 20) ? tiles : order_tiles(1 << 20);
  return align256((size_t)nq * 4) + align256((size_t)tiles * QO_CELLS * 4) +
         align256((size_t)QO_BLOCKS * 4) + QB_WORDS * 4 + 256;
}

template <int DC, int ITEMS>
static void launch_order(hipError_t &e, int32_t *order, uint32_t *th, uint32_t *tot,
                         const uint32_t *acc, int nblocks, const float *q, int nq, int tiles, hipStream_t s)
{
  CUKD_LAUNCH(e, (k_qcount<DC, ITEMS>), dim3(tiles), dim3(QO_NT), 0, s, th, q, nq, acc, nblocks);
  CUKD_LAUNCH(e, k_qcolscan, dim3(QO_BLOCKS), dim3(QO_SCAN_NT * QO_SPLIT), 0, s, th, tot,
              tiles);
  CUKD_LAUNCH(e, (k_qplace<DC, ITEMS>), dim3(tiles), dim3(QO_NT), 0, s, order,
              (const uint32_t *)th, (const uint32_t *)tot, q, nq, acc, nblocks);
}

// Writes the launch order of nq queries into the front of 'tmp' (which
// holds query_order_temp_bytes(nq) bytes) and returns it.  e as in CUKD_LAUNCH.
int32_t *make_query_order(hipError_t &e, void *tmp, const float *q, int nq, int D, hipStream_t s)
{
  uint8_t *t = (uint8_t *)tmp;
  int32_t *order = (int32_t *)t;
  if (nq <= 0) return order;
  const int tiles = order_tiles(nq), items = order_items(nq);
  t += align256((size_t)nq * 4);
  uint32_t *th = (uint32_t *)t;
  t += align256((size_t)tiles * QO_CELLS * 4);
  uint32_t *tot = (uint32_t *)t;
  t += align256((size_t)QO_BLOCKS * 4);
  uint32_t *acc = (uint32_t *)t;
  const long long E = (long long)nq * D;
  long long blocks = (E + QB_NT * 4 - 1) / (QB_NT * 4);
  if (blocks > QB_BLOCKS) blocks = QB_BLOCKS;
  long long T = blocks * QB_NT;
  T -= T % D;
  if (T < D) T = D;  // E >= D, and blocks * QB_NT >= 256 >= D
  CUKD_LAUNCH(e, k_qbounds, dim3((unsigned)blocks), dim3(QB_NT), 0, s, acc, q, E, D, T);
#define CUKD_QORDER_CASE(DCv)                                                                      \
  case DCv:                                                                                        \
    if (items == 4) launch_order<DCv, 4>(e, order, th, tot, acc, (int)blocks, q, nq, tiles, s);    \
    else if (items == 8) launch_order<DCv, 8>(e, order, th, tot, acc, (int)blocks, q, nq, tiles, s); \
    else launch_order<DCv, 16>(e, order, th, tot, acc, (int)blocks, q, nq, tiles, s);              \
    break
  switch (D) {
    CUKD_QORDER_CASE(1);
    CUKD_QORDER_CASE(2);
    CUKD_QORDER_CASE(3);
    CUKD_QORDER_CASE(4);
    CUKD_QORDER_CASE(5);
    CUKD_QORDER_CASE(6);
    CUKD_QORDER_CASE(7);
    default: CUKD_QORDER_CASE(8);
  }
#undef CUKD_QORDER_CASE
  return order;
}

}  // namespace cukd_amd
