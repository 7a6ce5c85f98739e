// query_impl.h -- batched FCP / kNN kernels over a left-balanced k-d tree.
//
// One query per lane.  k_query runs the public device-inline traversals of
// include/cukd/ (traverse.h, fcp.h, knn.h) through an accessor over the
// run-time element layout; k_query_box (query_box.h), the default over trees
// with round-robin split dims, gives the same results with fewer visits.
// ids and dist2 bits equal the CPU oracle's, ties included.
#pragma once
#pragma clang fp contract(off)

#include "cukd/knn.h"
#include "cukd_common.h"

namespace cukd_amd {

// node accessor over a cukd_layout-described array
struct TreeView {
  const uint8_t *base;
  int n;
  int stride;
  int point_offset;
  int dim_offset;
  int dim_bytes;
  int num_dims;

  __device__ inline int size() const { return n; }
  template <int D>
  __device__ inline void point(int i, float (&p)[D]) const
  {
    const float *src = (const float *)(base + (size_t)i * stride + point_offset);
#pragma unroll
    for (int d = 0; d < D; d++) p[d] = src[d];
  }
  __device__ inline int dim(int i) const
  {
    if (dim_offset < 0) {
      const int l = 31 - __clz(i + 1);
      return (num_dims & (num_dims - 1)) == 0 ? (l & (num_dims - 1)) : l % num_dims;
    }
    const uint8_t *p = base + (size_t)i * stride + dim_offset;
    if (dim_bytes == 1) return *p;
    if (dim_bytes == 2) return *(const uint16_t *)p;
    return *(const int32_t *)p;
  }
};

// TreeView with the query's dimension count known at compile time: the
// round-robin split dim of a node is then a constant-divisor modulo
template <int D>
struct TreeViewD : TreeView {
  __device__ inline int dim(int i) const
  {
    if (dim_offset >= 0) return TreeView::dim(i);
    const int l = 31 - __clz(i + 1);
    return (D & (D - 1)) == 0 ? (l & (D - 1)) : l % D;
  }
};

// The run-time-k lists (k <= 64) keep their entries in LDS, in columns:
// entry i of the lane's query at col[i * stride], col = base + lane and
// stride = the workgroup size, so the lanes of a wave touch consecutive
// words.  (A per-lane array indexed at run time lives in scratch memory:
// k = 64 took 304 ms for 1M queries over a 10M-point tree.)  The largest
// kept key is also held in a register, so rejected candidates -- most of them
// -- touch no LDS.
struct LdsCol {
  uint64_t *p;
  int stride;
  __device__ inline uint64_t &operator[](int i) const { return p[(size_t)i * stride]; }
};

__device__ inline uint64_t list_key(float d2, uint32_t id)
{
  return ((uint64_t)__float_as_uint(d2) << 32) | id;
}

// the reference's max-heap push (knn.h:456-483, as detail::heap_push) over
// an LDS column; top = e[0]
__device__ inline void lds_heap_push(const LdsCol &e, int k, uint64_t v, uint64_t &top)
{
  if (v >= top) return;
  int pos = 0;
  for (;;) {
    uint64_t largest_val = ~0ull;
    const int c0 = 2 * pos + 1;
    int largest = k;
    if (c0 < k) {
      largest = c0;
      largest_val = e[c0];
    }
    const int c1 = c0 + 1;
    if (c1 < k) {
      const uint64_t v1 = e[c1];
      if (v1 > largest_val) {
        largest = c1;
        largest_val = v1;
      }
    }
    if (largest == k || largest_val < v) {
      e[pos] = v;
      break;
    }
    e[pos] = largest_val;
    pos = largest;
  }
  top = e[0];
}

// in-place heapsort of a max-heap column into ascending order
__device__ inline void lds_heap_sort(const LdsCol &e, int k)
{
  for (int end = k - 1; end > 0; end--) {
    const uint64_t v = e[end];
    e[end] = e[0];
    int pos = 0;
    for (;;) {
      int c = 2 * pos + 1;
      if (c >= end) break;
      uint64_t cv = e[c];
      if (c + 1 < end) {
        const uint64_t v1 = e[c + 1];
        if (v1 > cv) {
          c++;
          cv = v1;
        }
      }
      if (!(cv > v)) break;
      e[pos] = cv;
      pos = c;
    }
    e[pos] = v;
  }
}

// Run-time-k candidate lists over an LDS column, as a max-heap (top = the
// k-th smallest key).
//  SORTED = false: HeapCandidateList / FlexHeapCandidateList (knn.h:240-
//    287), written out in heap order as the reference leaves it.
//  SORTED = true: FixedCandidateList with a run-time k (knn.h:214-232).  The
//    fixed list keeps the k smallest keys offered so far, ascending, and
//    culls with the largest of them; a max-heap given the same candidates
//    holds the same k keys with the same largest one, so every cull and
//    every accepted candidate is the same, and one heapsort at the end
//    gives the fixed list's ascending order.  (A sorted insert moves up to
//    k - 1 words per accepted candidate; the heap moves log2(k).)
template <bool SORTED> struct LdsList {
  static constexpr bool kSorted = SORTED;
  LdsCol e;
  int k;
  uint64_t top;  // e[0]
  __device__ inline void init_top(uint64_t v) { top = v; }
  __device__ inline float maxRadius2() const { return __uint_as_float((uint32_t)(top >> 32)); }
  __device__ inline float initialCullDist2() const { return maxRadius2(); }
  __device__ inline float processCandidate(int id, float d2)
  {
    lds_heap_push(e, k, list_key(d2, (uint32_t)id), top);
    return maxRadius2();
  }
};
using DynFixedList = LdsList<true>;
using LdsHeapList = LdsList<false>;

// persistent per-query candidate lists in HBM (multi-round kNN)
struct ListArgs {
  uint64_t *lists;  // nq * k entries, query q at lists[q*k]
  int init;         // fill with (cutoff^2, -1) before the traversal
  int id_offset;    // added to every candidate id
};

// The reference's global-memory FlexHeapCandidateList of a multi-round
// query (samples/mpiHugeQuery.cu:75-88, knn.h:360-421): the k entries are
// loaded from HBM into the LDS column, updated with the same heap push,
// and stored back, so they end as the reference's in-place list would.
struct AccumList {
  LdsCol e;
  int k;
  int id_offset;
  uint64_t top;
  __device__ inline float maxRadius2() const { return __uint_as_float((uint32_t)(top >> 32)); }
  __device__ inline float initialCullDist2() const { return maxRadius2(); }
  __device__ inline float processCandidate(int id, float d2)
  {
    lds_heap_push(e, k, list_key(d2, (uint32_t)(id + id_offset)), top);
    return maxRadius2();
  }
};

// ---------------------------------------------------------------------------
// per-result-type set-up and output
// ---------------------------------------------------------------------------
// kLds: the type keeps k 64-bit words per query in the kernel's dynamic
// LDS (init gets the lane's column; the others ignore it)
template <class R> struct ResultOps;

template <> struct ResultOps<AccumList> {
  static constexpr bool kLds = true;
  struct State { AccumList r; };
  __device__ static inline AccumList &init(State &s, float cutoff, int k, int q, const ListArgs &la,
                                           LdsCol col)
  {
    s.r.e = col;
    s.r.k = k;
    s.r.id_offset = la.id_offset;
    const uint64_t *src = la.lists + (size_t)q * k;
    const uint64_t v = list_key(cutoff * cutoff, 0xffffffffu);
    for (int i = 0; i < k; i++) col[i] = la.init ? v : src[i];
    s.r.top = col[0];
    return s.r;
  }
  __device__ static inline void write(const State &s, int q, int k, int32_t *, float *, float *,
                                      const ListArgs &la)
  {
    uint64_t *dst = la.lists + (size_t)q * k;
    for (int i = 0; i < k; i++) dst[i] = s.r.e[i];
  }
};

template <> struct ResultOps<cukd::FCPResult> {
  static constexpr bool kLds = false;
  struct State { cukd::FCPResult r; };
  __device__ static inline cukd::FCPResult &init(State &s, float cutoff, int, int, const ListArgs &,
                                                 LdsCol)
  {
    s.r.clear(cutoff * cutoff);
    return s.r;
  }
  __device__ static inline void write(const State &s, int q, int, int32_t *ids, float *dist2, float *,
                                      const ListArgs &)
  {
    ids[q] = s.r.closestPrimID;
    if (dist2) dist2[q] = s.r.closestDist2;
  }
};

template <int K> struct ResultOps<cukd::FixedCandidateList<K>> {
  static constexpr bool kLds = false;
  struct State { cukd::FixedCandidateList<K> r; __device__ State() : r(0.f) {} };
  __device__ static inline cukd::FixedCandidateList<K> &init(State &s, float cutoff, int, int,
                                                             const ListArgs &, LdsCol)
  {
    s.r = cukd::FixedCandidateList<K>(cutoff);
    return s.r;
  }
  __device__ static inline void write(const State &s, int q, int, int32_t *ids, float *dist2, float *ret,
                                      const ListArgs &)
  {
#pragma unroll
    for (int i = 0; i < K; i++) {
      ids[(size_t)q * K + i] = (int32_t)(uint32_t)s.r.entry[i];
      dist2[(size_t)q * K + i] = __uint_as_float((uint32_t)(s.r.entry[i] >> 32));
    }
    if (ret) ret[q] = s.r.maxRadius2();
  }
};

// the run-time-k fixed and heap lists: (cutoff^2, -1) in every entry, and
// the entries written out in storage order
template <class L> struct LdsListOps {
  static constexpr bool kLds = true;
  struct State { L r; };
  __device__ static inline L &init(State &s, float cutoff, int k, int, const ListArgs &, LdsCol col)
  {
    s.r.e = col;
    s.r.k = k;
    const uint64_t v = list_key(cutoff * cutoff, 0xffffffffu);
    for (int i = 0; i < k; i++) col[i] = v;
    s.r.init_top(v);
    return s.r;
  }
  __device__ static inline void write(const State &s, int q, int k, int32_t *ids, float *dist2, float *ret,
                                      const ListArgs &)
  {
    if (L::kSorted) lds_heap_sort(s.r.e, k);
    for (int i = 0; i < k; i++) {
      const uint64_t x = s.r.e[i];
      ids[(size_t)q * k + i] = (int32_t)(uint32_t)x;
      dist2[(size_t)q * k + i] = __uint_as_float((uint32_t)(x >> 32));
    }
    if (ret) ret[q] = s.r.maxRadius2();
  }
};
template <bool SORTED> struct ResultOps<LdsList<SORTED>> : LdsListOps<LdsList<SORTED>> {};

// Queries over a forest (many trees back to back in one array): query qi
// belongs to the segment s with seg_off[s] <= qi < seg_off[s+1] and runs
// against tree seg_tree[s] = elements tree_off[t] .. tree_off[t+1].
// seg_off == nullptr: one tree, the TreeView as given.
struct ForestQ {
  const int32_t *seg_off;
  const int32_t *seg_tree;
  int nseg;
  const int32_t *tree_off;
};

__device__ inline int segment_of(const int32_t *seg_off, int nseg, int qi)
{
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (seg_off[mid] <= qi) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// batch kernel: one query per lane
// ---------------------------------------------------------------------------
template <int D, int METHOD, class R>
__global__ __launch_bounds__(256) void k_query(TreeView t, const float *queries, int nq,
                                               const float *world_bounds, float cutoff,
                                               float eps, int k, const int32_t *order,
                                               int32_t *ids, float *dist2, float *ret,
                                               ListArgs la, ForestQ fq,
                                               unsigned long long *stats)
{
  // Workgroups are dispatched round-robin over the 8 XCDs, each with its
  // own L2: give every XCD one contiguous run of (Morton-ordered) queries,
  // so neighbouring queries share an L2 instead of fetching the same tree
  // nodes into eight of them.  A bijection of [0, gridDim.x).
  const int nb = (int)gridDim.x;
  const int xcd = (int)blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int lb = xcd * q8 + (xcd < r8 ? xcd : r8) + ((int)blockIdx.x >> 3);
  const int i = lb * (int)blockDim.x + (int)threadIdx.x;
  if (i >= nq) return;
  const int qi = order ? order[i] : i;
  if (fq.seg_off) {
    const int tr = fq.seg_tree[segment_of(fq.seg_off, fq.nseg, qi)];
    const int b = fq.tree_off[tr];
    t.base += (size_t)b * t.stride;
    t.n = fq.tree_off[tr + 1] - b;
    if (world_bounds) world_bounds += (size_t)tr * 2 * D;
  }
  float q[D];
#pragma unroll
  for (int d = 0; d < D; d++) q[d] = queries[(size_t)qi * D + d];
  HIP_DYNAMIC_SHARED(uint64_t, s_lists);
  typename ResultOps<R>::State st;
  R &res = ResultOps<R>::init(st, cutoff, k, qi, la, LdsCol{s_lists + threadIdx.x, (int)blockDim.x});
  unsigned visits = 0;
  TreeViewD<D> tv;
  static_cast<TreeView &>(tv) = t;
  if (METHOD == CUKD_STACK_BASED) {
    cukd::detail::traverse_stack_based<D>(res, q, tv, visits);
  } else if (METHOD == CUKD_STACK_FREE) {
    cukd::detail::traverse_stack_free<D>(res, q, tv, eps, visits);
  } else {
    float lo[D], hi[D];
#pragma unroll
    for (int d = 0; d < D; d++) { lo[d] = world_bounds[d]; hi[d] = world_bounds[D + d]; }
    cukd::detail::traverse_cct<D>(res, q, lo, hi, tv, visits);
  }
  ResultOps<R>::write(st, qi, k, ids, dist2, ret, la);
  // CUKD_STATS (common.h:348-360): one count per visited node
  if (stats) atomicAdd(stats, (unsigned long long)visits);
}

}  // namespace cukd_amd

#include "query_box.h"

namespace cukd_amd {

// ---------------------------------------------------------------------------
// per-dimension launchers
// ---------------------------------------------------------------------------
struct QueryArgs {
  TreeView t;
  const float *queries;
  int nq;
  const float *world_bounds;
  float cutoff;
  float eps;
  int k;
  int list_kind;   // -1 = FCP, CUKD_LIST_FIXED, CUKD_LIST_HEAP or LIST_ACCUM
  const int32_t *order;
  int32_t *ids;
  float *dist2;
  float *ret;
  ListArgs la;
  ForestQ fq;
  unsigned long long *stats;
  int block = 0;    // workgroup size: 64, 128 or 256 (0: the kernel's own default)
  bool box = true;  // k_query_box where the call allows it
  uint64_t tree_bytes = 0;  // bytes of the tree array (forests: all trees)
  int max_n = 0;            // forests: points of the largest tree
};

// persistent multi-round lists (cukd_knn_accumulate)
enum { LIST_ACCUM = 100 };

enum { LDS_PER_CU = 163840 };

template <int D, int METHOD, class R>
inline hipError_t launch_q(const QueryArgs &a, hipStream_t s)
{
  const int nt = a.block ? a.block : 128;
  const int blocks = (a.nq + nt - 1) / nt;
  // run-time-k lists: k words per lane of dynamic LDS (k <= 64 and nt <=
  // 256 keep it within one CU's 160 KiB)
  const size_t shm = ResultOps<R>::kLds ? (size_t)a.k * sizeof(uint64_t) * nt : 0;
  if (shm > LDS_PER_CU) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_query<D, METHOD, R>), dim3(blocks), dim3(nt), shm, s, a.t, a.queries,
                     a.nq, a.world_bounds, a.cutoff, a.eps, a.k, a.order, a.ids, a.dist2,
                     a.ret, a.la, a.fq, a.stats);
  return hipGetLastError();
}

template <int D, int METHOD, class L>
inline hipError_t launch_box(const QueryArgs &a, hipStream_t s)
{
  const int nt = a.block ? a.block : 64;
  const int rows = sd_rows(a.fq.seg_off ? a.max_n : a.t.n);
  const size_t shm = (size_t)rows * nt * sizeof(float);
  const int blocks = (a.nq + nt - 1) / nt;
  hipLaunchKernelGGL((k_query_box<D, METHOD, L>), dim3(blocks), dim3(nt), shm, s, a.t, a.queries,
                     a.nq, a.world_bounds, a.cutoff, a.eps, a.k, a.order, a.ids, a.dist2,
                     a.ret, a.la, a.fq, rows);
  return hipGetLastError();
}

// k_query_box serves trees with round-robin dims and 32-bit node offsets.
// Counted traversals (cukd_set_traversal_stats) run k_query, whose visits
// are the reference's, and so do NaN cutoffs, whose keys have no order as
// doubles.
inline bool box_ok(const QueryArgs &a)
{
  const uint64_t bytes = a.fq.seg_off ? a.tree_bytes : (uint64_t)a.t.n * (uint64_t)a.t.stride;
  return a.box && !a.stats && a.t.dim_offset < 0 && bytes <= 0xffffffffull &&
         a.cutoff == a.cutoff;
}

template <int D, int METHOD>
inline hipError_t launch_method(const QueryArgs &a, hipStream_t s)
{
  if (box_ok(a)) {
    if (a.list_kind < 0) return launch_box<D, METHOD, RegClosest>(a, s);
    if (a.list_kind == CUKD_LIST_FIXED) {
      if (a.k == 1) return launch_box<D, METHOD, RegSorted<1>>(a, s);
      if (a.k <= 4) return launch_box<D, METHOD, RegSorted<4>>(a, s);
      if (a.k <= 8) return launch_box<D, METHOD, RegSorted<8>>(a, s);
      if (a.k <= 16) return launch_box<D, METHOD, RegSorted<16>>(a, s);
      if (a.k <= 24) return launch_box<D, METHOD, RegSorted<24>>(a, s);
      if (a.k <= 32) return launch_box<D, METHOD, RegSorted<32>>(a, s);
      if (a.k <= 48) return launch_box<D, METHOD, RegSorted<48>>(a, s);
      return launch_box<D, METHOD, RegSorted<64>>(a, s);
    }
    // heap lists, also the persistent ones of a multi-round query
    if (a.k <= 8) return launch_box<D, METHOD, RegHeap<8>>(a, s);
    if (a.k <= 16) return launch_box<D, METHOD, RegHeap<16>>(a, s);
    if (a.k <= 24) return launch_box<D, METHOD, RegHeap<24>>(a, s);
    if (a.k <= 32) return launch_box<D, METHOD, RegHeap<32>>(a, s);
    if (a.k <= 48) return launch_box<D, METHOD, RegHeap<48>>(a, s);
    return launch_box<D, METHOD, RegHeap<64>>(a, s);
  }
  if (a.list_kind < 0) return launch_q<D, METHOD, cukd::FCPResult>(a, s);
  if (a.list_kind == CUKD_LIST_HEAP) return launch_q<D, METHOD, LdsHeapList>(a, s);
  if (a.list_kind == LIST_ACCUM) return launch_q<D, METHOD, AccumList>(a, s);
  switch (a.k) {
    case 1: return launch_q<D, METHOD, cukd::FixedCandidateList<1>>(a, s);
    case 4: return launch_q<D, METHOD, cukd::FixedCandidateList<4>>(a, s);
    case 8: return launch_q<D, METHOD, cukd::FixedCandidateList<8>>(a, s);
    case 16: return launch_q<D, METHOD, cukd::FixedCandidateList<16>>(a, s);
    default: return launch_q<D, METHOD, DynFixedList>(a, s);
  }
}

template <int D>
inline hipError_t launch_query_d(int method, const QueryArgs &a, hipStream_t s)
{
  if (method == CUKD_STACK_BASED) return launch_method<D, CUKD_STACK_BASED>(a, s);
  if (method == CUKD_STACK_FREE) return launch_method<D, CUKD_STACK_FREE>(a, s);
  return launch_method<D, CUKD_CCT>(a, s);
}

hipError_t launch_query(int D, int method, const QueryArgs &a, hipStream_t s);
hipError_t launch_knn_extract(const uint64_t *lists, int nq, int k, int32_t *ids, float *dist2,
                              float *radius, hipStream_t s);

// spatial-tree queries (spatial.hip)
struct SpatialBounds {
  float v[2 * CUKD_MAX_DIMS];
};
struct SpatialArgs {
  const cukd_spatial_node *nodes;
  const uint32_t *prim_ids;
  int num_nodes;
  TreeView data;
  SpatialBounds bounds;
  const float *queries;
  int nq;
  float cutoff;
  int k;
  int list_kind;  // -1 = FCP
  const int32_t *order;  // launch order (nullable)
  bool prune;            // box pruning allowed
  int32_t *ids;
  float *dist2;
  float *ret;
  unsigned long long *stats;  // node + leaf-point visits (fcp.h:294,327), nullable
};
// bytes of points from which large spatial batches run in Morton order: an
// L2's size
constexpr uint64_t SPATIAL_ORDER_MIN_BYTES = (uint64_t)4 << 20;
// what the build recorded in the tree for its queries
enum { SPATIAL_MAY_PRUNE = 1, SPATIAL_MAY_ALLOCATE = 2 };
int spatial_may(const cukd_spatial_tree *tree, int D);
hipError_t launch_spatial_query(int D, int method, const SpatialArgs &a, hipStream_t s);
int spatial_build_impl(cukd_spatial_tree *tree, const void *d_points, int n, const cukd_layout &L,
                       int leaf_threshold, hipStream_t s, const MemResource &mem);

}  // namespace cukd_amd
