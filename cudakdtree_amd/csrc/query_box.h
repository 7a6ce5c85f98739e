// query_box.h -- the batch query kernel over trees with round-robin split
// dims: box-pruned traversal, pending planes in LDS, lists in registers.
//
// One query per lane.  It returns bit for bit what the reference's three
// traversals return (include/cukd/traverse.h states them), heap order and
// ties included, while visiting fewer nodes:
//
//  Box pruning.  Beside the split plane's distance, a far subtree is skipped
//  when the distance to its cell -- the sum over the dims of the squared
//  distances to the planes that the path crossed, added in the order of the
//  point distance -- is above the cull distance.  Float subtraction,
//  squaring and ordered addition are monotone, so every point of such a
//  subtree has a computed dist2 of at least that sum: above the cull, where
//  no list accepts it.  Skipping it changes no accepted candidate, no later
//  cull and no order.  (An equal distance is not skipped: a smaller id could
//  still be accepted.)  CPU count over 10M uniform points: 96 visits per
//  query instead of 112 for kNN-8, 276 instead of 357 for k = 50, and a
//  fifth of them for queries far from clustered points.
//
//  Planes in LDS.  Row r of a lane's LDS column holds diff*diff of the far
//  child at depth r of its path, written when that child is pushed and
//  kept while the path runs below it.  So a pop costs no node load, and the
//  cell's plane distances at any ancestor are read back from the rows of
//  the far children on the path (mask 'far'), the deepest one per dim.
//
// What bounds it: vector issue at partial lane use (a wave runs 170
// iterations for 96 visits per lane at kNN-8) and one line access per lane
// and visit; a small batch is one chain of iterations of 0.3 .. 0.5 us.
// Measured on 1M Morton-ordered queries over 10M uniform float3, kernel time
// before (two queries per lane, planes only; k = 20 and up: lists in LDS,
// one query per lane) and now: FCP 312 -> 202 us, kNN-8 755 -> 485,
// kNN-16 1184 -> 710, kNN-20 3530 -> 774, kNN-64 28100 -> 2610,
// heap 50 14800 -> 2740; 100K FCP over 100K points 109 -> 45 us; 200K
// uniform queries over 1M clustered points 145 -> 6.7 ms.
// Also measured (kNN-8): refilling finished lanes within a wave 650 us and
// more; 16 resident waves per CU instead of 27, 550 us; a load in every
// iteration, popping or not, 564 us (the line accesses).
#pragma once
#pragma clang fp contract(off)

namespace cukd_amd {

__device__ inline double key_min(double a, double b)
{
#ifdef __HIP_DEVICE_COMPILE__
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return a < b ? a : b;
#endif
}
__device__ inline double key_max(double a, double b)
{
#ifdef __HIP_DEVICE_COMPILE__
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return a > b ? a : b;
#endif
}

// Writes entries [first, first + k) of e as ids and dist2 words.  A lane's row is
// its own lines, so every store instruction of a wave costs 64 line accesses:
// stores are 16 bytes wide, aligned or, where k or the rows do not allow that,
// at any word.  Those rows go out one array after the other, since fewer lines
// are then open at a time than the L2 holds: 400K empty lists of 50 take 111 us,
// 179 with both arrays in one pass, 483 a word at a time (33 entries 92, 133 and
// 364; 196 and 148 when a CU held 4 waves).
struct __align__(16) Word4 {
  uint32_t v[4];
};
struct __attribute__((packed, aligned(4))) AnyWord4 {
  uint32_t v[4];
};
template <int K, class T>
__device__ inline void write_words(const T (&e)[K], int first, int k, int shift, uint32_t *out)
{
#pragma unroll
  for (int i = 0; i < K; i += 4) {
    if (i + 4 <= K && i >= first && i + 4 <= first + k) {
      AnyWord4 a;
#pragma unroll
      for (int j = 0; j < 4; j++)
        a.v[j] = (uint32_t)(__builtin_bit_cast(uint64_t, e[i + j < K ? i + j : 0]) >> shift);
      *(AnyWord4 *)(out + (i - first)) = a;
    } else {
#pragma unroll
      for (int j = i; j < i + 4 && j < K; j++)
        if (j >= first && j < first + k)
          out[j - first] = (uint32_t)(__builtin_bit_cast(uint64_t, e[j]) >> shift);
    }
  }
}
template <int K, class T>
__device__ inline void write_row(const T (&e)[K], int first, int k, int32_t *ids, float *dist2)
{
  const bool quads = K % 4 == 0 && ((first | k) & 3) == 0 &&
                     (((uintptr_t)ids | (uintptr_t)dist2) & 15) == 0;
  if (quads) {
#pragma unroll
    for (int i = 0; i + 4 <= K; i += 4) {
      if (i < first || i >= first + k) continue;
      Word4 a, b;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint64_t x = __builtin_bit_cast(uint64_t, e[i + j]);
        a.v[j] = (uint32_t)x;
        b.v[j] = (uint32_t)(x >> 32);
      }
      *(Word4 *)(ids + (i - first)) = a;
      *(Word4 *)(dist2 + (i - first)) = b;
    }
  } else {
    write_words<K>(e, first, k, 0, (uint32_t *)ids);
    write_words<K>(e, first, k, 32, (uint32_t *)dist2);
  }
}

// Sorted list of the k <= K smallest keys (FixedCandidateList), in registers.
// A key (dist2 bits, id) read as a double orders like the integer: the
// largest, dist2 = +inf, has the exponent 0x7f8, a finite double.  Insertion
// is then one v_min_f64 and one v_max_f64 per slot, full-rate on gfx950,
// against a 64-bit compare and four selects; a key above all entries leaves
// them as they are.  The first K - k entries are -1.0, below every key, and
// are not written out.
template <int K> struct RegSorted {
  double e[K];
  __device__ inline void init(float cutoff, int k, const uint64_t *, bool, int)
  {
    const double v = __builtin_bit_cast(double, list_key(cutoff * cutoff, 0xffffffffu));
#pragma unroll
    for (int i = 0; i < K; i++) e[i] = i < K - k ? -1.0 : v;
  }
  __device__ inline float cull() const
  {
    return __uint_as_float((uint32_t)(__builtin_bit_cast(uint64_t, e[K - 1]) >> 32));
  }
  __device__ inline void offer(int id, float d2, float &c)
  {
    if (!(d2 <= c)) return;  // also a NaN dist2, which is above every key
    const double v = __builtin_bit_cast(double, list_key(d2, (uint32_t)id));
#pragma unroll
    for (int i = K - 1; i > 0; i--) e[i] = key_max(e[i - 1], key_min(e[i], v));
    e[0] = key_min(e[0], v);
    c = cull();
  }
  __device__ inline void write(int k, int32_t *ids, float *dist2, float *ret, uint64_t *) const
  {
    write_row<K>(e, K - k, k, ids, dist2);
    if (ret) *ret = cull();
  }
};

// closest point only (FCPResult): the first strictly closer one wins
struct RegClosest {
  int id;
  float d;
  __device__ inline void init(float cutoff, int, const uint64_t *, bool, int)
  {
    id = -1;
    d = cutoff * cutoff;
  }
  __device__ inline float cull() const { return d; }
  __device__ inline void offer(int i, float d2, float &c)
  {
    const bool closer = d2 < d;
    id = closer ? i : id;
    d = closer ? d2 : d;
    c = d;
  }
  __device__ inline void write(int, int32_t *ids, float *dist2, float *, uint64_t *) const
  {
    *ids = id;
    if (dist2) *dist2 = d;
  }
};

// Max-heap of k <= K keys (HeapCandidateList, FlexHeapCandidateList;
// knn.h:456-483) in registers, which cannot be indexed at run time: the sift
// walks every slot in order, and a slot is touched by the lanes whose path
// runs through it.  Slots from k on hold 0, which no child comparison picks:
// a missing child is skipped because its slot is not above its sibling's,
// and with both missing the sift ends at the parent.  Keys are unsigned
// integers here, since a multi-round list comes from the caller's memory.
template <int K> struct RegHeap {
  uint64_t e[K];
  int id_offset;
  __device__ inline void init(float cutoff, int k, const uint64_t *src, bool fill, int off)
  {
    const uint64_t v = list_key(cutoff * cutoff, 0xffffffffu);
    id_offset = off;
#pragma unroll
    for (int i = 0; i < K; i++) e[i] = i < k ? (fill ? v : src[i]) : 0ull;
  }
  __device__ inline float cull() const { return __uint_as_float((uint32_t)(e[0] >> 32)); }
  __device__ inline void offer(int id, float d2, float &c)
  {
    const uint64_t v = list_key(d2, (uint32_t)(id + id_offset));
    if (v >= e[0]) return;
    sift<0>(v, true);
    c = cull();
  }
  // reference: the larger child moves up while it is not below v (a child of
  // equal key moves, the later child only if strictly larger)
  template <int P> __device__ inline void sift(uint64_t v, bool here)
  {
    if constexpr (2 * P + 1 >= K) {
      e[P] = here ? v : e[P];
    } else {
      if (!here) return;
      constexpr int A = 2 * P + 1, B = 2 * P + 2;
      if constexpr (B < K) {
        const bool right = e[B] > e[A];
        const uint64_t m = right ? e[B] : e[A];
        const bool stop = m < v || m == 0;
        e[P] = stop ? v : m;
        sift<A>(v, !stop && !right);
        sift<B>(v, !stop && right);
      } else {
        const bool stop = e[A] < v || e[A] == 0;
        e[P] = stop ? v : e[A];
        sift<A>(v, !stop);
      }
    }
  }
  __device__ inline void write(int k, int32_t *ids, float *dist2, float *ret, uint64_t *list) const
  {
    if (list) {
#pragma unroll
      for (int i = 0; i < K; i++)
        if (i < k) list[i] = e[i];
    } else {
      write_row<K>(e, 0, k, ids, dist2);
    }
    if (ret) *ret = cull();
  }
};

// round-robin split dim of level l (0 <= l < 32)
template <int D>
__device__ inline int rr_dim(int l)
{
  if ((D & (D - 1)) == 0) return l & (D - 1);
  if (D == 3) return l - (int)__umul24((unsigned)__umul24((unsigned)l, 11u) >> 5, 3u);  // l / 3 for l < 32
  return l % D;
}

// depths whose far child was cut off by a plane of dim j
template <int D>
constexpr uint32_t depths_of_dim(int j)
{
  uint32_t m = 0;
  for (int d = 1; d < 32; d++)
    if ((d - 1) % D == j) m |= 1u << d;
  return m;
}

// rows of a query's LDS column: row 0, and row d for the far child at depth
// d, which exists only if 2^d <= n
__host__ __device__ inline int sd_rows(int n)
{
  int r = 0;
  while (r < 30 && (2ll << r) <= (long long)n) r++;
  return r + 1;
}

template <int D, int METHOD, class L>
__global__ __launch_bounds__(256) void k_query_box(TreeView t, const float *queries, int nq,
                                                   const float *world_bounds, float cutoff,
                                                   float eps, int k, const int32_t *order,
                                                   int32_t *ids, float *dist2, float *ret,
                                                   ListArgs la, ForestQ fq, int rows)
{
  HIP_DYNAMIC_SHARED(float, s_pd);
  // XCD-aware workgroup order, as in k_query
  const int nb = (int)gridDim.x;
  const int xcd = (int)blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int lb = xcd * q8 + (xcd < r8 ? xcd : r8) + ((int)blockIdx.x >> 3);
  const int i = lb * (int)blockDim.x + (int)threadIdx.x;
  if (i >= nq) return;
  const int qi = order ? order[i] : i;
  const unsigned stride = (unsigned)t.stride;
  unsigned base = (unsigned)t.point_offset;  // of the query's tree (under 4 GiB in all)
  int n = t.n;
  if (fq.seg_off) {
    const int tr = fq.seg_tree[segment_of(fq.seg_off, fq.nseg, qi)];
    const int b = fq.tree_off[tr];
    base += (unsigned)b * stride;
    n = fq.tree_off[tr + 1] - b;
    if (METHOD == CUKD_CCT) world_bounds += (size_t)tr * 2 * D;
  }
  // the wave's rows, 64 words each; row 0 holds the distance of a dim that
  // no plane of the path has cut (0)
  float *col = s_pd + (threadIdx.x >> 6) * (rows * 64) + (threadIdx.x & 63);
  col[0] = 0.f;
  float q[D], o[D], o0[D];
#pragma unroll
  for (int d = 0; d < D; d++) q[d] = queries[(size_t)qi * D + d];
  // squared distance from the query to the current cell, per dim; the
  // closest-corner traversal starts from the world bounds
  bool done = n <= 0;
  L list;
  list.init(cutoff, k, la.lists ? la.lists + (size_t)qi * k : nullptr, !la.lists || la.init,
            la.id_offset);
  float cull = list.cull();
#pragma unroll
  for (int d = 0; d < D; d++) {
    o0[d] = 0.f;
    if (METHOD == CUKD_CCT) {
      float v = q[d];
      const float lo = world_bounds[d], hi = world_bounds[D + d];
      v = v < lo ? lo : v;
      v = hi < v ? hi : v;
      const float df = v - q[d];
      o0[d] = df * df;
    }
    o[d] = o0[d];
  }
  if (METHOD == CUKD_CCT) {
    float s = o0[0];
#pragma unroll
    for (int d = 1; d < D; d++) s = s + o0[d];
    if (s > cull) done = true;
  }
  const float eps1 = 1.f + eps;
  int curr = 0, lvl = 0;
  unsigned off = 0;                   // byte offset of curr in its tree
  unsigned pending = 0;               // bit d: the far child at depth d is still to be visited
  unsigned far = 0;                   // bit d: the path's node at depth d is a far child
  float topd = 0.f;                   // plane distance of the deepest pending far child
  bool pop = false;
  float p[D];                         // coordinates of curr (not while popping)
  const uint8_t *tb = t.base;
  auto load = [&](unsigned at) {
    const float *src = (const float *)(tb + (size_t)(base + at));
#pragma unroll
    for (int d = 0; d < D; d++) p[d] = src[d];
  };
  if (!done) load(0);
  while (!done) {
    if (pop) {
      const int d = 31 - __clz((int)pending);
      pending &= ~(1u << d);
      bool enter = METHOD == CUKD_STACK_FREE ? topd * eps1 < cull : topd < cull;
      const unsigned up = far & ((1u << d) - 1u);
      float c[D];
      const int dim = rr_dim<D>(d - 1);
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < D; j++) {
        const unsigned m = up & depths_of_dim<D>(j);
        const float v = col[(31 - __clz((int)(m | 1u))) * 64];
        c[j] = dim == j ? topd : (METHOD == CUKD_CCT && !m ? o0[j] : v);
        s = j == 0 ? c[0] : s + c[j];
      }
      if (METHOD == CUKD_CCT) enter = s < cull;
      if (enter) {
        curr = (((curr + 1) >> (lvl - d)) ^ 1) - 1;
        lvl = d;
        off = (unsigned)curr * stride;
        far = up | (1u << d);
#pragma unroll
        for (int j = 0; j < D; j++) o[j] = c[j];
        load(off);
        pop = false;
      } else if (!pending) {
        done = true;
      }
      topd = col[(31 - __clz((int)(pending | 1u))) * 64];
    }
    if (!pop) {
      float df[D], sq[D];
#pragma unroll
      for (int d = 0; d < D; d++) df[d] = p[d] - q[d];
      const int dim = rr_dim<D>(lvl);
      // plane minus query, exactly the negated difference the reference
      // squares; its sign is the comparison of the two (denormals are kept)
      const float diff = cukd::detail::pick<D>(df, dim);
      const bool left_close = METHOD == CUKD_STACK_FREE ? !(diff < 0.f) : diff > 0.f;
      // The close child's load goes out before this node is offered, so
      // that the list, the box and the push run in its latency.
      const int l = 2 * curr + 1;
      const int close_c = left_close ? l : l + 1;
      const unsigned close_off = 2u * off + (left_close ? stride : 2u * stride);
      pop = close_c >= n;
      if (!pop) load(close_off);
#pragma unroll
      for (int d = 0; d < D; d++) sq[d] = df[d] * df[d];
      float d2 = sq[0];
#pragma unroll
      for (int d = 1; d < D; d++) d2 = d2 + sq[d];
      list.offer(curr, d2, cull);
      const float dd = diff * diff;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < D; j++) {
        const float v = dim == j ? dd : o[j];
        s = j == 0 ? v : s + v;
      }
      bool near;
      if (METHOD == CUKD_CCT) near = s < cull;
      else if (METHOD == CUKD_STACK_FREE) near = dd * eps1 < cull && !(s > cull);
      else near = dd < cull && !(s > cull);
      if (near && l + (left_close ? 1 : 0) < n) {
        pending |= 2u << lvl;
        col[(lvl + 1) * 64] = dd;
        topd = dd;
      }
      curr = close_c;
      off = close_off;
      lvl++;
      done = pop && !pending;
    }
  }
  const size_t out = (size_t)qi * k;
  list.write(k, ids ? ids + out : nullptr, dist2 ? dist2 + out : nullptr, ret ? ret + qi : nullptr,
             la.lists ? la.lists + out : nullptr);
}

}  // namespace cukd_amd
