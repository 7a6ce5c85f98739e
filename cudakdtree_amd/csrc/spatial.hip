// spatial.hip -- spatial k-d tree build and queries for gfx950.
//
// Build (spatial-kdtree.h:496-612 in the reference): spatial_build.h splits
// large nodes round by round and finishes small ones in LDS; the kernels here
// build trees too deep for that, one round per tree level over all open
// nodes at once.  Both give the same tree:
//   decide   : leaf if count <= threshold, else split the widest centroid
//              extent at its centre (ties pick the earlier dim; a centre
//              not between the ends makes a degenerate "dim -1" split)
//   number   : children of this round's split nodes get consecutive ids in
//              ascending parent order (exclusive scan; the reference takes
//              atomicAdd order, so its numbering is not reproducible)
//   partition: each node's prims stay contiguous and in ascending prim id;
//              a stable partition sends them to the two children ("coord >=
//              pos" goes right; a degenerate split alternates by rank)
//   bounds   : children's centroid boxes grow with int-encoded float
//              atomics (order independent)
// then primIDs are laid out leaf by leaf in node-id order.  The host reads
// one counter per round to know whether another round is needed, as the
// reference does (spatial-kdtree.h:545-567).
//
// Queries: stack-based and closest-corner traversal with the reference's
// results, its 50-entry stack's overflow included (fcp.h:256-427,
// knn.h:566-752).
#pragma clang fp contract(off)
#include <new>
#include <type_traits>

#include "cukd/spatial-kdtree.h"
#include "cukd_common.h"
#include "query_impl.h"

namespace cukd_amd {

// AtomicBox encoding (spatial-kdtree.h:172-188): float -> int32 whose
// signed order is the float order (-0.0 sorts below +0.0)
__device__ inline int32_t abox_enc(float f)
{
  int32_t b = __float_as_int(f);
  if (b & (int32_t)0x80000000) b ^= 0x7fffffff;
  return b;
}
__device__ inline float abox_dec(int32_t b)
{
  if (b & (int32_t)0x80000000) b ^= 0x7fffffff;
  return __int_as_float(b);
}

// A coordinate as the builder sees it: int coordinates go through the
// reference's implicit int -> float conversion (AtomicBox::encode(float),
// 'const float center = get_coord(point,split.dim)',
// spatial-kdtree.h:172-188, 427-429).
__device__ inline float sp_coord(const uint8_t *pts, uint32_t i, const cukd_layout &L, int d)
{
  const uint32_t b = load_coord_bits(pts + (size_t)i * L.stride, L, d);
  return L.scalar_type == CUKD_SCALAR_F32 ? __uint_as_float(b) : (float)(int32_t)b;
}

// Node::pos and the bounds hold scalar_t: a float result stored into an
// int one is truncated by C's conversion for int points
// (spatial-kdtree.h:75-77, 163-168, 489).
__device__ inline uint32_t sp_store(float f, bool isf)
{
  return isf ? __float_as_uint(f) : (uint32_t)(int32_t)f;
}

enum { SP_OPEN = 0, SP_LEAF = 1, SP_SPLIT = 2, SP_INNER = 3 };

struct SpNode {
  int32_t lo[CUKD_MAX_DIMS], hi[CUKD_MAX_DIMS];
  uint32_t count;
  uint32_t start;    // first position of this node's prims
  uint32_t offset;   // first child (inner)
  uint32_t lex;      // left points before this node's, and its own (spatial_build.h)
  uint32_t lcount;
  int32_t level;
  int32_t dim;
  float pos;
  int32_t state;
};

// ---------------------------------------------------------------------------
// exclusive scan of uint32 (multi-block, recursive over block sums)
// ---------------------------------------------------------------------------
enum { SCAN_NT = 256, SCAN_ITEMS = 8, SCAN_TILE = SCAN_NT * SCAN_ITEMS };

__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *s, uint32_t &total)
{
  s[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < SCAN_NT; off <<= 1) {
    const uint32_t t = threadIdx.x >= (unsigned)off ? s[threadIdx.x - off] : 0u;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  total = s[SCAN_NT - 1];
  const uint32_t r = s[threadIdx.x] - v;
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(SCAN_NT) void k_scan_tiles(const uint32_t *in, uint32_t *out,
                                                        uint32_t *tile_sums, long long n)
{
  __shared__ uint32_t s[SCAN_NT];
  const long long base = (long long)blockIdx.x * SCAN_TILE + (long long)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS], sum = 0;
  for (int i = 0; i < SCAN_ITEMS; i++) {
    v[i] = base + i < n ? in[base + i] : 0u;
    sum += v[i];
  }
  uint32_t total;
  uint32_t run = block_exclusive_scan(sum, s, total);
  for (int i = 0; i < SCAN_ITEMS; i++) {
    if (base + i < n) out[base + i] = run;
    run += v[i];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(SCAN_NT) void k_scan_add(uint32_t *out, const uint32_t *tile_offsets,
                                                      long long n)
{
  const long long base = (long long)blockIdx.x * SCAN_TILE;
  const uint32_t add = tile_offsets[blockIdx.x];
  for (int i = threadIdx.x; i < SCAN_TILE; i += SCAN_NT)
    if (base + i < n) out[base + i] += add;
}

// scratch: at least scan_scratch_words(n) uint32
size_t scan_scratch_words(long long n)
{
  size_t w = 0;
  while (n > 1) {
    n = (n + SCAN_TILE - 1) / SCAN_TILE;
    w += (size_t)n + 1;
  }
  return w + 1;
}

void scan_exclusive(hipError_t &e, const uint32_t *in, uint32_t *out, long long n,
                    uint32_t *scratch, hipStream_t s)
{
  if (n <= 0) return;
  const long long tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  uint32_t *sums = scratch;
  CUKD_LAUNCH(e, k_scan_tiles, dim3((unsigned)tiles), dim3(SCAN_NT), 0, s, in, out, sums, n);
  if (tiles > 1) {
    scan_exclusive(e, sums, sums, tiles, scratch + tiles + 1, s);
    CUKD_LAUNCH(e, k_scan_add, dim3((unsigned)tiles), dim3(SCAN_NT), 0, s, out,
                (const uint32_t *)sums, n);
  }
}

// ---------------------------------------------------------------------------
// build kernels
// ---------------------------------------------------------------------------
__global__ void k_sp_init(SpNode *nodes, uint32_t *pos_prim, uint32_t *pos_node, uint32_t *degen,
                          int n, int D)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *degen = 0u;
  if (i < 2) {
    SpNode &t = nodes[i];
    for (int d = 0; d < D; d++) { t.lo[d] = abox_enc(3.402823466e+38f); t.hi[d] = abox_enc(-3.402823466e+38f); }
    t.count = i == 0 ? (uint32_t)n : 0u;
    t.start = 0;
    t.offset = 0;
    t.dim = 0;
    t.pos = 0.f;
    t.state = i == 0 ? SP_OPEN : SP_LEAF;
  }
  if (i < n) {
    pos_prim[i] = (uint32_t)i;
    pos_node[i] = 0u;
  }
}

__global__ __launch_bounds__(256) void k_sp_root_bounds(SpNode *nodes, const uint8_t *pts, int n,
                                                        cukd_layout L)
{
  __shared__ int32_t s_lo[CUKD_MAX_DIMS][256], s_hi[CUKD_MAX_DIMS][256];
  const int D = L.num_dims;
  int32_t lo[CUKD_MAX_DIMS], hi[CUKD_MAX_DIMS];
  for (int d = 0; d < D; d++) { lo[d] = 0x7fffffff; hi[d] = (int32_t)0x80000000; }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    for (int d = 0; d < D; d++) {
      const int32_t e = abox_enc(sp_coord(pts, (uint32_t)i, L, d));
      lo[d] = min(lo[d], e);
      hi[d] = max(hi[d], e);
    }
  }
  for (int d = 0; d < D; d++) { s_lo[d][threadIdx.x] = lo[d]; s_hi[d][threadIdx.x] = hi[d]; }
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off)
      for (int d = 0; d < D; d++) {
        s_lo[d][threadIdx.x] = min(s_lo[d][threadIdx.x], s_lo[d][threadIdx.x + off]);
        s_hi[d][threadIdx.x] = max(s_hi[d][threadIdx.x], s_hi[d][threadIdx.x + off]);
      }
    __syncthreads();
  }
  if ((int)threadIdx.x < D) {
    atomicMin(&nodes[0].lo[threadIdx.x], s_lo[threadIdx.x][0]);
    atomicMax(&nodes[0].hi[threadIdx.x], s_hi[threadIdx.x][0]);
  }
}

// selectSplits' rule (spatial-kdtree.h:316-396): the widest extent at its
// centre, ties to the earlier dim; -1 (the points are dealt out in turn) where
// the centre is not strictly between the extent's ends.  The reference looks
// for a centre equal to an end only, and its build never ends where the sum of
// the ends overflows or is NaN: one child would keep every point.  The halves
// are added instead where the sum overflows, so both children of any split
// have points, which bounds the nodes of a subtree of m points by 2 m - 1.
// box(w): lower ends, then upper ends, encoded.
template <class F>
__device__ inline int sp_choose(int D, F box, float &pos)
{
  float widest_w = 0.f;
  int widest = -1;
  for (int d = 0; d < D; d++) {
    const float w = abox_dec(box(D + d)) - abox_dec(box(d));
    if (w <= widest_w) continue;
    widest_w = w;
    widest = d;
  }
  if (widest >= 0) {
    const float lo = abox_dec(box(widest)), hi = abox_dec(box(D + widest));
    pos = 0.5f * (lo + hi);
    if (isinf(pos)) pos = 0.5f * lo + 0.5f * hi;
    if (!(pos > lo && pos < hi)) widest = -1;
  }
  if (widest < 0) pos = abox_dec(box(0));
  return widest;
}

// selectSplits for the open nodes [a, b)
__global__ void k_sp_decide(SpNode *nodes, uint32_t *split_flag, uint32_t *degen, int a, int b,
                            int D, uint32_t threshold)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (a + i >= b) return;
  SpNode &t = nodes[a + i];
  uint32_t is_split = 0;
  if (t.count <= threshold) {
    t.state = SP_LEAF;
    t.offset = 0xffffffffu;
    t.dim = 0;
    t.pos = 0.f;
  } else {
    float pos;
    const int dim = sp_choose(D, [&](int w) { return w < D ? t.lo[w] : t.hi[w - D]; }, pos);
    if (dim < 0) *degen = 1u;  // same value from every writer
    t.dim = dim;
    t.pos = pos;
    t.state = SP_SPLIT;
    is_split = 1;
  }
  split_flag[i] = is_split;
}

// child ids and empty child boxes
__global__ void k_sp_alloc(SpNode *nodes, const uint32_t *split_excl, int a, int b, int next,
                           int D)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (a + i >= b) return;
  SpNode &t = nodes[a + i];
  if (t.state != SP_SPLIT) return;
  t.offset = (uint32_t)next + 2u * split_excl[i];
  for (int side = 0; side < 2; side++) {
    SpNode &c = nodes[t.offset + side];
    for (int d = 0; d < D; d++) { c.lo[d] = abox_enc(3.402823466e+38f); c.hi[d] = abox_enc(-3.402823466e+38f); }
    c.state = SP_OPEN;
    c.offset = 0;
    c.dim = 0;
    c.pos = 0.f;
    c.count = 0;
    c.start = t.start;
  }
}

// updatePrims (spatial-kdtree.h:398-436) part 1: side of every prim
__global__ void k_sp_classify(const SpNode *nodes, const uint32_t *pos_prim,
                              const uint32_t *pos_node, uint32_t *left_flag, const uint8_t *pts,
                              int n, cukd_layout L)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const SpNode &t = nodes[pos_node[p]];
  uint32_t left = 0;
  if (t.state == SP_SPLIT) {
    int side;
    if (t.dim < 0) {
      side = (int)(((uint32_t)p - t.start) & 1u);
    } else {
      side = sp_coord(pts, pos_prim[p], L, t.dim) >= t.pos;
    }
    left = side == 0;
  }
  left_flag[p] = left;
}

// updatePrims part 2: stable partition into the children, child boxes.
// The boxes grow with one atomic per (child, word) and wave: the lanes of a
// wave hold consecutive positions, so nearly always one or two children,
// and per-prim atomics on the few children of the top levels serialise
// (min and max are order-independent, so the boxes are the same).
__global__ __launch_bounds__(256) void k_sp_scatter(SpNode *nodes, const uint32_t *pos_prim,
                                                    const uint32_t *pos_node,
                                                    const uint32_t *left_flag,
                                                    const uint32_t *left_excl, uint32_t *npos_prim,
                                                    uint32_t *npos_node, const uint8_t *pts, int n,
                                                    cukd_layout L)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const int D = L.num_dims;
  const int lane = (int)threadIdx.x & 63;
  uint32_t mychild = 0xffffffffu;  // none: past the end, or not split this round
  int32_t e[CUKD_MAX_DIMS];
#pragma unroll
  for (int d = 0; d < CUKD_MAX_DIMS; d++) e[d] = 0;
  if (p < n) {
    const uint32_t node = pos_node[p];
    const SpNode &t = nodes[node];
    const uint32_t prim = pos_prim[p];
    if (t.state != SP_SPLIT) {
      npos_prim[p] = prim;
      npos_node[p] = node;
    } else {
      const uint32_t end = t.start + t.count;
      const uint32_t left_end =
          end < (uint32_t)n ? left_excl[end] : left_excl[n - 1] + left_flag[n - 1];
      const uint32_t lcount = left_end - left_excl[t.start];
      const uint32_t lrank = left_excl[p] - left_excl[t.start];
      uint32_t np, child;
      if (left_flag[p]) {
        np = t.start + lrank;
        child = t.offset;
      } else {
        np = t.start + lcount + ((uint32_t)p - t.start - lrank);
        child = t.offset + 1;
      }
      npos_prim[np] = prim;
      npos_node[np] = child;
      SpNode &c = nodes[child];
      if (lrank == 0 && left_flag[p]) {
        c.count = lcount;
        c.start = t.start;
      }
      if (!left_flag[p] && (uint32_t)p - t.start - lrank == 0) {
        c.count = t.count - lcount;
        c.start = t.start + lcount;
      }
      mychild = child;
#pragma unroll
      for (int d = 0; d < CUKD_MAX_DIMS; d++)
        if (d < D) e[d] = abox_enc(sp_coord(pts, prim, L, d));
    }
  }
  // every lane of the wave takes part: one child per trip
  uint64_t active = __ballot(mychild != 0xffffffffu);
  while (active) {
    const int leader = __ffsll((unsigned long long)active) - 1;
    const uint32_t c = (uint32_t)__shfl((int)mychild, leader);
    const bool peer = mychild == c;
    active &= ~__ballot(peer);
#pragma unroll
    for (int d = 0; d < CUKD_MAX_DIMS; d++) {
      if (d >= D) break;
      int32_t lo = peer ? e[d] : 0x7fffffff, hi = peer ? e[d] : (int32_t)0x80000000;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o));
        hi = max(hi, __shfl_xor(hi, o));
      }
      if (lane == leader) {
        atomicMin(&nodes[c].lo[d], lo);
        atomicMax(&nodes[c].hi[d], hi);
      }
    }
  }
}

// split nodes of this round become inner nodes; count the next round
__global__ void k_sp_close(SpNode *nodes, const uint32_t *split_flag, const uint32_t *split_excl,
                           int a, int b, uint32_t *num_split)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (a + i >= b) return;
  SpNode &t = nodes[a + i];
  if (t.state == SP_SPLIT) t.state = SP_INNER;
  if (a + i == b - 1) *num_split = split_excl[i] + split_flag[i];
}

// leaf offsets in node-id order, then primIDs leaf by leaf
__global__ void k_sp_leaf_counts(const SpNode *nodes, uint32_t *cnt, int num_nodes)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_nodes) return;
  cnt[i] = nodes[i].state == SP_LEAF ? nodes[i].count : 0u;
}

__global__ void k_sp_write_prims(const SpNode *nodes, const uint32_t *leaf_off,
                                 const uint32_t *pos_prim, const uint32_t *pos_node,
                                 uint32_t *prim_ids, int n)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t node = pos_node[p];
  prim_ids[leaf_off[node] + ((uint32_t)p - nodes[node].start)] = pos_prim[p];
}

// writeNodes (spatial-kdtree.h:477-494): dim -1 is stored as 0
__global__ void k_sp_write_nodes(const SpNode *nodes, const uint32_t *leaf_off,
                                 cukd_spatial_node *out, int num_nodes, bool isf)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_nodes) return;
  const SpNode &t = nodes[i];
  cukd_spatial_node o;
  if (t.state == SP_LEAF) {
    o.offset = t.count > 0 ? leaf_off[i] : (i == 1 ? 0u : 0xffffffffu);
    o.count = (uint16_t)t.count;
    o.dim = 0;
    o.pos = 0.f;
  } else {
    o.offset = t.offset;
    o.count = 0;
    o.dim = (int16_t)(t.dim < 0 ? 0 : t.dim);
    o.ipos = (int32_t)sp_store(t.pos, isf);
  }
  out[i] = o;
}

// saveBounds (spatial-kdtree.h:464-473): box_t of scalar_t
__global__ void k_sp_bounds_out(const SpNode *nodes, uint32_t *bounds, int D, bool isf)
{
  const int d = threadIdx.x;
  if (d < D) {
    bounds[d] = sp_store(abox_dec(nodes[0].lo[d]), isf);
    bounds[D + d] = sp_store(abox_dec(nodes[0].hi[d]), isf);
  }
}

// The bounds' last two words, unused below 8 dims, record what queries may do
// with the tree: prune by box (k_spatial_query), if it has no degenerate split
// and no path of 50 inner nodes, and take scratch from the library's memory,
// if the tree itself was built there and not with a caller's resource.  Without
// the record they do neither.
enum : int32_t { SP_MARK = 0x70727562, SP_MARK2 = 0x786f6200 };
static void spatial_record(cukd_spatial_tree *tree, int D, bool prunable, const MemResource &mem)
{
  if (D >= CUKD_MAX_DIMS) return;
  const bool scratch = !(mem.user && mem.user->malloc_fn);
  tree->ibounds[2 * CUKD_MAX_DIMS - 2] = SP_MARK;
  tree->ibounds[2 * CUKD_MAX_DIMS - 1] =
      SP_MARK2 | (prunable ? SPATIAL_MAY_PRUNE : 0) | (scratch ? SPATIAL_MAY_ALLOCATE : 0);
}

int spatial_may(const cukd_spatial_tree *tree, int D)
{
  const int32_t w = tree->ibounds[2 * CUKD_MAX_DIMS - 1];
  const int all = SPATIAL_MAY_PRUNE | SPATIAL_MAY_ALLOCATE;
  if (D >= CUKD_MAX_DIMS || tree->ibounds[2 * CUKD_MAX_DIMS - 2] != SP_MARK) return 0;
  return (w & ~all) == SP_MARK2 ? w & all : 0;
}

enum { SP_DEPTH = 50 };  // the reference's traversal stack (fcp.h:265)

}  // namespace cukd_amd

#include "spatial_build.h"

namespace cukd_amd {

static int spatial_build_rounds(cukd_spatial_tree *tree, const void *d_points, int n,
                                const cukd_layout &L, uint32_t thr, hipStream_t s,
                                const MemResource &mem);

int spatial_build_impl(cukd_spatial_tree *tree, const void *d_points, int n, const cukd_layout &L,
                       int leaf_threshold, hipStream_t s, const MemResource &mem)
{
  const uint32_t thr = leaf_threshold <= 0 ? 8u : (uint32_t)leaf_threshold;
  (void)hipGetLastError();  // an earlier call's error is no launch's below
  if (n > 0 && (uint32_t)n > thr) {  // one leaf takes fewer launches round by round
    const uint8_t *pts = (const uint8_t *)d_points;
    bool deep = false;
    int rc;
    switch (L.num_dims) {
      case 1: rc = spatial_build_items<1>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 2: rc = spatial_build_items<2>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 3: rc = spatial_build_items<3>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 4: rc = spatial_build_items<4>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 5: rc = spatial_build_items<5>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 6: rc = spatial_build_items<6>(tree, pts, n, L, thr, s, mem, &deep); break;
      case 7: rc = spatial_build_items<7>(tree, pts, n, L, thr, s, mem, &deep); break;
      default: rc = spatial_build_items<8>(tree, pts, n, L, thr, s, mem, &deep); break;
    }
    if (rc != CUKD_OK || !deep) return rc;
  }
  return spatial_build_rounds(tree, d_points, n, L, thr, s, mem);
}

// Round by round over all open nodes: trees of more than SPB_LEVELS levels, and
// those of one leaf (5 points 200 us, 228 the other way).
static int spatial_build_rounds(cukd_spatial_tree *tree, const void *d_points, int n,
                                const cukd_layout &L, uint32_t thr, hipStream_t s,
                                const MemResource &mem)
{
  const int D = L.num_dims;
  const size_t max_nodes = 2 * (size_t)(n > 0 ? n : 1) + 2;
  const size_t nn = (size_t)(n > 0 ? n : 1);
  const size_t scan_words = scan_scratch_words((long long)(max_nodes > nn ? max_nodes : nn));
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o = (o + bytes + 255) & ~(size_t)255; return at; };
  const size_t o_nodes = take(max_nodes * sizeof(SpNode));
  const size_t o_pp0 = take(nn * 4), o_pn0 = take(nn * 4), o_pp1 = take(nn * 4), o_pn1 = take(nn * 4);
  const size_t o_nflag = take(max_nodes * 4), o_nexcl = take(max_nodes * 4);
  const size_t o_pflag = take(nn * 4), o_pexcl = take(nn * 4);
  const size_t o_scan = take(scan_words * 4), o_misc = take(256);
  uint8_t *tmp = nullptr;
  if (mem.alloc((void **)&tmp, o, s) != 0) return CUKD_ERR_ALLOC;
  SpNode *nodes = (SpNode *)(tmp + o_nodes);
  uint32_t *pp[2] = {(uint32_t *)(tmp + o_pp0), (uint32_t *)(tmp + o_pp1)};
  uint32_t *pn[2] = {(uint32_t *)(tmp + o_pn0), (uint32_t *)(tmp + o_pn1)};
  uint32_t *nflag = (uint32_t *)(tmp + o_nflag), *nexcl = (uint32_t *)(tmp + o_nexcl);
  uint32_t *pflag = (uint32_t *)(tmp + o_pflag), *pexcl = (uint32_t *)(tmp + o_pexcl);
  uint32_t *scratch = (uint32_t *)(tmp + o_scan);
  uint32_t *num_split = (uint32_t *)(tmp + o_misc);
  uint32_t *bounds_dev = (uint32_t *)(tmp + o_misc + 64);  // 2 * D words, then degen
  uint32_t *degen = bounds_dev + 2 * D;
  const bool isf = L.scalar_type == CUKD_SCALAR_F32;
  const uint8_t *pts = (const uint8_t *)d_points;
  int rc = CUKD_OK;
  hipError_t e = hipSuccess;

  CUKD_LAUNCH(e, k_sp_init, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, s, nodes, pp[0],
              pn[0], degen, n, D);
  if (n > 0) {
    int blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    CUKD_LAUNCH(e, k_sp_root_bounds, dim3(blocks), dim3(256), 0, s, nodes, pts, n, L);
  }
  // open nodes [a, b); node 1 is the reference's reserved empty leaf, so
  // the first children are numbered from 2
  int cur = 0, a = 0, b = 1, next = 2, levels = 0;
  const int gp = (n + 255) / 256;
  while (a < b) {
    levels++;
    const int cnt = b - a;
    const int g = (cnt + 255) / 256;
    CUKD_LAUNCH(e, k_sp_decide, dim3(g), dim3(256), 0, s, nodes, nflag, degen, a, b, D,
                thr);
    scan_exclusive(e, nflag, nexcl, cnt, scratch, s);
    CUKD_LAUNCH(e, k_sp_alloc, dim3(g), dim3(256), 0, s, nodes, (const uint32_t *)nexcl, a, b, next,
                D);
    if (n > 0) {
      CUKD_LAUNCH(e, k_sp_classify, dim3(gp), dim3(256), 0, s, (const SpNode *)nodes,
                  (const uint32_t *)pp[cur], (const uint32_t *)pn[cur], pflag, pts, n, L);
      scan_exclusive(e, pflag, pexcl, n, scratch, s);
      CUKD_LAUNCH(e, k_sp_scatter, dim3(gp), dim3(256), 0, s, nodes, (const uint32_t *)pp[cur],
                  (const uint32_t *)pn[cur], (const uint32_t *)pflag, (const uint32_t *)pexcl,
                  pp[cur ^ 1], pn[cur ^ 1], pts, n, L);
      cur ^= 1;
    }
    CUKD_LAUNCH(e, k_sp_close, dim3(g), dim3(256), 0, s, nodes, (const uint32_t *)nflag,
                (const uint32_t *)nexcl, a, b, num_split);
    uint32_t h_split = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&h_split, num_split, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) break;
    a = next;
    b = next + 2 * (int)h_split;
    next = b;
  }
  const int num_nodes = next;
  cukd_spatial_node *out_nodes = nullptr;
  uint32_t *out_prims = nullptr;
  if (e == hipSuccess) {
    if (mem.alloc((void **)&out_nodes, (size_t)num_nodes * sizeof(cukd_spatial_node), s) != 0 ||
        mem.alloc((void **)&out_prims, nn * 4, s) != 0) {
      rc = CUKD_ERR_ALLOC;
    } else {
      const int g = (num_nodes + 255) / 256;
      CUKD_LAUNCH(e, k_sp_leaf_counts, dim3(g), dim3(256), 0, s, (const SpNode *)nodes, nflag,
                  num_nodes);
      scan_exclusive(e, nflag, nexcl, num_nodes, scratch, s);
      if (n > 0)
        CUKD_LAUNCH(e, k_sp_write_prims, dim3(gp), dim3(256), 0, s, (const SpNode *)nodes,
                    (const uint32_t *)nexcl, (const uint32_t *)pp[cur],
                    (const uint32_t *)pn[cur], out_prims, n);
      CUKD_LAUNCH(e, k_sp_write_nodes, dim3(g), dim3(256), 0, s, (const SpNode *)nodes,
                  (const uint32_t *)nexcl, out_nodes, num_nodes, isf);
      CUKD_LAUNCH(e, k_sp_bounds_out, dim3(1), dim3(64), 0, s, (const SpNode *)nodes,
                  bounds_dev, D, isf);
      uint32_t hb[2 * CUKD_MAX_DIMS + 1];
      if (e == hipSuccess) e = hipMemcpyAsync(hb, bounds_dev, 4 * (2 * D + 1), hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e == hipSuccess) {
        for (int i = 0; i < 2 * CUKD_MAX_DIMS; i++) tree->ibounds[i] = i < 2 * D ? (int32_t)hb[i] : 0;
        spatial_record(tree, D, levels <= SP_DEPTH && hb[2 * D] == 0u, mem);
        tree->nodes = out_nodes;
        tree->prim_ids = out_prims;
        tree->data = d_points;
        tree->num_prims = n;
        tree->num_nodes = num_nodes;
      }
    }
  }
  mem.release(tmp, s);
  if (e != hipSuccess) {
    if (out_nodes) mem.release(out_nodes, s);
    if (out_prims) mem.release(out_prims, s);
    set_last_error("spatial build failed: %s", hipGetErrorString(e));
    return CUKD_ERR_HIP;
  }
  if (rc != CUKD_OK) {
    if (out_nodes) mem.release(out_nodes, s);
    if (out_prims) mem.release(out_prims, s);
  }
  return rc;
}

// ---------------------------------------------------------------------------
// spatial queries
// ---------------------------------------------------------------------------

// One query per lane, with the results of the reference's traversals
// (fcp.h:256-427, knn.h:566-752; cukd/spatial-kdtree.h states them) bit for
// bit.
//
// Each iteration of a wave pops, takes up to SP_STEPS steps down, and offers
// SP_POINTS points of a leaf: ids and points are loaded together, the
// distances that may be accepted are offered in order, one per trip and lane.
// A chunk's missing points repeat its first (branches around single loads
// cost more than the loads).
//
// Box pruning (prune), as in k_query_box: the stack-based traversal also skips
// a far child whose cell is beyond the cull distance, which no list accepts
// from.  The host allows it where the tree is known to have no degenerate
// split, whose children may lie on either side of the plane, and to be
// shallower than the reference's stack, so that no skipped subtree could have
// overflowed it.  Otherwise, and while visits are counted, nothing is
// skipped beyond the reference's own test.
//
// Bound by lane use (15 of 64 per vector instruction: lanes pop, step and read
// leaves at different times) and by a line access per point.  kNN-16 within
// 0.05, 2M queries over 4M float4: 12.2 -> 3.8 ms with the Morton order (2.2
// ms of it the order, 1.7 ms the box); closest-corner 13.5 -> 3.8; heap 16
// 14.5 -> 3.9; kNN-64 over 4M float3, 1M queries: 28.7 -> 6.9 ms.  One step
// per iteration 3.9 ms; node, ids and points loaded an iteration ahead, one
// round trip each, 5.2 ms.
//
// The stack is indexed at run time: its first COLS entries (a node with its
// parent's split dim in the top bits, and the cell's squared distance per
// dim) are LDS columns, only deeper ones a per-lane array in scratch.
enum { SP_POINTS = 4, SP_STEPS = 3, SP_DIM_SHIFT = 29 };
enum { SP_POP = 0, SP_NODE = 1, SP_PTS = 2 };
// 10 KB a wave: at 7.5 KB kNN-16 loses 3 % to scratch, at 5 KB 20 %, at 15 KB
// 40 % to the waves that no longer fit
template <int D> constexpr int sp_cols() { return 40 / (D + 1) < 16 ? 40 / (D + 1) : 16; }

template <int D, bool CCT, class L>
__global__ __launch_bounds__(256) void k_spatial_query(const cukd_spatial_node *nodes,
                                                       const uint32_t *prim_ids, TreeView data,
                                                       SpatialBounds bounds, const float *queries,
                                                       int nq, float cutoff, int k, bool prune,
                                                       const int32_t *order, int32_t *ids,
                                                       float *dist2, float *ret,
                                                       unsigned long long *stats)
{
  constexpr int W = D + 1, COLS = sp_cols<D>();
  HIP_DYNAMIC_SHARED(uint32_t, s_stack);
  // XCD-aware workgroup order, as in k_query
  const int nb = (int)gridDim.x;
  const int xcd = (int)blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int lb = xcd * q8 + (xcd < r8 ? xcd : r8) + ((int)blockIdx.x >> 3);
  const int i = lb * (int)blockDim.x + (int)threadIdx.x;
  if (i >= nq) return;
  const int qi = order ? order[i] : i;
  uint32_t *col = s_stack + (threadIdx.x >> 6) * (COLS * W * 64) + (threadIdx.x & 63);
  uint32_t deep[(SP_DEPTH - COLS) * W];  // entries COLS and up
  float q[D], o[D];                      // o: squared distance to the current cell, per dim
#pragma unroll
  for (int d = 0; d < D; d++) q[d] = queries[(size_t)qi * D + d];
  L list;
  list.init(cutoff, k, nullptr, true, 0);
  float cull = list.cull();
  unsigned visits = 0;
  int sp = 0, stage = SP_NODE;
  bool done = false, ok = true;
#pragma unroll
  for (int d = 0; d < D; d++) {
    o[d] = 0.f;
    if (CCT) {
      float v = q[d];
      v = v < bounds.v[d] ? bounds.v[d] : v;
      v = bounds.v[D + d] < v ? bounds.v[D + d] : v;
      const float df = v - q[d];
      o[d] = df * df;
    }
  }
  if (CCT) {
    float s = o[0];
#pragma unroll
    for (int d = 1; d < D; d++) s = s + o[d];
    done = s > cull;
  }
  uint32_t li = 0, le = 0;  // points of the current leaf still to be offered
  int node = 0;
  while (!done) {
    if (stage == SP_POP) {
      if (sp == 0) {
        done = true;
      } else {
        --sp;
        uint32_t e[W];
        if (sp < COLS) {
#pragma unroll
          for (int w = 0; w < W; w++) e[w] = col[(sp * W + w) * 64];
        } else {
#pragma unroll
          for (int w = 0; w < W; w++) e[w] = deep[(sp - COLS) * W + w];
        }
        float c[D], s = 0.f;
#pragma unroll
        for (int d = 0; d < D; d++) {
          c[d] = __uint_as_float(e[1 + d]);
          s = d == 0 ? c[0] : s + c[d];
        }
        const float plane2 = cukd::detail::pick<D>(c, (int)(e[0] >> SP_DIM_SHIFT));
        if (!((CCT ? s : plane2) >= cull) && !(!CCT && prune && s > cull)) {
          node = (int)(e[0] & ((1u << SP_DIM_SHIFT) - 1u));
#pragma unroll
          for (int d = 0; d < D; d++) o[d] = c[d];
          stage = SP_NODE;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < SP_STEPS; u++) {
      if (stage != SP_NODE || done) break;
      visits++;
      const cukd_spatial_node nd = nodes[node];
      // an empty root leaf (no points) has count 0 and offset ~0u
      if (nd.count || nd.offset == 0xffffffffu) {
        li = nd.offset;
        le = nd.offset + nd.count;
        stage = nd.count ? SP_PTS : SP_POP;
      } else {
        const int dim = nd.dim;
        const float qc = cukd::detail::pick<D>(q, dim);
        const bool left_close = qc < nd.pos;
        const float diff = qc - nd.pos;
        const float plane2 = diff * diff;
        const uint32_t far_c = nd.offset + (left_close ? 1u : 0u);
        node = (int)(nd.offset + (left_close ? 0u : 1u));
        uint32_t e[W];
        float s = 0.f;
        e[0] = far_c | (uint32_t)dim << SP_DIM_SHIFT;
#pragma unroll
        for (int d = 0; d < D; d++) {
          const float v = d == dim ? plane2 : o[d];
          e[1 + d] = __float_as_uint(v);
          s = d == 0 ? v : s + v;
        }
        if (CCT ? s < cull : plane2 < cull && !(prune && s > cull)) {
          if (sp < COLS) {
#pragma unroll
            for (int w = 0; w < W; w++) col[(sp * W + w) * 64] = e[w];
          } else {
#pragma unroll
            for (int w = 0; w < W; w++) deep[(sp - COLS) * W + w] = e[w];
          }
          if (++sp >= SP_DEPTH) {
            ok = false;
            done = true;
          }
        }
      }
    }
    if (stage == SP_PTS && !done) {
      const uint32_t m = le - li < SP_POINTS ? le - li : SP_POINTS;
      visits += m;
      uint32_t prim[SP_POINTS];
      float p[SP_POINTS][D], d2[SP_POINTS];
#pragma unroll
      for (int j = 0; j < SP_POINTS; j++)
        prim[j] = prim_ids[li + ((uint32_t)j < m ? j : 0)];
#pragma unroll
      for (int j = 0; j < SP_POINTS; j++) data.template point<D>((int)prim[j], p[j]);
      unsigned in = 0;  // bit j: point j may be accepted
#pragma unroll
      for (int j = 0; j < SP_POINTS; j++) {
        d2[j] = cukd::detail::sqr_dist<D>(p[j], q);
        if ((uint32_t)j < m && d2[j] <= cull) in |= 1u << j;
      }
      // in order, one per trip and lane: most lanes take none or one
      while (in) {
        float v = d2[0];
        uint32_t id = prim[0];
        const unsigned low = in & (0u - in);
#pragma unroll
        for (int j = 1; j < SP_POINTS; j++) {
          v = low == 1u << j ? d2[j] : v;
          id = low == 1u << j ? prim[j] : id;
        }
        list.offer((int)id, v, cull);
        in &= in - 1;
      }
      li += m;
      if (li == le) stage = SP_POP;
    }
  }
  if (stats) atomicAdd(stats, (unsigned long long)visits);
  const size_t out = (size_t)qi * k;
  list.write(k, ids + out, dist2 ? dist2 + out : nullptr, ret ? ret + qi : nullptr, nullptr);
  // stack overflow: fcp reports no result, knn returns -1 (fcp.h:317-320,
  // knn.h:620-623 print "STACK OVERFLOW" and return -1) where the caller takes
  // the radii, and leaves the row as found
  if (!ok) {
    if (std::is_same<L, RegClosest>::value) ids[qi] = -1;
    else if (ret) ret[qi] = -1.f;
  }
}

// The traversals of cukd/spatial-kdtree.h as they stand, with lists whose
// keys are compared as integers: for NaN cutoffs, whose keys have no order
// as doubles, for trees of 2^29 nodes and more, and where reading single points
// wins:
//  * one dim, few entries, below 2^18 queries, over 1K .. 1M points: FCP takes
//    0.72 .. 1.02 times the kernel above, k = 1 and 2 0.74 .. 1.1, k = 4 0.71 ..
//    1.2 with the list in registers; k = 3, and 5 and more, 1.0 .. 2.2 times;
//  * the closest point of 2^19 queries and more in a small tree, if half of
//    them find none: 1M queries over 100K float4 330 us here, 386 above.  Where
//    most find one it is 563 against 359 (2^19 queries), but never slower than
//    it has been.
// The first 16 entries of the stack-based FCP's stack are LDS columns.
template <bool CCT, class R> struct SpStackCols {
  enum { value = (CCT || ResultOps<R>::kLds) ? 0 : 16 };
};

template <int D, bool CCT, class R>
__global__ __launch_bounds__(128) void k_spatial_query_any(const cukd_spatial_node *nodes,
                                                       const uint32_t *prim_ids, TreeView data,
                                                       SpatialBounds bounds, const float *queries,
                                                       int nq, float cutoff, int k,
                                                       int32_t *ids, float *dist2, float *ret,
                                                       unsigned long long *stats)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  float q[D];
#pragma unroll
  for (int d = 0; d < D; d++) q[d] = queries[(size_t)i * D + d];
  HIP_DYNAMIC_SHARED(uint64_t, s_lists);
  typename ResultOps<R>::State st;
  const ListArgs no_lists{nullptr, 0, 0};
  R &res = ResultOps<R>::init(st, cutoff, k, i, no_lists,
                              LdsCol{s_lists + threadIdx.x, (int)blockDim.x});
  float lo[D], hi[D];
#pragma unroll
  for (int d = 0; d < D; d++) { lo[d] = bounds.v[d]; hi[d] = bounds.v[D + d]; }
  unsigned visits = 0;
  // stack columns: COLS node words, then as many dist2 words, each row
  // blockDim.x wide
  constexpr int COLS = SpStackCols<CCT, R>::value;
  uint32_t *stk = (uint32_t *)s_lists + threadIdx.x;
  const cukd::detail::SpatialStackCols cols{
      (int *)stk, (float *)(stk + (size_t)COLS * blockDim.x), (int)blockDim.x};
  const bool ok = cukd::detail::spatial_traverse<D, CCT, COLS>(res, q, nodes, prim_ids, lo, hi,
                                                                data, visits, cols);
  if (stats) atomicAdd(stats, (unsigned long long)visits);
  ResultOps<R>::write(st, i, k, ids, dist2, ret, no_lists);
  // stack overflow: fcp reports no result, knn returns -1 (fcp.h:317-320,
  // knn.h:620-623 print "STACK OVERFLOW" and return -1) where the caller takes
  // the radii, and leaves the row as found
  if (!ok) {
    if (std::is_same<R, cukd::FCPResult>::value) ids[i] = -1;
    else if (ret) ret[i] = -1.f;
  }
}

template <int D, bool CCT, class L>
static void launch_spatial_l(const SpatialArgs &a, hipStream_t s)
{
  const int nt = 64, blocks = (a.nq + nt - 1) / nt;
  const size_t shm = (size_t)(D + 1) * sp_cols<D>() * nt * 4;
  hipLaunchKernelGGL((k_spatial_query<D, CCT, L>), dim3(blocks), dim3(nt), shm, s, a.nodes,
                     a.prim_ids, a.data, a.bounds, a.queries, a.nq, a.cutoff, a.k, a.prune, a.order, a.ids,
                     a.dist2, a.ret, a.stats);
}

template <int D, bool CCT>
static hipError_t launch_spatial_m(const SpatialArgs &a, hipStream_t s)
{
  const bool small_fcp = !CCT && a.list_kind < 0 && a.nq >= (1 << 19) &&
                         (uint64_t)a.data.n * (uint64_t)a.data.stride < SPATIAL_ORDER_MIN_BYTES;
  const bool line = D == 1 && a.nq < (1 << 18) &&
                    (a.k <= 2 || (a.k == 4 && a.list_kind == CUKD_LIST_FIXED));
  if (a.cutoff != a.cutoff || a.num_nodes > (1 << SP_DIM_SHIFT) || small_fcp || line) {
    const int nt = 128, blocks = (a.nq + nt - 1) / nt;
    // dynamic LDS: k 64-bit words per lane (64 KiB at k = 64), or the stack
    // columns (16 KiB)
#define CUKD_SPQ(R)                                                                             \
  hipLaunchKernelGGL((k_spatial_query_any<D, CCT, R>), dim3(blocks), dim3(nt),                  \
                     ((ResultOps<R>::kLds ? (size_t)a.k : (size_t)SpStackCols<CCT, R>::value) * \
                      8 * nt),                                                                  \
                     s, a.nodes, a.prim_ids,                                                    \
                     a.data, a.bounds, a.queries, a.nq, a.cutoff, a.k, a.ids, a.dist2, a.ret,   \
                     a.stats)
    if (a.list_kind < 0) CUKD_SPQ(cukd::FCPResult);
    else if (a.list_kind == CUKD_LIST_HEAP) CUKD_SPQ(LdsHeapList);
    else if (D == 1 && a.k == 4) CUKD_SPQ(cukd::FixedCandidateList<D == 1 ? 4 : 1>);
    else CUKD_SPQ(DynFixedList);
#undef CUKD_SPQ
    return hipGetLastError();
  }
  if (a.list_kind < 0) launch_spatial_l<D, CCT, RegClosest>(a, s);
  else if (a.list_kind == CUKD_LIST_FIXED) {
    if (a.k <= 4) launch_spatial_l<D, CCT, RegSorted<4>>(a, s);
    else if (a.k <= 8) launch_spatial_l<D, CCT, RegSorted<8>>(a, s);
    else if (a.k <= 16) launch_spatial_l<D, CCT, RegSorted<16>>(a, s);
    else if (a.k <= 32) launch_spatial_l<D, CCT, RegSorted<32>>(a, s);
    else launch_spatial_l<D, CCT, RegSorted<64>>(a, s);
  } else {
    if (a.k <= 8) launch_spatial_l<D, CCT, RegHeap<8>>(a, s);
    else if (a.k <= 16) launch_spatial_l<D, CCT, RegHeap<16>>(a, s);
    else if (a.k <= 32) launch_spatial_l<D, CCT, RegHeap<32>>(a, s);
    else launch_spatial_l<D, CCT, RegHeap<64>>(a, s);
  }
  return hipGetLastError();
}

template <int D>
static hipError_t launch_spatial_d(int method, const SpatialArgs &a, hipStream_t s)
{
  return method == CUKD_CCT ? launch_spatial_m<D, true>(a, s) : launch_spatial_m<D, false>(a, s);
}

hipError_t launch_spatial_query(int D, int method, const SpatialArgs &a, hipStream_t s)
{
  switch (D) {
    case 1: return launch_spatial_d<1>(method, a, s);
    case 2: return launch_spatial_d<2>(method, a, s);
    case 3: return launch_spatial_d<3>(method, a, s);
    case 4: return launch_spatial_d<4>(method, a, s);
    case 5: return launch_spatial_d<5>(method, a, s);
    case 6: return launch_spatial_d<6>(method, a, s);
    case 7: return launch_spatial_d<7>(method, a, s);
    default: return launch_spatial_d<8>(method, a, s);
  }
}

}  // namespace cukd_amd
