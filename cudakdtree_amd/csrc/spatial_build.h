// spatial_build.h -- spatial k-d tree build in two phases, included by
// spatial.hip (which states the tree's rules and holds the round-by-round
// build that very deep trees fall back to).
//
// Large nodes, more than SPB_T points, are split round by round over the
// whole array, four launches a round: decide and number the children (one
// workgroup), count each tile's left points, scan the tile counts and set
// the children's ranges (one workgroup), and move the points while the
// children's boxes grow.  The round state lives on the device, so several
// rounds are launched between two looks at it.
//
// Every node of at most SPB_T points ("item") is then finished by one
// workgroup in LDS: its points are loaded once, and every level is decided,
// scanned and partitioned there.  The result is a list of records per item,
// level by level, and its nodes per level.
//
// Node ids are level by level, left to right, over the whole tree.  With the
// items in position order, a node's id is its level's first id, plus the
// nodes of that level in the items before its own, plus its place in the
// item.  A large node counts, at its level, for the item that starts where it
// starts, and its left child for the same one.  So one exclusive scan per
// level over the items numbers everything.
//
// Bound by launches, waits and allocations (0.7 of 1.45 ms at 1M) and, in the
// item kernel (0.23 ms), by barriers and LDS.  1M float4 with 1 % duplicates:
// 7.4 -> 1.45 ms, where the round-by-round build spent 4.8 ms in wave-wide box
// reductions of nodes of a few points and 2.4 ms in 200 launches and 21 waits;
// 4M: 24.2 -> 3.0 ms; 10M float3: 48.4 -> 6.9 ms; 1000 points: 0.80 -> 0.28 ms.
#pragma once

namespace cukd_amd {

enum { SPB_T = 2048, SPB_NT = 256, SPB_TILE = SPB_T, SPB_LEVELS = 64 };
// the item kernel: 256 and 512 threads within 3 %, 1024 5 .. 10 % slower
enum { SPB_SNT = 512, SPB_ITEMS = SPB_T / SPB_SNT };
enum { SPB_LEAF = -2 };  // SpRec::dim of a leaf

// device state of the rounds
struct SpRounds {
  int32_t a, b;          // open nodes
  int32_t split_a, split_b;  // nodes the last round looked at
  int32_t next;          // first unused node
  int32_t level;         // of the open nodes
  int32_t cur;           // buffer the last round read
  int32_t active;        // the last round split something (its points are in buffer cur ^ 1)
  int32_t nitems;
  int32_t deep;          // a level beyond SPB_LEVELS: nothing here is valid
  uint32_t degen;        // some split was degenerate
};

struct SpRec {
  float pos;
  int32_t dim;     // SPB_LEAF, -1 (degenerate) or the split dim
  uint32_t start;  // first position
  uint32_t count;
  uint32_t child;  // place of the left child in its level of the item
};

struct SpLevelBase {
  uint32_t v[SPB_LEVELS + 1];
};

// exclusive scan over the NT threads of a workgroup; s_w: NT / 64 + 1 words.
// The caller separates two uses of s_w by a barrier.
template <int NT>
__device__ inline uint32_t spb_scan(uint32_t v, uint32_t *s_w, uint32_t &total)
{
  const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = (uint32_t)__shfl_up((int)incl, o);
    if (lane >= o) incl += u;
  }
  if (lane == 63) s_w[w] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; i++) {
    const uint32_t x = s_w[i];
    if (i < w) before += x;
    all += x;
  }
  total = all;
  return before + incl - v;
}

// ---------------------------------------------------------------------------
// rounds over large nodes
// ---------------------------------------------------------------------------

// box copies of a large node: [copy][lo 0 .. D-1, hi 0 .. D-1]
enum { SPB_COPIES = 8 };
__device__ inline int32_t *box_copy(int32_t *boxes, uint32_t node, int copy, int D)
{
  return boxes + ((size_t)node * SPB_COPIES + (unsigned)copy % SPB_COPIES) * 2 * D;
}
__device__ inline void box_clear(int32_t *boxes, uint32_t node, int count, int D, int tid, int nt)
{
  int32_t *b = box_copy(boxes, node, 0, D);
  for (int i = tid; i < count * SPB_COPIES * 2 * D; i += nt)
    b[i] = abox_enc(i % (2 * D) < D ? 3.402823466e+38f : -3.402823466e+38f);
}

// The box of the whole array into the root's copies
__global__ __launch_bounds__(SPB_NT) void k_spb_root(int32_t *boxes, const uint8_t *pts, int n,
                                                     cukd_layout L)
{
  __shared__ int32_t s_box[2 * CUKD_MAX_DIMS];
  const int D = L.num_dims, tid = (int)threadIdx.x;
  int32_t lo[CUKD_MAX_DIMS], hi[CUKD_MAX_DIMS];
#pragma unroll
  for (int d = 0; d < CUKD_MAX_DIMS; d++) {
    lo[d] = 0x7fffffff;
    hi[d] = (int32_t)0x80000000;
  }
  if (tid < 2 * CUKD_MAX_DIMS) s_box[tid] = tid < CUKD_MAX_DIMS ? 0x7fffffff : (int32_t)0x80000000;
  for (int i = (int)blockIdx.x * SPB_NT + tid; i < n; i += (int)gridDim.x * SPB_NT) {
#pragma unroll
    for (int d = 0; d < CUKD_MAX_DIMS; d++) {
      if (d >= D) break;
      const int32_t e = abox_enc(sp_coord(pts, (uint32_t)i, L, d));
      lo[d] = min(lo[d], e);
      hi[d] = max(hi[d], e);
    }
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < CUKD_MAX_DIMS; d++) {
    if (d >= D) break;
    int32_t l = lo[d], h = hi[d];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      l = min(l, __shfl_xor(l, o));
      h = max(h, __shfl_xor(h, o));
    }
    if ((tid & 63) == 0) {
      atomicMin(&s_box[d], l);
      atomicMax(&s_box[CUKD_MAX_DIMS + d], h);
    }
  }
  __syncthreads();
  if (tid < 2 * D) {
    int32_t *b = box_copy(boxes, 0, (int)blockIdx.x, D) + tid;
    if (tid < D) atomicMin(b, s_box[tid]);
    else atomicMax(b, s_box[CUKD_MAX_DIMS + tid - D]);
  }
}

__global__ void k_spb_init(SpNode *nodes, int32_t *boxes, SpRounds *st, uint32_t *pos_prim,
                           uint32_t *pos_node, int n, int D)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0) box_clear(boxes, 0, 1, D, (int)threadIdx.x, (int)blockDim.x);
  if (i == 0) {
    SpNode &t = nodes[0];
    t.count = (uint32_t)n;
    t.start = 0;
    t.level = 0;
    t.state = SP_OPEN;
    *st = SpRounds{0, 1, 0, 0, 1, 0, 0, 0, 0, 0, 0u};
  }
  if (i < n) {
    pos_prim[i] = (uint32_t)i;
    pos_node[i] = 0u;
  }
}

// decides the open nodes and makes the children; one workgroup
enum { SPB_LNT = 1024 };
__global__ __launch_bounds__(SPB_LNT) void k_spb_level(SpNode *nodes, int32_t *boxes,
                                                       SpRounds *st, int D, uint32_t small)
{
  __shared__ uint32_t s_w[SPB_LNT / 64];
  const int a = st->a, b = st->b, next = st->next, level = st->level;
  const int cur = st->cur ^ st->active;
  __syncthreads();  // the state is read before it is rewritten
  // the boxes from their copies, one word a thread
  for (int j = (int)threadIdx.x; j < (b - a) * 2 * D; j += SPB_LNT) {
    const int i = a + j / (2 * D), w = j % (2 * D);
    const int32_t *c = box_copy(boxes, (uint32_t)i, 0, D) + w;
    int32_t v = c[0];
#pragma unroll
    for (int x = 1; x < SPB_COPIES; x++) {
      const int32_t u = c[x * 2 * D];
      v = w < D ? min(v, u) : max(v, u);
    }
    if (w < D) nodes[i].lo[w] = v;
    else nodes[i].hi[w - D] = v;
  }
  __syncthreads();
  uint32_t splits = 0, items = 0;
  for (int i0 = a; i0 < b; i0 += SPB_LNT) {
    const int i = i0 + (int)threadIdx.x;
    const bool open = i < b;
    const bool split = open && nodes[i].count > small;
    uint32_t total;
    const uint32_t e = spb_scan<SPB_LNT>(split ? 1u : 0u, s_w, total);
    if (split) {
      SpNode &t = nodes[i];
      float pos;
      const int dim = sp_choose(D, [&](int w) { return w < D ? t.lo[w] : t.hi[w - D]; }, pos);
      if (dim < 0) st->degen = 1u;  // same value from every writer
      t.dim = dim;
      t.pos = pos;
      t.state = SP_SPLIT;
      t.offset = (uint32_t)next + 2u * (splits + e);
      for (int side = 0; side < 2; side++) {
        SpNode &c = nodes[t.offset + side];
        c.state = SP_OPEN;
        c.level = level + 1;
      }
    } else if (open) {
      nodes[i].state = SP_LEAF;  // an item
    }
    splits += total;
    items += (uint32_t)min(b - i0, (int)SPB_LNT) - total;
    __syncthreads();
  }
  box_clear(boxes, (uint32_t)next, 2 * (int)splits, D, (int)threadIdx.x, SPB_LNT);
  if (threadIdx.x == 0) {
    // an item's last level is two below the table's end at most
    const bool deep = splits > 0 && level + 1 >= SPB_LEVELS - 2;
    st->cur = cur;
    st->active = splits > 0 && !deep;
    st->split_a = a;
    st->split_b = b;
    st->a = next;
    st->b = deep ? next : next + 2 * (int)splits;
    st->next = next + 2 * (int)splits;
    st->level = level + 1;
    st->nitems += (int)items;
    if (deep) st->deep = 1;
  }
}

// Left flags of a tile's points (START: of items' first positions) with
// their exclusive prefix inside the tile: loc = prefix | flag << 15
template <bool START>
__global__ __launch_bounds__(SPB_NT) void k_spb_flags(const SpNode *nodes, const SpRounds *st,
                                                      const uint32_t *pp0, const uint32_t *pp1,
                                                      const uint32_t *pn0, const uint32_t *pn1,
                                                      uint16_t *loc, uint32_t *tile_sum,
                                                      const uint8_t *pts, int n, cukd_layout L)
{
  enum { E = SPB_TILE / SPB_NT, W = SPB_NT / 64 };
  __shared__ uint32_t s_cnt[E * W];
  if (!START && !st->active) return;
  const bool alt = ((START ? st->cur ^ st->active : st->cur) & 1) != 0;
  const uint32_t *pp = alt ? pp1 : pp0, *pn = alt ? pn1 : pn0;
  const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const int p0 = (int)blockIdx.x * SPB_TILE + (int)threadIdx.x;
  uint32_t mine = 0, rank[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int p = p0 + e * SPB_NT;
    bool f = false;
    if (p < n) {
      const SpNode &t = nodes[pn[p]];
      if (START) {
        f = t.start == (uint32_t)p;
      } else if (t.state == SP_SPLIT) {
        if (t.dim < 0) f = (((uint32_t)p - t.start) & 1u) == 0;
        else f = !(sp_coord(pts, pp[p], L, t.dim) >= t.pos);
      }
    }
    const uint64_t m = __ballot(f);
    rank[e] = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    if (f) mine |= 1u << e;
    if (lane == 0) s_cnt[e * W + w] = (uint32_t)__popcll(m);
  }
  __syncthreads();
  uint32_t run = 0;
#pragma unroll
  for (int e = 0; e < E; e++) {
#pragma unroll
    for (int j = 0; j < W; j++) {
      if (j == w) {
        const int p = p0 + e * SPB_NT;
        if (p < n) loc[p] = (uint16_t)((run + rank[e]) | ((mine >> e) & 1u) << 15);
      }
      run += s_cnt[e * W + j];
    }
  }
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = run;
}

__device__ inline uint32_t spb_before(const uint32_t *tile_base, const uint16_t *loc, uint32_t p)
{
  return tile_base[p / SPB_TILE] + (loc[p] & 0x7fffu);
}

// exclusive scan of the tile sums in place (tile_base[tiles] = total), then
// the ranges of the round's children; one workgroup
template <bool START>
__global__ __launch_bounds__(SPB_LNT) void k_spb_scan(SpNode *nodes, const SpRounds *st,
                                                      uint32_t *tile_base, const uint16_t *loc,
                                                      int tiles, int n)
{
  __shared__ uint32_t s_w[SPB_LNT / 64];
  if (!START && !st->active) return;
  uint32_t run = 0;
  for (int i0 = 0; i0 < tiles; i0 += SPB_LNT) {
    const int i = i0 + (int)threadIdx.x;
    const uint32_t v = i < tiles ? tile_base[i] : 0u;
    uint32_t total;
    const uint32_t e = spb_scan<SPB_LNT>(v, s_w, total);
    if (i < tiles) tile_base[i] = run + e;
    run += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) tile_base[tiles] = run;
  if (START) return;
  __syncthreads();
  for (int i = st->split_a + (int)threadIdx.x; i < st->split_b; i += SPB_LNT) {
    SpNode &t = nodes[i];
    if (t.state != SP_SPLIT) continue;
    const uint32_t end = t.start + t.count;
    t.lex = spb_before(tile_base, loc, t.start);
    t.lcount = (end < (uint32_t)n ? spb_before(tile_base, loc, end) : run) - t.lex;
    SpNode &l = nodes[t.offset], &r = nodes[t.offset + 1];
    l.start = t.start;
    l.count = t.lcount;
    r.start = t.start + t.lcount;
    r.count = t.count - t.lcount;
  }
}

// Moves the points to their children (stable) and grows the children's
// boxes.  A wave takes 64 consecutive positions at a time, so its lanes
// nearly always share a node: they fold into registers, a left and a right
// box, until the node changes, then into the tile's table, and each tile into
// one of SPB_COPIES copies of a box: atomics on one word take 7 ns each, and
// the first round's tiles all meet in two boxes (234 us with one atomic per
// wave and word).
template <int D>
__global__ __launch_bounds__(SPB_NT) void k_spb_scatter(const SpNode *nodes, int32_t *boxes,
                                                        const SpRounds *st,
                                                        uint32_t *pp0, uint32_t *pp1,
                                                        uint32_t *pn0, uint32_t *pn1,
                                                        const uint16_t *loc,
                                                        const uint32_t *tile_base,
                                                        const uint8_t *pts, int n, cukd_layout L)
{
  if (!st->active) return;
  const bool alt = (st->cur & 1) != 0;
  const uint32_t *pp = alt ? pp1 : pp0, *pn = alt ? pn1 : pn0;
  uint32_t *npp = alt ? pp0 : pp1, *npn = alt ? pn0 : pn1;
  __shared__ uint32_t s_node[2];             // left children of the tile's split nodes
  __shared__ int32_t s_box[2 * 2 * 2 * D];   // [node][side][lo, hi][dim]
  const int lane = (int)threadIdx.x & 63;
  int32_t lo[2][D], hi[2][D];
  uint32_t held = 0xffffffffu;  // the left child whose boxes the wave folds
  for (int i = (int)threadIdx.x; i < 2 * 4 * D; i += SPB_NT)
    s_box[i] = (i / D) & 1 ? (int32_t)0x80000000 : 0x7fffffff;
  if (threadIdx.x < 2) s_node[threadIdx.x] = 0xffffffffu;
  __syncthreads();
  auto flush = [&]() {
    if (held == 0xffffffffu) return;
    // the tile's table: split nodes have more points than a tile, so it
    // meets at most two, neighbours in their level, whose left children's
    // ids differ by 2
    const uint32_t row = (held >> 1) & 1u;
    if (lane == 0) s_node[row] = held;  // the same from every wave
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        int32_t l = lo[s][d], h = hi[s][d];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          l = min(l, __shfl_xor(l, o));
          h = max(h, __shfl_xor(h, o));
        }
        if (lane == 0) {
          int32_t *b = s_box + (row * 2 + s) * 2 * D;
          atomicMin(&b[d], l);
          atomicMax(&b[D + d], h);
        }
      }
    }
  };
  for (int e = 0; e < SPB_TILE / SPB_NT; e++) {
    const int p = (int)blockIdx.x * SPB_TILE + e * SPB_NT + (int)threadIdx.x;
    uint32_t child = 0xffffffffu;  // left child of the point's node
    bool left = false;
    int32_t c[D];
#pragma unroll
    for (int d = 0; d < D; d++) c[d] = 0;
    if (p < n) {
      const uint32_t node = pn[p], prim = pp[p];
      const SpNode &t = nodes[node];
      if (t.state != SP_SPLIT) {
        npp[p] = prim;
        npn[p] = node;
      } else {
        left = (loc[p] >> 15) != 0;
        const uint32_t lrank = spb_before(tile_base, loc, (uint32_t)p) - t.lex;
        const uint32_t np = left ? t.start + lrank : (uint32_t)p - lrank + t.lcount;
        child = t.offset;
        npp[np] = prim;
        npn[np] = child + (left ? 0u : 1u);
#pragma unroll
        for (int d = 0; d < D; d++) c[d] = abox_enc(sp_coord(pts, prim, L, d));
      }
    }
    uint64_t todo = __ballot(child != 0xffffffffu);
    while (todo) {
      const int leader = __ffsll((unsigned long long)todo) - 1;
      const uint32_t ch = (uint32_t)__shfl((int)child, leader);
      const bool peer = child == ch;
      todo &= ~__ballot(peer);
      if (ch != held) {
        flush();
        held = ch;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int d = 0; d < D; d++) {
            lo[s][d] = 0x7fffffff;
            hi[s][d] = (int32_t)0x80000000;
          }
      }
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const bool take = peer && left == (s == 0);
#pragma unroll
        for (int d = 0; d < D; d++) {
          lo[s][d] = take && c[d] < lo[s][d] ? c[d] : lo[s][d];
          hi[s][d] = take && c[d] > hi[s][d] ? c[d] : hi[s][d];
        }
      }
    }
  }
  flush();
  __syncthreads();
  for (int i = (int)threadIdx.x; i < 2 * 4 * D; i += SPB_NT) {
    const uint32_t left_child = s_node[i / (4 * D)];
    const int side = (i / (2 * D)) & 1, w = i % (2 * D);
    if (left_child == 0xffffffffu) continue;
    int32_t *b = box_copy(boxes, left_child + side, (int)blockIdx.x, D) + w;
    if (w < D) {
      if (s_box[i] != 0x7fffffff) atomicMin(b, s_box[i]);
    } else {
      if (s_box[i] != (int32_t)0x80000000) atomicMax(b, s_box[i]);
    }
  }
}

// items in position order, and the rank of the item starting at a position
__global__ void k_spb_items(const SpRounds *st, const uint32_t *pn0, const uint32_t *pn1,
                            const uint16_t *loc, const uint32_t *tile_base, uint32_t *items,
                            uint32_t *rank_at, int n)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !(loc[p] >> 15)) return;
  const uint32_t r = spb_before(tile_base, loc, (uint32_t)p);
  items[r] = (((st->cur ^ st->active) & 1) ? pn1 : pn0)[p];
  rank_at[p] = r;
}

// ---------------------------------------------------------------------------
// items: one workgroup each
// ---------------------------------------------------------------------------

// open-node slots an item needs at once, and the kernel's dynamic LDS
__host__ __device__ inline int spb_slots(uint32_t thr) { return SPB_T / (int)(thr + 1 < SPB_T ? thr + 1 : SPB_T) + 1; }
inline size_t spb_lds(int D, uint32_t thr)
{
  const size_t S = (size_t)spb_slots(thr);
  return (size_t)SPB_T * 4 * D            // coordinates
         + S * 4 * 2 * D                  // boxes
         + S * 4 * 2                      // split dim, pos
         + 2 * ((S * 3 + 1) & ~(size_t)1) * 2  // start, count, place: this level and the next
         + S * 2 * 4                      // lcount, children's slots (padded)
         + SPB_T * 2 * 2 + (SPB_T + 2) * 2;    // order, slot of a position, left prefix
}

template <int D>
__global__ __launch_bounds__(SPB_SNT) void k_spb_small(const SpNode *nodes, SpRounds *st,
                                                      const uint32_t *items, uint32_t *pp0,
                                                      uint32_t *pp1, const uint8_t *pts,
                                                      cukd_layout L, uint32_t thr, SpRec *recs,
                                                      uint32_t *pos_rec, uint32_t *M, int nitems)
{
  enum : uint16_t { NONE = 0xffff };
  HIP_DYNAMIC_SHARED(uint32_t, s_mem);
  __shared__ uint32_t s_w[SPB_SNT / 64], s_levels[SPB_LEVELS];
  const int r = (int)blockIdx.x, tid = (int)threadIdx.x;
  const SpNode &t = nodes[items[r]];
  const int m = (int)t.count, level0 = t.level;
  const uint32_t g0 = t.start, base = 2 * g0;  // at most 2 m - 1 records
  const bool alt = ((st->cur ^ st->active) & 1) != 0;
  const uint32_t *prim = (alt ? pp1 : pp0) + g0;
  uint32_t *out = (alt ? pp0 : pp1) + g0;
  if (tid < SPB_LEVELS) s_levels[tid] = tid == level0 ? 1u : 0u;
  if ((uint32_t)m <= thr) {  // a leaf, of any size
    if (tid == 0) recs[base] = SpRec{0.f, SPB_LEAF, g0, (uint32_t)m, 0u};
    for (int p = tid; p < m; p += SPB_SNT) {
      pos_rec[g0 + p] = base;
      out[p] = prim[p];
    }
  } else {
    const int S = spb_slots(thr);
    float *crd = (float *)s_mem;                       // [D][SPB_T] by slot of the point
    int32_t *box = (int32_t *)(crd + D * SPB_T);       // [2 D][S]
    int32_t *ndim = box + 2 * D * S;
    float *npos = (float *)(ndim + S);
    uint16_t *cur = (uint16_t *)(npos + S);            // start, count, place: [3][S]
    uint16_t *nxt = cur + ((S * 3 + 1) & ~1);
    uint16_t *lcnt = nxt + ((S * 3 + 1) & ~1);
    uint16_t *slot = lcnt + S;                         // the children's slots: [2][S]
    uint16_t *ord = lcnt + S * 4;
    uint16_t *own = ord + SPB_T;                       // slot of the position's open node
    uint16_t *lex = own + SPB_T;
    for (int i = tid; i < m; i += SPB_SNT) {
      const uint32_t id = prim[i];
#pragma unroll
      for (int d = 0; d < D; d++) crd[d * SPB_T + i] = sp_coord(pts, id, L, d);
      ord[i] = (uint16_t)i;
      own[i] = 0;
    }
    if (tid < D) {
      box[tid * S] = t.lo[tid];
      box[(D + tid) * S] = t.hi[tid];
    }
    if (tid == 0) {
      cur[0] = 0;
      cur[S] = (uint16_t)m;
      cur[2 * S] = 0;
    }
    int k = 1, level = level0;
    uint32_t lstart = base, lnext = base + 1;  // records of this level and the next
    __syncthreads();
    for (;;) {
      // split every open node
      for (int i = tid; i < k; i += SPB_SNT) {
        float pos;
        const int dim = sp_choose(D, [&](int w) { return box[w * S + i]; }, pos);
        if (dim < 0) st->degen = 1u;
        ndim[i] = dim;
        npos[i] = pos;
        recs[lstart + cur[2 * S + i]] =
            SpRec{pos, dim, g0 + cur[i], (uint32_t)cur[S + i], 2u * (uint32_t)i};
      }
      __syncthreads();
      // left points before every position
      const int p0 = tid * SPB_ITEMS;
      uint32_t bits = 0, total;
#pragma unroll
      for (int e = 0; e < SPB_ITEMS; e++) {
        const int p = p0 + e;
        if (p >= m || own[p] == NONE) continue;
        const int i = own[p], dim = ndim[i];
        const bool left = dim < 0 ? ((p - cur[i]) & 1) == 0
                                  : !(crd[dim * SPB_T + ord[p]] >= npos[i]);
        if (left) bits |= 1u << e;
      }
      uint32_t run = spb_scan<SPB_SNT>((uint32_t)__popc(bits), s_w, total);
#pragma unroll
      for (int e = 0; e < SPB_ITEMS; e++) {
        if (p0 + e < m) lex[p0 + e] = (uint16_t)run;
        run += (bits >> e) & 1u;
      }
      if (tid == 0) lex[m] = (uint16_t)total;
      __syncthreads();
      // the children: leaves are recorded, the others take slots in order
      uint32_t open = 0;
      for (int i0 = 0; i0 < k; i0 += SPB_SNT) {
        const int i = i0 + tid;
        uint32_t l = 0, c = 0, start = 0;
        if (i < k) {
          start = cur[i];
          c = cur[S + i];
          l = (uint32_t)lex[start + c] - lex[start];
          lcnt[i] = (uint16_t)l;
        }
        const uint32_t f0 = l > thr ? 1u : 0u, f1 = c - l > thr ? 1u : 0u;
        uint32_t got;
        const uint32_t at = open + spb_scan<SPB_SNT>(f0 + f1, s_w, got);
        if (i < k) {
#pragma unroll
          for (uint32_t side = 0; side < 2; side++) {
            const uint32_t cs = side ? start + l : start, cc = side ? c - l : l;
            const uint32_t place = 2u * (uint32_t)i + side;
            if (side ? f1 : f0) {
              const uint32_t sl = side ? at + f0 : at;
              slot[side * S + i] = (uint16_t)sl;
              nxt[sl] = (uint16_t)cs;
              nxt[S + sl] = (uint16_t)cc;
              nxt[2 * S + sl] = (uint16_t)place;
#pragma unroll
              for (int d = 0; d < D; d++) {
                box[d * S + sl] = abox_enc(3.402823466e+38f);
                box[(D + d) * S + sl] = abox_enc(-3.402823466e+38f);
              }
            } else {
              slot[side * S + i] = NONE;
              recs[lnext + place] = SpRec{0.f, SPB_LEAF, g0 + cs, cc, 0u};
            }
          }
        }
        open += got;
        __syncthreads();
      }
      // move the points (in registers over the barrier) and grow the boxes
      uint16_t to[SPB_ITEMS], pt[SPB_ITEMS], sl[SPB_ITEMS];
      uint32_t moved = 0;
#pragma unroll
      for (int e = 0; e < SPB_ITEMS; e++) {
        const int p = p0 + e;
        to[e] = pt[e] = sl[e] = 0;
        if (p >= m || own[p] == NONE) continue;
        moved |= 1u << e;
        const int i = own[p], start = cur[i];
        const int lrank = (int)lex[p] - (int)lex[start];
        const bool left = ((bits >> e) & 1u) != 0;
        to[e] = (uint16_t)(left ? start + lrank : p - lrank + lcnt[i]);
        pt[e] = ord[p];
        sl[e] = slot[(left ? 0 : S) + i];
        if (sl[e] == NONE) pos_rec[g0 + to[e]] = lnext + 2u * (uint32_t)i + (left ? 0u : 1u);
      }
      __syncthreads();
#pragma unroll
      for (int e = 0; e < SPB_ITEMS; e++) {
        if (!((moved >> e) & 1u)) continue;
        ord[to[e]] = pt[e];
        own[to[e]] = sl[e];
        if (sl[e] == NONE) continue;
#pragma unroll
        for (int d = 0; d < D; d++) {
          const int32_t v = abox_enc(crd[d * SPB_T + pt[e]]);
          atomicMin(&box[d * S + sl[e]], v);
          atomicMax(&box[(D + d) * S + sl[e]], v);
        }
      }
      level++;
      lstart = lnext;
      lnext += 2u * (uint32_t)k;
      if (tid == 0) s_levels[level] = 2u * (uint32_t)k;
      k = (int)open;
      uint16_t *x = cur;
      cur = nxt;
      nxt = x;
      __syncthreads();
      if (k == 0) break;
      if (level >= SPB_LEVELS - 1) {
        if (tid == 0) st->deep = 1;
        break;
      }
    }
    for (int p = tid; p < m; p += SPB_SNT) out[p] = prim[ord[p]];
  }
  __syncthreads();
  if (tid < SPB_LEVELS) M[(size_t)tid * nitems + r] = s_levels[tid];
}

// ---------------------------------------------------------------------------
// numbering and output
// ---------------------------------------------------------------------------

// a large node counts for the item that starts where it starts
__global__ void k_spb_large(const SpNode *nodes, const SpRounds *st, const uint32_t *rank_at,
                            uint32_t *M, int nitems)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st->next || nodes[i].state != SP_SPLIT) return;
  M[(size_t)nodes[i].level * nitems + rank_at[nodes[i].start]] = 1u;
}

// exclusive scan of one level's counts over the items, one workgroup a level
__global__ __launch_bounds__(SPB_LNT) void k_spb_number(uint32_t *M, uint32_t *level_total,
                                                        int nitems)
{
  __shared__ uint32_t s_w[SPB_LNT / 64];
  uint32_t *row = M + (size_t)blockIdx.x * nitems;
  uint32_t run = 0;
  for (int i0 = 0; i0 < nitems; i0 += SPB_LNT) {
    const int i = i0 + (int)threadIdx.x;
    const uint32_t v = i < nitems ? row[i] : 0u;
    uint32_t total;
    const uint32_t e = spb_scan<SPB_LNT>(v, s_w, total);
    if (i < nitems) row[i] = run + e;
    run += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) level_total[blockIdx.x] = run;
}

// Ids of every record, and the points of every leaf by node id (WRITE: the
// nodes themselves, once the leaves' offsets are known).  Workgroup r < nitems
// takes item r, the others large nodes.
template <bool WRITE>
__global__ __launch_bounds__(SPB_NT) void k_spb_ids(const SpNode *nodes, const SpRounds *st,
                                                    const uint32_t *items,
                                                    const uint32_t *rank_at, const SpRec *recs,
                                                    const uint32_t *M, SpLevelBase lb, int nitems,
                                                    uint32_t *rec_id, uint32_t *leaf_cnt,
                                                    const uint32_t *leaf_off,
                                                    cukd_spatial_node *out, bool isf)
{
  const int tid = (int)threadIdx.x;
  auto inner = [&](uint32_t id, uint32_t child, int dim, float pos) {
    if (WRITE) {
      cukd_spatial_node o;
      o.offset = child;
      o.count = 0;
      o.dim = (int16_t)(dim < 0 ? 0 : dim);  // dim -1 is stored as 0 (spatial-kdtree.h:477-494)
      o.ipos = (int32_t)sp_store(pos, isf);
      out[id] = o;
    } else {
      leaf_cnt[id] = 0u;
    }
  };
  auto leaf = [&](uint32_t id, uint32_t off, uint32_t count) {
    if (WRITE) {
      cukd_spatial_node o;
      o.offset = off;
      o.count = (uint16_t)count;
      o.dim = 0;
      o.pos = 0.f;
      out[id] = o;
    } else {
      leaf_cnt[id] = count;
    }
  };
  if ((int)blockIdx.x < nitems) {
    const int r = (int)blockIdx.x;
    const SpNode &t = nodes[items[r]];
    uint32_t first = 2 * t.start;
    for (int l = t.level; l < SPB_LEVELS; l++) {
      const uint32_t *row = M + (size_t)l * nitems;
      const uint32_t before = row[r];
      const uint32_t after = r + 1 < nitems ? row[r + 1] : lb.v[l + 1] - lb.v[l] - (l == 0);
      const uint32_t cnt = after - before;
      if (cnt == 0) break;
      const uint32_t id0 = lb.v[l] + before;
      const uint32_t child0 = l + 1 < SPB_LEVELS ? lb.v[l + 1] + row[nitems + r] : 0u;
      for (uint32_t j = (uint32_t)tid; j < cnt; j += SPB_NT) {
        const SpRec e = recs[first + j];
        const uint32_t id = id0 + j;
        if (!WRITE) rec_id[first + j] = id;
        if (e.dim == SPB_LEAF) leaf(id, WRITE ? leaf_off[id] : 0u, e.count);
        else inner(id, child0 + e.child, e.dim, e.pos);
      }
      first += cnt;
    }
    return;
  }
  const int i = ((int)blockIdx.x - nitems) * SPB_NT + tid;
  if (i == 0) leaf(1u, 0u, 0u);  // node 1 is the reference's reserved empty leaf
  if (i >= st->next || nodes[i].state != SP_SPLIT) return;
  const SpNode &t = nodes[i];
  const uint32_t r = rank_at[t.start];
  inner(lb.v[t.level] + M[(size_t)t.level * nitems + r],
        lb.v[t.level + 1] + M[(size_t)(t.level + 1) * nitems + r], t.dim, t.pos);
}

__global__ void k_spb_prims(const SpRounds *st, const SpRec *recs, const uint32_t *pos_rec,
                            const uint32_t *rec_id, const uint32_t *leaf_off, const uint32_t *pp0,
                            const uint32_t *pp1, uint32_t *prim_ids, int n)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t e = pos_rec[p];
  // the items left their points in the buffer they did not read
  prim_ids[leaf_off[rec_id[e]] + ((uint32_t)p - recs[e].start)] =
      (((st->cur ^ st->active) & 1) ? pp0 : pp1)[p];
}

// Builds the tree; *deep (and no tree) when a level would pass SPB_LEVELS, or
// when an item's slots do not fit LDS (8 dims and leaves of one point).
template <int D>
static int spatial_build_items(cukd_spatial_tree *tree, const uint8_t *pts, int n,
                               const cukd_layout &L, uint32_t thr, hipStream_t s,
                               const MemResource &mem, bool *deep)
{
  if (spb_lds(D, thr) > (size_t)LDS_PER_CU - 1024) {
    *deep = true;
    return CUKD_OK;
  }
  const size_t nn = (size_t)n;
  const int tiles = (n + SPB_TILE - 1) / SPB_TILE;
  // splits have more than SPB_T points, so a level has at most n / SPB_T
  const size_t cap = nn / 16 + 256;
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o = (o + bytes + 255) & ~(size_t)255; return at; };
  const size_t o_box = take(cap * SPB_COPIES * 2 * D * 4);
  const size_t o_nodes = take(cap * sizeof(SpNode)), o_items = take(cap * 4), o_st = take(1024);
  const size_t o_pp0 = take(nn * 4), o_pp1 = take(nn * 4), o_pn0 = take(nn * 4), o_pn1 = take(nn * 4);
  const size_t o_loc = take(nn * 2), o_tile = take(((size_t)tiles + 1) * 4);
  const size_t o_rank = take(nn * 4), o_recs = take(2 * nn * sizeof(SpRec));
  const size_t o_prec = take(nn * 4), o_id = take(2 * nn * 4);
  const size_t max_nodes = 2 * nn + 2;
  const size_t o_cnt = take(max_nodes * 4), o_off = take(max_nodes * 4);
  const size_t o_scan = take(scan_scratch_words((long long)max_nodes) * 4);
  uint8_t *tmp = nullptr;
  if (mem.alloc((void **)&tmp, o, s) != 0) return CUKD_ERR_ALLOC;
  SpNode *nodes = (SpNode *)(tmp + o_nodes);
  int32_t *boxes = (int32_t *)(tmp + o_box);
  uint32_t *items = (uint32_t *)(tmp + o_items);
  SpRounds *st = (SpRounds *)(tmp + o_st);
  uint32_t *out_words = (uint32_t *)(tmp + o_st + 256);  // level totals, then the bounds
  uint32_t *pp0 = (uint32_t *)(tmp + o_pp0), *pp1 = (uint32_t *)(tmp + o_pp1);
  uint32_t *pn0 = (uint32_t *)(tmp + o_pn0), *pn1 = (uint32_t *)(tmp + o_pn1);
  uint16_t *loc = (uint16_t *)(tmp + o_loc);
  uint32_t *tile = (uint32_t *)(tmp + o_tile), *rank_at = (uint32_t *)(tmp + o_rank);
  SpRec *recs = (SpRec *)(tmp + o_recs);
  uint32_t *pos_rec = (uint32_t *)(tmp + o_prec), *rec_id = (uint32_t *)(tmp + o_id);
  uint32_t *leaf_cnt = (uint32_t *)(tmp + o_cnt), *leaf_off = (uint32_t *)(tmp + o_off);
  uint32_t *scratch = (uint32_t *)(tmp + o_scan);
  const uint32_t small = thr > (uint32_t)SPB_T ? thr : (uint32_t)SPB_T;
  const bool isf = L.scalar_type == CUKD_SCALAR_F32;
  const int gn = (n + 255) / 256;
  hipError_t e = hipSuccess;
  if (spb_lds(D, thr) > 65536)  // more than a kernel may take unasked
    e = hipFuncSetAttribute((const void *)k_spb_small<D>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)spb_lds(D, thr));

  CUKD_LAUNCH(e, k_spb_init, dim3(gn), dim3(256), 0, s, nodes, boxes, st, pp0, pn0,
              n, D);
  CUKD_LAUNCH(e, k_spb_root, dim3(gn < 512 ? gn : 512), dim3(SPB_NT), 0, s, boxes, pts, n, L);
  // Halving n points down to SPB_T takes log2(n / SPB_T) rounds where the
  // points are even, and one more to see that nothing is open; more are
  // launched, two at a time, while nodes remain.
  int rounds = 1;
  while (((long long)SPB_T << (rounds - 1)) < (long long)n && rounds < SPB_LEVELS) rounds++;
  SpRounds h;
  for (;;) {
    for (int i = 0; i < rounds; i++) {
      CUKD_LAUNCH(e, k_spb_level, dim3(1), dim3(SPB_LNT), 0, s, nodes, boxes, st, D,
                  small);
      if ((uint32_t)n <= small) break;
      CUKD_LAUNCH(e, k_spb_flags<false>, dim3(tiles), dim3(SPB_NT), 0, s, (const SpNode *)nodes,
                  (const SpRounds *)st, (const uint32_t *)pp0, (const uint32_t *)pp1,
                  (const uint32_t *)pn0, (const uint32_t *)pn1, loc, tile, pts, n, L);
      CUKD_LAUNCH(e, k_spb_scan<false>, dim3(1), dim3(SPB_LNT), 0, s, nodes,
                  (const SpRounds *)st, tile, (const uint16_t *)loc, tiles, n);
      CUKD_LAUNCH(e, k_spb_scatter<D>, dim3(tiles), dim3(SPB_NT), 0, s,
                  (const SpNode *)nodes, boxes, (const SpRounds *)st, pp0, pp1, pn0, pn1,
                  (const uint16_t *)loc, (const uint32_t *)tile, pts, n, L);
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&h, st, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess || h.deep || h.a >= h.b) break;
    rounds = 2;
  }
  uint32_t *M = nullptr;
  cukd_spatial_node *out_nodes = nullptr;
  uint32_t *out_prims = nullptr;
  int rc = CUKD_OK, num_nodes = 0;
  uint32_t hw[SPB_LEVELS + 2 * CUKD_MAX_DIMS];
  SpLevelBase lb;
  *deep = e == hipSuccess && h.deep;
  if (e == hipSuccess && !*deep) {
    const int ni = h.nitems, gl = (h.next + SPB_NT - 1) / SPB_NT;
    if (mem.alloc((void **)&M, (size_t)SPB_LEVELS * ni * 4, s) != 0) rc = CUKD_ERR_ALLOC;
    if (rc == CUKD_OK) {
      CUKD_LAUNCH(e, k_spb_flags<true>, dim3(tiles), dim3(SPB_NT), 0, s, (const SpNode *)nodes,
                  (const SpRounds *)st, (const uint32_t *)pp0, (const uint32_t *)pp1,
                  (const uint32_t *)pn0, (const uint32_t *)pn1, loc, tile, pts, n, L);
      CUKD_LAUNCH(e, k_spb_scan<true>, dim3(1), dim3(SPB_LNT), 0, s, nodes,
                  (const SpRounds *)st, tile, (const uint16_t *)loc, tiles, n);
      CUKD_LAUNCH(e, k_spb_items, dim3(gn), dim3(256), 0, s, (const SpRounds *)st,
                  (const uint32_t *)pn0, (const uint32_t *)pn1, (const uint16_t *)loc,
                  (const uint32_t *)tile, items, rank_at, n);
      CUKD_LAUNCH(e, k_spb_small<D>, dim3(ni), dim3(SPB_SNT), spb_lds(D, thr), s,
                  (const SpNode *)nodes, st, (const uint32_t *)items, pp0, pp1, pts, L, thr,
                  recs, pos_rec, M, ni);
      CUKD_LAUNCH(e, k_spb_large, dim3(gl), dim3(SPB_NT), 0, s, (const SpNode *)nodes,
                  (const SpRounds *)st, (const uint32_t *)rank_at, M, ni);
      CUKD_LAUNCH(e, k_sp_bounds_out, dim3(1), dim3(64), 0, s, (const SpNode *)nodes,
                  out_words + SPB_LEVELS, D, isf);
      CUKD_LAUNCH(e, k_spb_number, dim3(SPB_LEVELS), dim3(SPB_LNT), 0, s, M, out_words, ni);
      if (e == hipSuccess)
        e = hipMemcpyAsync(hw, out_words, 4 * (SPB_LEVELS + 2 * D), hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipMemcpyAsync(&h, st, sizeof(h), hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      *deep = e == hipSuccess && h.deep;
      if (e == hipSuccess && !*deep) {
        // node 1 is reserved, so level 1 starts at 2
        uint32_t run = 0;
        for (int l = 0; l < SPB_LEVELS; l++) {
          lb.v[l] = run;
          run += hw[l] + (l == 0 ? 1u : 0u);
        }
        lb.v[SPB_LEVELS] = run;
        num_nodes = (int)run;
        if (mem.alloc((void **)&out_nodes, (size_t)num_nodes * sizeof(cukd_spatial_node), s) != 0 ||
            mem.alloc((void **)&out_prims, nn * 4, s) != 0)
          rc = CUKD_ERR_ALLOC;
      }
    }
    if (rc == CUKD_OK && e == hipSuccess && !*deep) {
      CUKD_LAUNCH(e, k_spb_ids<false>, dim3(ni + gl), dim3(SPB_NT), 0, s, (const SpNode *)nodes,
                  (const SpRounds *)st, (const uint32_t *)items, (const uint32_t *)rank_at,
                  (const SpRec *)recs, (const uint32_t *)M, lb, ni, rec_id, leaf_cnt,
                  (const uint32_t *)leaf_off, out_nodes, isf);
      scan_exclusive(e, leaf_cnt, leaf_off, num_nodes, scratch, s);
      CUKD_LAUNCH(e, k_spb_ids<true>, dim3(ni + gl), dim3(SPB_NT), 0, s, (const SpNode *)nodes,
                  (const SpRounds *)st, (const uint32_t *)items, (const uint32_t *)rank_at,
                  (const SpRec *)recs, (const uint32_t *)M, lb, ni, rec_id, leaf_cnt,
                  (const uint32_t *)leaf_off, out_nodes, isf);
      CUKD_LAUNCH(e, k_spb_prims, dim3(gn), dim3(256), 0, s, (const SpRounds *)st,
                  (const SpRec *)recs, (const uint32_t *)pos_rec, (const uint32_t *)rec_id,
                  (const uint32_t *)leaf_off, (const uint32_t *)pp0, (const uint32_t *)pp1,
                  out_prims, n);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
    }
  }
  mem.release(M, s);
  mem.release(tmp, s);
  if (e != hipSuccess || rc != CUKD_OK) {
    mem.release(out_nodes, s);
    mem.release(out_prims, s);
    if (e != hipSuccess) {
      set_last_error("spatial build failed: %s", hipGetErrorString(e));
      return CUKD_ERR_HIP;
    }
    return rc;
  }
  if (*deep) return CUKD_OK;
  for (int i = 0; i < 2 * CUKD_MAX_DIMS; i++)
    tree->ibounds[i] = i < 2 * D ? (int32_t)hw[SPB_LEVELS + i] : 0;
  int levels = 0;
  while (levels < SPB_LEVELS && hw[levels]) levels++;
  spatial_record(tree, D, levels <= SP_DEPTH && h.degen == 0u, mem);
  tree->nodes = out_nodes;
  tree->prim_ids = out_prims;
  tree->data = pts;
  tree->num_prims = n;
  tree->num_nodes = num_nodes;
  return CUKD_OK;
}

}  // namespace cukd_amd
