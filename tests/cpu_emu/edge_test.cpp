// CPU kernel-emulator tests of edge cases of the C ABI (test infrastructure;
// see emu_test.cpp): inputs, launches and runtime states that a GPU test
// cannot or must not bring about.
//
//   edge_test [case-name-substring]
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "cukd_amd.h"
#include "../../oracle/cukd_oracle.h"

// query kernels are compiled for dims 2, 3 and 4 only
namespace cukd_amd {
struct QueryArgs;
#define CUKD_EMU_NO_DIM(d)                                                          \
  hipError_t launch_query_##d(int, const QueryArgs &, hipStream_t) { return hipErrorInvalidValue; }
CUKD_EMU_NO_DIM(1)
CUKD_EMU_NO_DIM(5)
CUKD_EMU_NO_DIM(6)
CUKD_EMU_NO_DIM(7)
CUKD_EMU_NO_DIM(8)
}  // namespace cukd_amd

namespace {

uint64_t sm(uint64_t &x)
{
  uint64_t z = (x += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
float unit(uint64_t &x) { return (float)(sm(x) >> 40) * (1.f / 16777216.f); }

// device memory of a vector's size and contents
template <class T> struct Dev {
  T *p = nullptr;
  size_t n;
  explicit Dev(size_t n_) : n(n_) { hipMalloc((void **)&p, n * sizeof(T) + 4); }
  explicit Dev(const std::vector<T> &v) : Dev(v.size()) { if (n) memcpy(p, v.data(), n * sizeof(T)); }
  ~Dev() { hipFree(p); }
  bool same(const std::vector<T> &v) const { return !n || !memcmp(p, v.data(), n * sizeof(T)); }
};

oc_layout ocl(const cukd_layout &L)
{
  return oc_layout{L.num_dims, L.scalar_type, L.stride, L.point_offset, L.dim_offset, L.dim_bytes};
}
cukd_layout floats(int D) { return cukd_layout{D, CUKD_SCALAR_F32, 4 * D, 0, -1, 4}; }

struct SpatialRef {
  std::vector<oc_spatial_node> nodes;
  std::vector<uint32_t> prims;
  std::vector<float> box;
  SpatialRef(const std::vector<float> &pts, const cukd_layout &L, int leaf)
  {
    const int n = (int)pts.size() / L.num_dims;
    const oc_layout O = ocl(L);
    nodes.resize(oc_spatial_build(pts.data(), n, &O, leaf, nullptr, nullptr, nullptr));
    prims.resize(n);
    box.resize(2 * L.num_dims);
    oc_spatial_build(pts.data(), n, &O, leaf, nodes.data(), prims.data(), box.data());
  }
  bool same(const cukd_spatial_tree &t) const
  {
    return (size_t)t.num_nodes == nodes.size() &&
           !memcmp(t.nodes, nodes.data(), nodes.size() * sizeof(nodes[0])) &&
           !memcmp(t.prim_ids, prims.data(), prims.size() * 4) &&
           !memcmp(t.bounds, box.data(), box.size() * 4);
  }
};

// Extents whose centre does not lie strictly between their ends as a float:
// ends whose sum overflows, and infinite ones.
bool spatial_centre_case(const char *kind, int n, int D, int leaf)
{
  uint64_t seed = 7 + n;
  std::vector<float> pts((size_t)n * D);
  for (int i = 0; i < n; i++)
    for (int d = 0; d < D; d++) {
      float v = unit(seed);
      const uint32_t r = (uint32_t)(sm(seed) % 5);
      if (!strcmp(kind, "sum overflows")) v = d == 0 ? 1.8e38f + 1.6e38f * v : v;
      if (!strcmp(kind, "negative sum overflows")) v = -1.8e38f - 1.6e38f * v;
      if (!strcmp(kind, "opposite infinities")) v = r == 0 ? -INFINITY : r == 1 ? INFINITY : v;
      if (!strcmp(kind, "infinity in one dim")) v = d == D - 1 && r < 3 ? INFINITY : v;
      if (!strcmp(kind, "minus infinity")) v = r < 2 ? -INFINITY : v;
      if (!strcmp(kind, "all infinite")) v = r < 2 ? -INFINITY : INFINITY;
      pts[(size_t)i * D + d] = v;
    }
  const cukd_layout L = floats(D);
  const oc_layout O = ocl(L);
  const SpatialRef ref(pts, L, leaf);
  Dev<float> dp(pts);
  cukd_spatial_tree t;
  if (cukd_spatial_build(&t, dp.p, n, &L, leaf, nullptr, nullptr) != CUKD_OK) return false;
  bool ok = ref.same(t);
  // queries beside the points, at infinity and in the ordinary range
  std::vector<float> q(pts.begin(), pts.begin() + (size_t)(n < 60 ? n : 60) * D);
  for (int i = 0; i < 20 * D; i++) q.push_back(unit(seed));
  const int nq = (int)q.size() / D, k = 5;
  Dev<float> dq(q), dd((size_t)nq * k);
  Dev<int32_t> di((size_t)nq * k);
  std::vector<int32_t> ri((size_t)nq * k);
  std::vector<float> rd((size_t)nq * k);
  for (int m : {CUKD_STACK_BASED, CUKD_CCT}) {
    oc_spatial_knn(m, OC_LIST_FIXED, k, ref.nodes.data(), ref.prims.data(), ref.box.data(),
                   pts.data(), &O, q.data(), nq, INFINITY, ri.data(), rd.data(), nullptr, 1);
    ok = ok && cukd_spatial_knn(m, CUKD_LIST_FIXED, k, &t, &L, dq.p, nq, INFINITY, di.p, dd.p,
                                nullptr, nullptr) == CUKD_OK &&
         di.same(ri) && dd.same(rd);
  }
  cukd_spatial_free(&t, nullptr, nullptr);
  return ok;
}

// A kNN query that overflows the reference's traversal stack, without an
// array for the radii: every row is the oracle's, its own and the others'.
// plain: through the kernel that trees of 2^29 nodes and more take.
bool spatial_overflow_case(bool plain, int method, int list)
{
  const int n = 120, nq = 70, k = 4;
  const cukd_layout L = floats(3);
  const oc_layout O = ocl(L);
  std::vector<float> pts(3 * n, 0.f), q;
  for (int i = 0; i < n; i++) pts[3 * i] = std::ldexp(1.f, -i);
  uint64_t seed = 5;
  for (int i = 0; i < 3 * nq; i++) q.push_back(unit(seed));
  for (int i = 40; i < nq; i += 9) q[3 * i] = q[3 * i + 1] = q[3 * i + 2] = 0.f;
  const SpatialRef ref(pts, L, 1);
  Dev<float> dp(pts), dq(q), dd((size_t)nq * k);
  Dev<int32_t> di((size_t)nq * k);
  cukd_spatial_tree t;
  if (cukd_spatial_build(&t, dp.p, n, &L, 1, nullptr, nullptr) != CUKD_OK) return false;
  const int nodes = t.num_nodes;
  if (plain) t.num_nodes = (1 << 29) + 1;  // read for the choice of the kernel only
  std::vector<int32_t> ri((size_t)nq * k);
  std::vector<float> rd((size_t)nq * k), rr(nq);
  oc_spatial_knn(method, list, k, ref.nodes.data(), ref.prims.data(), ref.box.data(), pts.data(),
                 &O, q.data(), nq, INFINITY, ri.data(), rd.data(), rr.data(), 1);
  bool ok = rr[49] == -1.f && rr[0] != -1.f;  // some overflow, some do not
  ok = ok && cukd_spatial_knn(method, list, k, &t, &L, dq.p, nq, INFINITY, di.p, dd.p, nullptr,
                              nullptr) == CUKD_OK &&
       di.same(ri) && dd.same(rd);
  t.num_nodes = nodes;
  cukd_spatial_free(&t, nullptr, nullptr);
  return ok;
}

// launches since 'from' that name the kernel
int launches_of(const char *kernel, size_t from)
{
  int c = 0;
  for (size_t i = from; i < emu_launches.size(); i++)
    c += emu_launches[i].find(kernel) != std::string::npos;
  return c;
}

// An autotuned call that may not prune by box leaves nothing behind that keeps
// a later one of the same sizes from it, and a call with
// CUKD_QUERY_ONE_PER_LANE never prunes, whatever is cached.
bool autotune_case(const char *first, int k)
{
  const int n = 700, nq = 90;
  const bool expl = !strcmp(first, "explicit dims");
  const cukd_layout L = floats(3), X{3, CUKD_SCALAR_F32, 20, 0, 16, 4};
  const oc_layout O = ocl(L), OX = ocl(X);
  uint64_t seed = 3 + k;
  std::vector<float> pts, q, rows, box(6);
  for (int i = 0; i < 3 * n; i++) pts.push_back(unit(seed));
  for (int i = 0; i < 3 * nq; i++) q.push_back(unit(seed));
  for (int i = 0; i < n; i++) {
    rows.insert(rows.end(), pts.begin() + 3 * i, pts.begin() + 3 * i + 3);
    rows.insert(rows.end(), 2, 0.f);
  }
  oc_build_host(pts.data(), n, &O, nullptr);
  oc_build_host(rows.data(), n, &OX, box.data());
  Dev<float> dt(pts), dx(rows), dq(q), dd((size_t)nq * k);
  Dev<int32_t> di((size_t)nq * k);
  std::vector<int32_t> ri((size_t)nq * k);
  std::vector<float> rd((size_t)nq * k);
  oc_knn(OC_STACK_BASED, OC_LIST_HEAP, k, pts.data(), n, &O, nullptr, q.data(), nq, INFINITY,
         ri.data(), rd.data(), nullptr, nullptr, 1);
  auto knn = [&](const float *tree, const cukd_layout &lay, float cutoff, int flags) {
    return cukd_knn(CUKD_STACK_BASED, CUKD_LIST_HEAP, k, tree, n, &lay, nullptr, dq.p, nq, cutoff,
                    di.p, dd.p, nullptr, CUKD_QUERY_AUTOTUNE | flags, nullptr,
                    nullptr) == CUKD_OK;
  };
  Dev<unsigned long long> count(1);
  if (!strcmp(first, "counted")) cukd_set_traversal_stats(count.p);
  bool ok = expl ? knn(dx.p, X, INFINITY, 0)
                 : knn(dt.p, L, !strcmp(first, "NaN cutoff") ? NAN : INFINITY,
                       !strcmp(first, "one per lane") ? CUKD_QUERY_ONE_PER_LANE : 0);
  cukd_set_traversal_stats(nullptr);
  ok = ok && launches_of("k_query_box", 0) == 0;
  // the plain call: pruned, now and once it is tuned
  for (int rep = 0; rep < 2; rep++) {
    const size_t from = emu_launches.size();
    ok = ok && knn(dt.p, L, INFINITY, 0) && di.same(ri) && dd.same(rd) &&
         launches_of("k_query_box", from) > 0 &&
         emu_launches.back().find("k_query_box") != std::string::npos;
  }
  const size_t from = emu_launches.size();
  ok = ok && knn(dt.p, L, INFINITY, CUKD_QUERY_ONE_PER_LANE) && di.same(ri) && dd.same(rd) &&
       launches_of("k_query_box", from) == 0;
  return ok;
}

// Runs 'call' again and again, with its first launch refused, then its second,
// ..., until it runs through: each refusal is its error, and no launch of the
// call works on what a refused one did not write.  'done' follows a success.
bool refusals_reported(const std::function<int()> &call, const std::function<bool()> &done)
{
  for (int i = 0;; i++) {
    emu_refuse_in = i;
    const int rc = call();
    const bool refused = emu_refuse_in < 0;
    emu_refuse_in = -1;
    if (!refused) return i > 0 && rc == CUKD_OK && done();
    if (rc != CUKD_ERR_HIP || hipGetLastError() != hipSuccess) {
      printf("  launch %d: rc %d\n", i, rc);
      return false;
    }
  }
}

// deep: points that peel off one by one, more than the level table holds
bool refused_spatial_build_case(int n, int D, bool deep)
{
  const cukd_layout L = floats(D);
  uint64_t seed = 9;
  std::vector<float> pts((size_t)n * D, 0.f);
  for (int i = 0; i < n * D; i++)
    pts[i] = !deep ? unit(seed) : i % D ? 0.f : std::ldexp(1.f, -(i / D));
  const int leaf = deep ? 1 : 0;
  const SpatialRef ref(pts, L, leaf);
  Dev<float> dp(pts);
  cukd_spatial_tree t;
  return refusals_reported(
      [&] { return cukd_spatial_build(&t, dp.p, n, &L, leaf, nullptr, nullptr); },
      [&] {
        const bool ok = ref.same(t);
        cukd_spatial_free(&t, nullptr, nullptr);
        return ok;
      });
}

bool refused_sorted_query_case()
{
  const int n = 500, nq = 100, k = 4;
  const cukd_layout L = floats(3);
  const oc_layout O = ocl(L);
  uint64_t seed = 9;
  std::vector<float> pts, q;
  for (int i = 0; i < 3 * n; i++) pts.push_back(unit(seed));
  for (int i = 0; i < 3 * nq; i++) q.push_back(unit(seed));
  oc_build_host(pts.data(), n, &O, nullptr);
  Dev<float> dt(pts), dq(q), dd((size_t)nq * k);
  Dev<int32_t> di((size_t)nq * k);
  std::vector<int32_t> ri((size_t)nq * k);
  std::vector<float> rd((size_t)nq * k);
  oc_knn(OC_STACK_BASED, OC_LIST_FIXED, k, pts.data(), n, &O, nullptr, q.data(), nq, INFINITY,
         ri.data(), rd.data(), nullptr, nullptr, 1);
  return refusals_reported(
      [&] {
        return cukd_knn(CUKD_STACK_BASED, CUKD_LIST_FIXED, k, dt.p, n, &L, nullptr, dq.p, nq,
                        INFINITY, di.p, dd.p, nullptr, CUKD_QUERY_SORT, nullptr, nullptr);
      },
      [&] { return di.same(ri) && dd.same(rd); });
}

// Temporaries come from memory of the stream's device, and from the pool that
// the program chose for it where it chose one.
bool pool_case(const char *what)
{
  const int n = 600;
  const cukd_layout L = floats(3);
  uint64_t seed = 21;
  std::vector<float> pts;
  for (int i = 0; i < 3 * n; i++) pts.push_back(unit(seed));
  Dev<float> dp(pts);
  const bool other = !strcmp(what, "stream of another device");
  const int dev = other ? 1 : 0;
  hipSetDevice(dev);
  hipStream_t own_stream = nullptr;
  hipStreamCreateWithFlags(&own_stream, hipStreamNonBlocking);
  hipSetDevice(0);
  hipStream_t s = own_stream;
  if (!strcmp(what, "null stream")) s = nullptr;
  if (!strcmp(what, "legacy stream")) s = hipStreamLegacy;
  if (!strcmp(what, "per-thread stream")) s = hipStreamPerThread;
  hipMemPool_t def = nullptr, own = nullptr;
  hipDeviceGetDefaultMemPool(&def, dev);
  const hipMemPoolProps props{hipMemAllocationTypePinned, {hipMemLocationTypeDevice, dev}};
  hipMemPoolCreate(&own, &props);
  uint64_t keep = 1 << 20, none = 0;
  if (!strcmp(what, "a current pool")) hipDeviceSetMemPool(dev, own);
  if (!strcmp(what, "a default pool that keeps")) hipMemPoolSetAttribute(def, hipMemPoolAttrReleaseThreshold, &keep);
  emu_last_pool = nullptr;
  bool ok = cukd_build_tree(dp.p, n, &L, CUKD_BUILDER_ID_DEFAULT, nullptr, s, nullptr) == CUKD_OK;
  ok = ok && emu_last_pool && emu_last_pool->device == dev;
  if (!strcmp(what, "a current pool")) ok = ok && emu_last_pool == own;
  else if (!strcmp(what, "a default pool that keeps")) ok = ok && emu_last_pool == def;
  else ok = ok && emu_last_pool != def && emu_last_pool->threshold > 0;  // the library's
  hipDeviceSetMemPool(dev, def);
  hipMemPoolSetAttribute(def, hipMemPoolAttrReleaseThreshold, &none);
  hipStreamDestroy(own_stream);
  return ok;
}

// A batch of one wave is never ordered and allocates nothing; larger ones are.
bool small_batch_case(int nq, int flags)
{
  const int n = 400, k = 2 + flags;  // its own tuned choice
  const cukd_layout L = floats(3);
  const oc_layout O = ocl(L);
  uint64_t seed = 17;
  std::vector<float> pts, q;
  for (int i = 0; i < 3 * n; i++) pts.push_back(unit(seed));
  for (int i = 0; i < 3 * nq; i++) q.push_back(unit(seed));
  oc_build_host(pts.data(), n, &O, nullptr);
  Dev<float> dt(pts), dq(q), dd((size_t)nq * k);
  Dev<int32_t> di((size_t)nq * k);
  std::vector<int32_t> ri((size_t)nq * k);
  std::vector<float> rd((size_t)nq * k);
  oc_knn(OC_STACK_BASED, OC_LIST_FIXED, k, pts.data(), n, &O, nullptr, q.data(), nq, INFINITY,
         ri.data(), rd.data(), nullptr, nullptr, 1);
  emu_last_pool = nullptr;
  return cukd_knn(CUKD_STACK_BASED, CUKD_LIST_FIXED, k, dt.p, n, &L, nullptr, dq.p, nq, INFINITY,
                  di.p, dd.p, nullptr, flags, nullptr, nullptr) == CUKD_OK &&
         di.same(ri) && dd.same(rd) && (launches_of("k_qplace", 0) > 0) == (nq > 64) &&
         (emu_last_pool != nullptr) == (nq > 64);
}

int own_malloc(void *, void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
int own_free(void *, void *p, hipStream_t) { return hipFree(p); }

// A large batch over a spatial tree built with the caller's memory resource
// allocates nothing; over one built without, it is Morton-ordered.
bool spatial_scratch_case(bool own)
{
  const int n = 16400, nq = 1 << 18;
  const cukd_layout L{3, CUKD_SCALAR_F32, 256, 0, -1, 4};
  const cukd_mem_resource res{nullptr, own_malloc, own_free};
  uint64_t seed = 33;
  std::vector<float> pts((size_t)n * 64, 0.f), q;
  for (int i = 0; i < n; i++)
    for (int d = 0; d < 3; d++) pts[(size_t)i * 64 + d] = unit(seed);
  for (int i = 0; i < 3 * nq; i++) q.push_back(unit(seed));
  Dev<float> dp(pts), dq(q);
  Dev<int32_t> di((size_t)nq);
  cukd_spatial_tree t;
  if (cukd_spatial_build(&t, dp.p, n, &L, 0, nullptr, own ? &res : nullptr) != CUKD_OK) return false;
  const size_t from = emu_launches.size();
  emu_last_pool = nullptr;
  bool ok = cukd_spatial_fcp(CUKD_STACK_BASED, &t, &L, dq.p, nq, 0.001f, di.p, nullptr,
                             nullptr) == CUKD_OK &&
            (emu_last_pool == nullptr) == own && (launches_of("k_qplace", from) == 0) == own;
  cukd_spatial_free(&t, nullptr, own ? &res : nullptr);
  return ok;
}

}  // namespace

int main(int argc, char **argv)
{
  const std::string only = argc > 1 ? argv[1] : "";
  struct Case {
    std::string name;
    std::function<bool()> run;
  };
  std::vector<Case> cases;
  for (const char *kind : {"sum overflows", "negative sum overflows", "opposite infinities",
                           "infinity in one dim", "minus infinity", "all infinite"})
    for (int n : {9, 40, 2500, 5000})
      for (int leaf : {0, 1})
        for (int D : {2, 3})
          cases.push_back({std::string("spatial centre, ") + kind + " n=" + std::to_string(n) +
                               " leaf=" + std::to_string(leaf) + " D=" + std::to_string(D),
                           [=] { return spatial_centre_case(kind, n, D, leaf); }});
  for (bool plain : {false, true})
    for (int list : {CUKD_LIST_FIXED, CUKD_LIST_HEAP})
      cases.push_back({std::string("spatial overflow without radii") + (plain ? ", plain" : "") +
                           (list == CUKD_LIST_HEAP ? ", heap" : ""),
                       [=] { return spatial_overflow_case(plain, CUKD_STACK_BASED, list); }});
  int k = 20;
  for (const char *first : {"counted", "NaN cutoff", "explicit dims", "one per lane"}) {
    k++;
    cases.push_back({std::string("autotune after ") + first, [=] { return autotune_case(first, k); }});
  }
  cases.push_back({"refused launch, spatial build", [] { return refused_spatial_build_case(5000, 3, false); }});
  cases.push_back({"refused launch, spatial build of one leaf", [] { return refused_spatial_build_case(5, 3, false); }});
  cases.push_back({"refused launch, deep spatial build", [] { return refused_spatial_build_case(110, 2, true); }});
  cases.push_back({"refused launch, sorted query", [] { return refused_sorted_query_case(); }});
  for (const char *what : {"nothing chosen", "stream of another device", "a current pool",
                           "a default pool that keeps", "null stream", "legacy stream",
                           "per-thread stream", "nothing chosen"})
    cases.push_back({std::string("memory pool, ") + what, [=] { return pool_case(what); }});
  for (int nq : {1, 63, 64, 65})
    for (int flags : {CUKD_QUERY_SORT, CUKD_QUERY_AUTOTUNE, CUKD_QUERY_SORT | CUKD_QUERY_AUTOTUNE})
      cases.push_back({"order of small batches, nq=" + std::to_string(nq) + " flags=" + std::to_string(flags),
                       [=] { return small_batch_case(nq, flags); }});
  for (bool own : {false, true})
    cases.push_back({std::string("scratch of spatial queries, ") + (own ? "caller's" : "library's") + " memory",
                     [=] { return spatial_scratch_case(own); }});
  int fail = 0;
  for (auto &c : cases)
    if (only.empty() || c.name.find(only) != std::string::npos) {
      emu_launches.clear();
      const bool ok = c.run();
      printf("%-66s %s\n", c.name.c_str(), ok ? "ok" : "FAILED");
      fflush(stdout);
      fail += !ok;
    }
  printf(fail ? "%d FAILED\n" : "ALL OK\n", fail);
  return fail ? 1 : 0;
}
