// Memory that contexts can do without (dgx_pool.cpp), on a stand-in for the HIP
// runtime with two devices of limited memory: the adjoint's workspace is kept
// and grown on the context's own device, is not shared by calls that overlap, is
// given back when another allocation needs the room, and is not kept above its
// bound; the stored geometry is given back likewise, but not under a launch, a
// captured one or a table that keeps it.
#include <atomic>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include "dgx_pool.hpp"

using namespace dgx;

static int g_failed = 0;
#define CHECK(x)                                               \
  do                                                           \
    if (!(x))                                                  \
    {                                                          \
      ++g_failed;                                              \
      std::printf("line %d: %s\n", __LINE__, #x);              \
    }                                                          \
  while (0)

static dgx_ctx* context(int device)
{
  dgx_ctx* c = new dgx_ctx();
  std::memset(c, 0, sizeof(*c));
  c->device    = device;
  c->geo_users = -1;
  pool_add(c);
  return c;
}

static void destroy(dgx_ctx* c)
{
  pool_remove(c);
  workspace_release(c);
  delete c;
}

static void store(dgx_ctx* c, size_t bytes)
{
  CHECK(hipMalloc((void**)&c->geo, bytes) == hipSuccess);
  c->geo_bytes = bytes;
  c->nelem = c->nbf = 1;
  __atomic_store_n(&c->geo_users, 0, __ATOMIC_RELEASE);
}

static void geometry()
{
  g_hip.capacity[0] = (size_t)100 << 20;
  dgx_ctx *a = context(0), *b = context(0);
  {
    MeshLease m(MeshArgs{}, b);  // nothing stored
    CHECK(!m.geov && !m.geof && b->geo_users == -1);
  }
  store(a, (size_t)30 << 20);
  store(b, (size_t)30 << 20);
  void* p = nullptr;
  {
    MeshLease m(MeshArgs{}, a);
    CHECK(m.geov == a->geo && m.geof == a->geo + GEOV);
    CHECK(pool_malloc(&p, (size_t)60 << 20, 0) == hipSuccess);  // b's goes, a's is being read
    CHECK(a->geo && !b->geo && b->geo_users == -1 && b->geo_bytes == 0);
    CHECK(!geometry_release(a));
    MeshLease n(MeshArgs{}, b);
    CHECK(!n.geov && !n.geof);
    hipFree(p);
  }
  CHECK(a->geo_users == 0 && geometry_release(a) && !a->geo && !geometry_release(a));

  // recorded into a graph, or kept in a table: held for good
  for (int k = 0; k < 2; ++k)
  {
    dgx_ctx* c = context(0);
    store(c, (size_t)30 << 20);
    MeshArgs kept{};
    g_capturing = k == 0;
    {
      MeshLease m(MeshArgs{}, c);
      if (k == 1)
        kept = m.keep();
    }
    g_capturing = false;
    CHECK(k == 0 || kept.geov == c->geo);
    CHECK(!pool_reclaim(0) && c->geo);
    hipFree(c->geo);
    destroy(c);
  }

  // threads that launch while others need the room
  store(a, (size_t)1 << 20);
  std::atomic<int> bad{0};
  std::atomic<bool> stop{false};
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; ++t)
    ts.emplace_back([&] {
      while (!stop)
      {
        MeshLease m(MeshArgs{}, a);
        std::lock_guard<std::mutex> lk(g_hip.mx);
        if (m.geov && !g_hip.blocks.count((void*)m.geov))
          ++bad;
      }
    });
  for (int it = 0; it < 200; ++it)
  {
    while (!geometry_release(a))
      std::this_thread::yield();
    store(a, (size_t)1 << 20);
  }
  stop = true;
  for (auto& t : ts)
    t.join();
  CHECK(bad == 0 && a->geo_users == 0 && geometry_release(a));
  destroy(a);
  destroy(b);
  CHECK(g_hip.blocks.empty());
}

int main()
{
  constexpr size_t MB = (size_t)1 << 17;  // doubles of a megabyte
  g_hip.capacity[0] = g_hip.capacity[1] = (size_t)100 << 20;
  dgx_ctx *a = context(0), *b = context(1);

  // kept between calls, grown, on the context's device whatever the current one is
  for (int device : {0, 1})
  {
    hipSetDevice(device);
    for (size_t n : {10 * MB, 20 * MB, 5 * MB})
      for (dgx_ctx* c : {a, b})
      {
        Workspace w(c);
        CHECK(w.open(n) == hipSuccess);
        double* p = w.take(n);
        CHECK(g_hip.blocks.count(p) && g_hip.blocks[p].device == c->device);
        CHECK(((size_t)(w.take(1) - p) == Workspace::padded(n)));
      }
    CHECK(t_device == device);
  }
  hipSetDevice(0);
  CHECK(g_hip.mallocs == 4 && g_hip.used[0] == (20u << 20) && g_hip.used[1] == (20u << 20));

  // an allocation that does not fit takes idle workspaces of its device
  void* p = nullptr;
  CHECK(pool_malloc(&p, (size_t)90 << 20, 0) == hipSuccess && a->adj_ws == nullptr);
  CHECK(b->adj_ws != nullptr && b->adj_ws_bytes == (20u << 20));
  void* q = &p;
  CHECK(pool_malloc(&q, (size_t)90 << 20, 0) == hipErrorOutOfMemory && q == nullptr);
  hipFree(p);

  // but not one that a call is using, and the calls go on
  {
    Workspace w(a);
    CHECK(w.open(20 * MB) == hipSuccess);
    CHECK(pool_malloc(&p, (size_t)90 << 20, 0) == hipErrorOutOfMemory);
    workspace_release(a);
    CHECK(a->adj_ws != nullptr);
    // a second call on the context meanwhile has memory of its own
    {
      Workspace v(a);
      CHECK(v.open(30 * MB) == hipSuccess);
      double *x = v.take(30 * MB), *y = w.take(20 * MB);
      CHECK(x >= y + 20 * MB || y >= x + 30 * MB);
    }
    CHECK(g_hip.used[0] == (20u << 20));
  }
  workspace_release(a);
  CHECK(g_hip.used[0] == 0);

  // a failed call leaves the context usable
  {
    Workspace w(a);
    CHECK(w.open(200 * MB) == hipErrorOutOfMemory);
  }
  {
    Workspace w(a);
    CHECK(w.open(MB) == hipSuccess);
  }

  // threads on one context and one that needs the room: no two calls share memory
  std::atomic<int> clashes{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; ++t)
    ts.emplace_back([&, t] {
      for (int it = 0; it < 300; ++it)
      {
        Workspace w(a);
        const size_t n = (1 + (it + t) % 5) * 1000;
        if (w.open(n) != hipSuccess)
          continue;
        double* x = w.take(n);
        for (size_t i = 0; i < n; ++i)
          x[i] = t;
        std::this_thread::yield();
        for (size_t i = 0; i < n; ++i)
          if (x[i] != t)
            ++clashes;
      }
    });
  for (int it = 0; it < 300; ++it)
    (void)pool_reclaim(0);
  for (auto& t : ts)
    t.join();
  CHECK(clashes == 0);

  // above the bound it goes back after the call
  g_hip.capacity[0] = (size_t)3 << 30;
  {
    Workspace w(a);
    CHECK(w.open((WORKSPACE_KEEP >> 3) + 32) == hipSuccess);
  }
  CHECK(a->adj_ws == nullptr && g_hip.used[0] == 0);

  destroy(a);
  destroy(b);
  CHECK(g_hip.blocks.empty() && g_hip.mallocs == g_hip.frees);

  geometry();
  return g_failed ? 1 : 0;
}
