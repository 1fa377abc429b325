// The block pools (csrc/rsg_pool.hip) against a device of counted bytes: hipMalloc, hipFree and
// operator new are this program's, so both kinds of memory run out where a case wants them to.
#include "../../r-scape_amd/csrc/rsg_pool.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <new>
#include <random>
#include <thread>

static std::atomic<long> g_new_left{-1};                // allocations until one fails; < 0: none does
void *operator new(size_t n)
{
  long k = g_new_left.load();
  while (k > 0 && !g_new_left.compare_exchange_weak(k, k - 1)) {}
  if (k == 0) throw std::bad_alloc();
  if (void *p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

static std::mutex g_mu;
static std::map<char *, size_t> g_live;                 // device blocks
static size_t g_cap = (size_t)1 << 40, g_total = 0;
static char *g_next = (char *)0x1000;                   // addresses only: nothing is read or written there
struct NoFail { long k; NoFail() : k(g_new_left.exchange(-1)) {} ~NoFail() { g_new_left = k; } };

extern "C" hipError_t hipMalloc(void **p, size_t n)
{
  std::lock_guard<std::mutex> lk(g_mu);
  NoFail f;
  if (g_total + n > g_cap) { *p = nullptr; return hipErrorOutOfMemory; }
  g_live[g_next] = n; g_total += n;
  *p = g_next; g_next += n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p)
{
  std::lock_guard<std::mutex> lk(g_mu);
  NoFail f;
  const auto it = g_live.find((char *)p);
  if (it == g_live.end()) { printf("hipFree of a block that is not one\n"); exit(1); }
  g_total -= it->second;
  g_live.erase(it);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)

// blocks come back by size class, within the bounds, and with the pool
static void reuse()
{
  {
    RsgPool p;
    void *a, *b;
    CHECK(p.get(&a, 1000) == hipSuccess); p.put(a);
    CHECK(p.get(&b, 1010) == hipSuccess && b == a); p.put(b);
    CHECK(p.get(&b, 5000) == hipSuccess && b != a); p.put(b);
    CHECK(g_live.size() == 2);
    void *big;
    CHECK(p.get(&big, RSG_POOL_BLOCK + 1) == hipSuccess); p.put(big);
    CHECK(g_live.size() == 2);                          // over the block size: given back at once
    void *v[8];
    for (auto &q : v) CHECK(p.get(&q, RSG_POOL_BLOCK) == hipSuccess);
    for (auto &q : v) p.put(q);
    CHECK(g_total <= RSG_POOL_KEEP);
    p.trim();
    CHECK(g_live.empty());
    void *w[RSG_POOL_COUNT + 5];
    for (auto &q : w) CHECK(p.get(&q, 512) == hipSuccess);
    for (auto &q : w) p.put(q);
    CHECK(g_live.size() == RSG_POOL_COUNT);
    CHECK(p.get(&a, 512) == hipSuccess);
    p.close();
    CHECK(g_live.size() == 1);
    p.put(a);                                           // a block that outlives its context
    CHECK(g_live.empty());
  }
  CHECK(g_live.empty());
}

// an allocation that does not fit takes the idle blocks of every pool back
static void pressure()
{
  RsgPool p, q;
  void *a, *b, *c;
  g_cap = 10000;
  CHECK(p.get(&a, 4096) == hipSuccess && q.get(&b, 4096) == hipSuccess);
  p.put(a); q.put(b);
  CHECK(rsg_dev_malloc(&c, 9000) == hipSuccess && g_live.size() == 1);
  CHECK(q.get(&b, 4096) == hipErrorOutOfMemory && b == nullptr);
  CHECK(hipFree(c) == hipSuccess);
  g_cap = (size_t)1 << 40;
}

// host memory that runs out anywhere: an error from get, nothing from put, no block lost
static void host_memory()
{
  for (long k = 0; k < 400; k++) {
    {
      std::unique_ptr<RsgPool> p;
      try { g_new_left = k; p.reset(new RsgPool()); } catch (const std::bad_alloc &) {}
      if (p) {
        void *v[300];
        for (int rep = 0; rep < 2; rep++) {
          int n = 0;
          for (; n < 300; n++) if (p->get(&v[n], 512 + 64 * (size_t)(n % 7)) != hipSuccess) { CHECK(v[n] == nullptr); break; }
          for (int i = 0; i < n; i++) p->put(v[i]);
          if (rep == 0) p->trim();
        }
        p->close();
      }
      g_new_left = -1;
    }
    CHECK(g_live.empty() && g_total == 0);
  }
}

// several threads on two pools: a block has one owner at a time
static void threads()
{
  RsgPool p[2];
  std::mutex mu;
  std::map<void *, int> owner;
  std::vector<std::thread> th;
  for (int t = 0; t < 8; t++)
    th.emplace_back([&, t] {
      std::mt19937 rng(t);
      std::vector<std::pair<int, void *>> mine;
      for (int i = 0; i < 4000; i++) {
        if (mine.size() < 12 && rng() % 2) {
          const int w = rng() % 2;
          void *b = nullptr;
          CHECK(p[w].get(&b, 1 + rng() % 4000) == hipSuccess);
          { std::lock_guard<std::mutex> lk(mu); CHECK(owner.emplace(b, t).second); }
          mine.emplace_back(w, b);
        } else if (!mine.empty()) {
          const size_t k = rng() % mine.size();
          { std::lock_guard<std::mutex> lk(mu); CHECK(owner.erase(mine[k].second) == 1); }
          p[mine[k].first].put(mine[k].second);
          mine.erase(mine.begin() + (ptrdiff_t)k);
        }
        if (i % 500 == 499) p[rng() % 2].trim();
      }
      for (auto &m : mine) {
        { std::lock_guard<std::mutex> lk(mu); owner.erase(m.second); }
        p[m.first].put(m.second);
      }
    });
  for (auto &x : th) x.join();
}

int main()
{
  reuse(); printf("reuse ok\n");
  pressure(); printf("pressure ok\n");
  host_memory(); printf("host memory ok\n");
  threads(); CHECK(g_live.empty()); printf("threads ok\n");
  return 0;
}
