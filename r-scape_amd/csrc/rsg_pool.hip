// rsg_pool.hip -- pools of device blocks (host code: no kernels here)
#include "rsg_pool.h"
#include <algorithm>
#include <new>

static std::mutex g_pools_mu;
static std::vector<RsgPool *> g_pools;                 // those alive

RsgPool::RsgPool()
{
  idle.reserve(RSG_POOL_COUNT);
  std::lock_guard<std::mutex> lk(g_pools_mu);
  g_pools.push_back(this);
}
RsgPool::~RsgPool()
{
  { std::lock_guard<std::mutex> lk(g_pools_mu); g_pools.erase(std::find(g_pools.begin(), g_pools.end(), this)); }
  trim();
}

// Size classes of eight steps per power of two, 512 bytes and up: at most an eighth is unused.
static size_t pool_class(size_t n)
{
  if (n <= 512) return 512;
  size_t s = (size_t)1 << (60 - __builtin_clzll(n));  // an eighth of the power of two at or under n
  if (s < 64) s = 64;
  return (n + s - 1) / s * s;
}

hipError_t RsgPool::get(void **p, size_t bytes)
{
  *p = nullptr;
  const size_t n = bytes > RSG_POOL_BLOCK ? bytes : pool_class(bytes);
  try {
    std::lock_guard<std::mutex> lk(mu);
    for (size_t k = idle.size(); k-- > 0;)             // the last one put back is the likeliest in cache
      if (idle[k].first == n) {
        used.emplace(idle[k].second, n);               // (if this throws the block stays idle)
        *p = idle[k].second;
        idle.erase(idle.begin() + (ptrdiff_t)k);
        kept -= n;
        return hipSuccess;
      }
  } catch (const std::bad_alloc &) { return hipErrorOutOfMemory; }
  const hipError_t e = rsg_dev_malloc(p, n);
  if (e != hipSuccess) { *p = nullptr; return e; }
  try {
    std::lock_guard<std::mutex> lk(mu);
    used.emplace(*p, n);
  } catch (const std::bad_alloc &) {
    (void)hipFree(*p);
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  return hipSuccess;
}

void RsgPool::put(void *p)
{
  if (!p) return;
  {
    std::lock_guard<std::mutex> lk(mu);
    const auto it = used.find(p);
    const size_t n = it->second;
    used.erase(it);
    if (open && n <= RSG_POOL_BLOCK && kept + n <= RSG_POOL_KEEP && idle.size() < RSG_POOL_COUNT) {
      idle.emplace_back(n, p);
      kept += n;
      return;
    }
  }
  (void)hipFree(p);
}

void RsgPool::trim()
{
  void *v[RSG_POOL_COUNT];
  size_t n = 0;
  {
    std::lock_guard<std::mutex> lk(mu);
    for (auto &b : idle) v[n++] = b.second;
    idle.clear();                                      // (its room stays)
    kept = 0;
  }
  for (size_t k = 0; k < n; k++) (void)hipFree(v[k]);
}

void RsgPool::close()
{
  { std::lock_guard<std::mutex> lk(mu); open = false; }
  trim();
}

hipError_t rsg_dev_malloc(void **p, size_t bytes)
{
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  { std::lock_guard<std::mutex> lk(g_pools_mu); for (RsgPool *q : g_pools) q->trim(); }
  return hipMalloc(p, bytes);
}
