// rsg_pool.h -- pools of device blocks
#pragma once
#include <hip/hip_runtime_api.h>
#include <cstddef>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

// Device blocks of short-lived objects, kept for the next ones: hipMalloc and hipFree of a dozen
// buffers cost more than scoring a family does (score of 600 x 300 on a new alignment object,
// R-scape's own call: 236 us with them, 174 us without).  A block put back is handed out again for
// a request of its size class; at most RSG_POOL_KEEP bytes are kept (the rest, and blocks over
// RSG_POOL_BLOCK, go back to the device at once), all of them are given back with the context, and
// by every pool when a device allocation of the library fails (rsg_dev_malloc makes them all).  Any
// thread may call.
// A pool does not wait for the device: its user keeps one of two rules.  `tmp` of a context holds
// blocks that only work on that context's stream touches (RsgTmp), so stream order covers their
// reuse; `pool` holds blocks of alignments, which any context may have used: they are put back
// when the device is idle (as hipFree waits for it).
#define RSG_POOL_KEEP  ((size_t)1 << 30)
#define RSG_POOL_BLOCK ((size_t)1 << 28)
#define RSG_POOL_COUNT 256               // idle blocks at most
struct RsgPool {
  RsgPool();                             // std::bad_alloc only; nothing below throws
  ~RsgPool();
  hipError_t get(void **p, size_t bytes);
  void put(void *p);
  void close();                          // gives back the idle blocks and keeps none from here on
  void trim();                           // gives back the idle blocks
private:
  std::mutex mu;
  std::unordered_map<void *, size_t> used;            // size classes of the blocks handed out
  std::vector<std::pair<size_t, void *>> idle;        // never past the RSG_POOL_COUNT reserved
  size_t kept = 0;
  bool open = true;
};
// Every device allocation of the library: hipMalloc; when the device is full, again after every pool has
// given back its idle blocks
hipError_t rsg_dev_malloc(void **p, size_t bytes);
template <typename T> static inline hipError_t rsg_dev_malloc(T **p, size_t bytes) { return rsg_dev_malloc((void **)p, bytes); }
