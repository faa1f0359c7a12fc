// Device workspaces kept between solves.
//
// Mapping and unmapping device memory costs more than short solves do (two
// vectors of 64 MiB: 0.43 ms of hipMalloc and hipFree a call, two of 256 MiB
// 0.72 ms), so blocks that a solve, a batch or one of its instances is finished
// with wait here for the next one of their size (to the page: a block is never
// larger than what its user counts).  At most kPoolBytes are kept, the least
// recently returned ones are freed beyond that, all of a device's are freed
// before one of the library's allocations on it is allowed to fail, and all of
// them by rkx_release_workspaces.  A block is returned only when no stream uses
// it any more (its owner has waited for its stream), so the next owner may use
// it on any stream and from any thread.
#include "rkx_internal.hpp"

#include <algorithm>
#include <list>
#include <mutex>

namespace rkx {
namespace {

constexpr size_t kPoolBytes = size_t(1) << 30;

struct block {
  void *p;
  size_t bytes;
  int dev;
};

struct pool_t {
  std::mutex mu;
  std::list<block> kept;          // least recently returned first
  size_t bytes = 0;
};
// never destroyed: the runtime may be gone when static destructors run
pool_t &pool()
{
  static pool_t *p = new pool_t;
  return *p;
}

// Frees the kept blocks of one device (dev < 0: of all).
void free_kept(int dev)
{
  pool_t &P = pool();
  std::list<block> drop;
  {
    std::lock_guard<std::mutex> lk(P.mu);
    for (auto it = P.kept.begin(); it != P.kept.end();) {
      const auto nx = std::next(it);
      if (dev < 0 || it->dev == dev) {
        P.bytes -= it->bytes;
        drop.splice(drop.end(), P.kept, it);
      }
      it = nx;
    }
  }
  for (const block &b : drop)
    (void) hipFree(b.p);
}

}  // namespace

void pool_release() { free_kept(-1); }

int device_alloc(void **out, size_t bytes)
{
  if (hipMalloc(out, bytes) == hipSuccess)
    return RKX_OK;
  (void) hipGetLastError();
  int dev = 0;
  RKX_HIP(hipGetDevice(&dev));
  free_kept(dev);
  if (hipMalloc(out, bytes) == hipSuccess)
    return RKX_OK;
  (void) hipGetLastError();
  *out = nullptr;
  return fail(RKX_ENOMEM, "hipMalloc of " + std::to_string(bytes) + " bytes failed");
}

int pool_take(void **out, size_t bytes, size_t *got)
{
  int dev = 0;
  RKX_HIP(hipGetDevice(&dev));
  bytes = (bytes + 4095) & ~size_t(4095);
  pool_t &P = pool();
  {
    std::lock_guard<std::mutex> lk(P.mu);
    const auto it = std::find_if(P.kept.begin(), P.kept.end(), [&](const block &b) {
      return b.dev == dev && b.bytes == bytes;
    });
    if (it != P.kept.end()) {
      *out = it->p;
      *got = bytes;
      P.bytes -= bytes;
      P.kept.erase(it);
      return RKX_OK;
    }
  }
  if (int rc = device_alloc(out, bytes))
    return rc;
  *got = bytes;
  return RKX_OK;
}

void pool_give(void *p, size_t bytes)
{
  int dev = 0;
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, p) == hipSuccess)
    dev = at.device;
  else
    (void) hipGetLastError();
  pool_t &P = pool();
  std::list<block> drop;
  {
    std::lock_guard<std::mutex> lk(P.mu);
    P.kept.push_back(block{p, bytes, dev});
    P.bytes += bytes;
    while (P.bytes > kPoolBytes) {
      P.bytes -= P.kept.front().bytes;
      drop.splice(drop.end(), P.kept, P.kept.begin());
    }
  }
  for (const block &b : drop)
    (void) hipFree(b.p);
}

}  // namespace rkx
