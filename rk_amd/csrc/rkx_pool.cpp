// Device workspaces kept between solves.
//
// Mapping and unmapping device memory costs more than short solves do (two
// vectors of 64 MiB: 0.43 ms of hipMalloc and hipFree a call, two of 256 MiB
// 0.72 ms), so blocks that a solve or a batch instance is finished with wait
// here for the next one of their size (to the page: a block is never larger
// than what its user counts).  At most kPoolBytes are kept, the least recently
// returned ones are freed beyond that, and all of a device's are freed before
// an allocation on it is allowed to fail.  A block is returned only when no
// stream uses it any more (its owner has waited for its stream), so the next
// owner may use it on any stream and from any thread.
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

}  // namespace

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
  void *p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void) hipGetLastError();
    std::list<block> drop;
    {
      std::lock_guard<std::mutex> lk(P.mu);
      for (auto it = P.kept.begin(); it != P.kept.end();) {
        auto nx = std::next(it);
        if (it->dev == dev) {
          P.bytes -= it->bytes;
          drop.splice(drop.end(), P.kept, it);
        }
        it = nx;
      }
    }
    for (const block &b : drop)
      (void) hipFree(b.p);
    if (hipMalloc(&p, bytes) != hipSuccess) {
      (void) hipGetLastError();
      return fail(RKX_ENOMEM, "hipMalloc of " + std::to_string(bytes) + " bytes failed");
    }
  }
  *out = p;
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
