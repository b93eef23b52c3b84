// PoolArena against a stand-in for the HIP runtime (tests/test_pool.py): an owner of buffers of device 0 goes away
// while device 1 is current.  Its buffers must not be handed out before the work of their own device is
// done: the wait, the frees and the return of what is not kept happen on device 0, in that order, and device
// 1 is current again afterwards.
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "ddf_pool.h"

static int g_dev = 0;
static std::vector<std::string> g_log;
static void note(const char* what) { g_log.push_back(std::string(what) + std::to_string(g_dev)); }

hipError_t hipGetDevice(int* d) { return *d = g_dev, hipSuccess; }
hipError_t hipSetDevice(int d) { return g_dev = d, hipSuccess; }
hipError_t hipDeviceSynchronize() { return note("wait"), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return note("sync"), hipSuccess; }
hipError_t hipFreeAsync(void* p, hipStream_t) { return note("free"), free(p), hipSuccess; }
namespace ddf {
hipError_t pool_alloc(void** p, size_t bytes, hipStream_t) { return *p = malloc(bytes), hipSuccess; }
hipError_t pool_trim(size_t keep) { return note(keep == kPoolKeep ? "trim" : "bad"), hipSuccess; }
}  // namespace ddf

int main() {
  ddf::PoolArena a, none, list;
  // a slab, and a buffer of its own, made as an optional list's that the owner then takes over
  if (!list.get(100, nullptr) || !list.get(size_t(40) << 20, nullptr)) return 1;
  a.take(list);
  if (!list.empty() || list.bytes() != 0) return 3;
  // what is held is whole slabs and whole buffers, until the end
  if (a.bytes() != (size_t(42) << 20) || none.bytes() != 0) return 2;
  hipSetDevice(1);
  a.close();
  none.close();
  std::string all;
  for (const std::string& s : g_log) all += s + " ";
  printf("%s-> %d\n", all.c_str(), g_dev);
  return all == "wait0 free0 free0 sync0 trim0 " && g_dev == 1 && a.empty() && a.bytes() == 0 ? 0 : 1;
}
