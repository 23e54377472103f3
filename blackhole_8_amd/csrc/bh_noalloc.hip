// bh_noalloc.hip — device memory of the allocation-free render entry point
// (bh_render_device_noalloc): one file-scope array per GPU holds the scene
// record and the FP64 queue of a frame, so the entry point needs no hipMalloc.
// Its address on each device is resolved once, when a context is created on
// that device (noalloc_scratch), and only that address is used on the host.
// Every call on a GPU shares that GPU's array: calls that overlap on one GPU
// race.
#include "bh_internal.h"

namespace bh {
namespace {

// Layout: scene record, queue count words, queue items.
constexpr size_t kSceneBytes = (sizeof(DevScene) + 255) / 256 * 256;
constexpr size_t kCountBytes = (kQueueCountWords * sizeof(uint32_t) + 255) / 256 * 256;
constexpr size_t kScratchBytes = kSceneBytes + kCountBytes + kNoallocQueueItems * sizeof(uint64_t);

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

}  // namespace

hipError_t noalloc_scratch(void** ptr) {
  return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch));
}

NoallocLayout noalloc_layout(void* base) {
  unsigned char* b = static_cast<unsigned char*>(base);
  NoallocLayout l;
  l.scene = reinterpret_cast<DevScene*>(b);
  l.count = reinterpret_cast<uint32_t*>(b + kSceneBytes);
  l.items = reinterpret_cast<uint64_t*>(b + kSceneBytes + kCountBytes);
  return l;
}

}  // namespace bh
