// workspace.cpp -- device and pinned host memory of the stage operators' calls.
//
// An operator needs temporaries for one call.  Allocating and freeing them took most of a
// small call's time (a hipMalloc of 64 MiB or more costs about 300 us here, one of 2 MiB 20 to
// 40, each hipFree 2 to 100), so the blocks of a finished call are kept for the next one.
//   - A block belongs to one call at a time: it is taken from the free list and goes back only
//     when the call has waited for its stream (Workspace::done), so no other stream or thread
//     can meet work that still uses it.  A call that ends early frees its blocks instead.
//   - Per device at most KEEP_BYTES in KEEP_BLOCKS are kept, the oldest freed first (a block
//     above KEEP_BYTES is freed and evicts none); all of them are freed when a context is
//     destroyed, when a context needs the memory, and when an allocation here fails (which is
//     then tried once more).
//   - The list itself is never destroyed: the runtime may be gone when the process ends.
#include <algorithm>
#include <mutex>

#include "engine.h"

namespace pic {

namespace {

constexpr size_t KEEP_BYTES = 256ull << 20;
constexpr size_t KEEP_BLOCKS = 32;

struct Pool {
  std::mutex mu;
  std::vector<Workspace::Block> kept;  // oldest first
};
Pool& pool() {
  static Pool* p = new Pool();
  return *p;
}

void give_back(const std::vector<Workspace::Block>& blocks) {
  for (const Workspace::Block& b : blocks) {
    if (b.host) (void)hipHostFree(b.p);
    else (void)hipFree(b.p);
  }
}

// power-of-two sizes up to 1 MiB, whole MiB above
size_t block_size(size_t bytes) {
  if (bytes > (1u << 20)) return (bytes + (1u << 20) - 1) >> 20 << 20;
  size_t s = 4096;
  while (s < bytes) s *= 2;
  return s;
}

}  // namespace

void workspace_trim(int device) {
  std::vector<Workspace::Block> out;
  {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    auto it = std::stable_partition(q.kept.begin(), q.kept.end(), [&](const Workspace::Block& b) {
      return b.device != device;
    });
    out.assign(it, q.kept.end());
    q.kept.erase(it, q.kept.end());
  }
  give_back(out);
}

hipError_t Workspace::raw(void** p, size_t bytes, bool host) {
  *p = nullptr;
  Block b;
  b.host = host;
  hipError_t e = hipGetDevice(&b.device);
  if (e != hipSuccess) return e;
  const size_t want = block_size(bytes);
  {
    // the smallest kept block that holds it, of at most twice the size
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    size_t best = q.kept.size();
    for (size_t i = 0; i < q.kept.size(); ++i) {
      const Block& k = q.kept[i];
      if (k.device == b.device && k.host == host && k.bytes >= want && k.bytes <= 2 * want &&
          (best == q.kept.size() || k.bytes < q.kept[best].bytes))
        best = i;
    }
    if (best < q.kept.size()) {
      blocks.push_back(q.kept[best]);
      q.kept.erase(q.kept.begin() + (long)best);
      *p = blocks.back().p;
      return hipSuccess;
    }
  }
  b.bytes = want;
  e = host ? hipHostMalloc(&b.p, want, hipHostMallocDefault) : hipMalloc(&b.p, want);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    workspace_trim(b.device);
    b.bytes = bytes ? bytes : 1;
    e = host ? hipHostMalloc(&b.p, b.bytes, hipHostMallocDefault) : hipMalloc(&b.p, b.bytes);
  }
  if (e != hipSuccess) return e;
  blocks.push_back(b);
  *p = b.p;
  return hipSuccess;
}

Workspace::~Workspace() {
  if (!finished) {
    give_back(blocks);  // frees wait for the device
    return;
  }
  // blocks that evict each other go back the largest first, so that the small ones stay
  size_t total = 0;
  for (const Block& b : blocks) total += b.bytes;
  if (total > KEEP_BYTES)
    std::sort(blocks.begin(), blocks.end(),
              [](const Block& a, const Block& b) { return a.bytes > b.bytes; });
  std::vector<Block> out;
  {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    for (const Block& b : blocks) {
      if (b.bytes > KEEP_BYTES) {  // would evict all the others and not fit itself
        out.push_back(b);
        continue;
      }
      size_t held = b.bytes, count = 1;
      for (const Block& k : q.kept)
        if (k.device == b.device) {
          held += k.bytes;
          ++count;
        }
      for (size_t i = 0; i < q.kept.size() && (held > KEEP_BYTES || count > KEEP_BLOCKS);) {
        if (q.kept[i].device != b.device) {
          ++i;
          continue;
        }
        held -= q.kept[i].bytes;
        --count;
        out.push_back(q.kept[i]);
        q.kept.erase(q.kept.begin() + (long)i);
      }
      q.kept.push_back(b);
    }
  }
  give_back(out);
}

}  // namespace pic
