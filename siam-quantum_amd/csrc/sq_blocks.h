// sq_blocks.h - cache of device and pinned host blocks.
//
// Mem gives the memory: malloc(&p, bytes, host) and free(p, host) with 0 for
// success, clear_error() which forgets the error that a failed call leaves
// behind, device() (the current one, negative on error) and total(), the
// current device's memory in bytes.
#pragma once
#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

template <class Mem>
class BlockCache {
 public:
  explicit BlockCache(Mem m = Mem()) : mem(m) {}

  // Device and pinned host blocks released by a context are kept for the next
  // one (an SCF creates and releases its context once per solve; hipFree and
  // hipHostFree synchronise the device and cost more than the work they end).
  // A request takes the smallest cached block of the same kind and device that
  // holds it, at most twice its size.  The cache keeps 4 GiB, and an eighth of
  // the device's memory while any context is alive: the MP2 path works in
  // blocks of tens of gigabytes, and the driver clears such an allocation
  // before it hands it out again ((H2O)16/6-31G*, 22 GB: 0.5 s a call, where
  // the transform takes 0.05 s).  A failed allocation empties the cache and
  // tries again.  Null if that fails too; either way no error is left for the
  // next check of the runtime's last error, which may follow any launch.
  void* get(size_t bytes, bool host) {
    const int dev = mem.device();
    if (dev < 0) return nullptr;
    std::lock_guard<std::mutex> lk(mu);
    size_t best = kept.size();
    for (size_t i = 0; i < kept.size(); ++i) {
      const Block& b = kept[i];
      if (b.host == host && (host || b.device == dev) && b.bytes >= bytes && b.bytes <= 2 * bytes &&
          (best == kept.size() || b.bytes < kept[best].bytes))
        best = i;
    }
    if (best < kept.size()) {
      const Block b = kept[best];
      kept.erase(kept.begin() + (long)best);
      kept_bytes -= b.bytes;
      live.push_back(b);
      return b.p;
    }
    void* p = nullptr;
    if (mem.malloc(&p, bytes, host)) {
      mem.clear_error();
      trim_locked();
      if (mem.malloc(&p, bytes, host)) {
        mem.clear_error();
        return nullptr;
      }
    }
    live.push_back({p, bytes, dev, host});
    return p;
  }

  void put(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lk(mu);
    for (size_t i = 0; i < live.size(); ++i)
      if (live[i].p == p) {
        const Block b = live[i];
        live.erase(live.begin() + (long)i);
        if (kept_bytes + b.bytes <= most_locked()) {
          kept.push_back(b);
          kept_bytes += b.bytes;
        } else {
          (void)mem.free(b.p, b.host);
        }
        return;
      }
  }

  void trim() {
    std::lock_guard<std::mutex> lk(mu);
    trim_locked();
  }

  // A context comes to life or goes; without any, the cache shrinks to its
  // ordinary size, largest blocks first.
  void count_context(int d) {
    std::lock_guard<std::mutex> lk(mu);
    contexts += d;
    while (contexts == 0 && kept_bytes > kMost) {
      auto it = std::max_element(kept.begin(), kept.end(),
                                 [](const Block& x, const Block& y) { return x.bytes < y.bytes; });
      (void)mem.free(it->p, it->host);
      kept_bytes -= it->bytes;
      kept.erase(it);
    }
  }

  size_t cached() {
    std::lock_guard<std::mutex> lk(mu);
    return kept_bytes;
  }

 private:
  struct Block { void* p; size_t bytes; int device; bool host; };
  static constexpr size_t kMost = size_t(4) << 30;

  size_t most_locked() { return contexts > 0 ? std::max(kMost, mem.total() / 8) : kMost; }
  void trim_locked() {
    for (const Block& b : kept) (void)mem.free(b.p, b.host);
    kept.clear();
    kept_bytes = 0;
  }

  Mem mem;
  std::mutex mu;
  std::vector<Block> kept;  // cached, free
  std::vector<Block> live;  // handed out
  size_t kept_bytes = 0;
  int contexts = 0;
};
