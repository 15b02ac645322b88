// sq_blocks.h - cache of device and pinned host blocks.
//
// Mem gives the memory: malloc(&p, bytes, host) and free(p, host) with 0 for
// success, clear_error() which forgets the error that a failed call leaves
// behind, device() (the current one, negative on error), and total() and
// available(), the current device's memory and what is free of it, in bytes.
#pragma once
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
  // holds it, at most twice its size.  The cache keeps 4 GiB, and large device
  // blocks beside them for as long as someone works with such blocks (see
  // large_user).  A failed allocation empties the cache and tries again.  Null
  // if that fails too; either way no error is left for the next check of the
  // runtime's last error, which may follow any launch.
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
      if (!b.large) small_bytes -= b.bytes;
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
    live.push_back({p, bytes, dev, host, false});
    return p;
  }

  void put(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lk(mu);
    for (size_t i = 0; i < live.size(); ++i)
      if (live[i].p == p) {
        Block b = live[i];
        live.erase(live.begin() + (long)i);
        b.large = keep_large_locked(b);
        if (b.large || small_bytes + b.bytes <= kMost) {
          kept.push_back(b);
          if (!b.large) small_bytes += b.bytes;
        } else {
          (void)mem.free(b.p, b.host);
        }
        return;
      }
  }

  // Frees every cached block; returns their bytes.
  size_t trim() {
    std::lock_guard<std::mutex> lk(mu);
    return trim_locked();
  }

  // Someone who works in large device blocks call after call comes (+1) or
  // goes (-1).  Meanwhile device blocks above 256 MiB are kept beside the
  // others, up to an eighth of their device, and only while half of it is
  // free, so that neither another process nor another allocator in this one
  // finds the device full of cached blocks.  They go with the last such user.
  // Why: the driver clears an allocation before it hands it out ((H2O)16/6-31G*
  // MP2, 22 GB: 0.5 s a call, where the transform takes 0.05 s).
  void large_user(int d) {
    std::lock_guard<std::mutex> lk(mu);
    users += d;
    if (users > 0) return;
    for (size_t i = kept.size(); i-- > 0;)
      if (kept[i].large) {
        (void)mem.free(kept[i].p, false);
        kept.erase(kept.begin() + (long)i);
      }
  }

  // Cached bytes of a device: what a request finds beside its free memory.
  size_t cached(int device) {
    std::lock_guard<std::mutex> lk(mu);
    return bytes_locked([&](const Block& k) { return !k.host && k.device == device; });
  }

 private:
  struct Block { void* p; size_t bytes; int device; bool host, large; };
  static constexpr size_t kMost = size_t(4) << 30, kLarge = size_t(256) << 20;

  template <class F>
  size_t bytes_locked(F&& f) const {
    size_t n = 0;
    for (const Block& k : kept)
      if (f(k)) n += k.bytes;
    return n;
  }
  bool keep_large_locked(const Block& b) {
    if (users <= 0 || b.host || b.bytes <= kLarge || mem.device() != b.device) return false;
    const size_t total = mem.total(), have = bytes_locked([&](const Block& k) { return k.large && k.device == b.device; });
    return have + b.bytes <= total / 8 && mem.available() >= total / 2;
  }
  size_t trim_locked() {
    const size_t n = bytes_locked([](const Block&) { return true; });
    for (const Block& b : kept) (void)mem.free(b.p, b.host);
    kept.clear();
    small_bytes = 0;
    return n;
  }

  Mem mem;
  std::mutex mu;
  std::vector<Block> kept;  // cached, free
  std::vector<Block> live;  // handed out
  size_t small_bytes = 0;   // of the kept blocks that are not large
  int users = 0;
};
