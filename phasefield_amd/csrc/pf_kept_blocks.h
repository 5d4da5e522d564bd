// pf_kept_blocks.h — device memory that handles keep from one adjoint run to the next, and its way
// back when something else needs it.
#pragma once
#include <cstddef>
#include <mutex>
#include <vector>

namespace pfamd {

// At most one block per owner.  A block is in use from `take` to `done` and idle otherwise; an idle one
// is freed when its owner takes a larger one or is dropped, and by `release`, which the library's
// allocations call before they report a full device.  Safe with owners on several threads.
// Mem: `static void *alloc(size_t)` on the current device (null: out of memory), `static void free(void *)`.
template <class Mem> class KeptBlocks {
 public:
  // a block of at least `bytes` on the current device, which is `device`; null: out of memory
  void *take(const void *owner, int device, size_t bytes) {
    std::lock_guard<std::mutex> lock(mutex_);
    for (size_t q = 0; q < blocks_.size(); ++q)
      if (blocks_[q].owner == owner) {
        if (blocks_[q].bytes >= bytes) {
          blocks_[q].in_use = true;
          return blocks_[q].ptr;
        }
        remove(q);
        break;
      }
    void *p = Mem::alloc(bytes);
    if (!p && release_locked(device)) p = Mem::alloc(bytes);
    if (p) blocks_.push_back({owner, device, p, bytes, true});
    return p;
  }
  // the owner's work on its block has ended; a block of more than `most` bytes is not kept
  void done(const void *owner, size_t most) {
    std::lock_guard<std::mutex> lock(mutex_);
    for (size_t q = 0; q < blocks_.size(); ++q)
      if (blocks_[q].owner == owner) {
        blocks_[q].in_use = false;
        if (blocks_[q].bytes > most) remove(q);
        return;
      }
  }
  // give the owner's block back (not one in use, but for an owner that ends)
  void drop(const void *owner, bool ends) {
    std::lock_guard<std::mutex> lock(mutex_);
    for (size_t q = 0; q < blocks_.size(); ++q)
      if (blocks_[q].owner == owner) {
        if (ends || !blocks_[q].in_use) remove(q);
        return;
      }
  }
  // bytes of the idle blocks on `device`, which `take` and `release` can free
  size_t idle(int device) {
    std::lock_guard<std::mutex> lock(mutex_);
    size_t n = 0;
    for (const Block &b : blocks_)
      if (b.device == device && !b.in_use) n += b.bytes;
    return n;
  }
  // free the idle blocks on `device`; whether there was one
  bool release(int device) {
    std::lock_guard<std::mutex> lock(mutex_);
    return release_locked(device);
  }

 private:
  struct Block {
    const void *owner;
    int device;
    void *ptr;
    size_t bytes;
    bool in_use;
  };
  void remove(size_t q) {
    Mem::free(blocks_[q].ptr);
    blocks_.erase(blocks_.begin() + long(q));
  }
  bool release_locked(int device) {
    bool any = false;
    for (size_t q = blocks_.size(); q-- > 0;)
      if (blocks_[q].device == device && !blocks_[q].in_use) {
        remove(q);
        any = true;
      }
    return any;
  }
  std::mutex mutex_;
  std::vector<Block> blocks_;
};

}  // namespace pfamd
