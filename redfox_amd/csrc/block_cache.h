// block_cache.h - device blocks that rfx_free keeps for rfx_malloc: a text
// load allocates and frees a column per field, each call of the runtime's
// allocator 10 to 40 us (a million-row text load with 9 columns: 720 -> 500
// us, with the passes over the text).
//
// A block is kept only once the device is idle, as hipFree waits too: no
// queued work of any stream or thread can still touch it, so it may be
// handed to any of them.  Blocks of up to kKeepBlock bytes, kKeepTotal in
// all; they go back to the runtime when an allocation fails (any of the
// library's: alloc) and when the last context is destroyed.  Other pointers, other devices' blocks and frees
// while a graph is being captured (no waiting then) go straight to the
// runtime.
//
// Rt is the runtime's side, so that the rules can be checked on a host
// without a device:
//   bool alloc(void** p, uint64_t bytes), void release(void* p);
//   int device()            the current device, negative if unknown
//   bool idle()             waits for the device; false if it could not
//   uint64_t extent(void*)  bytes of the allocation that starts there, or 0
//   bool capturing()        some context is between graph_begin and graph_end
#pragma once

#include <cstdint>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace rfx {

template <class Rt>
class BlockCache {
 public:
  static constexpr uint64_t kKeepBlock = 64ull << 20, kKeepTotal = 512ull << 20;
  enum Given { kKept, kCallerFrees, kFreedBefore };

  explicit BlockCache(Rt rt = Rt()) : rt_(rt) {}

  bool take(void** ptr, uint64_t bytes) {
    const uint64_t size = rounded(bytes);
    const int dev = rt_.device();
    if (dev < 0) return false;
    if (size <= kKeepBlock) {
      std::lock_guard<std::mutex> hold(mu_);
      auto it = free_.find({dev, size});
      if (it != free_.end()) {
        *ptr = it->second.back();
        it->second.pop_back();
        if (it->second.empty()) free_.erase(it);
        kept_ -= size;
        blocks_[*ptr].kept = false;
        return true;
      }
    }
    if (!rt_.alloc(ptr, size)) {
      if (!alloc(ptr, bytes)) return false;
      std::lock_guard<std::mutex> hold(mu_);
      blocks_.erase(*ptr);  // of its own size: not kept when freed
      return true;
    }
    std::lock_guard<std::mutex> hold(mu_);
    if (size <= kKeepBlock) blocks_[*ptr] = {dev, size, false};
    else blocks_.erase(*ptr);
    return true;
  }

  // Memory of the caller's own, which the caller releases: the kept blocks
  // make room for it.  (Not while capturing: hipFree waits.)
  bool alloc(void** ptr, uint64_t bytes) {
    if (rt_.alloc(ptr, bytes)) return true;
    return !rt_.capturing() && drop() && rt_.alloc(ptr, bytes);
  }

  // kFreedBefore: the block is kept already, so this is its second free.
  // The block that it is stays kept, and the caller must not free it.
  Given give(void* ptr) {
    Block b;
    {
      std::lock_guard<std::mutex> hold(mu_);
      auto it = blocks_.find(ptr);
      if (it == blocks_.end()) return kCallerFrees;
      if (it->second.kept) return kFreedBefore;
      if (kept_ + it->second.size > kKeepTotal) {  // no room: no need to wait
        blocks_.erase(it);
        return kCallerFrees;
      }
      // Marked before the wait below: of two threads that free it, one does.
      it->second.kept = true;
      b = it->second;
    }
    // A block of another extent is not the one that was handed out (the
    // runtime freed that one and gave its address to somebody else).
    const bool keep = !rt_.capturing() && rt_.device() == b.dev && rt_.extent(ptr) == b.size &&
                      rt_.idle();
    std::lock_guard<std::mutex> hold(mu_);
    if (!keep || kept_ + b.size > kKeepTotal) {
      blocks_.erase(ptr);
      return kCallerFrees;
    }
    free_[{b.dev, b.size}].push_back(ptr);
    kept_ += b.size;
    return kKept;
  }

  // Contexts come and go while others work (a server makes one per slot), so
  // the blocks stay until none is left: giving them back waits for the device
  // block by block.
  void context_made() {
    std::lock_guard<std::mutex> hold(mu_);
    ++contexts_;
  }
  void context_gone() {
    {
      std::lock_guard<std::mutex> hold(mu_);
      if (--contexts_) return;
    }
    drop();
  }

  // Bytes kept on a device.
  uint64_t kept(int dev) {
    std::lock_guard<std::mutex> hold(mu_);
    uint64_t sum = 0;
    for (auto& f : free_)
      if (f.first.first == dev) sum += f.first.second * f.second.size();
    return sum;
  }

  // Gives every kept block back to the runtime; false if there was none.
  bool drop() {
    std::vector<void*> all;
    {
      std::lock_guard<std::mutex> hold(mu_);
      for (auto& f : free_) {
        for (void* p : f.second) {
          blocks_.erase(p);
          all.push_back(p);
        }
      }
      free_.clear();
      kept_ = 0;
    }
    for (void* p : all) rt_.release(p);
    return !all.empty();
  }

 private:
  struct Block {
    int dev = 0;
    uint64_t size = 0;
    bool kept = false;  // in free_, or on its way there
  };
  // Steps of an eighth of the size below, so that a block that held nearly
  // as much is found again; sizes that are not kept stay as they are.
  static uint64_t rounded(uint64_t bytes) {
    if (bytes > kKeepBlock) return bytes;
    uint64_t step = 256;
    while (step * 16 < bytes) step *= 2;
    return (bytes + step - 1) / step * step;
  }
  Rt rt_;
  std::mutex mu_;
  std::map<std::pair<int, uint64_t>, std::vector<void*>> free_;  // by device and size
  std::map<void*, Block> blocks_;                                // handed out or kept
  uint64_t kept_ = 0;
  int64_t contexts_ = 0;
};

}  // namespace rfx
