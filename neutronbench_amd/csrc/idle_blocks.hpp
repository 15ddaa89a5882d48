// Device memory that is kept between the objects that use it.  Host logic only: `Api` names the runtime
// calls, so that the rules below are tested without a device.
//   Error (kSuccess)
//   Error current_device(int *)       Error wait_for_device(int)    waits for all work queued on that device
//   Error allocate(void **, size_t)   Error release(void *)         release waits for the block's device itself
//   bool out_of_memory(Error)         void clear_error()
#pragma once
#include <stddef.h>

#include <mutex>
#include <utility>
#include <vector>

namespace nts {

struct BlockRef {
  void *ptr = nullptr;
  size_t bytes = 0;
  int device = 0;
};

template <class Api>
class IdleBlocks {
 public:
  using Error = typename Api::Error;

  IdleBlocks(size_t keep_bytes, size_t keep_blocks) : keep_bytes_(keep_bytes), keep_blocks_(keep_blocks) {}

  // An idle block of the current device of want .. want + want / 2 bytes, or a new one.
  Error take(size_t want, BlockRef &block) {
    block = BlockRef();
    if (want == 0) return Api::kSuccess;
    Error err = Api::current_device(&block.device);
    if (err != Api::kSuccess) return err;
    std::lock_guard<std::mutex> lock(mutex_);
    size_t best = idle_.size();
    for (size_t i = 0; i < idle_.size(); ++i)
      if (idle_[i].device == block.device && idle_[i].bytes >= want && idle_[i].bytes - want <= want / 2 &&
          (best == idle_.size() || idle_[i].bytes < idle_[best].bytes))
        best = i;
    if (best < idle_.size()) {
      block = idle_[best];
      idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(best));
      return Api::kSuccess;
    }
    err = Api::allocate(&block.ptr, want);
    if (Api::out_of_memory(err) && idle_bytes(block.device) != 0) {  // what lies idle may be what is missing
      Api::clear_error();
      (void)drop(block.device, 0, 0);
      err = Api::allocate(&block.ptr, want);
    }
    if (err != Api::kSuccess) block.ptr = nullptr;
    else block.bytes = want;
    return err;
  }

  // Gives a block back.  `unused`: the caller has waited, with success, for all work that uses it.  Otherwise it
  // must not reach another taker and goes to the driver, which waits by itself.
  Error give(BlockRef &block, bool unused) {
    if (!block.ptr) return Api::kSuccess;
    const BlockRef b = block;
    block = BlockRef();
    if (!unused) return Api::release(b.ptr);
    std::lock_guard<std::mutex> lock(mutex_);
    idle_.push_back(b);
    return drop(b.device, keep_bytes_, keep_blocks_);
  }

  // Waits once for every device that the blocks lie on (which need not be the current one) and gives them
  // back; the first error is returned.
  Error retire(BlockRef *const *blocks, size_t n) {
    Error first = Api::kSuccess;
    std::vector<std::pair<int, bool>> waited;
    for (size_t i = 0; i < n; ++i) {
      if (!blocks[i]->ptr) continue;
      size_t w = 0;
      while (w < waited.size() && waited[w].first != blocks[i]->device) ++w;
      if (w == waited.size()) {
        const Error err = Api::wait_for_device(blocks[i]->device);
        if (err != Api::kSuccess) {
          Api::clear_error();
          if (first == Api::kSuccess) first = err;
        }
        waited.emplace_back(blocks[i]->device, err == Api::kSuccess);
      }
      const Error given = give(*blocks[i], waited[w].second);
      if (first == Api::kSuccess) first = given;
    }
    return first;
  }

  // An allocation of another kind on the current device: `allocate` is tried again without the idle blocks
  // where it runs out of memory.
  template <class Allocate>
  Error with_idle_memory(Allocate allocate) {
    Error err = allocate();
    int device = 0;
    if (!Api::out_of_memory(err) || Api::current_device(&device) != Api::kSuccess || held(device) == 0) return err;
    Api::clear_error();
    (void)trim(device);
    return allocate();
  }

  // Bytes that lie idle on `device`.
  size_t held(int device) {
    std::lock_guard<std::mutex> lock(mutex_);
    return idle_bytes(device);
  }

  Error trim(int device) {
    std::lock_guard<std::mutex> lock(mutex_);
    return drop(device, 0, 0);
  }

 private:
  size_t idle_bytes(int device) const {
    size_t total = 0;
    for (const BlockRef &b : idle_) total += b.device == device ? b.bytes : 0;
    return total;
  }

  // Frees the idle blocks of `device`, the ones that have lain longest first, until at most `keep_bytes` and
  // `keep_blocks` are left.  A block that the driver refuses to free stays listed.  Caller holds mutex_.
  Error drop(int device, size_t keep_bytes, size_t keep_blocks) {
    while (true) {
      size_t count = 0, oldest = idle_.size();
      for (size_t i = 0; i < idle_.size(); ++i) {
        if (idle_[i].device != device) continue;
        if (count++ == 0) oldest = i;
      }
      if (count == 0 || (idle_bytes(device) <= keep_bytes && count <= keep_blocks)) return Api::kSuccess;
      const Error err = Api::release(idle_[oldest].ptr);
      if (err != Api::kSuccess) return err;
      idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(oldest));
    }
  }

  const size_t keep_bytes_, keep_blocks_;
  std::mutex mutex_;
  std::vector<BlockRef> idle_;  // in the order in which they were given back
};

}  // namespace nts
