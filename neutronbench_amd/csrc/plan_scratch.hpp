// The scratch of a schedule: the partial sums of its cut rows and, for some widths, a copy of the input with padded rows.
// Host logic only: `Memory` says where blocks come from, so that the rules below are tested without a device.
//   Error (kSuccess)
//   Block        .ptr, .bytes, Error take(size_t bytes); holds nothing at first, gives its memory back at the end
//   Error retire(Block &)    gives a block back after the work that uses it
//   bool out_of_memory(Error)         void clear_error()
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace nts {

// What a call needs: `slots` partial rows of F floats, of `padded` floats where it gathers from a copy of `copy_rows` rows of
// that many (padded 0: its width takes no copy).
struct ScratchNeed {
  size_t slots, F, padded, copy_rows;
};

template <class Memory>
class PlanScratch {
 public:
  using Error = typename Memory::Error;
  using Block = typename Memory::Block;

  float *partial() const { return static_cast<float *>(partial_.ptr); }
  float *copy() const { return static_cast<float *>(copy_.ptr); }
  Block *partial_block() { return &partial_; }
  Block *copy_block() { return &copy_; }

  // Makes room for a call and leaves the stride of its rows in *stride: `padded`, or 0 where the call does not gather from the
  // copy (it does not want one, there is no memory for it, or the call is `recorded` by a capture and no room was made before).
  // A recorded call keeps the address of its partial sums, so a width's partial rows are placed once, as wide as a copy would make them, whichever
  // of its calls comes first; and what a recorded call found stays for all calls that it is enough for.
  Error place(const ScratchNeed &need, bool want_copy, bool recorded, size_t *stride) {
    *stride = 0;
    const size_t least = need.slots * need.F * sizeof(float);
    const size_t wide = need.padded ? need.slots * need.padded * sizeof(float) : least;
    if (partial_.bytes < least || (partial_.bytes < wide && !recorded && !recorded_)) {
      recorded_ = false;
      Error err = grow(partial_, wide);
      if (err != Memory::kSuccess && wide > least) {
        Memory::clear_error();
        err = grow(copy_, 0);  // the copy has taken the memory that the partial sums need more
        if (err == Memory::kSuccess) err = grow(partial_, least);
      }
      if (err != Memory::kSuccess) return err;
    }
    recorded_ = recorded_ || recorded;
    if (!want_copy || !need.padded || partial_.bytes < wide) return Memory::kSuccess;
    const size_t bytes = need.copy_rows * need.padded * sizeof(float);
    if (copy_.bytes < bytes) {
      if (recorded) return Memory::kSuccess;
      if (grow(copy_, bytes) != Memory::kSuccess) {
        Memory::clear_error();
        return Memory::kSuccess;
      }
    }
    *stride = need.padded;
    return Memory::kSuccess;
  }

 private:
  // A buffer that grows may still be read by work queued earlier, on any stream.
  static Error grow(Block &block, size_t bytes) {
    const Error err = Memory::retire(block);
    return err != Memory::kSuccess ? err : block.take(bytes);
  }

  Block partial_, copy_;
  bool recorded_ = false;  // a capture holds the address of the partial sums
};

}  // namespace nts
