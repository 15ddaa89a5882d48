// The scratch of a schedule: the partial sums of its cut rows and, for some widths, a copy of the input with padded rows.
// Host logic only: `Memory` says where blocks come from, so that the rules below are tested without a device.
//   Error (kSuccess)
//   Block        .ptr, .bytes, Error take(size_t bytes), swap(Block &); holds nothing at first, gives its memory back at the end
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
  // of its calls comes first; and what a recorded call found stays for all calls that it is enough for.  Sizes for which there was
  // no memory are not asked for again (an allocation that fails empties the list of idle blocks) until ask_again().
  Error place(const ScratchNeed &need, bool want_copy, bool recorded, size_t *stride) {
    *stride = 0;
    const size_t least = need.slots * need.F * sizeof(float);
    const size_t wide = need.padded ? need.slots * need.padded * sizeof(float) : least;
    if (partial_.bytes < least || (partial_.bytes < wide && !recorded && !recorded_ && wide < partial_refused_)) {
      recorded_ = false;
      const size_t want = wide < partial_refused_ ? wide : least;
      Error err = Memory::retire(partial_);  // work queued earlier, on any stream, may still use it
      if (err == Memory::kSuccess) err = partial_.take(want);
      if (Memory::out_of_memory(err) && copy_.ptr) {  // the copy has taken the memory that the partial sums need more
        Memory::clear_error();
        if (copy_.bytes < copy_refused_) copy_refused_ = copy_.bytes;
        err = Memory::retire(copy_);
        if (err == Memory::kSuccess) err = partial_.take(want);
      }
      if (Memory::out_of_memory(err) && want > least) {
        Memory::clear_error();
        partial_refused_ = want;
        err = partial_.take(least);
      }
      if (err != Memory::kSuccess) return err;
    }
    recorded_ = recorded_ || recorded;
    if (!want_copy || !need.padded || partial_.bytes < wide) return Memory::kSuccess;
    const size_t bytes = need.copy_rows * need.padded * sizeof(float);
    if (copy_.bytes < bytes) {
      if (recorded || bytes >= copy_refused_) return Memory::kSuccess;
      Block larger;  // the one there is, for narrower rows, goes only when this is had
      Error err = larger.take(bytes);
      if (Memory::out_of_memory(err)) {
        Memory::clear_error();
        copy_refused_ = bytes;
        return Memory::kSuccess;
      }
      if (err == Memory::kSuccess) {
        copy_.swap(larger);
        err = Memory::retire(larger);
      }
      if (err != Memory::kSuccess) return err;
    }
    *stride = need.padded;
    return Memory::kSuccess;
  }

  // The stride that an ordinary call's rows would have as things are.
  size_t stride_of(const ScratchNeed &need) const {
    const size_t least = need.slots * need.F * sizeof(float), wide = need.slots * need.padded * sizeof(float);
    const size_t bytes = need.copy_rows * need.padded * sizeof(float);
    const bool sums = partial_.bytes >= wide || (wide < partial_refused_ && (partial_.bytes < least || !recorded_));
    return need.padded && sums && (copy_.bytes >= bytes || bytes < copy_refused_) ? need.padded : 0;
  }

  void ask_again() { partial_refused_ = copy_refused_ = kNone; }

 private:
  static constexpr size_t kNone = ~static_cast<size_t>(0);

  Block partial_, copy_;
  bool recorded_ = false;  // a capture holds the address of the partial sums
  size_t partial_refused_ = kNone, copy_refused_ = kNone;  // bytes for which there was no memory; as many and more are not asked for
};

}  // namespace nts
