// The rules of a schedule's scratch (csrc/plan_scratch.hpp) on a made-up device of `g_free` bytes that counts what is asked of
// it.  Prints "ok" and returns 0, or names the line.
#include "plan_scratch.hpp"

#include <stdio.h>

#include <utility>

namespace {
size_t g_free = 0;
int g_asked = 0, g_refused = 0, g_retired = 0;
uintptr_t g_next = 4096;

struct Memory {
  using Error = int;
  static constexpr int kSuccess = 0;
  struct Block {
    void *ptr = nullptr;
    size_t bytes = 0;
    void swap(Block &o) { std::swap(*this, o); }
    int take(size_t want) {
      if (want == 0) return 0;
      ++g_asked;
      if (want > g_free) {
        ++g_refused;
        return 2;
      }
      g_free -= want;
      bytes = want;
      ptr = reinterpret_cast<void *>(g_next += 4096);
      return 0;
    }
  };
  static int retire(Block &b) {
    if (b.ptr) ++g_retired;
    g_free += b.bytes;
    b = Block();
    return 0;
  }
  static bool out_of_memory(int e) { return e == 2; }
  static void clear_error() {}
};
using Scratch = nts::PlanScratch<Memory>;
constexpr size_t kSlots = 10, kRows = 100;
constexpr bool kCopy = true, kNoCopy = false, kRecorded = true, kEager = false;

// A call of F floats: 257 to 768 floats off whole lines have a copy.
nts::ScratchNeed need(size_t F) {
  const size_t padded = (F + 31) / 32 * 32;
  return {kSlots, F, F > 256 && F <= 768 && F != padded ? padded : 0, kRows};
}
void fresh(size_t floats) {
  g_free = floats * 4;
  g_asked = g_refused = g_retired = 0;
}

#define CHECK(cond)                                  \
  do {                                               \
    if (!(cond)) {                                   \
      printf("line %d: %s\n", __LINE__, #cond);      \
      return 1;                                      \
    }                                                \
  } while (0)

// A graph holds the address of its partial sums: an ordinary call of the same width must not move them.
int a_widths_partial_sums_stay_where_a_capture_found_them() {
  size_t ld = 9;
  {  // heads first: no copy; then the capture, then a call that takes the copy
    fresh(1 << 20);
    Scratch s;
    CHECK(s.place(need(300), kNoCopy, kEager, &ld) == 0 && ld == 0 && !s.copy());
    const float *at = s.partial();
    CHECK(s.place(need(300), kCopy, kRecorded, &ld) == 0 && ld == 0 && s.partial() == at && !s.copy());
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320 && s.partial() == at && s.copy());
    CHECK(g_retired == 0 && g_asked == 2);
  }
  {  // room from a width of whole lines
    fresh(1 << 20);
    Scratch s;
    CHECK(s.place(need(320), kCopy, kEager, &ld) == 0 && ld == 0);
    const float *at = s.partial();
    CHECK(s.place(need(300), kCopy, kRecorded, &ld) == 0 && ld == 0);
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320 && s.partial() == at);
  }
  {  // enough for the sums, too few for those beside a copy: what a capture found stays, also for the other calls
    fresh(1 << 20);
    Scratch s;
    const nts::ScratchNeed plain{kSlots, 304, 0, kRows};
    CHECK(s.place(plain, kNoCopy, kEager, &ld) == 0);
    const float *at = s.partial();
    CHECK(s.place(need(300), kNoCopy, kRecorded, &ld) == 0 && ld == 0 && s.partial() == at);
    for (int i = 0; i < 3; ++i) CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && s.partial() == at);
    for (size_t F = 257; F <= 304; ++F) CHECK(s.place(need(F), kCopy, kEager, &ld) == 0 && s.partial() == at);
    CHECK(g_retired == 0);
  }
  {  // a capture of a width without a copy, then narrower calls with one
    fresh(1 << 20);
    Scratch s;
    const nts::ScratchNeed plain{kSlots, 300, 0, kRows}, narrower{kSlots, 299, 320, kRows};
    CHECK(s.place(plain, kCopy, kEager, &ld) == 0);
    const float *at = s.partial();
    CHECK(s.place(plain, kCopy, kRecorded, &ld) == 0 && s.place(narrower, kCopy, kEager, &ld) == 0 && s.partial() == at);
    CHECK(s.place(need(500), kCopy, kEager, &ld) == 0 && ld == 512 && s.partial() != at);  // a greater width moves them
    CHECK(s.place(narrower, kCopy, kEager, &ld) == 0 && ld == 320);
  }
  {  // without a capture they move once and the copy is made
    fresh(1 << 20);
    Scratch s;
    const nts::ScratchNeed plain{kSlots, 304, 0, kRows};
    CHECK(s.place(plain, kNoCopy, kEager, &ld) == 0 && s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320);
  }
  return 0;
}

// Memory that was not there is asked for once, and what there is stays.
int a_refusal_is_remembered() {
  size_t ld = 9;
  {  // no room for the copy: one attempt for any number of calls, one more for a reservation
    fresh(kSlots * 320 + kRows * 320 - 1);
    Scratch s;
    for (int i = 0; i < 4; ++i) CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && s.partial() && !s.copy());
    CHECK(g_asked == 2 && g_refused == 1 && g_retired == 0 && s.stride_of(need(300)) == 0);
    g_free += 1;
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && g_asked == 2);
    s.ask_again();
    CHECK(s.stride_of(need(300)) == 320 && s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && g_refused == 2);  // (3 bytes short)
    g_free += 4;
    s.ask_again();
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320 && s.copy() && s.stride_of(need(300)) == 320);
  }
  {  // a wider copy that does not fit leaves the narrower one; narrower ones than refused are still had
    fresh(kSlots * 640 + kRows * 320 + kRows * 500);
    Scratch s;
    CHECK(s.place(need(640), kCopy, kEager, &ld) == 0 && ld == 0);
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320);
    const float *at = s.copy();
    for (int i = 0; i < 3; ++i) CHECK(s.place(need(602), kCopy, kEager, &ld) == 0 && ld == 0 && s.copy() == at);
    CHECK(g_refused == 1 && g_retired == 0);
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320 && s.copy() == at && g_refused == 1);
    CHECK(s.place(need(420), kCopy, kEager, &ld) == 0 && ld == 448 && g_refused == 1 && g_retired == 1);
  }
  {  // the partial sums of a wider call need the memory that the copy has
    fresh(kSlots * 320 + kRows * 320 + kSlots * 320);
    Scratch s;
    const nts::ScratchNeed wider{kSlots, 1000, 0, kRows};
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 320);
    CHECK(s.place(wider, kCopy, kEager, &ld) == 0 && ld == 0 && !s.copy() && s.partial());
    const int asked = g_asked;
    for (int i = 0; i < 3; ++i) CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && s.place(wider, kCopy, kEager, &ld) == 0);
    CHECK(g_asked == asked);  // (the copy's size is known to be too much)
  }
  {  // room for the sums as they are and not for those beside a copy
    fresh(kSlots * 300);
    Scratch s;
    for (int i = 0; i < 3; ++i) CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && s.partial());
    CHECK(g_asked == 2 && g_refused == 1 && g_retired == 0 && s.stride_of(need(300)) == 0);
  }
  {  // none for these either: an error, each time
    fresh(kSlots * 300 - 1);
    Scratch s;
    for (int i = 0; i < 2; ++i) CHECK(s.place(need(300), kCopy, kEager, &ld) == 2 && ld == 0 && !s.partial());
    g_free += 4;
    CHECK(s.place(need(300), kCopy, kEager, &ld) == 0 && ld == 0 && s.partial());
  }
  return 0;
}
}  // namespace

int main() {
  if (a_widths_partial_sums_stay_where_a_capture_found_them() || a_refusal_is_remembered()) return 1;
  printf("ok\n");
  return 0;
}
