// The rules of a schedule's scratch (csrc/plan_scratch.hpp) on a made-up device of `g_free` bytes that counts what is asked of
// it.  Prints "ok" and returns 0, or names the line.
#include "plan_scratch.hpp"

#include <stdio.h>

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
}  // namespace

int main() {
  if (a_widths_partial_sums_stay_where_a_capture_found_them()) return 1;
  printf("ok\n");
  return 0;
}
