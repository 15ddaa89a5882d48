// The rules of the kept device memory (csrc/idle_blocks.hpp) against a made-up runtime of two devices: every
// call is recorded, waits and allocations fail on demand.  Prints "ok" and returns 0, or names the line.
#include "idle_blocks.hpp"

#include <stdint.h>
#include <stdio.h>

#include <string>

namespace {
int g_device = 0, g_fail_wait = -1, g_allocations_that_fail = 0;
uintptr_t g_next = 4096;
std::string g_log;

struct Api {
  using Error = int;
  static constexpr int kSuccess = 0;
  static int current_device(int *d) {
    *d = g_device;
    return 0;
  }
  static int wait_for_device(int d) {
    g_log += "w" + std::to_string(d) + " ";
    return d == g_fail_wait ? 7 : 0;
  }
  static int allocate(void **p, size_t bytes) {
    g_log += "a" + std::to_string(bytes) + " ";
    if (g_allocations_that_fail > 0) {
      --g_allocations_that_fail;
      return 2;
    }
    *p = reinterpret_cast<void *>(g_next += 4096);
    return 0;
  }
  static int release(void *) {
    g_log += "f ";
    return 0;
  }
  static bool out_of_memory(int e) { return e == 2; }
  static void clear_error() { g_log += "c "; }
};
using Pool = nts::IdleBlocks<Api>;
using nts::BlockRef;

std::string take_log() {
  std::string s;
  s.swap(g_log);
  return s;
}

#define CHECK(cond)                                  \
  do {                                               \
    if (!(cond)) {                                   \
      printf("line %d: %s\n", __LINE__, #cond);      \
      return 1;                                      \
    }                                                \
  } while (0)

// A schedule of device 0 is dropped while device 1 is current: device 0 is waited for, once for its two blocks.
int waits_for_the_blocks_own_device() {
  Pool pool(1 << 20, 8);
  BlockRef a, b, c;
  g_device = 0;
  CHECK(pool.take(100, a) == 0 && pool.take(200, b) == 0);
  g_device = 1;
  CHECK(pool.take(300, c) == 0);
  take_log();
  BlockRef *both[] = {&a, &b};
  CHECK(pool.retire(both, 2) == 0);
  CHECK(take_log() == "w0 ");
  CHECK(!a.ptr && !b.ptr);
  BlockRef *all[] = {&c};
  CHECK(pool.retire(all, 1) == 0 && take_log() == "w1 ");
  CHECK(pool.take(100, a) == 0 && take_log() == "a100 ");  // device 0's block is not for device 1
  g_device = 0;
  CHECK(pool.take(100, b) == 0 && take_log() == "");       // and is for device 0
  return 0;
}

// The wait fails (the thread captures a graph, an earlier error stands): the driver gets the block, nobody else.
int a_block_whose_wait_failed_is_not_handed_on() {
  Pool pool(1 << 20, 8);
  BlockRef a, b;
  g_device = 0;
  CHECK(pool.take(100, a) == 0);
  take_log();
  g_fail_wait = 0;
  BlockRef *one[] = {&a};
  CHECK(pool.retire(one, 1) == 7);
  g_fail_wait = -1;
  CHECK(take_log() == "w0 c f " && !a.ptr);
  CHECK(pool.take(100, b) == 0 && take_log() == "a100 ");
  CHECK(pool.give(b, false) == 0 && take_log() == "f ");
  CHECK(pool.take(100, a) == 0 && take_log() == "a100 ");
  return 0;
}

int sizes_and_bounds() {
  Pool pool(1000, 2);
  BlockRef a, b, c;
  g_device = 0;
  CHECK(pool.take(0, a) == 0 && !a.ptr && take_log() == "");
  CHECK(pool.take(300, a) == 0 && pool.take(300, b) == 0 && pool.take(900, c) == 0);
  take_log();
  CHECK(pool.give(a, true) == 0 && take_log() == "");
  CHECK(pool.take(199, b) == 0 && take_log() == "a199 ");   // 300 is more than half above 199
  CHECK(pool.take(200, b) == 0 && take_log() == "" && b.bytes == 300);
  CHECK(pool.give(b, true) == 0 && pool.give(c, true) == 0);  // 1,200 bytes: the one that has lain longer goes
  CHECK(take_log() == "f " && pool.held(0) == 900 && pool.held(1) == 0);
  CHECK(pool.take(100, a) == 0 && pool.take(100, b) == 0 && take_log() == "a100 a100 ");
  CHECK(pool.give(a, true) == 0 && take_log() == "" && pool.held(0) == 1000);
  CHECK(pool.give(b, true) == 0 && take_log() == "f " && pool.held(0) == 200);  // three blocks: the oldest, not the smallest
  CHECK(pool.trim(1) == 0 && take_log() == "");
  CHECK(pool.trim(0) == 0 && take_log() == "f f " && pool.held(0) == 0);
  return 0;
}

int an_allocation_that_fails_gets_the_idle_memory() {
  Pool pool(1 << 20, 8);
  BlockRef a, b;
  g_device = 0;
  CHECK(pool.take(100, a) == 0 && pool.give(a, true) == 0);
  take_log();
  g_allocations_that_fail = 1;
  CHECK(pool.take(5000, b) == 0 && take_log() == "a5000 c f a5000 ");
  CHECK(pool.give(b, true) == 0);
  g_allocations_that_fail = 2;
  CHECK(pool.take(6000, a) == 2 && !a.ptr);
  take_log();
  g_allocations_that_fail = 1;
  CHECK(pool.take(6000, a) == 2 && take_log() == "a6000 ");  // nothing idle: not tried again
  return 0;
}

// Scratch and the allocations of the C interface, which do not come from the list.
int other_allocations_get_the_idle_memory() {
  Pool pool(1 << 20, 8);
  BlockRef a;
  void *p = nullptr;
  auto other = [&] { return Api::allocate(&p, 77); };
  g_device = 0;
  CHECK(pool.take(100, a) == 0 && pool.give(a, true) == 0);
  take_log();
  CHECK(pool.with_idle_memory(other) == 0 && take_log() == "a77 " && pool.held(0) == 100);
  g_device = 1;  // the other device's idle memory would not help
  g_allocations_that_fail = 1;
  CHECK(pool.with_idle_memory(other) == 2 && take_log() == "a77 " && pool.held(0) == 100);
  g_device = 0;
  g_allocations_that_fail = 1;
  CHECK(pool.with_idle_memory(other) == 0 && take_log() == "a77 c f a77 " && pool.held(0) == 0);
  g_allocations_that_fail = 1;
  CHECK(pool.with_idle_memory(other) == 2 && take_log() == "a77 ");
  return 0;
}
}  // namespace

int main() {
  if (waits_for_the_blocks_own_device() || a_block_whose_wait_failed_is_not_handed_on() || sizes_and_bounds() ||
      an_allocation_that_fails_gets_the_idle_memory() || other_allocations_get_the_idle_memory())
    return 1;
  printf("ok\n");
  return 0;
}
