// kept_blocks_main.cpp — CPU check of the kept device blocks (phasefield_amd/csrc/pf_kept_blocks.h) on an
// allocator of limited size.  tests/test_kept_blocks.py builds it with g++ and runs it.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>

#include "../phasefield_amd/csrc/pf_kept_blocks.h"

static std::atomic<long> room{0};

struct Mem {
  static void *alloc(size_t bytes) {
    if ((room -= long(bytes)) < 0) {
      room += long(bytes);
      return nullptr;
    }
    size_t *p = static_cast<size_t *>(std::malloc(bytes + sizeof(size_t)));
    *p = bytes;
    return p + 1;
  }
  static void free(void *q) {
    size_t *p = static_cast<size_t *>(q) - 1;
    room += long(*p);
    std::free(p);
  }
};

#define CHECK(x)                                                  \
  do {                                                            \
    if (!(x)) {                                                   \
      std::fprintf(stderr, "line %d: %s\n", __LINE__, #x);        \
      return 1;                                                   \
    }                                                             \
  } while (0)

int main() {
  pfamd::KeptBlocks<Mem> kept;
  int a, b, c;
  room = 1000;
  // kept between runs, and the same block again when it is large enough
  void *p = kept.take(&a, 0, 600);
  CHECK(p && room == 400 && kept.idle(0) == 0);
  kept.done(&a, 700);
  CHECK(room == 400 && kept.idle(0) == 600 && kept.idle(1) == 0);
  CHECK(kept.take(&a, 0, 500) == p);
  // in use: neither another owner, nor a full device, nor its own release takes it
  CHECK(!kept.take(&b, 0, 500));
  CHECK(!kept.release(0));
  kept.drop(&a, false);
  CHECK(room == 400);
  kept.done(&a, 700);
  // idle: another owner's run that needs it gets it, on the same device only
  CHECK(!kept.take(&b, 1, 500));
  CHECK(room == 400);
  CHECK(kept.take(&b, 0, 500) && room == 500 && kept.idle(0) == 0);
  // too large to keep
  kept.done(&b, 400);
  CHECK(room == 1000);
  // a larger one frees the owner's own first
  CHECK(kept.take(&c, 0, 600));
  kept.done(&c, 1000);
  CHECK(kept.take(&c, 0, 900) && room == 100);
  kept.done(&c, 1000);
  // an allocation elsewhere, its owner, and the owner's end give it back
  CHECK(kept.release(0) && room == 1000 && !kept.release(0));
  CHECK(kept.take(&c, 0, 900));
  kept.done(&c, 1000);
  kept.drop(&c, false);
  CHECK(room == 1000);
  CHECK(kept.take(&c, 0, 900));
  kept.drop(&c, true);
  CHECK(room == 1000);
  // owners on several threads: what a thread holds stays its own
  std::atomic<int> bad{0};
  room = 3000;
  std::thread t[4];
  for (int k = 0; k < 4; ++k)
    t[k] = std::thread([&, k] {
      int owner;
      for (int it = 0; it < 20000; ++it) {
        volatile char *q = static_cast<volatile char *>(kept.take(&owner, 0, size_t(400 + 100 * (it % 4))));
        if (!q) {
          ++bad;
          continue;
        }
        for (int n = 0; n < 400; n += 40) q[n] = char(k);
        for (int n = 0; n < 400; n += 40) bad += q[n] != char(k);
        kept.done(&owner, 650);
        if (it % 7 == 0) kept.release(0);
      }
      kept.drop(&owner, true);
    });
  for (auto &x : t) x.join();
  CHECK(bad == 0 && room == 3000);
  std::printf("kept_blocks_main: ok\n");
  return 0;
}
