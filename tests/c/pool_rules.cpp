// The rules of the device memory pool (device_memory.hpp) over a fake HIP runtime.
#include "device_memory.hpp"

#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>

using namespace cuvs::detail;

#define REQUIRE(x)                                                   \
  if (!(x)) {                                                        \
    std::printf("line %d: %s\n", __LINE__, #x);                      \
    std::exit(1);                                                    \
  }

constexpr size_t MiB = size_t(1) << 20, GiB = size_t(1) << 30;

struct buffer {
  void* p;
  size_t capacity;
  int device;
  explicit buffer(size_t n) : p(device_allocate(n, &capacity, &device)) {}
  void release() { device_release(p, capacity, device); }
};

int main()
{
  // a released block serves the next request of its size, and one of three quarters of it
  buffer a(200 * MiB);
  a.release();
  REQUIRE(fake_used == 200 * MiB);
  buffer b(160 * MiB);
  REQUIRE(b.p == a.p && b.capacity == 200 * MiB && fake_mallocs == 1);
  buffer c(100 * MiB);
  REQUIRE(fake_mallocs == 2);
  b.release();
  buffer d(140 * MiB);  // less than three quarters of 200 MiB
  REQUIRE(fake_mallocs == 3 && d.p != a.p);
  c.release();
  d.release();
  REQUIRE(fake_used == 440 * MiB);
  device_trim(0);
  REQUIRE(fake_used == 0 && fake_blocks.empty());
  // at most kPoolBytes stay, the newest ones; a larger block never does
  buffer large(kPoolBytes + GiB);
  large.release();
  REQUIRE(fake_used == 0);
  buffer x(2 * GiB), y(2 * GiB), z(1 * GiB);
  x.release();
  y.release();
  z.release();
  REQUIRE(fake_used == 3 * GiB && fake_blocks.count(x.p) == 0);
  // an allocation that the device refuses empties the pool first
  fake_foreign = fake_total - fake_used;
  buffer w(512 * MiB);
  REQUIRE(w.p != nullptr && fake_used == 512 * MiB);
  // on a device short of memory (less than a sixteenth free) nothing stays, also of what came in before
  fake_foreign = 0;
  w.release();
  buffer s(256 * MiB), t(256 * MiB);
  s.release();
  REQUIRE(fake_used == GiB);
  std::this_thread::sleep_for(std::chrono::milliseconds(2));
  fake_foreign = fake_total - fake_used - fake_total / 16 + 1;
  t.release();
  REQUIRE(fake_used == 0);
  // and every release asks again until there is memory
  fake_foreign = fake_total - fake_total / 16;
  buffer u(16 * MiB), u2(16 * MiB);
  u.release();
  u2.release();
  REQUIRE(fake_used == 0);
  fake_foreign = 0;
  buffer v(16 * MiB);
  v.release();
  REQUIRE(fake_used == 16 * MiB);
  // blocks released under a device_idle enter without a wait each
  device_trim(0);
  buffer m(1 * MiB), n(1 * MiB);
  fake_syncs = 0;
  {
    device_idle idle;
    idle.enter(0);
    m.release();
    n.release();
  }
  REQUIRE(fake_syncs == 1 && fake_used == 4 * MiB);
  std::puts("ok");
  return 0;
}
