#include "device_memory.hpp"

#include <hip/hip_runtime.h>

#include <chrono>
#include <map>
#include <mutex>
#include <new>
#include <unordered_map>

namespace cuvs::detail {

namespace {

struct block {
  void* p;
  unsigned long long age;  // the pool's count when it came in
};
struct pool {
  std::multimap<size_t, block> blocks;
  size_t held             = 0;
  size_t unchecked        = 0;  // bytes that came in since the device's free memory was asked for
  std::chrono::steady_clock::time_point checked{};
  unsigned long long ages = 0;
};

std::mutex g_mutex;
/** Never destroyed: at the process's end the driver takes the memory back. */
auto pools() -> std::unordered_map<int, pool>&
{
  static auto* p = new std::unordered_map<int, pool>();
  return *p;
}

/** The device that a device_idle of this thread covers (-1: none). */
thread_local int t_idle = -1;

/** hipSetDevice(device) for a scope, when it is not the current one. */
struct on_device {
  int before = -1;
  explicit on_device(int device)
  {
    int now = -1;
    if (hipGetDevice(&now) == hipSuccess && now != device && hipSetDevice(device) == hipSuccess) { before = now; }
  }
  ~on_device()
  {
    if (before >= 0) { (void)hipSetDevice(before); }
  }
};

/** Sizes that allocations are rounded up to: 2 MiB pages from 1 MiB on, else 4 KiB. */
auto rounded(size_t bytes) -> size_t
{
  const size_t unit = bytes >= (size_t(1) << 20) ? size_t(2) << 20 : size_t(4) << 10;
  return (bytes + unit - 1) / unit * unit;
}

/** Whether a block of `capacity` may enter the pool of the current device, `device`: its free memory
 *  is asked for once kPoolCheckBytes came in, at most once in a millisecond (it takes 5 us, and an index
 *  of 250,000 x 960 bytes built, searched and dropped 370). */
auto has_room(size_t capacity, int device) -> bool
{
  const auto now = std::chrono::steady_clock::now();
  {
    std::lock_guard lk(g_mutex);
    pool& q = pools()[device];
    q.unchecked += capacity;
    if (q.unchecked < kPoolCheckBytes || now - q.checked < std::chrono::milliseconds(1)) { return true; }
  }
  size_t free = 0, total = 0;
  if (hipMemGetInfo(&free, &total) != hipSuccess || free < total / 16) { return false; }  // and asks again next time
  std::lock_guard lk(g_mutex);
  pools()[device].unchecked = 0;
  pools()[device].checked   = now;
  return true;
}

}  // namespace

void* device_allocate(size_t bytes, size_t* capacity, int* device)
{
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { return nullptr; }
  const size_t n = rounded(bytes);
  {
    std::lock_guard lk(g_mutex);
    pool& p = pools()[dev];
    auto it = p.blocks.lower_bound(n);
    if (it != p.blocks.end() && it->first - it->first / 4 <= n) {
      void* ptr = it->second.p;
      *capacity = it->first;
      *device   = dev;
      p.held -= it->first;
      p.blocks.erase(it);
      return ptr;
    }
  }
  void* ptr = nullptr;
  if (hipMalloc(&ptr, n) != hipSuccess) {
    (void)hipGetLastError();
    device_trim(dev);
    if (hipMalloc(&ptr, n) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  *capacity = n;
  *device   = dev;
  return ptr;
}

void device_release(void* p, size_t capacity, int device) noexcept
{
  if (p == nullptr) { return; }
  on_device at(device);
  bool keep = capacity <= kPoolBytes && (t_idle == device || hipDeviceSynchronize() == hipSuccess);
  try {
    if (keep && !has_room(capacity, device)) {
      keep = false;
      device_trim(device);
    }
  } catch (std::bad_alloc const&) {
    keep = false;
  }
  if (keep) {
    // the newest block stays, the oldest ones make room: what was freed last is what a program
    // that builds and drops alike indexes asks for next
    while (true) {
      void* oldest = nullptr;
      try {
        std::lock_guard lk(g_mutex);
        pool& q = pools()[device];
        if (q.held + capacity <= kPoolBytes) {
          q.blocks.emplace(capacity, block{p, q.ages++});
          q.held += capacity;
          return;
        }
        auto it = q.blocks.begin();
        for (auto b = q.blocks.begin(); b != q.blocks.end(); ++b) {
          if (b->second.age < it->second.age) { it = b; }
        }
        oldest = it->second.p;
        q.held -= it->first;
        q.blocks.erase(it);
      } catch (std::bad_alloc const&) {  // no host memory for the entry: the block goes back
        break;
      }
      (void)hipFree(oldest);
    }
  }
  (void)hipGetLastError();
  (void)hipFree(p);
}

void device_trim(int device) noexcept
{
  std::multimap<size_t, block> blocks;
  {
    std::lock_guard lk(g_mutex);
    pool& p = pools()[device];
    blocks.swap(p.blocks);
    p.held = 0;
  }
  on_device at(device);
  for (auto const& b : blocks) { (void)hipFree(b.second.p); }
}

void device_idle::enter(int device) noexcept
{
  on_device at(device);
  if (entered_ || hipDeviceSynchronize() != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  outer_   = t_idle;
  t_idle   = device;
  entered_ = true;
}

device_idle::~device_idle()
{
  if (entered_) { t_idle = outer_; }
}

}  // namespace cuvs::detail
