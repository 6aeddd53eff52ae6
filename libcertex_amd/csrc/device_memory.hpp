// Device memory of the library: allocations that outlive a call come from a bounded pool.
#pragma once

#include <cstddef>

namespace cuvs::detail {

/**
 * Device memory on the current device. hipMalloc and hipFree map and unmap the memory (about 5 ms
 * for the 256 MB of a 250,000 x 960 byte index, built, searched and dropped in 0.5 ms of kernels),
 * so a freed block waits in a pool for the next allocation of its size:
 * - a block enters the pool only when the device is idle of every use of it: device_release waits
 *   for the device, as hipFree does, or the caller has (device_idle). Any thread and any stream
 *   may then take it;
 * - the pool of a device holds at most kPoolBytes: its oldest blocks go back to the driver to make
 *   room, a larger block at once, and an allocation the driver refuses empties the pool and is tried
 *   again;
 * - other allocators of the process cannot empty it, so that it keeps nothing on a device that is short
 *   of memory: with less than a sixteenth free (asked for after every kPoolCheckBytes that come in,
 *   once in a millisecond) the released block and the whole pool go back to the driver;
 * - device_trim gives the pool of a device back to the driver (cuvsCertexTrimPool).
 * A block serves requests of at least three quarters of its size, so that little of it is unused.
 */
constexpr size_t kPoolBytes      = size_t(4) << 30;
constexpr size_t kPoolCheckBytes = size_t(64) << 20;

/** At least `bytes` bytes on the current device (*capacity: how many, *device: where), or null when
 *  the device has no memory left. The contents are undefined. */
void* device_allocate(size_t bytes, size_t* capacity, int* device);
/** Gives back a block of device_allocate (its capacity and device), after waiting for the device
 *  unless a device_idle of this thread covers it. */
void device_release(void* p, size_t capacity, int device) noexcept;
/** Gives every pooled block of `device` back to the driver. */
void device_trim(int device) noexcept;

/**
 * Between enter() and the guard's end, blocks of `device` that this thread releases enter the pool
 * without a wait each: enter() has waited for the device once, and the thread queues no work on
 * them in between. A member of a structure of device buffers, declared before them (so that it ends
 * after them) and entered by the structure's destructor.
 */
class device_idle {
 public:
  device_idle() = default;
  device_idle(device_idle const&)            = delete;
  device_idle& operator=(device_idle const&) = delete;
  ~device_idle();
  void enter(int device) noexcept;

 private:
  int outer_    = -1;
  bool entered_ = false;
};

}  // namespace cuvs::detail
