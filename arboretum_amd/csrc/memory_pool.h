// Work memory that outlives the objects that use it: device blocks and pinned host blocks.
#ifndef ARBORETUM_AMD_MEMORY_POOL_H_
#define ARBORETUM_AMD_MEMORY_POOL_H_

#include <hip/hip_runtime.h>

#include <cstddef>

namespace arb {

// Device memory of the current device.  A booster takes some forty blocks when it is created and
// gives them back when it goes; hipMalloc and hipFree of them cost up to milliseconds (a free waits
// for the device and unmaps), so blocks given back are kept and handed out again.
//   - Bounded: at most kDevicePoolBytes of idle blocks per device, the oldest go first.
//   - Given back to the driver: when a hipMalloc here fails (everything idle is freed, then it is tried
//     again), when the bound is passed, when a block has been idle for kPoolIdleSeconds (looked at
//     on every call of the pool, so not while nobody calls it), by DevicePoolTrim() and by TrimPools().
//     An allocation that fails elsewhere in the process gets nothing back by itself: TrimPools() (AReleaseMemory)
//     is for a program that needs the memory for something else.
//   - Safe with several threads and streams: one lock; a block may only be given back when no work
//     that uses it is pending on any stream.
// The contents of a block are undefined.
void *DevicePoolTake(size_t bytes);
void DevicePoolGive(void *p) noexcept;  // p may be null
void DevicePoolTrim() noexcept;         // frees every idle block of the current device

// Pinned host memory, by the same rules (at most kPinnedPoolBytes idle).
void *PinnedPoolTake(size_t bytes);
void PinnedPoolGive(void *p) noexcept;

// Ordinary host memory for large buffers, by the same rules (at most kHostPoolBytes idle): a fresh
// allocation of this size comes from the kernel page by page, and touching it the first time costs
// more than filling it.
void *HostPoolTake(size_t bytes);
void HostPoolGive(void *p) noexcept;

// Whether this process has taken memory or a stream of a GPU from these pools (a child made by fork
// has not).
bool GpuInUse() noexcept;

// Streams (non-blocking, default priority) of the current device that are kept and handed out again;
// nothing may be pending on one that is given back.  Blocks and streams return to the device they came
// from, whichever one is current when they are given back.
hipStream_t StreamPoolTake();
void StreamPoolGive(hipStream_t s) noexcept;  // s may be null

// Frees everything idle in the pools above, on every device.
void TrimPools() noexcept;

}  // namespace arb
#endif  // ARBORETUM_AMD_MEMORY_POOL_H_
