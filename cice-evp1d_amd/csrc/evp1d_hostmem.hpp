// evp1d_hostmem.hpp - results written straight into a caller's page-locked
// memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

// The address at which kernels write `bytes` at dst when dst is page-locked
// host memory (evp1d_host_alloc, hipHostMalloc) of the current device that
// holds them; null for any other memory, which takes a copy.  A gather that
// writes there needs no copy behind it and no second wait for the queue: launch
// and wait take 11 us in place of 14 for 100 values, 16 in place of 21 for
// 20 000, 40 in place of 47 for 200 000, 155 in place of 163 for a million (the
// query takes 0.2 us).  From two million values on the copy is 1 to 2 % faster
// (53 GB/s): null for those.
inline double *page_locked(double *dst, size_t bytes) {
  if (bytes > ((size_t)16 << 20) || reinterpret_cast<uintptr_t>(dst) % alignof(double)) return nullptr;
  hipPointerAttribute_t a{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  int dev = -1;
  if (hipPointerGetAttributes(&a, dst) != hipSuccess || a.type != hipMemoryTypeHost || !a.devicePointer ||
      hipGetDevice(&dev) != hipSuccess || a.device != dev ||
      hipMemGetAddressRange(&base, &size, a.devicePointer) != hipSuccess) {
    (void)hipGetLastError();   // not this memory: no error
    return nullptr;
  }
  const size_t off = (size_t)(static_cast<char *>(a.devicePointer) - static_cast<char *>(base));
  return off + bytes <= size ? static_cast<double *>(a.devicePointer) : nullptr;
}
