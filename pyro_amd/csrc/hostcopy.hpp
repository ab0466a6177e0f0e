// hostcopy.hpp -- large copies between pageable host arrays and the device.
//
// A pageable hipMemcpy is staged by the runtime on one thread (27 GB/s in and
// 10 GB/s out into fresh memory, whose pages it also faults in).  These
// copies run through pinned slots filled and emptied by a few threads, each
// moving its own chunks, so the host side keeps up with the link.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace pyro {

// The slots and threads are one pool for the process, made by the first large
// copy and given back when the last handle that holds a HostCopyUse is
// destroyed.  A copy that finds the pool in use by another host thread takes
// the runtime's path, so several threads never wait for one another.
struct HostCopyUse {
  HostCopyUse();
  ~HostCopyUse();
  HostCopyUse(const HostCopyUse &) = delete;
  HostCopyUse &operator=(const HostCopyUse &) = delete;
};

// Copy to the device, ordered on s: src may be changed on return, or with
// `later` not before s is synchronised (a small copy then waits for nothing).
hipError_t copy_in(void *dst, const void *src, size_t bytes, hipStream_t s, bool later = false);
// Copy from the device, ordered on s: complete on return.
hipError_t copy_out(void *dst, const void *src, size_t bytes, hipStream_t s);

}  // namespace pyro
