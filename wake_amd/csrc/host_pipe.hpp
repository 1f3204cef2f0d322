// host_pipe.hpp -- device arrays into pageable host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace wake_hip {

// Copies `bytes` from device memory to host memory after the work enqueued on
// `stream`, and returns when they are there.  Throws HipError.
void device_to_host(void* dst, const void* src, size_t bytes, hipStream_t stream);

// Frees the idle pinned buffers (called when the last domain goes).
void trim_host_pipe() noexcept;

}  // namespace wake_hip
