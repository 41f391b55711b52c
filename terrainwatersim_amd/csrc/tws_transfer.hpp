// tws_transfer.hpp -- copies between the caller's host arrays and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace tws {

// Copies of `bytes` in stream order.  The host array may be reused (upload) or
// read (download) once the stream has been synchronised.
hipError_t copy_to_device(void* device, const void* host, size_t bytes, hipStream_t s);
hipError_t copy_to_host(void* host, const void* device, size_t bytes, hipStream_t s);

// A handle that makes such copies: the pinned memory they go through is kept
// while any is alive.
struct TransferUser {
    TransferUser();
    ~TransferUser();
    TransferUser(const TransferUser&) = delete;
    TransferUser& operator=(const TransferUser&) = delete;
};

}  // namespace tws
