// host_copy.h -- copies between pageable host memory and the device for the
// entry points that take host arrays.
#pragma once

#include <cstddef>

namespace perks {

// As hipMemcpy on the default stream: the host array may be reused, and holds
// the data, when they return.  PERKS_OK or PERKS_ERR_HIP.
int copy_to_device(void* dst, const void* src, size_t bytes);
int copy_to_host(void* dst, const void* src, size_t bytes);
// Frees the pinned buffers that no copy is using.
void release_host_copy();

}  // namespace perks
