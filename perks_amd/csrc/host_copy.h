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

// A copy goes in pieces through kStagingBuffers pinned buffers: up to 36 MiB in as
// many pieces as buffers, beyond in pieces of 4 MiB (17 us of the link go by
// between two: 64 MiB in pieces of 1, 2 and 4 MiB take 2.16, 1.73 and 1.55 ms; 3 or
// 8 buffers or threads, the same).  The thirds are for a program's first call: with
// more pieces than three the runtime stands still once for some 6 ms, which the
// copies of a program that moves little then never pay.  First call of a process
// (10 steps, FP32 3D) at 8, 16, 24 and 32 MiB: hipMemcpy 6.3, 7.3, 8.5 and 9.2 ms,
// pieces of 4 MiB 2.9, 10.0, 10.4 and 11.1, thirds 2.3, 4.2, 5.8 and 7.7; the tenth
// 1.0, 1.8, 2.6, 3.5; 0.83, 1.25, 1.68, 2.0; 0.77, 1.27, 1.70, 2.15.  Beyond, thirds
// would cost every call for the sake of the first: 48 MiB first call 11.2, 11.5 and
// 10.9, tenth 5.5, 3.0 and 3.5.
constexpr int kStagingBuffers = 3;
constexpr size_t kStagingPiece = (size_t)4 << 20;
constexpr size_t kStagingThirds = (size_t)36 << 20;
// Bytes of a buffer of a set made for a copy of `bytes`, and of the pieces of a copy
// through buffers of `capacity`.
constexpr size_t staging_third(size_t bytes)
{
    return (bytes / kStagingBuffers + 4095) / 4096 * 4096 + (bytes % kStagingBuffers ? 4096 : 0);
}
constexpr size_t staging_capacity(size_t bytes)
{
    const size_t third = bytes <= kStagingThirds ? staging_third(bytes) : 0;
    return third > kStagingPiece ? third : kStagingPiece;
}
constexpr size_t staging_piece(size_t capacity, size_t bytes)
{
    const size_t third = staging_third(bytes);
    return third <= capacity ? third : kStagingPiece;
}

}  // namespace perks
