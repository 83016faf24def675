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
// (10 steps, FP32 3D) at 8, 16, 24, 30 and 36 MiB: hipMemcpy 6.1, 7.5, 8.4, 9.2 and
// 10.1 ms, pieces of 4 MiB 2.7, 10.1, 10.4, 10.8 and 11.4, thirds 2.4, 4.2, 5.4, 6.7
// and 8.2; later ones 0.93, 1.78, 2.84, 3.40 and 4.36; 0.80, 1.25, 1.65, 1.88 and
// 2.31; 0.68, 1.10, 1.50, 1.84 and 2.46.  Beyond, thirds would cost every call for
// the sake of the first.
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
