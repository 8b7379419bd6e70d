// Copies from the device to a caller's pageable host array.
//
// hipMemcpyAsync takes a pageable array through one staging buffer and one
// host thread: 17 GB/s into an array in use and 4 to 9 into a fresh one, whose
// page faults that thread takes too, where the link moves 57 GB/s.  Here
// several host threads empty the pinned slots that the DMA fills.  Measured,
// direct / staged: 4 MB fresh 0.92 / 0.64 ms, in use 0.23 / 0.20; 9.7 MB fresh
// 2.2 / 0.9, in use 0.55 / 0.42; 250 MB fresh 58 / 9.9, in use 14.6 / 6.8.  To
// the device hipMemcpyAsync is as fast from 64 MB on and faster below.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace misa {

constexpr size_t kStagedBytes = size_t(4) << 20;

// Copies `bytes` from device to host memory, ordered on `st` after the work
// before it, and returns when the copy is done.  Any host memory, any
// alignment.  Arrays below kStagedBytes, pinned memory, and calls that find
// the slots in use by another thread go through hipMemcpyAsync.
hipError_t copyToHost(void* host, const void* dev, size_t bytes, hipStream_t st);

// The pinned slots belong to the process: 32 MB, allocated by the first staged
// copy and freed with the last StageUser (every handle holds one).
struct StageUser {
  StageUser();
  ~StageUser();
  StageUser(const StageUser&) = delete;
  StageUser& operator=(const StageUser&) = delete;
};

}  // namespace misa
