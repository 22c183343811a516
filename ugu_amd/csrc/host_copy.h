// Copies between the device and host arrays, through pinned slots if pageable: a
// copy kernel moves chunks between the device and the slots while host threads
// move them between the slots and the caller's arrays.
//
// What bounds it is PCIe: 57 GB/s. hipMemcpy to and from pageable memory reaches
// 18 GB/s out of the device and 30 GB/s into it (one thread copies, one slot at a
// time, and takes a fresh destination's page faults one by one). Copy engine
// commands of 1 MB into pinned memory cost 10 us each beside their 18 us of
// transfer; the kernel writes pinned memory at 53 GB/s and reads it at 55 GB/s
// with 32 blocks, in one launch, and tells the host of each 32 KB as it is done.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace ugu_hip {

struct HostCopy {
  void* host;
  void* dev;
  size_t bytes;
};

struct HostJob;

// The slots of one context; allocated by the first copy that uses them.
class CopyRing {
 public:
  static constexpr int kGroups = 2;           // launches in flight
  static constexpr int kGroupChunks = 128;    // chunks of a launch
  static constexpr size_t kChunkBytes = 32768;
  static constexpr int kSlots = kGroups * kGroupChunks;

  // Queues the copies after the stream's work. to_host returns when the host
  // arrays hold the data, to_device when the pageable host arrays have been read
  // (pinned ones are read in the stream's order).
  hipError_t to_host(hipStream_t st, const HostCopy* c, int n);
  hipError_t to_device(hipStream_t st, const HostCopy* c, int n);
  void release();

 private:
  friend class Prefault;
  hipError_t prepare();
  hipError_t wait_groups();
  unsigned char* pinned_ = nullptr;
  hipEvent_t ev_[kGroups] = {};
  bool used_[kGroups] = {};  // the group's event has been recorded
  uint32_t seq_ = 0;         // sequence number of the last chunk
};

// Populates the pages of host arrays that are about to be written, on the pool's
// threads, while the device still works on what goes there. Changes no byte. To be
// made after the call's allocations: both need the process's memory map (a
// context's first 801 x 603 pass took up to 1 ms longer with its buffers allocated
// beside it), so the ring's
// slots are allocated first.
class Prefault {
 public:
  Prefault(CopyRing& ring, const HostCopy* c, int n);
  ~Prefault();
  Prefault(const Prefault&) = delete;
  Prefault& operator=(const Prefault&) = delete;

 private:
  HostJob* job_ = nullptr;
};

}  // namespace ugu_hip
