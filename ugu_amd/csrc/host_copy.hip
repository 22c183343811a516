#include "host_copy.h"

#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace ugu_hip {
namespace {

constexpr size_t kChunkBytes = CopyRing::kChunkBytes;
constexpr int kCopyThreads = 256;
constexpr int kCopyBlocks = 32;

// Copies below these many bytes in all are plain hipMemcpyAsync calls: 8 KB to the
// host take 22 us so and 8.5 us through the slots, 128 KB 60 and 15 us; to the
// device 8 KB take 14 us either way, 128 KB 57 and 22 us.
constexpr size_t kMinToHost = size_t(4) << 10;
constexpr size_t kMinToDevice = size_t(64) << 10;
// Pinned arrays of this many bytes in all are copied by the engine: it takes no
// page fault (a CPU's first touch of pinned pages costs 1 us each, populating them
// 0.1 ms per MB) and the CPU moves nothing. Outputs in pinned memory, first and later
// passes: 74 KB 131 / 90 us so, 139 / 71 through the slots; 460 KB 117 / 110 and
// 249 / 87; 11.6 MB 348 / 343 and 1342 / 418; 302 MB 5670 / 5630 and 30800 / 7450.
constexpr size_t kMinDirect = size_t(128) << 10;
// Jobs below this many bytes are not given to the pool: its threads take 50 us to
// wake, in which the caller moves 512 KB itself.
constexpr size_t kPoolBytes = size_t(512) << 10;
// Pages are populated in pieces of the large page size, so that no two threads
// clear the same page.
constexpr size_t kPageStep = size_t(2) << 20;

struct DevChunk {
  unsigned char* dev;
  uint32_t bytes;
  uint32_t seq;  // to the host: the value the slot's flag takes
};

// Slots and, by queue_direct's check, device addresses are multiples of 16.
__device__ __forceinline__ void copy_chunk(unsigned char* dst, const unsigned char* src,
                                           uint32_t bytes) {
  const uint32_t words = bytes / 16;
  for (uint32_t i = threadIdx.x; i < words; i += kCopyThreads)
    reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  const uint32_t i = words * 16 + threadIdx.x;
  if (i < bytes) dst[i] = src[i];
}

// A block per chunk in turn; `slots`, `table` and `flags` are pinned host memory.
// Few blocks, so that a chunk is whole after 20 us and not after the launch.
__global__ __launch_bounds__(kCopyThreads) void k_to_slots(const DevChunk* table, int n,
                                                           unsigned char* slots, uint32_t* flags) {
  for (int k = blockIdx.x; k < n; k += gridDim.x) {
    const DevChunk c = table[k];
    copy_chunk(slots + size_t(k) * kChunkBytes, c.dev, c.bytes);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(flags + k, c.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ __launch_bounds__(kCopyThreads) void k_from_slots(const DevChunk* table, int n,
                                                             const unsigned char* slots) {
  for (int k = blockIdx.x; k < n; k += gridDim.x) {
    const DevChunk c = table[k];
    copy_chunk(c.dev, slots + size_t(k) * kChunkBytes, c.bytes);
  }
}

void relax(int* spins) {
  if (++*spins < 2000)
    __builtin_ia32_pause();
  else if (*spins < 10000)
    std::this_thread::yield();
  else
    std::this_thread::sleep_for(std::chrono::microseconds(50));
}

constexpr size_t kSlotBytes = size_t(CopyRing::kSlots) * kChunkBytes;
constexpr size_t kTableOff = kSlotBytes;
constexpr size_t kFlagOff = kTableOff + size_t(CopyRing::kSlots) * sizeof(DevChunk);
constexpr size_t kPinnedBytes = kFlagOff + size_t(CopyRing::kSlots) * 4;

}  // namespace

// Work the pool's threads take part in: populating pages (`ranges`) or moving
// chunks. Chunk k goes through slot k % kSlots. A thread takes the next chunk and
// waits for it: to the host until the device has flagged it, to the device until
// the slot is free (`open` exceeds k). The caller takes only chunks that need no
// wait, so it completes the job without the pool too.
struct HostJob {
  struct Chunk {
    unsigned char* host;
    unsigned char* dev;
    size_t bytes;
  };
  std::vector<HostCopy> ranges;
  std::vector<Chunk> chunks;
  unsigned char* pinned = nullptr;
  bool out = false;
  uint32_t seq0 = 0;
  std::atomic<int> take{0}, open{0}, helpers{0};
  std::atomic<bool> stop{false};
  std::atomic<int> moved[CopyRing::kSlots / CopyRing::kGroupChunks];  // per group, running count

  HostJob() {
    for (auto& m : moved) m.store(0);
  }
  int size() const { return static_cast<int>(ranges.empty() ? chunks.size() : ranges.size()); }
  int group_of(int k) const { return k / CopyRing::kGroupChunks % CopyRing::kGroups; }

  bool ready(int k) const {
    if (!ranges.empty()) return true;
    if (!out) return open.load(std::memory_order_acquire) > k;
    const uint32_t* flag = reinterpret_cast<const uint32_t*>(pinned + kFlagOff) + k % CopyRing::kSlots;
    return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq0 + uint32_t(k);
  }
  void run(int k) {
    if (!ranges.empty()) {
      const HostCopy& r = ranges[size_t(k)];
      (void)madvise(r.host, r.bytes, MADV_POPULATE_WRITE);  // a hint: older kernels refuse it
      return;
    }
    const Chunk& c = chunks[size_t(k)];
    unsigned char* slot = pinned + size_t(k % CopyRing::kSlots) * kChunkBytes;
    if (out)
      std::memcpy(c.host, slot, c.bytes);
    else
      std::memcpy(slot, c.host, c.bytes);
    moved[group_of(k)].fetch_add(1, std::memory_order_release);
  }
  void help() {
    for (;;) {
      const int k = take.fetch_add(1);
      if (k >= size()) return;
      for (int spins = 0; !ready(k);) {
        if (stop.load(std::memory_order_acquire)) return;
        relax(&spins);
      }
      run(k);
    }
  }
  bool help_once() {
    int k = take.load();
    while (k < size() && ready(k))
      if (take.compare_exchange_weak(k, k + 1)) {
        run(k);
        return true;
      }
    return false;
  }
};

namespace {

// Threads shared by every context of the process, started by the first job and
// asleep between jobs. Never destroyed: they may be waiting when the process
// ends.
class Pool {
 public:
  static Pool& get() {
    static Pool* p = new Pool();
    return *p;
  }
  void add(HostJob* j) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      jobs_.push_back(j);
    }
    cv_.notify_all();
  }
  // after this no pool thread holds the job
  void remove(HostJob* j) {
    j->stop.store(true, std::memory_order_release);
    {
      std::lock_guard<std::mutex> lk(mu_);
      jobs_.erase(std::remove(jobs_.begin(), jobs_.end(), j), jobs_.end());
    }
    for (int spins = 0; j->helpers.load(std::memory_order_acquire) != 0;) relax(&spins);
  }

 private:
  Pool() {
    const int hw = static_cast<int>(std::thread::hardware_concurrency());
    const int n = std::max(0, std::min(7, hw / 2 - 1));
    try {
      for (int i = 0; i < n; i++) std::thread([this] { run(); }).detach();
    } catch (...) {
      // fewer threads: the callers move what these would have
    }
  }
  void run() {
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      HostJob* job = nullptr;
      for (HostJob* j : jobs_)
        if (j->take.load() < j->size()) {
          job = j;
          break;
        }
      if (!job) {
        cv_.wait(lk);
        continue;
      }
      job->helpers.fetch_add(1);
      lk.unlock();
      job->help();
      job->helpers.fetch_sub(1, std::memory_order_release);
      lk.lock();
    }
  }
  std::mutex mu_;
  std::condition_variable cv_;
  std::vector<HostJob*> jobs_;
};

// Takes the job out of the pool on every way out of a scope.
struct Posted {
  HostJob* job = nullptr;
  void add(HostJob* j) {
    Pool::get().add(j);
    job = j;
  }
  ~Posted() {
    if (job) Pool::get().remove(job);
  }
};

enum class Memory { kPageable, kPinned, kOther };

// What an array is: at both ends, as the caller may have a part of an allocation.
Memory memory_of(const HostCopy& c) {
  for (size_t at : {size_t(0), c.bytes - 1}) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, static_cast<const unsigned char*>(c.host) + at) != hipSuccess)
      (void)hipGetLastError();  // not known to HIP
    else if (a.type != hipMemoryTypeUnregistered)
      return a.type == hipMemoryTypeHost ? Memory::kPinned : Memory::kOther;
  }
  return Memory::kPageable;
}

hipError_t queue(hipStream_t st, const HostCopy& c, bool out) {
  return out ? hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, st)
             : hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, st);
}

// Whether two of the host arrays share bytes. Copies out are then made in their
// order, so that the last one's bytes stay, as in a loop of copies.
bool overlap(const HostCopy* c, int n) {
  std::vector<std::pair<uintptr_t, uintptr_t>> r;
  for (int i = 0; i < n; i++) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(c[i].host);
    if (c[i].bytes > 0) r.emplace_back(at, at + c[i].bytes);
  }
  std::sort(r.begin(), r.end());
  for (size_t i = 1; i < r.size(); i++)
    if (r[i].first < r[i - 1].second) return true;
  return false;
}

// Queues the copies that the engine makes: of pinned arrays (from kMinDirect bytes
// of them in all on), of memory that is not the host's or not aligned on the device, and,
// where fewer than `least` bytes would be left or results overlap, all of them. The others are
// returned in *slots.
hipError_t queue_direct(hipStream_t st, const HostCopy* c, int n, bool out, size_t least,
                        std::vector<HostCopy>* slots) {
  std::vector<Memory> kind(static_cast<size_t>(n), Memory::kOther);
  size_t pinned = 0, left = 0;
  for (int i = 0; i < n; i++) {
    if (c[i].bytes == 0) continue;
    if (reinterpret_cast<uintptr_t>(c[i].dev) % 16 == 0) kind[size_t(i)] = memory_of(c[i]);
    if (kind[size_t(i)] == Memory::kPinned) pinned += c[i].bytes;
    if (kind[size_t(i)] == Memory::kPageable) left += c[i].bytes;
  }
  if (pinned < kMinDirect) left += pinned;
  const bool use = left >= least && !(out && overlap(c, n));
  for (int i = 0; i < n; i++) {
    if (c[i].bytes == 0) continue;
    if (use && (kind[size_t(i)] == Memory::kPageable ||
                (kind[size_t(i)] == Memory::kPinned && pinned < kMinDirect))) {
      slots->push_back(c[i]);
    } else if (hipError_t e = queue(st, c[i], out)) {
      return e;
    }
  }
  return hipSuccess;
}

// Returns the bytes of all chunks.
size_t split(const std::vector<HostCopy>& copies, std::vector<HostJob::Chunk>* out) {
  size_t bytes = 0;
  for (const HostCopy& c : copies) bytes += c.bytes;
  out->reserve(bytes / kChunkBytes + copies.size());
  for (const HostCopy& c : copies)
    for (size_t at = 0; at < c.bytes; at += kChunkBytes)
      out->push_back(HostJob::Chunk{static_cast<unsigned char*>(c.host) + at,
                                    static_cast<unsigned char*>(c.dev) + at,
                                    std::min(kChunkBytes, c.bytes - at)});
  return bytes;
}

}  // namespace

Prefault::Prefault(CopyRing& ring, const HostCopy* c, int n) {
  size_t bytes = 0;
  for (int i = 0; i < n; i++) bytes += c[i].bytes;
  if (bytes < kPoolBytes) return;
  if (ring.prepare() != hipSuccess) (void)hipGetLastError();
  auto job = std::make_unique<HostJob>();
  for (int i = 0; i < n; i++) {
    if (c[i].bytes == 0 || memory_of(c[i]) != Memory::kPageable) continue;
    uintptr_t at = reinterpret_cast<uintptr_t>(c[i].host);
    const uintptr_t end = at + c[i].bytes;
    at = (at + 4095) & ~uintptr_t(4095);
    while (at < end) {
      const uintptr_t to = std::min(end, (at & ~uintptr_t(kPageStep - 1)) + kPageStep);
      if (to - at >= 65536) job->ranges.push_back(HostCopy{reinterpret_cast<void*>(at), nullptr, to - at});
      at = to;
    }
  }
  if (job->ranges.empty()) return;
  Pool::get().add(job.get());
  job_ = job.release();
}

Prefault::~Prefault() {
  if (!job_) return;
  Pool::get().remove(job_);
  delete job_;
}

hipError_t CopyRing::prepare() {
  if (pinned_) return hipSuccess;
  void* p = nullptr;
  hipError_t e = hipHostMalloc(&p, kPinnedBytes, hipHostMallocDefault);
  if (e != hipSuccess) return e;
  for (int g = 0; g < kGroups; g++)
    if ((e = hipEventCreateWithFlags(&ev_[g], hipEventDisableTiming)) != hipSuccess) {
      while (--g >= 0) (void)hipEventDestroy(ev_[g]);
      (void)hipHostFree(p);
      return e;
    }
  pinned_ = static_cast<unsigned char*>(p);
  std::memset(pinned_ + kFlagOff, 0, size_t(kSlots) * 4);
  seq_ = 0;
  return hipSuccess;
}

hipError_t CopyRing::wait_groups() {
  for (int g = 0; g < kGroups; g++)
    if (used_[g])
      if (hipError_t e = hipEventSynchronize(ev_[g])) return e;
  return hipSuccess;
}

void CopyRing::release() {
  if (!pinned_) return;
  (void)wait_groups();
  for (int g = 0; g < kGroups; g++) {
    (void)hipEventDestroy(ev_[g]);
    ev_[g] = nullptr;
    used_[g] = false;
  }
  (void)hipHostFree(pinned_);
  pinned_ = nullptr;
}

hipError_t CopyRing::to_host(hipStream_t st, const HostCopy* c, int n) {
  std::vector<HostCopy> slots;
  hipError_t err = queue_direct(st, c, n, true, kMinToHost, &slots);
  if (err != hipSuccess) return err;
  if (!slots.empty() && prepare() != hipSuccess) {
    (void)hipGetLastError();
    for (const HostCopy& x : slots)
      if ((err = queue(st, x, true)) != hipSuccess) return err;
    slots.clear();
  }
  if (slots.empty()) return hipStreamSynchronize(st);
  if ((err = wait_groups()) != hipSuccess) return err;
  HostJob job;
  const size_t bytes = split(slots, &job.chunks);
  job.pinned = pinned_;
  job.out = true;
  const int count = job.size();
  if (seq_ > UINT32_MAX - uint32_t(count) - 1) seq_ = 0;
  job.seq0 = seq_ + 1;
  seq_ += uint32_t(count);
  Posted posted;
  if (bytes >= kPoolBytes) posted.add(&job);
  DevChunk* table = reinterpret_cast<DevChunk*>(pinned_ + kTableOff);
  uint32_t* flags = reinterpret_cast<uint32_t*>(pinned_ + kFlagOff);
  int sent = 0, done = 0;  // chunks launched, chunks of the groups known to be empty again
  for (int idle = 0; done < count;) {
    // a group's slots are written again once its chunks have been moved out
    if (sent < count && sent - done < kSlots) {
      const int g = job.group_of(sent), first = g * kGroupChunks;
      const int m = std::min(kGroupChunks, count - sent);
      for (int k = 0; k < m; k++) {
        const HostJob::Chunk& h = job.chunks[size_t(sent + k)];
        table[first + k] = DevChunk{h.dev, uint32_t(h.bytes), job.seq0 + uint32_t(sent + k)};
      }
      k_to_slots<<<std::min(m, kCopyBlocks), kCopyThreads, 0, st>>>(
          table + first, m, pinned_ + size_t(first) * kChunkBytes, flags + first);
      if ((err = hipGetLastError()) != hipSuccess) return err;
      sent += m;
      continue;
    }
    const int g = job.group_of(done), m = std::min(kGroupChunks, count - done);
    if (job.moved[g].load(std::memory_order_acquire) == m) {
      job.moved[g].store(0);
      done += m;
      continue;
    }
    if (job.help_once()) {
      idle = 0;
      continue;
    }
    // nothing arrives: the stream is still busy, or it has failed
    if (++idle % 4096 == 0) {
      const hipError_t q = hipStreamQuery(st);
      if (q == hipErrorNotReady)
        (void)hipGetLastError();
      else if (q != hipSuccess)
        return q;
      else
        for (int k = done; k < sent; k++)
          if (!job.ready(k)) return hipErrorLaunchFailure;  // finished without its flags
    }
    __builtin_ia32_pause();
  }
  return hipSuccess;  // the direct copies were queued before the chunks
}

hipError_t CopyRing::to_device(hipStream_t st, const HostCopy* c, int n) {
  std::vector<HostCopy> slots;
  hipError_t err = queue_direct(st, c, n, false, kMinToDevice, &slots);
  if (err != hipSuccess) return err;
  if (!slots.empty() && prepare() != hipSuccess) {
    (void)hipGetLastError();
    for (const HostCopy& x : slots)
      if ((err = queue(st, x, false)) != hipSuccess) return err;
    slots.clear();
  }
  if (slots.empty()) return hipSuccess;
  if ((err = wait_groups()) != hipSuccess) return err;
  HostJob job;
  const size_t bytes = split(slots, &job.chunks);
  job.pinned = pinned_;
  const int count = job.size();
  int open = std::min(count, kSlots);
  job.open.store(open);
  Posted posted;
  if (bytes >= kPoolBytes) posted.add(&job);
  DevChunk* table = reinterpret_cast<DevChunk*>(pinned_ + kTableOff);
  for (int sent = 0; sent < count;) {
    const int g = job.group_of(sent), first = g * kGroupChunks;
    const int m = std::min(kGroupChunks, count - sent);
    if (job.moved[g].load(std::memory_order_acquire) == m) {
      job.moved[g].store(0);
      for (int k = 0; k < m; k++) {
        const HostJob::Chunk& h = job.chunks[size_t(sent + k)];
        table[first + k] = DevChunk{h.dev, uint32_t(h.bytes), 0};
      }
      k_from_slots<<<std::min(m, kCopyBlocks), kCopyThreads, 0, st>>>(
          table + first, m, pinned_ + size_t(first) * kChunkBytes);
      if ((err = hipGetLastError()) != hipSuccess) return err;
      if ((err = hipEventRecord(ev_[g], st)) != hipSuccess) return err;
      used_[g] = true;
      sent += m;
      continue;
    }
    // the group whose copy has left opens for the chunks after the open ones
    if (open < count && open - kSlots < sent) {
      const hipError_t q = hipEventQuery(ev_[job.group_of(open)]);
      if (q == hipSuccess) {
        open = std::min(count, open + kGroupChunks);
        job.open.store(open, std::memory_order_release);
        continue;
      }
      (void)hipGetLastError();
      if (q != hipErrorNotReady) return q;
    }
    if (!job.help_once()) __builtin_ia32_pause();
  }
  return hipSuccess;
}

}  // namespace ugu_hip
