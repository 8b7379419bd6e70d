// Copies from the device to pageable host arrays (host_copy.hpp).
#include "host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace misa {

namespace {

// A chunk's DMA takes 20 us and 17 us a MB: 250 MB into an array in use take
// 8.6 ms in chunks of 1 MB, 6.8 ms in chunks of 2.
constexpr size_t kStageChunk = size_t(2) << 20;
constexpr size_t kStageSlots = 16;    // chunks on their way at once
constexpr size_t kStageThreads = 12;  // workers; fewer than 16 processors are often there
constexpr size_t kHelpBacklog = 4;    // arrived chunks that wait before the calling thread helps

// A copy in chunks c = 0, 1, ..., chunk c through slot c % kStageSlots.  The
// calling thread makes every HIP call, and helps to empty the slots where the
// workers fall behind: on a machine whose processors are busy a worker may not
// run for milliseconds, and then nothing waits for it.
struct StagedCopy {
  char* host;
  char* slots;
  size_t bytes, chunks;
  std::atomic<size_t> arrived{0};  // chunks in their slots so far, in order
  std::atomic<size_t> next{0};     // the first chunk nobody has taken yet
  std::atomic<size_t> done{0};     // chunks copied out
  std::atomic<size_t> emptied[kStageSlots] = {};  // chunks that have left a slot

  size_t length(size_t c) const { return std::min(kStageChunk, bytes - c * kStageChunk); }

  // Takes an arrived chunk and copies it out of its slot; false without one.
  bool copyOne() {
    size_t c = next.load(std::memory_order_relaxed);
    do {
      if (c >= arrived.load(std::memory_order_acquire)) return false;
    } while (!next.compare_exchange_weak(c, c + 1, std::memory_order_relaxed));
    const size_t k = c % kStageSlots;
    std::memcpy(host + c * kStageChunk, slots + k * kStageChunk, length(c));
    emptied[k].fetch_add(1, std::memory_order_release);
    done.fetch_add(1, std::memory_order_release);
    return true;
  }

  void work() {
    int idle = 0;
    while (next.load(std::memory_order_relaxed) < chunks) pause(copyOne() ? idle = 0 : ++idle);
  }

  // A chunk's DMA takes tens of microseconds; work queued before the copy may take long.
  static void pause(int idle) {
    if (idle > 5000) std::this_thread::sleep_for(std::chrono::microseconds(20));
    else if (idle > 0) std::this_thread::yield();
  }

  // Sends the chunks to their slots as these fall free, and hands on what has
  // arrived, until every chunk is copied.
  hipError_t drive(const char* dev, hipEvent_t* ev, hipStream_t st) {
    size_t sent = 0, in = 0;
    int idle = 0;
    while (done.load(std::memory_order_acquire) < chunks) {
      bool moved = false;
      const size_t k = sent % kStageSlots;
      if (sent < chunks && emptied[k].load(std::memory_order_acquire) == sent / kStageSlots) {
        hipError_t e = hipMemcpyAsync(slots + k * kStageChunk, dev + sent * kStageChunk, length(sent),
                                      hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev[k], st);
        if (e != hipSuccess) return e;
        sent++;
        moved = true;
      }
      if (in < sent) {
        const hipError_t e = hipEventQuery(ev[in % kStageSlots]);
        if (e == hipSuccess) {
          arrived.store(++in, std::memory_order_release);
          moved = true;
        } else if (e != hipErrorNotReady) {
          return e;
        }
      }
      if (!moved && (in == chunks || in - next.load(std::memory_order_relaxed) >= kHelpBacklog)) moved = copyOne();
      pause(moved ? idle = 0 : ++idle);
    }
    return hipSuccess;
  }
};

// The pinned slots and the worker threads, which sleep between copies.
struct Stage {
  std::mutex busy;  // held through a staged copy
  char* slots = nullptr;
  std::vector<std::thread> threads;
  std::mutex lock;  // of what follows
  std::condition_variable wake;
  std::shared_ptr<StagedCopy> job;
  uint64_t jobs = 0;
  bool quit = false;

  void worker() {
    uint64_t seen = 0;
    for (;;) {
      std::shared_ptr<StagedCopy> j;
      {
        std::unique_lock<std::mutex> l(lock);
        wake.wait(l, [&] { return quit || (jobs != seen && job); });
        if (quit) return;
        seen = jobs;
        j = job;
      }
      j->work();
    }
  }

  // With busy held.  False without pinned memory or a thread.
  bool open() {
    if (!slots && hipHostMalloc(reinterpret_cast<void**>(&slots), kStageSlots * kStageChunk, hipHostMallocPortable) !=
                      hipSuccess) {
      slots = nullptr;
      (void)hipGetLastError();
      return false;
    }
    try {
      threads.reserve(kStageThreads);
      while (threads.size() < kStageThreads) threads.emplace_back([this] { worker(); });
    } catch (const std::exception&) {  // no more threads: those there share the work
    }
    return true;
  }

  void close() {
    std::lock_guard<std::mutex> b(busy);
    {
      std::lock_guard<std::mutex> l(lock);
      quit = true;
    }
    wake.notify_all();
    for (std::thread& t : threads) t.join();
    threads.clear();
    quit = false;
    if (slots) (void)hipHostFree(slots);
    slots = nullptr;
  }

  hipError_t copy(char* host, const char* dev, size_t bytes, hipStream_t st) {
    std::shared_ptr<StagedCopy> s;
    try {
      s = std::make_shared<StagedCopy>();
    } catch (const std::bad_alloc&) {
      return hipErrorOutOfMemory;
    }
    s->host = host;
    s->slots = slots;
    s->bytes = bytes;
    s->chunks = (bytes + kStageChunk - 1) / kStageChunk;
    hipEvent_t ev[kStageSlots] = {};
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < std::min(kStageSlots, s->chunks) && e == hipSuccess; k++)
      e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    if (e == hipSuccess) {
      {
        std::lock_guard<std::mutex> l(lock);
        job = s;
        jobs++;
      }
      for (size_t t = std::min(threads.size(), s->chunks); t > 0; t--) wake.notify_one();
      e = s->drive(dev, ev, st);
      // nobody takes another chunk, and those taken (after an error) leave their slots
      const size_t taken = s->next.exchange(s->chunks);
      while (s->done.load(std::memory_order_acquire) < taken) std::this_thread::yield();
      std::lock_guard<std::mutex> l(lock);
      job.reset();
    }
    // every DMA into the slots has ended before they are given up
    const hipError_t w = hipStreamSynchronize(st);
    (void)hipGetLastError();  // hipErrorNotReady of the queries
    for (hipEvent_t x : ev)
      if (x) (void)hipEventDestroy(x);
    return e != hipSuccess ? e : w;
  }
};

// Never destroyed: its threads end with the last StageUser.
Stage& stage() {
  alignas(Stage) static unsigned char room[sizeof(Stage)];
  static Stage* s = new (room) Stage();
  return *s;
}
std::mutex stageUsersLock;
int stageUsers = 0;

// Pinned or managed memory, which the DMA reaches without staging.
bool reachable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

}  // namespace

hipError_t copyToHost(void* host, const void* dev, size_t bytes, hipStream_t st) {
  if (bytes >= kStagedBytes && !reachable(host)) {
    Stage& s = stage();
    std::unique_lock<std::mutex> busy(s.busy, std::try_to_lock);
    if (busy.owns_lock() && s.open())
      return s.copy(static_cast<char*>(host), static_cast<const char*>(dev), bytes, st);
  }
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

StageUser::StageUser() {
  std::lock_guard<std::mutex> g(stageUsersLock);
  stageUsers++;
}
StageUser::~StageUser() {
  std::lock_guard<std::mutex> g(stageUsersLock);
  if (--stageUsers == 0) stage().close();
}

}  // namespace misa
