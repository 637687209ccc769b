// Copies between the caller's ordinary (pageable) host memory and the device.
//
// hipMemcpy to pageable memory is one thread's work: the runtime moves
// ~1 MB at a time into its own pinned buffer and copies it out before the
// next.  Measured: device to host 18 GB/s, 10.6 into memory the caller has
// just allocated (its pages are first touched by that one thread), and host
// to device 7 GB/s at 1 MB (35 at 8 MB), while the link carries 56 GB/s each
// way.  A HostPool has a ring of pinned slots and a few threads: the link fills
// or empties one slot while the threads copy others.  Measured with it: 955 MB
// to the host 20.1 ms (47 GB/s; 21.4 into new memory, ~90 before), from it 20.8
// (25 before); 25 MB to the host 0.58 ms (1.4), from it 0.60 (0.66).  Slots of
// 2 MB: 24.4, 23.8, 0.64 and 0.66.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace ane {

// One per device, shared by the objects that copy (host_pool); freed with
// the last of them.  One HostCopy uses it at a time; a copy that finds it in
// use (another thread's) goes through hipMemcpyAsync instead.
class HostPool {
 public:
  static constexpr int kSlots = 8;
  static constexpr size_t kSlotBytes = (size_t)4 << 20;
  static constexpr size_t kTaskBytes = (size_t)256 << 10;  // one thread's piece of a slot
  static constexpr int kThreads = 6;
  // Below this a copy is left to hipMemcpyAsync: waking the threads costs more
  // (us a call, hipMemcpyAsync / pool, to the host 368 KB 25 / 45, 880 KB 46 /
  // 56, 1.1 MB 73 / 62, 2.1 MB 133 / 87; from it 33 / 46, 52 / 56, 73 / 62, 102 /
  // 82).  A call of many copies, or one that has the pool already, uses it
  // from kMoreBytes on (one layer's forward with its ten taps, 512 wide, 128
  // positions, 256 KB a copy: 465 / 398).
  static constexpr size_t kMinBytes = (size_t)1 << 20;
  static constexpr size_t kMoreBytes = (size_t)256 << 10;
  // what an object has to copy before a pool is made for it (one that is
  // there already is used at once): making it, 32 MB of pinned memory and the
  // threads, costs about what the pool saves on 8 MB.  Opening and closing a
  // model of 1.6 MB: 310 us without one, 500 with it
  static constexpr size_t kMakeBytes = (size_t)8 << 20;
  // How long a thread looks for pieces before it sleeps: past the gap between
  // two slots' arrivals (75 us on the link) and past short kernels between a
  // call's copies in and out (MoE of 8192 tokens, 280 us of kernels, against
  // threads that never sleep: 1753 / 1714 us with 300 us here, 1708 / 1715 with
  // 600), below a wait for long ones.
  static constexpr int kIdleUs = 600;

  ~HostPool();

 private:
  friend class HostCopy;
  friend std::shared_ptr<HostPool> host_pool(int device, bool make);
  struct Task {  // (read by threads that may then fail to claim it, hence atomic)
    std::atomic<void*> dst;
    std::atomic<const void*> src;
    std::atomic<size_t> n;
    std::atomic<std::atomic<int>*> left;
  };
  struct Slot {
    char* mem = nullptr;
    hipEvent_t ev = nullptr;
    bool in_flight = false;      // a copy between the slot and the device is queued; ev follows it
    std::atomic<int> left{0};    // pieces between the slot and the host not yet copied
    char* host = nullptr;        // device to host: where the slot's bytes go once ev has passed
    size_t n = 0;
  };
  HostPool() = default;
  bool init(int device);
  void run();                    // a thread's loop
  bool step();                   // copies one queued piece; false if there is none
  void push(void* dst, const void* src, size_t n, std::atomic<int>* left);
  void wake();                   // sleeping threads look for pieces again, for kIdleUs at least

  static constexpr int kRing = 256;
  std::mutex use_;               // held by the HostCopy in hand
  char* mem_ = nullptr;
  Slot slots_[kSlots];
  int next_ = 0;
  std::atomic<int> touched_{0};  // first touches queued and not yet done
  Task ring_[kRing];
  std::atomic<unsigned> head_{0}, tail_{0};
  std::mutex mu_;
  std::condition_variable cv_;
  std::atomic<int> asleep_{0};
  std::atomic<unsigned> calls_{0};  // wake()s so far
  std::atomic<bool> stop_{false};
  hipEvent_t ahead_ = nullptr;      // after what a call's first copy to the host waits for
  std::vector<std::thread> threads_;
};

// The device's pool; null if there is none and it is not to be (or cannot be)
// made: then hipMemcpyAsync serves.
std::shared_ptr<HostPool> host_pool(int device, bool make);

// An object's hold on its device's pool, and the large copies it had without one.
struct HostPoolRef {
  std::shared_ptr<HostPool> pool;
  size_t bytes = 0;
};

// The copies of one call, on one stream.  up() returns once the source may be
// reused; down() queues, and finish() waits until every destination is
// written.  Copies take their place in the stream's order.
class HostCopy {
 public:
  // ref: the calling object's, filled by the copy from which the pool pays
  // many: the call has eight copies or more, or larger ones to come
  HostCopy(HostPoolRef* ref, int device, hipStream_t st, bool many = false)
      : ref_(ref), device_(device), st_(st), min_(many ? HostPool::kMoreBytes : HostPool::kMinBytes) {}
  ~HostCopy();
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  hipError_t up(void* dst, const void* src, size_t n);
  hipError_t down(void* dst, const void* src, size_t n);
  // poll: wait for the stream as stream_wait does; else hipStreamSynchronize,
  // which is quicker (by 6 us) where only short kernels follow an upload
  hipError_t finish(bool poll = true);

 private:
  bool take(const void* host, size_t n);          // whether this copy goes through the pool
  hipError_t free_slot(HostPool::Slot** s);       // the next slot, once nothing uses it
  hipError_t pass(HostPool::Slot* s);             // a device-to-host slot whose event has passed: hand out its pieces
  void drain(std::atomic<int>* left);             // copy pieces until *left is 0
  hipError_t pass_first();
  hipError_t wait(hipEvent_t ev);                 // copies pieces meanwhile
  void split(char* dst, const char* src, size_t n, std::atomic<int>* left);
  HostPoolRef* ref_;
  int device_;
  hipStream_t st_;
  size_t min_;                                    // least copy for which the pool is taken
  HostPool* p_ = nullptr;                         // locked
  bool busy_ = false;                             // another thread has the pool, or there is none: not asked again
  int pending_[HostPool::kSlots];                 // slots queued to the host: n_pending_ from first_, oldest first
  int first_ = 0, n_pending_ = 0;
  bool down_ = false;                             // p_->ahead_ is recorded, by the first copy to the host ...
  bool ahead_ = false;                            // ... and not yet waited for
};

}  // namespace ane
