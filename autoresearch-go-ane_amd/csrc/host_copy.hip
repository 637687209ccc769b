#include "host_copy.h"

#include "hip_common.h"

#include <string.h>

#include <algorithm>
#include <chrono>

namespace ane {

namespace {
inline void pause_cpu() { __builtin_ia32_pause(); }

// First touch of a page about to be written: a write that changes nothing.
// One locked instruction, so that a copy which another thread has meanwhile
// made to this byte stays (a load and a store could put the old byte back);
// in asm, as the compiler turns an atomic "or 0" into a fence and a load,
// which gives the page no memory of its own.
inline void touch_page(void* p) {
  asm volatile("lock orb $0, %0" : "+m"(*(char*)p) : : "memory", "cc");
}

std::mutex g_pools_mu;
constexpr int kMaxDevices = 64;
constexpr uintptr_t kPage = (uintptr_t)2 << 20;  // a transparent huge page
std::weak_ptr<HostPool> g_pools[kMaxDevices];
}  // namespace

std::shared_ptr<HostPool> host_pool(int device, bool make) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_pools_mu);
  if (auto p = g_pools[device].lock()) return p;
  if (!make) return nullptr;
  try {
    std::shared_ptr<HostPool> p(new HostPool());
    if (!p->init(device)) return nullptr;
    g_pools[device] = p;
    return p;
  } catch (...) {
    return nullptr;
  }
}

bool HostPool::init(int device) {
  // (a failure is cleared: the copy that asked goes through hipMemcpyAsync)
  int prev = -1;
  if (hipGetDevice(&prev) != hipSuccess || (prev != device && hipSetDevice(device) != hipSuccess)) {
    (void)hipGetLastError();
    return false;
  }
  struct Restore {
    int prev, now;
    ~Restore() {
      if (prev != now) (void)hipSetDevice(prev);
    }
  } restore{prev, device};
  if (hipHostMalloc((void**)&mem_, kSlots * kSlotBytes, hipHostMallocDefault) != hipSuccess) {
    mem_ = nullptr;
    (void)hipGetLastError();
    return false;
  }
  auto event = [](hipEvent_t* ev) {
    if (hipEventCreateWithFlags(ev, hipEventDisableTiming | (spin_waits() ? 0 : hipEventBlockingSync)) == hipSuccess)
      return true;
    *ev = nullptr;
    (void)hipGetLastError();
    return false;
  };
  if (!event(&ahead_)) return false;
  for (int i = 0; i < kSlots; i++) {
    slots_[i].mem = mem_ + i * kSlotBytes;
    if (!event(&slots_[i].ev)) return false;
  }
  try {
    const unsigned hw = std::thread::hardware_concurrency();
    const int n = std::max(1, std::min(kThreads, hw > 2 ? (int)hw - 2 : 1));
    for (int i = 0; i < n; i++) threads_.emplace_back([this] { run(); });
  } catch (...) {
    // fewer threads (or none): the copying thread works too
  }
  return true;
}

HostPool::~HostPool() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    stop_ = true;
  }
  cv_.notify_all();
  for (std::thread& t : threads_) t.join();
  for (Slot& s : slots_)
    if (s.ev) {
      if (s.in_flight) (void)hipEventSynchronize(s.ev);
      (void)hipEventDestroy(s.ev);
    }
  if (ahead_) (void)hipEventDestroy(ahead_);
  if (mem_) (void)hipHostFree(mem_);
}

// Looks for pieces while there are any and for kIdleUs after the last one or
// the last wake(), then sleeps: a call that waits for kernels keeps no thread busy.
void HostPool::run() {
  using clock = std::chrono::steady_clock;
  unsigned seen = 0;
  for (;;) {
    for (clock::time_point since = clock::now();;) {
      const unsigned c = calls_.load(std::memory_order_acquire);
      const bool worked = step();
      if (worked || c != seen) {
        seen = c;
        since = clock::now();
        continue;
      }
      if (stop_ || clock::now() - since > std::chrono::microseconds(kIdleUs)) break;
      for (int i = 0; i < 32; i++) pause_cpu();
    }
    {
      std::unique_lock<std::mutex> lk(mu_);
      asleep_.fetch_add(1);
      cv_.wait(lk, [&] { return stop_ || calls_.load() != seen; });
      asleep_.fetch_sub(1);
      if (stop_) return;
    }
    // the next two sleepers (the caller wakes one thread, not all: ~12 us each)
    cv_.notify_one();
    cv_.notify_one();
  }
}

bool HostPool::step() {
  unsigned h = head_.load(std::memory_order_acquire);
  while (h != tail_.load(std::memory_order_acquire)) {
    const Task& t = ring_[h % kRing];  // what is read is this piece's if the claim succeeds: push() reuses no entry that head has not passed
    void* dst = t.dst.load(std::memory_order_relaxed);
    const void* src = t.src.load(std::memory_order_relaxed);
    const size_t n = t.n.load(std::memory_order_relaxed);
    std::atomic<int>* left = t.left.load(std::memory_order_relaxed);
    if (head_.compare_exchange_weak(h, h + 1, std::memory_order_acq_rel)) {
      if (src) {
        memcpy(dst, src, n);
      } else {
        touch_page(dst);
      }
      left->fetch_sub(1, std::memory_order_release);
      return true;
    }
  }
  return false;
}

void HostPool::push(void* dst, const void* src, size_t n, std::atomic<int>* left) {
  const unsigned t = tail_.load(std::memory_order_relaxed);
  while (t - head_.load(std::memory_order_acquire) >= kRing) step();  // full: this thread works too
  Task& k = ring_[t % kRing];
  k.dst.store(dst, std::memory_order_relaxed);
  k.src.store(src, std::memory_order_relaxed);
  k.n.store(n, std::memory_order_relaxed);
  k.left.store(left, std::memory_order_relaxed);
  tail_.store(t + 1, std::memory_order_release);
}

// A thread counts itself asleep before it reads calls_ for the last time, and
// here calls_ changes before asleep_ is read: one of the two sees the other.
void HostPool::wake() {
  calls_.fetch_add(1);
  if (asleep_.load() == 0) return;
  { std::lock_guard<std::mutex> lk(mu_); }  // (a thread between its read and its wait)
  cv_.notify_one();
}

// ---- one call's copies ---------------------------------------------------------

bool HostCopy::take(const void* host, size_t n) {
  if (n < (p_ ? HostPool::kMoreBytes : min_) || busy_) return false;
  // memory the runtime already has pinned (or managed) is copied directly
  hipPointerAttribute_t at;
  memset(&at, 0, sizeof at);
  if (hipPointerGetAttributes(&at, host) != hipSuccess) (void)hipGetLastError();
  else if (at.type != hipMemoryTypeUnregistered) return false;
  if (p_) return true;
  if (!ref_->pool) {
    ref_->bytes = std::min(ref_->bytes + n, HostPool::kMakeBytes);
    const bool make = ref_->bytes == HostPool::kMakeBytes;
    ref_->pool = host_pool(device_, make);
    if (!ref_->pool) {
      busy_ = make;  // (it cannot be made: not tried again by this call)
      return false;
    }
  }
  if (!ref_->pool->use_.try_lock()) {
    busy_ = true;
    return false;
  }
  p_ = ref_->pool.get();
  p_->next_ = 0;  // (the slots of small calls stay in the caches, and later ones are not paged in for them)
  return true;
}

void HostCopy::drain(std::atomic<int>* left) {
  while (left->load(std::memory_order_acquire) > 0)
    if (!p_->step()) pause_cpu();
}

void HostCopy::split(char* dst, const char* src, size_t n, std::atomic<int>* left) {
  const int k = (int)((n + HostPool::kTaskBytes - 1) / HostPool::kTaskBytes);
  left->fetch_add(k, std::memory_order_relaxed);
  for (size_t o = 0; o < n; o += HostPool::kTaskBytes)
    p_->push(dst + o, src + o, std::min(HostPool::kTaskBytes, n - o), left);
  p_->wake();
}

hipError_t HostCopy::wait(hipEvent_t ev) {
  hipError_t h;
  while ((h = hipEventQuery(ev)) == hipErrorNotReady) {
    if (p_->step()) continue;
    if (!spin_waits()) return hipEventSynchronize(ev);
    pause_cpu();
  }
  return h;
}

hipError_t HostCopy::pass(HostPool::Slot* s) {
  hipError_t h = hipSuccess;
  if (ahead_) {  // the link starts now: threads that slept through the kernels wake meanwhile
    h = wait(p_->ahead_);
    ahead_ = false;
    p_->wake();
  }
  if (h == hipSuccess) h = wait(s->ev);
  s->in_flight = false;
  if (h == hipSuccess && s->host) split(s->host, s->mem, s->n, &s->left);
  s->host = nullptr;
  return h;
}

hipError_t HostCopy::pass_first() {
  HostPool::Slot* s = &p_->slots_[pending_[first_]];
  first_ = (first_ + 1) % HostPool::kSlots;
  n_pending_--;
  return pass(s);
}

hipError_t HostCopy::free_slot(HostPool::Slot** out) {
  HostPool::Slot* s = &p_->slots_[p_->next_];
  p_->next_ = (p_->next_ + 1) % HostPool::kSlots;
  hipError_t h = hipSuccess;
  if (s->in_flight) {  // the oldest: slots are used in turn
    h = n_pending_ > 0 && &p_->slots_[pending_[first_]] == s ? pass_first() : pass(s);
  }
  drain(&s->left);
  *out = s;
  return h;
}

hipError_t HostCopy::up(void* dst, const void* src, size_t n) {
  if (!take(src, n)) return hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st_);
  for (size_t o = 0; o < n; o += HostPool::kSlotBytes) {
    const size_t k = std::min(HostPool::kSlotBytes, n - o);
    HostPool::Slot* s;
    hipError_t h = free_slot(&s);
    if (h != hipSuccess) return h;
    split(s->mem, (const char*)src + o, k, &s->left);
    drain(&s->left);
    if ((h = hipMemcpyAsync((char*)dst + o, s->mem, k, hipMemcpyHostToDevice, st_)) != hipSuccess) return h;
    if ((h = hipEventRecord(s->ev, st_)) != hipSuccess) return h;
    s->in_flight = true;
    s->host = nullptr;
  }
  return hipSuccess;
}

hipError_t HostCopy::down(void* dst, const void* src, size_t n) {
  if (!take(dst, n)) return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st_);
  if (!down_) {
    const hipError_t h = hipEventRecord(p_->ahead_, st_);
    if (h != hipSuccess) return h;
    down_ = ahead_ = true;
  }
  // A buffer the caller has just allocated has no pages yet.  Each is touched
  // by one thread before its bytes arrive: left to the copies, several
  // threads would fault the same 2 MB page and each clear one for it.
  const uintptr_t end = (uintptr_t)dst + n;
  uintptr_t touch = n >= 2 * kPage ? (uintptr_t)dst : end;
  auto touch_to = [&](uintptr_t upto) {
    if (touch >= std::min(upto, end)) return;
    for (; touch < std::min(upto, end); touch = (touch | (kPage - 1)) + 1) {
      p_->touched_.fetch_add(1, std::memory_order_relaxed);
      p_->push((void*)touch, nullptr, 0, &p_->touched_);
    }
    p_->wake();
  };
  for (size_t o = 0; o < n; o += HostPool::kSlotBytes) {
    const size_t k = std::min(HostPool::kSlotBytes, n - o);
    touch_to((uintptr_t)dst + o + 8 * kPage);
    HostPool::Slot* s;
    hipError_t h = free_slot(&s);
    if (h != hipSuccess) return h;
    if ((h = hipMemcpyAsync(s->mem, (const char*)src + o, k, hipMemcpyDeviceToHost, st_)) != hipSuccess) return h;
    if ((h = hipEventRecord(s->ev, st_)) != hipSuccess) return h;
    s->in_flight = true;
    s->host = (char*)dst + o;
    s->n = k;
    pending_[(first_ + n_pending_++) % HostPool::kSlots] = (int)(s - p_->slots_);
    // hand out what has arrived meanwhile
    while (n_pending_ > 0 && hipEventQuery(p_->slots_[pending_[first_]].ev) == hipSuccess)
      if ((h = pass_first()) != hipSuccess) return h;
  }
  return hipSuccess;
}

hipError_t HostCopy::finish(bool poll) {
  hipError_t h = hipSuccess;
  if (p_) {
    while (n_pending_ > 0) {
      const hipError_t r = pass_first();
      if (h == hipSuccess) h = r;
    }
    for (HostPool::Slot& s : p_->slots_) drain(&s.left);
    drain(&p_->touched_);
  }
  const hipError_t r = poll ? stream_wait(st_) : hipStreamSynchronize(st_);
  return h == hipSuccess ? r : h;
}

HostCopy::~HostCopy() {
  if (!p_) return;
  // after an error: no destination is written once the call has returned
  for (; n_pending_ > 0; n_pending_--, first_ = (first_ + 1) % HostPool::kSlots) {
    HostPool::Slot& s = p_->slots_[pending_[first_]];
    (void)hipEventSynchronize(s.ev);
    s.in_flight = false;
    s.host = nullptr;
  }
  for (HostPool::Slot& s : p_->slots_) drain(&s.left);
  drain(&p_->touched_);
  p_->use_.unlock();
}

}  // namespace ane
