// hostcopy.hip -- see hostcopy.hpp (host code only).
#include "hostcopy.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace pyro {
namespace {

// Four threads with two 4 MiB slots each.  Two arrays of 256^3 doubles in (268
// MB) and one back (134 MB) took 9.9 + 13.4 ms through the runtime and 5.9 + 3.7
// ms this way, 6.9 + 4.7 with eight 2 MiB pairs and 12.4 + 6.4 with 512 KiB ones
// (each chunk costs the link about 20 us); eight 4 MiB pairs gain nothing.
// Making the pool and giving it back costs about 0.4 ms, so a handle that is
// made, solves once and is closed breaks even at 9 MB an array (104^3: its
// copies and its closing 3.00 ms before, 3.05 now) and gains from there (128^3
// 4.7, 4.2; 160^3 8.2, 6.4).
constexpr unsigned THREADS = 4;      // workers, the calling thread among them
constexpr size_t CHUNK = 4u << 20;   // bytes of a slot; two slots a worker
constexpr size_t SMALL = 8u << 20;   // below this the runtime's copy is as fast

class Pool {
 public:
  // nullptr where threads or pinned memory cannot be had
  static std::unique_ptr<Pool> make() {
    std::unique_ptr<Pool> p(new (std::nothrow) Pool);
    if (!p) return nullptr;
    if (hipHostMalloc(&p->slots_, 2 * CHUNK * THREADS, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      p->slots_ = nullptr;
      return nullptr;
    }
    try {
      for (unsigned k = 1; k < THREADS; k++) p->threads_.emplace_back(&Pool::loop, p.get(), k);
    } catch (const std::exception &) {
      return nullptr;  // the destructor ends those that started
    }
    return p;
  }
  ~Pool() {
    {
      std::lock_guard<std::mutex> l(m_);
      end_ = true;
    }
    go_.notify_all();
    for (std::thread &t : threads_) t.join();
    // copies in still read their slots
    for (Event &e : ev_)
      if (e.e) {
        (void)hipEventSynchronize(e.e);
        (void)hipEventDestroy(e.e);
      }
    if (slots_) (void)hipHostFree(slots_);
  }
  hipError_t run(char *dst, const char *src, size_t bytes, hipStream_t s, bool in) {
    // the slots' events are of the stream's device, which the caller need not
    // have made current
    int cur = 0;
    hipDevice_t dev = 0;
    hipError_t e = hipStreamGetDevice(s, &dev);
    if (e == hipSuccess) e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
    if (e != hipSuccess) return e;
    {
      std::lock_guard<std::mutex> l(m_);
      job_ = Job{dst, src, bytes, s, in, dev};
      err_ = hipSuccess;
      left_ = THREADS - 1;
      seq_++;
    }
    go_.notify_all();
    work(0);
    std::unique_lock<std::mutex> l(m_);
    done_.wait(l, [&] { return left_ == 0; });
    if (cur != dev) note_locked(hipSetDevice(cur));
    return err_;
  }

 private:
  struct Job {
    char *dst;
    const char *src;
    size_t bytes;
    hipStream_t s;
    bool in;
    int dev;
  };
  struct Event {
    hipEvent_t e = nullptr;
    int dev = -1;
    bool pending = false;  // a copy recorded before it may still use the slot
  };
  void loop(unsigned k) {
    unsigned long seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> l(m_);
        go_.wait(l, [&] { return end_ || seq_ != seen; });
        if (end_) return;
        seen = seq_;
      }
      (void)hipSetDevice(job_.dev);
      work(k);
      std::lock_guard<std::mutex> l(m_);
      if (--left_ == 0) done_.notify_one();
    }
  }
  void note_locked(hipError_t e) {
    if (err_ == hipSuccess) err_ = e;
  }
  void note(hipError_t e) {
    if (e == hipSuccess) return;
    std::lock_guard<std::mutex> l(m_);
    note_locked(e);
  }
  // waits until slot j is free, and has an event of the job's device for it
  hipError_t ready(unsigned j, int dev) {
    Event &v = ev_[j];
    if (v.pending) {
      v.pending = false;
      hipError_t e = hipEventSynchronize(v.e);
      if (e != hipSuccess) return e;
    }
    if (v.e && v.dev != dev) {
      (void)hipEventDestroy(v.e);
      v.e = nullptr;
    }
    if (!v.e) {
      v.dev = dev;
      return hipEventCreateWithFlags(&v.e, hipEventDisableTiming);
    }
    return hipSuccess;
  }
  // chunks k, k + THREADS, ... of the job, alternating between two slots
  void work(unsigned k) {
    const Job j = job_;
    size_t behind = 0, blen = 0;  // copy out: the chunk whose slot is still to be emptied
    int bslot = -1;
    auto empty = [&]() -> hipError_t {
      if (bslot < 0) return hipSuccess;
      ev_[bslot].pending = false;
      hipError_t e = hipEventSynchronize(ev_[bslot].e);
      if (e == hipSuccess) std::memcpy(j.dst + behind, slot(bslot), blen);
      bslot = -1;
      return e;
    };
    unsigned turn = 0;
    for (size_t off = k * CHUNK; off < j.bytes; off += CHUNK * THREADS, turn ^= 1u) {
      const unsigned sl = 2 * k + turn;
      const size_t len = std::min(CHUNK, j.bytes - off);
      hipError_t e = ready(sl, j.dev);
      if (e == hipSuccess && j.in) {
        std::memcpy(slot(sl), j.src + off, len);
        e = hipMemcpyAsync(j.dst + off, slot(sl), len, hipMemcpyHostToDevice, j.s);
      } else if (e == hipSuccess) {
        e = hipMemcpyAsync(slot(sl), j.src + off, len, hipMemcpyDeviceToHost, j.s);
      }
      if (e == hipSuccess) {
        e = hipEventRecord(ev_[sl].e, j.s);
        ev_[sl].pending = e == hipSuccess;
      }
      if (e == hipSuccess && !j.in) {
        e = empty();
        bslot = (int)sl;
        behind = off;
        blen = len;
      }
      if (e != hipSuccess) {
        note(e);
        return;
      }
    }
    if (!j.in) note(empty());
  }
  char *slot(unsigned j) { return static_cast<char *>(slots_) + j * CHUNK; }

  std::mutex m_;
  std::condition_variable go_, done_;
  std::vector<std::thread> threads_;
  Job job_{};
  hipError_t err_ = hipSuccess;
  unsigned left_ = 0;
  unsigned long seq_ = 0;
  bool end_ = false;
  void *slots_ = nullptr;
  Event ev_[2 * THREADS];
};

std::mutex g_mu;                // the pool's life and its use: one copy at a time
Pool *g_pool = nullptr;         // plain: never destroyed by the process's end, when the runtime may be gone
std::atomic<int> g_uses{0};

hipError_t copy(void *dst, const void *src, size_t bytes, hipStream_t s, bool in, bool later) {
  if (bytes >= SMALL) {
    std::unique_lock<std::mutex> l(g_mu, std::try_to_lock);
    if (l.owns_lock() && g_uses.load() > 0) {
      if (!g_pool) g_pool = Pool::make().release();
      if (g_pool) return g_pool->run(static_cast<char *>(dst), static_cast<const char *>(src), bytes, s, in);
    }
  }
  hipError_t e = hipMemcpyAsync(dst, src, bytes, in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
  return e == hipSuccess && !later ? hipStreamSynchronize(s) : e;
}
}  // namespace

HostCopyUse::HostCopyUse() { g_uses.fetch_add(1); }
HostCopyUse::~HostCopyUse() {
  if (g_uses.fetch_sub(1) != 1) return;
  std::lock_guard<std::mutex> l(g_mu);
  if (g_uses.load() != 0) return;
  delete g_pool;
  g_pool = nullptr;
}

hipError_t copy_in(void *dst, const void *src, size_t bytes, hipStream_t s, bool later) {
  return copy(dst, src, bytes, s, true, later);
}
hipError_t copy_out(void *dst, const void *src, size_t bytes, hipStream_t s) {
  return copy(dst, src, bytes, s, false, false);
}

}  // namespace pyro
