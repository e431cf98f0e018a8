// Copies between the caller's host arrays and the device, and the device
// blocks of the per-call entry points.
//
// The caller's arrays are ordinary pageable memory.  hipMemcpy moves those
// through the runtime's own bounce buffers on one host thread, which also
// takes the page faults of a freshly allocated destination: 10 GB/s out of a
// link that carries 57 GB/s from pinned memory (520 MB of a 100^3 system's
// state: 50 ms, as long as 50 collision intervals).  Here the link works from
// a ring of pinned slots and several host threads move the slots to or from
// the caller's memory.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <deque>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>
#include "mpcx_host.h"
#include "mpcx_stage.h"
#include "../../include/mpcx.h"

namespace mpcx {
namespace {

constexpr size_t SLOT = 2u << 20;        // bytes of a slot (device side)
constexpr int NSLOT = 16;                // 32 MB pinned, one ring a process
constexpr size_t MIN_STAGED = 1u << 20;  // below this hipMemcpy's latency is the smaller one
constexpr size_t PER_WORKER = 4u << 20;  // bytes that pay for starting one more host thread (about 20 us)
constexpr int MAX_WORKERS = 8;

struct Ring {
  std::mutex mu;   // one staged copy at a time; a second caller takes hipMemcpy
  char* pin = nullptr;
  hipEvent_t ev[NSLOT] = {nullptr};
  int dev = -1;
};
Ring g_ring;

void events_release() {
  for (auto& e : g_ring.ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  g_ring.dev = -1;
}
void ring_release() {
  if (g_ring.pin) (void)hipHostFree(g_ring.pin);
  g_ring.pin = nullptr;
  events_release();
}
// the ring on the current device, or false (the caller copies plainly): no
// pinned memory to be had, or a stream of another device, whose work the
// ring's events cannot mark.  The slots serve every device; only the events
// are made anew for another one.
bool ring_ready(hipStream_t st) {
  int dev = -1, sdev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  if (st && (hipStreamGetDevice(st, &sdev) != hipSuccess || sdev != dev)) {
    (void)hipGetLastError();
    return false;
  }
  if (!g_ring.pin && hipHostMalloc((void**)&g_ring.pin, SLOT * NSLOT, hipHostMallocPortable) != hipSuccess) {
    g_ring.pin = nullptr;
    (void)hipGetLastError();
    return false;
  }
  if (g_ring.dev == dev) return true;
  events_release();
  for (auto& e : g_ring.ev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      e = nullptr;
      (void)hipGetLastError();
      events_release();
      return false;
    }
  g_ring.dev = dev;
  return true;
}

struct Chunk {
  char* host;
  char* dev;
  size_t n;      // bytes on the device
  bool widen;    // int32 on the device, int64 on the host
};
void move_out(const Chunk& c, const char* slot) {
  if (!c.widen) {
    memcpy(c.host, slot, c.n);
    return;
  }
  const int32_t* s = (const int32_t*)slot;
  int64_t* d = (int64_t*)c.host;
  for (size_t i = 0; i < c.n / 4; i++) d[i] = s[i];
}

// Host threads that move slots; with none (small copies, or no thread to be
// had) the caller's thread does it in post().  Nothing here allocates once the
// threads run: a slot has at most one job.
class Movers {
 public:
  explicit Movers(int n) {
    for (auto& b : busy_) b.store(0);
    for (; n_ < n; n_++) {
      try {
        th_[n_] = std::thread([this] { work(); });
      } catch (const std::exception&) {   // no thread or no memory for it
        break;
      }
    }
  }
  ~Movers() {
    {
      std::lock_guard<std::mutex> l(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (int i = 0; i < n_; i++) th_[i].join();
  }
  void post(int slot, const Chunk& c, bool out) {
    if (n_ == 0) {
      run(slot, c, out);
      return;
    }
    busy_[slot].store(1);
    {
      std::lock_guard<std::mutex> l(mu_);
      q_[tail_++ % NSLOT] = Job{slot, c, out};
    }
    cv_.notify_one();
  }
  void wait(int slot) {
    if (!busy_[slot].load()) return;
    std::unique_lock<std::mutex> l(mu_);
    done_.wait(l, [&] { return !busy_[slot].load(); });
  }

 private:
  struct Job {
    int slot;
    Chunk c;
    bool out;
  };
  static void run(int slot, const Chunk& c, bool out) {
    char* p = g_ring.pin + (size_t)slot * SLOT;
    if (out) move_out(c, p);
    else memcpy(p, c.host, c.n);
  }
  void work() {
    std::unique_lock<std::mutex> l(mu_);
    while (true) {
      cv_.wait(l, [&] { return stop_ || head_ != tail_; });
      if (head_ == tail_) return;
      const Job j = q_[head_++ % NSLOT];
      l.unlock();
      run(j.slot, j.c, j.out);
      l.lock();
      busy_[j.slot].store(0);
      done_.notify_all();
    }
  }
  std::thread th_[MAX_WORKERS];
  int n_ = 0;
  Job q_[NSLOT];
  unsigned head_ = 0, tail_ = 0;
  std::mutex mu_;
  std::condition_variable cv_, done_;
  bool stop_ = false;
  std::atomic<int> busy_[NSLOT];
};

int plain(const std::vector<HostCopy>& v, bool out, hipStream_t st) {
  std::vector<int32_t> narrow;
  for (const HostCopy& c : v) {
    if (!c.host || !c.bytes) continue;
    hipError_t r;
    if (c.widen) {
      narrow.resize(c.bytes / 4);
      r = hipMemcpyAsync(narrow.data(), c.dev, c.bytes, hipMemcpyDeviceToHost, st);
      if (r == hipSuccess) r = hipStreamSynchronize(st);
      if (r == hipSuccess)
        for (size_t i = 0; i < narrow.size(); i++) ((int64_t*)c.host)[i] = narrow[i];
    } else {
      r = out ? hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, st)
              : hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, st);
    }
    if (r != hipSuccess) {
      (void)hipStreamSynchronize(st);
      return set_error(MPCX_E_HIP, hipGetErrorString(r));
    }
  }
  const hipError_t r = hipStreamSynchronize(st);
  return r == hipSuccess ? 0 : set_error(MPCX_E_HIP, hipGetErrorString(r));
}

int staged(const std::vector<HostCopy>& v, bool out, hipStream_t st, size_t total) {
  std::vector<Chunk> ch;
  for (const HostCopy& c : v) {
    if (!c.host) continue;
    for (size_t o = 0; o < c.bytes; o += SLOT)
      ch.push_back(Chunk{(char*)c.host + (c.widen ? 2 * o : o), (char*)c.dev + o, std::min(SLOT, c.bytes - o), c.widen});
  }
  const int n = (int)ch.size();
  hipError_t r = hipSuccess;
  {
    const int w = total < 2 * PER_WORKER ? 0 : (int)std::min<size_t>(MAX_WORKERS, total / PER_WORKER);
    Movers mv(w);
    auto slot = [](int i) { return i % NSLOT; };
    if (out) {
      constexpr int AHEAD = NSLOT / 2;   // link copies in flight; the other half of the ring is with the movers
      for (int i = 0; i < n + AHEAD && r == hipSuccess; i++) {
        if (i < n) {
          mv.wait(slot(i));
          r = hipMemcpyAsync(g_ring.pin + (size_t)slot(i) * SLOT, ch[i].dev, ch[i].n, hipMemcpyDeviceToHost, st);
          if (r == hipSuccess) r = hipEventRecord(g_ring.ev[slot(i)], st);
        }
        const int j = i - AHEAD;
        if (r == hipSuccess && j >= 0 && j < n) {
          r = hipEventSynchronize(g_ring.ev[slot(j)]);
          if (r == hipSuccess) mv.post(slot(j), ch[j], true);
        }
      }
    } else {
      for (int i = 0; i < n + NSLOT / 2 && r == hipSuccess; i++) {
        if (i < n) {
          if (i >= NSLOT) r = hipEventSynchronize(g_ring.ev[slot(i)]);   // the slot's last chunk has left it
          if (r == hipSuccess) mv.post(slot(i), ch[i], false);
        }
        const int j = i - NSLOT / 2;
        if (r == hipSuccess && j >= 0 && j < n) {
          mv.wait(slot(j));
          r = hipMemcpyAsync(ch[j].dev, g_ring.pin + (size_t)slot(j) * SLOT, ch[j].n, hipMemcpyHostToDevice, st);
          if (r == hipSuccess) r = hipEventRecord(g_ring.ev[slot(j)], st);
        }
      }
    }
  }   // the movers are done
  const hipError_t s = hipStreamSynchronize(st);   // the ring is free for the next copy
  if (r == hipSuccess) r = s;
  return r == hipSuccess ? 0 : set_error(MPCX_E_HIP, hipGetErrorString(r));
}

// Memory that the runtime knows (pinned, managed, a device's) goes over the link
// as it is: the ring is for pageable memory, and its host threads are slower
// than the link (67 MB read into a pinned array: 1.86 ms through the ring, 1.19 ms so).
bool pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

int copy(const std::vector<HostCopy>& v, bool out, hipStream_t st) {
  size_t all = 0, total = 0;
  for (const HostCopy& c : v)
    if (c.host) all += c.bytes;
  if (all < MIN_STAGED) return plain(v, out, st);
  std::vector<HostCopy> ring, rest;
  for (const HostCopy& c : v) {
    if (!c.host || !c.bytes) continue;
    const bool r = c.widen || pageable(c.host);   // (widening is host work whatever the memory)
    (r ? ring : rest).push_back(c);
    if (r) total += c.bytes;
  }
  if (total >= MIN_STAGED) {
    std::unique_lock<std::mutex> l(g_ring.mu, std::try_to_lock);
    if (l.owns_lock() && ring_ready(st)) {
      const int rc = rest.empty() ? 0 : plain(rest, out, st);
      return rc ? rc : staged(ring, out, st, total);
    }
  }
  return plain(v, out, st);
}

// ------------------------------------------------------------ device blocks
struct Block {
  void* p;
  size_t n;
  int dev;
};
std::mutex g_blocks_mu;
std::deque<Block> g_blocks;   // free blocks, the longest unused first, at most CACHE_MAX bytes
size_t g_blocks_bytes = 0;
constexpr size_t CACHE_MAX = 512u << 20;

size_t block_bytes(size_t n) { return (std::max<size_t>(n, 256) + 255) / 256 * 256; }

}  // namespace

// (called below C entry points: no exception may pass)
static int copy_noexcept(const std::vector<HostCopy>& v, bool out, hipStream_t st) {
  try {
    return copy(v, out, st);
  } catch (const std::bad_alloc&) {
    (void)hipStreamSynchronize(st);   // copies on their way still use the caller's arrays
    return set_error(MPCX_E_HIP, "out of host memory");
  }
}
int copy_out(const std::vector<HostCopy>& v, hipStream_t st) { return copy_noexcept(v, true, st); }
int copy_in(const std::vector<HostCopy>& v, hipStream_t st) { return copy_noexcept(v, false, st); }

// Every device allocation of the library comes through here: memory that only
// the cache holds must not make one fail.
hipError_t device_alloc_bytes(void** p, size_t n) {
  hipError_t r = hipMalloc(p, n);
  if (r == hipSuccess) return r;
  (void)hipGetLastError();
  {
    std::lock_guard<std::mutex> l(g_blocks_mu);
    if (g_blocks.empty()) return r;
  }
  blocks_release();
  r = hipMalloc(p, n);
  if (r != hipSuccess) (void)hipGetLastError();
  return r;
}

// The smallest free block that holds n bytes and is at most twice that (a new
// one otherwise).  The entry points that use these run on the null stream, so
// a block's next user is ordered after its last.
void* block_get(size_t n, size_t* got) {
  n = block_bytes(n);
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  {
    std::lock_guard<std::mutex> l(g_blocks_mu);
    size_t best = g_blocks.size();
    for (size_t i = 0; i < g_blocks.size(); i++)
      if (g_blocks[i].dev == dev && g_blocks[i].n >= n && g_blocks[i].n <= 2 * n &&
          (best == g_blocks.size() || g_blocks[i].n < g_blocks[best].n))
        best = i;
    if (best < g_blocks.size()) {
      void* p = g_blocks[best].p;
      *got = g_blocks[best].n;
      g_blocks_bytes -= g_blocks[best].n;
      g_blocks.erase(g_blocks.begin() + (long)best);
      return p;
    }
  }
  void* p = nullptr;
  if (device_alloc_bytes(&p, n) != hipSuccess) return nullptr;
  *got = n;
  return p;
}
// A block that does not fit drives out the longest unused ones: a driver that
// goes on with another system's sizes keeps those, not the last system's.
void block_put(void* p, size_t n) {
  if (!p) return;
  int dev = -1;
  bool kept = false;
  if (n <= CACHE_MAX && hipGetDevice(&dev) == hipSuccess) {
    std::lock_guard<std::mutex> l(g_blocks_mu);
    while (g_blocks_bytes + n > CACHE_MAX) {
      (void)hipFree(g_blocks.front().p);
      g_blocks_bytes -= g_blocks.front().n;
      g_blocks.pop_front();
    }
    try {
      g_blocks.push_back(Block{p, n, dev});
      g_blocks_bytes += n;
      kept = true;
    } catch (const std::bad_alloc&) {   // (called by destructors)
    }
  }
  if (!kept) (void)hipFree(p);
}
void blocks_release() {
  std::lock_guard<std::mutex> l(g_blocks_mu);
  for (const Block& b : g_blocks) (void)hipFree(b.p);
  g_blocks.clear();
  g_blocks_bytes = 0;
}
void stage_release() {
  std::lock_guard<std::mutex> l(g_ring.mu);
  ring_release();
}

}  // namespace mpcx
