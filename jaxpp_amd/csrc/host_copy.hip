// Copies between pageable host memory and the device: many tensors a call, converted on the way.
//
// hipMemcpy takes 10 - 20 us for a tensor of up to 256 KB and moves 25 GB/s of a large one to the device, 10 into a fresh
// host array, on one host thread; packing small tensors for it and converting to bf16 are more passes over host memory on the
// caller's thread, and fresh result arrays are paged in there.  Here a call's tensors are cut into chunks that are
// contiguous on the device, and lanes - the caller's thread and up to seven more - take the next chunk each,
// pack it into pinned memory of their own (or unpack it from there, converting) and run its copy on a
// stream of their own, with a second chunk in flight meanwhile.  What is left is the link and the
// host's memory: 8 MB 340 -> 275 us to the device and 495 -> 260 into a fresh host array, 128 MB 27 -> 37 - 49 GB/s and 10 -> 34
// (a single tensor of up to 2 MB stays within 15 % of hipMemcpy).  A train step over host arrays of four layers of
// hidden 256 (118 MB both ways) spent 9 of its 13 ms on these copies, now 4 of 7.
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <map>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include <sched.h>

#include "common.h"

namespace {

constexpr int kLanes = 8;                 // at most; half of the process's CPUs
constexpr size_t kSlot = 1 << 20;         // pinned bytes of a chunk, two per lane
constexpr size_t kLeast = 256 << 10;      // no chunk smaller: an asynchronous copy takes 10 us to issue, one lane at a time
constexpr size_t kAlone = 8 << 20;        // a chunk of a job without lanes

struct Piece {   // consecutive elements of one item
  uint8_t* host;
  int64_t count;
};
struct Chunk {   // pieces that lie one behind the other on the device
  uint8_t* device;
  size_t bytes;
  int first, last;
};
struct Lane {
  hipStream_t stream = nullptr;
  hipEvent_t done[2] = {nullptr, nullptr};
  uint8_t* slot[2] = {nullptr, nullptr};
};
struct Job {
  Lane* lanes = nullptr;
  std::vector<Piece> pieces;
  std::vector<Chunk> chunks;
  bool up = false, bf16 = false;
  int device = 0;
  std::atomic<size_t> next{0};
  std::atomic<int> error{hipSuccess};
};

void pack(uint8_t* dst, const Piece& p, bool bf16) {
  if (!bf16) {
    memcpy(dst, p.host, (size_t)p.count * 4);
    return;
  }
  const uint32_t* src = (const uint32_t*)p.host;
  uint16_t* out = (uint16_t*)dst;
  for (int64_t i = 0; i < p.count; ++i) out[i] = (uint16_t)((src[i] + 0x7fffu + ((src[i] >> 16) & 1u)) >> 16);
}
void unpack(const uint8_t* src, const Piece& p, bool bf16) {
  if (!bf16) {
    memcpy(p.host, src, (size_t)p.count * 4);
    return;
  }
  const uint16_t* in = (const uint16_t*)src;
  uint32_t* out = (uint32_t*)p.host;
  for (int64_t i = 0; i < p.count; ++i) out[i] = (uint32_t)in[i] << 16;
}
void walk(const Job& j, const Chunk& c, uint8_t* slot) {
  const size_t es = j.bf16 ? 2 : 4;
  for (int i = c.first; i < c.last; ++i) {
    if (j.up) pack(slot, j.pieces[i], j.bf16);
    else unpack(slot, j.pieces[i], j.bf16);
    slot += (size_t)j.pieces[i].count * es;
  }
}

// Cuts the items into chunks of at most `cut` bytes (a multiple of 4).
void cut_items(Job& j, int n, const jpp_copy_item* items, size_t cut) {
  const size_t es = j.bf16 ? 2 : 4;
  j.pieces.clear();
  j.chunks.clear();
  for (int i = 0; i < n; ++i) {
    int64_t left = items[i].count;
    uint8_t *h = (uint8_t*)items[i].host, *d = (uint8_t*)items[i].device;
    while (left > 0) {
      if (j.chunks.empty() || j.chunks.back().bytes + es > cut || j.chunks.back().device + j.chunks.back().bytes != d)
        j.chunks.push_back({d, 0, (int)j.pieces.size(), (int)j.pieces.size()});
      Chunk& c = j.chunks.back();
      const int64_t take = std::min(left, (int64_t)((cut - c.bytes) / es));
      j.pieces.push_back({h, take});
      c.last = (int)j.pieces.size();
      c.bytes += (size_t)take * es;
      h += take * 4;
      d += (size_t)take * es;
      left -= take;
    }
  }
}

// A whole job on the caller's thread and the null stream, without lanes: a chunk straight between host and device
// where it is one tensor's words, else through pageable memory.
hipError_t work_alone(const Job& j) {
  std::vector<uint8_t> slot;
  for (const Chunk& c : j.chunks) {
    const bool direct = !j.bf16 && c.last - c.first == 1;
    if (!direct && slot.size() < c.bytes) slot.resize(c.bytes);
    uint8_t* const at = direct ? j.pieces[c.first].host : slot.data();
    if (j.up && !direct) walk(j, c, at);
    const hipError_t e = j.up ? hipMemcpy(c.device, at, c.bytes, hipMemcpyHostToDevice)
                              : hipMemcpy(at, c.device, c.bytes, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return e;
    if (!j.up && !direct) walk(j, c, at);
  }
  return hipSuccess;
}

// One lane's share of a job.  Ends with nothing of it in flight, whatever failed.
void work(Job& j, Lane& l) {
  auto ok = [&](hipError_t e) {
    int none = hipSuccess;
    if (e != hipSuccess) j.error.compare_exchange_strong(none, e);
    return j.error.load() == hipSuccess;
  };
  auto take = [&]() -> const Chunk* {
    const size_t i = j.next.fetch_add(1);
    return i < j.chunks.size() ? &j.chunks[i] : nullptr;
  };
  // (events only where a slot is waited for with something behind it in flight)
  if (j.up) {
    int turn = 0;
    for (const Chunk* c = take(); c; ++turn) {
      const int s = turn & 1;
      if (turn >= 2 && !ok(hipEventSynchronize(l.done[s]))) break;
      walk(j, *c, l.slot[s]);
      if (!ok(hipMemcpyAsync(c->device, l.slot[s], c->bytes, hipMemcpyHostToDevice, l.stream))) break;
      c = take();
      if (c && !ok(hipEventRecord(l.done[s], l.stream))) break;
    }
  } else {
    auto start = [&](const Chunk* c, int s) {
      return ok(hipMemcpyAsync(l.slot[s], c->device, c->bytes, hipMemcpyDeviceToHost, l.stream));
    };
    const Chunk* c = take();
    if (c && start(c, 0))
      for (int s = 0; c; s ^= 1) {
        const Chunk* after = take();
        if (after && !(ok(hipEventRecord(l.done[s], l.stream)) && start(after, s ^ 1))) break;
        if (!ok(after ? hipEventSynchronize(l.done[s]) : hipStreamSynchronize(l.stream))) break;
        walk(j, *c, l.slot[s]);
        c = after;
      }
  }
  ok(hipStreamSynchronize(l.stream));
}

// The lanes' threads, and for every device that is copied to or from the lanes' streams and pinned memory: made by the
// first copy that needs them and given back by jpp_copy_release (at the latest; the last stage's end is one).  One job
// has them at a time; who finds them taken copies without (work_alone).
struct Pool {
  struct Device {
    Lane lanes[kLanes];
    int n = 0;                     // those that are complete
  };
  std::mutex call_mu;              // held for a whole job, and by release
  std::mutex mu;                   // guards what follows
  std::condition_variable wake, idle;
  std::vector<std::thread> threads;
  uint64_t ticket = 0;
  std::atomic<uint64_t> hint{0};   // ticket, for a look without the lock
  int lanes_wanted = 0, busy = 0;
  bool stop = false;
  Job* job = nullptr;
  std::map<int, Device> devices;   // (call_mu) by device
  std::atomic<pid_t> pid{0};       // of the first copy

  static int most_lanes() {
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 2;
    return std::max(1, std::min(kLanes, cpus / 2));
  }
  // Whether the pool is this process's own: the threads and streams of the one it was forked from are not here, and
  // its locks may be held by nobody.
  bool own() {
    pid_t first = 0;
    const pid_t here = getpid();
    return pid.compare_exchange_strong(first, here) || first == here;
  }
  // the device's lanes, up to `n` of them: as many as there is memory for
  Device& open(int dev, int n) {
    Device& d = devices[dev];
    for (; d.n < n; ++d.n) {
      Lane& l = d.lanes[d.n];
      hipError_t e = l.stream ? hipSuccess : hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
      for (int s = 0; s < 2; ++s) {
        if (e == hipSuccess && !l.done[s]) e = hipEventCreateWithFlags(&l.done[s], hipEventDisableTiming);
        if (e == hipSuccess && !l.slot[s]) e = hipHostMalloc((void**)&l.slot[s], kSlot, hipHostMallocDefault);
      }
      if (e != hipSuccess) {
        (void)hipGetLastError();   // (not for the next launch to report)
        break;
      }
    }
    return d;
  }
  void close() {
    for (auto& [dev, d] : devices)
      for (Lane& l : d.lanes) {
        for (int s = 0; s < 2; ++s) {
          if (l.done[s]) (void)hipEventDestroy(l.done[s]);
          if (l.slot[s]) (void)hipHostFree(l.slot[s]);
        }
        if (l.stream) (void)hipStreamDestroy(l.stream);
      }
    devices.clear();
  }
  void helper(int lane, uint64_t seen) {
    for (;;) {
      Job* j;
      {
        // (the next call of a train step follows within some 10 us, a sleeping thread wakes in 50)
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(100);
        while (hint.load(std::memory_order_relaxed) == seen && std::chrono::steady_clock::now() < until)
          std::this_thread::yield();
        std::unique_lock<std::mutex> lock(mu);
        wake.wait(lock, [&] { return stop || ticket != seen; });
        if (stop) return;
        seen = ticket;
        if (lane >= lanes_wanted) continue;
        j = job;
      }
      if (hipSetDevice(j->device) == hipSuccess) work(*j, j->lanes[lane]);
      std::lock_guard<std::mutex> lock(mu);
      if (--busy == 0) idle.notify_one();
    }
  }
  // (call_mu held) every lane's share of `j`, the caller's among them
  void run(Job& j, int n) {
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = false;
      try {
        while ((int)threads.size() < n - 1)
          threads.emplace_back(&Pool::helper, this, (int)threads.size() + 1, ticket);
      } catch (const std::exception&) {   // (no more threads to be had: those there are do it)
      }
      n = std::min(n, (int)threads.size() + 1);
      job = &j;
      lanes_wanted = n;
      busy = n - 1;
      if (n > 1) hint = ++ticket;
    }
    if (n > 1) wake.notify_all();
    work(j, j.lanes[0]);
    std::unique_lock<std::mutex> lock(mu);
    idle.wait(lock, [&] { return busy == 0; });
    job = nullptr;
  }
  void release() {
    std::vector<std::thread> ended;
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = true;
      ended.swap(threads);
    }
    wake.notify_all();
    for (auto& t : ended) t.join();
    close();
  }
};

Pool& pool() {
  static Pool* p = new Pool;   // (never destroyed: its threads may wait in it when the process ends)
  return *p;
}

int copy(int n, const jpp_copy_item* items, int kind, bool up) {
  JPP_REQUIRE(n >= 0 && (n == 0 || items), "copy: null items");
  JPP_REQUIRE(kind == JPP_COPY_WORDS || kind == JPP_COPY_BF16, "copy: unknown kind %d", kind);
  const size_t es = kind == JPP_COPY_BF16 ? 2 : 4;
  size_t total = 0;
  for (int i = 0; i < n; ++i) {
    JPP_REQUIRE(items[i].count >= 0 && items[i].count < (int64_t)1 << 48 &&
                    (items[i].count == 0 || (items[i].host && items[i].device)),
                "copy: item %d is null or has a bad count", i);
    total += (size_t)items[i].count * es;
  }
  if (total == 0) return JPP_OK;
  try {
    Pool& p = pool();
    if (!p.own()) return jpp_set_error(JPP_ERR_STATE, "copy: the process was forked after its first copy");
    Job j;
    j.up = up;
    j.bf16 = kind == JPP_COPY_BF16;
    JPP_CHECK_HIP(hipGetDevice(&j.device));
    std::unique_lock<std::mutex> call(p.call_mu, std::try_to_lock);
    Pool::Device* d = nullptr;
    if (call.owns_lock()) {
      const int most = Pool::most_lanes();
      cut_items(j, n, items, std::min(kSlot, std::max(kLeast, (total / most + 4095) / 4096 * 4096)));
      d = &p.open(j.device, (int)std::min<size_t>(most, j.chunks.size()));
    }
    hipError_t e;
    if (d && d->n > 0) {
      j.lanes = d->lanes;
      // as a copy on the null stream: behind everything queued there, over when this returns
      JPP_CHECK_HIP(hipStreamSynchronize(nullptr));
      p.run(j, (int)std::min({(size_t)Pool::most_lanes(), (size_t)d->n, j.chunks.size()}));
      e = (hipError_t)j.error.load();
    } else {
      if (d) call.unlock();
      cut_items(j, n, items, kAlone);
      e = work_alone(j);
    }
    if (e != hipSuccess) return jpp_set_error(JPP_ERR_HIP, "copy: %s", hipGetErrorString(e));
    return JPP_OK;
  } catch (const std::exception& e) {
    return jpp_set_error(JPP_ERR_STATE, "copy: %s", e.what());
  }
}

}  // namespace

extern "C" {

int jpp_copy_h2d(int n, const jpp_copy_item* items, int kind) { return copy(n, items, kind, true); }
int jpp_copy_d2h(int n, const jpp_copy_item* items, int kind) { return copy(n, items, kind, false); }
int jpp_copy_release(void) {
  Pool& p = pool();
  if (!p.pid || !p.own()) return JPP_OK;
  std::lock_guard<std::mutex> call(p.call_mu);
  p.release();
  return JPP_OK;
}

}  // extern "C"
