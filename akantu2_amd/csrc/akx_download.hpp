// akx_download.hpp -- device fields to host arrays.
//
// A field is packed by a kernel that writes the caller's layout straight into
// pinned host memory, and copied from there.  What a plain device-to-host
// copy into the caller's (pageable, often untouched) array spent its time on
// was the host: the runtime's own staging at 10 GB/s or less, the page faults
// of a new array, one synchronisation and one copy command per field.  Here
// several fields share one synchronisation, and large ones go in chunks of
// 1 MB that one to eight threads claim in turn: each launches the next chunk's
// kernel into one of its two pinned slots while it copies the one before out
// (to the array and, where asked, to a second one), so the link, the copies
// and the page faults overlap.  Threads beside the caller's join once the
// stream's earlier work is done: before, they waited for it in the runtime, which
// spins, took CPUs from an OpenMP team of the caller's that still spun too, and
// its next parallel region waited for a scheduler's slice or two (torch's cast of
// a 28 MB field to FP32 after the read-back, 0.5 ms, 5 to 12 ms every other time).
// Times: Downloader::get.
#pragma once

#include "akx_host.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace akx {

// Threads that help with copies, for the whole process: at most seven, started
// when more work is there than threads are idle, gone after two idle seconds.  Waiting
// threads are scheduled at once when they are woken; a new thread waits a
// scheduler's slice (3 ms) where the CPUs are busy, as they are for a while
// after an OpenMP loop.  Never destroyed: a thread may wait in it at exit.
class CopyThreads {
  static constexpr int MOST = 7;
  std::mutex mutex;
  std::condition_variable wake;
  std::deque<std::function<void()>> queue;
  int threads = 0, idle = 0;

  void loop() {
    std::unique_lock<std::mutex> lock(mutex);
    for (;;) {
      ++idle;
      const bool work = wake.wait_for(lock, std::chrono::seconds(2),
                                      [&] { return !queue.empty(); });
      --idle;
      if (!work) {
        --threads;
        return;
      }
      std::function<void()> f = std::move(queue.front());
      queue.pop_front();
      lock.unlock();
      f(); // does not throw
      f = nullptr;
      lock.lock();
    }
  }

public:
  static CopyThreads &get() {
    static CopyThreads *p = new CopyThreads;
    return *p;
  }
  void submit(const std::function<void()> &f, int copies) {
    std::lock_guard<std::mutex> lock(mutex);
    for (int k = 0; k < copies; ++k)
      queue.push_back(f);
    for (int more = (int)queue.size() - idle; more > 0 && threads < MOST; --more) {
      std::thread([this] { loop(); }).detach();
      ++threads;
    }
    wake.notify_all();
  }
};

// Chunks 0 .. n - 1 claimed by the calling thread and up to threads - 1
// others.  The caller waits for every claimed chunk, not for the threads: one
// that has not been scheduled yet is not waited for, and finds nothing to
// claim when it is.
struct ChunkJob {
  std::atomic<int64_t> next{0}, done{0};
  int64_t n = 0;
  std::mutex mutex;
  std::exception_ptr error;

  // the error, then what it leaves undone: the caller returns once that is
  // counted.  No further chunk is claimed.
  void fail(std::exception_ptr e, int64_t open) {
    {
      std::lock_guard<std::mutex> lock(mutex);
      if (!error)
        error = e;
    }
    const int64_t c = next.exchange(n);
    done.fetch_add(open + (c < n ? n - c : 0));
  }
};

// One thread's chunks: those it has claimed and not finished are its own to
// finish, or to give up by throwing
class Claims {
  ChunkJob &job;
  int64_t open = 0;

public:
  explicit Claims(ChunkJob &j) : job(j) {}
  int64_t claim() { // -1: none left
    const int64_t c = job.next.fetch_add(1);
    if (c >= job.n)
      return -1;
    ++open;
    return c;
  }
  void finish() { // the caller may return: nothing of its is touched after the last
    --open;
    job.done.fetch_add(1);
  }
  void fail(std::exception_ptr e) { job.fail(e, open); }
};

// work(claims, c, start) does chunk c and claims and does others until none is
// left.  In the calling thread (*start)(k) lets up to k others help from then
// on; in these start is null.
using StartHelp = std::function<void(int)>;
template <class F> void run_chunks(int64_t n, const F &work) {
  auto job = std::make_shared<ChunkJob>();
  job->n = n;
  // the threads hold the job alive and copies of what work refers to only
  // through it: work itself is run by a thread that has claimed a chunk
  std::shared_ptr<const F *> body = std::make_shared<const F *>(&work);
  auto loop = [job, body](const StartHelp *start) {
    Claims claims(*job);
    const int64_t c = claims.claim();
    if (c < 0)
      return; // the caller may have returned: work is not touched
    try {
      (**body)(claims, c, start);
    } catch (...) {
      claims.fail(std::current_exception());
    }
  };
  const StartHelp start = [loop](int others) {
    try {
      CopyThreads::get().submit([loop] { loop(nullptr); }, others);
    } catch (...) { // no thread to be had: their share is done by the caller
    }
  };
  loop(&start);
  while (job->done.load() < n)
    std::this_thread::yield();
  std::lock_guard<std::mutex> lock(job->mutex);
  if (job->error)
    std::rethrow_exception(job->error);
}

constexpr size_t COPY_CHUNK = 1u << 20;

// Threads for a copy: one per 8 MB, at most eight.  More did not pay for what
// a thread costs where the CPUs are busy: an 8 MB field by four threads 0.4 ms
// on idle CPUs, but 3.5 ms (a scheduler's slice) beside 16 spinning ones; by
// one thread 0.6 to 0.8 ms.
inline int copy_threads(size_t bytes) {
  const size_t hw = std::max(1u, std::thread::hardware_concurrency());
  return (int)std::max<size_t>(1, std::min<size_t>({8, hw, bytes >> 23}));
}

// whether two host arrays differ
inline bool host_differs(const void *a, const void *b, size_t bytes) {
  const int T = copy_threads(bytes);
  if (T == 1)
    return std::memcmp(a, b, bytes) != 0;
  std::atomic<bool> differ{false};
  run_chunks((int64_t)((bytes + COPY_CHUNK - 1) / COPY_CHUNK),
             [&](Claims &claims, int64_t c, const StartHelp *start) {
               if (start)
                 (*start)(T - 1);
               for (; c >= 0; c = claims.claim()) {
                 const size_t o = (size_t)c * COPY_CHUNK;
                 if (!differ.load(std::memory_order_relaxed) &&
                     std::memcmp((const char *)a + o, (const char *)b + o,
                                 std::min(COPY_CHUNK, bytes - o)) != 0)
                   differ = true;
                 claims.finish();
               }
             });
  return differ;
}

class Downloader {
  unsigned char *pin = nullptr;
  size_t cap = 0;
  // A model's first few small copies go through device memory: they cost 40 us
  // more each, but pinning and unpinning a buffer costs a model 0.3 ms.
  static constexpr int UNPINNED = 4;
  int small_copies = 0;
  DevBuf<unsigned char> dev;
  std::vector<hipEvent_t> events; // two per thread

  void reserve(size_t bytes) {
    if (bytes <= cap)
      return;
    size_t want = 64u << 10;
    while (want < bytes)
      want *= 2;
    if (pin)
      (void)hipHostFree(pin);
    pin = nullptr;
    cap = 0;
    HIPCHECK(hipHostMalloc((void **)&pin, want, hipHostMallocCoherent));
    cap = want;
  }

public:
  // n items of `item` bytes; pack(p, first, count) launches, on the stream,
  // the kernel that writes items first .. first + count - 1 to p (16-byte
  // aligned); copy: a second destination, or null
  struct Field {
    int64_t n;
    size_t item;
    void *host, *copy;
    std::function<void(void *, int64_t, int64_t)> pack;
    size_t bytes() const { return (size_t)n * item; }
  };

  Downloader() = default;
  Downloader(const Downloader &) = delete;
  Downloader &operator=(const Downloader &) = delete;
  ~Downloader() {
    for (hipEvent_t e : events)
      (void)hipEventDestroy(e);
    if (pin)
      (void)hipHostFree(pin);
  }

  // Waits for the stream's work and delivers the fields.  (device is current.)
  // Per field: 525 nodes 50-100 -> 19 us; 2 M nodes (49 MB) 5.2 -> 1.2 ms, with
  // the second copy 9.1 -> 1.6 ms (arrays used before; the comparison of two
  // such pairs at the next call 4.4 -> 1.7 ms).
  void get(int device, hipStream_t stream, std::vector<Field> &fields) {
    try {
      deliver(device, stream, fields);
    } catch (...) { // kernels that were launched still write the buffers
      (void)hipStreamSynchronize(stream);
      throw;
    }
  }

private:
  void deliver(int device, hipStream_t stream, std::vector<Field> &fields) {
    size_t total = 0;
    for (auto &f : fields)
      total += (f.bytes() + 63) / 64 * 64;
    if (total <= COPY_CHUNK && total > cap && ++small_copies <= UNPINNED) {
      dev.reserve(total);
      size_t o = 0;
      for (auto &f : fields) {
        if (f.n > 0) {
          f.pack(dev.p + o, 0, f.n);
          HIPCHECK(hipMemcpyAsync(f.host, dev.p + o, f.bytes(), hipMemcpyDeviceToHost, stream));
        }
        o += (f.bytes() + 63) / 64 * 64;
      }
      HIPCHECK(hipStreamSynchronize(stream));
      for (auto &f : fields)
        if (f.copy)
          std::memcpy(f.copy, f.host, f.bytes());
      return;
    }
    if (total <= COPY_CHUNK) {
      reserve(std::max<size_t>(total, 64));
      size_t o = 0;
      for (auto &f : fields) {
        if (f.n > 0)
          f.pack(pin + o, 0, f.n);
        o += (f.bytes() + 63) / 64 * 64;
      }
      HIPCHECK(hipStreamSynchronize(stream));
      o = 0;
      for (auto &f : fields) {
        if (f.n > 0) {
          std::memcpy(f.host, pin + o, f.bytes());
          if (f.copy)
            std::memcpy(f.copy, pin + o, f.bytes());
        }
        o += (f.bytes() + 63) / 64 * 64;
      }
      return;
    }
    struct Chunk {
      const Field *f;
      int64_t first, count;
    };
    const int T = copy_threads(total);
    std::vector<Chunk> chunks;
    for (auto &f : fields) {
      const int64_t per = std::max<int64_t>(1, (int64_t)(COPY_CHUNK / f.item));
      for (int64_t i = 0; i < f.n; i += per)
        chunks.push_back({&f, i, std::min(per, f.n - i)});
    }
    reserve((size_t)T * 2 * COPY_CHUNK);
    while ((int)events.size() < 2 * T) {
      hipEvent_t e;
      HIPCHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      events.push_back(e);
    }
    std::atomic<int> workers{0};
    run_chunks((int64_t)chunks.size(), [&](Claims &claims, int64_t c, const StartHelp *start) {
      // the thread's chunks in flight: claimed, the kernel launched
      const int w = workers.fetch_add(1);
      struct Flight {
        hipEvent_t ev;
        int64_t c;
      } fl[2] = {{events[2 * w], -1}, {events[2 * w + 1], -1}};
      unsigned char *slots = pin + (size_t)w * 2 * COPY_CHUNK;
      HIPCHECK(hipSetDevice(device));
      for (int k = 0;; k ^= 1) {
        if (c >= 0) {
          const Chunk &h = chunks[c];
          h.f->pack(slots + k * COPY_CHUNK, h.first, h.count);
          HIPCHECK(hipEventRecord(fl[k].ev, stream));
          fl[k].c = c;
        }
        Flight &o = fl[k ^ 1]; // the one before
        if (o.c >= 0) {
          HIPCHECK(hipEventSynchronize(o.ev));
          if (start && T > 1) // the stream's earlier work is done
            (*start)(T - 1);
          start = nullptr;
          const Chunk &h = chunks[o.c];
          const size_t at = (size_t)h.first * h.f->item, b = (size_t)h.count * h.f->item;
          const unsigned char *slot = slots + (k ^ 1) * COPY_CHUNK;
          std::memcpy((char *)h.f->host + at, slot, b);
          if (h.f->copy)
            std::memcpy((char *)h.f->copy + at, slot, b);
          o.c = -1;
          claims.finish();
        }
        c = claims.claim();
        if (c < 0 && fl[0].c < 0 && fl[1].c < 0)
          break;
      }
    });
  }
};

} // namespace akx
