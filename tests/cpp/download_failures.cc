// Downloads of 16 MB on two threads (akx_download.hpp over the host
// stand-in of HIP) whose helper thread fails on its last chunk, while the
// calling thread has nothing left but to wait for it: the call has to end in
// the error, every time, and to have waited for the stream (the failed chunk's
// kernel may be running).  argv[1]: "pack" (the launch throws) or "record" (the
// event cannot be recorded after the launch) or "none"; "late": nothing
// fails, the stream's earlier work takes 10 ms, and a helper that comes before it
// is done counts.  Prints the trials, those
// in which the helper had a chunk (it has none where the CPUs are busy), the
// errors, the calls that returned without one although bytes are missing, and the
// errors that had not waited for the stream.
#include "../../akantu2_amd/csrc/akx_download.hpp"

#include <cstdio>

namespace akx {
thread_local std::string g_last_error;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) {
  return std::memcpy(d, s, n), 0;
}

int main(int, char **argv) {
  const std::string mode = argv[1];
  fake::helper = false; // this thread
  const int64_t n = 16ll << 20;
  std::vector<unsigned char> host(n), copy(n);
  akx::Downloader down;
  int helped = 0, errors = 0, silent = 0, unwaited = 0;
  const bool fails = mode == "pack" || mode == "record";
  const int trials = fails ? 150 : 20;
  for (int t = 0; t < trials; ++t) {
    std::memset(host.data(), 0, n);
    std::memset(copy.data(), 0, n);
    std::atomic<int64_t> packed{0};
    std::atomic<int> taken{0}, calls{0};
    fake::stream_waits = 0;
    fake::records_to_fail = 0;
    fake::event_waits = 0;
    fake::slow_waits = mode == "late" ? 10 : 0;
    std::vector<akx::Downloader::Field> f{
        {n, 1, host.data(), copy.data(), [&](void *p, int64_t first, int64_t count) {
           if (fake::helper && mode == "late" && !fake::event_waits)
             taken = 1;
           if (fake::helper && fails) {
             taken = 1;
             // the calling thread does the others and waits
             while (packed.load() < n - count)
               std::this_thread::yield();
             std::this_thread::sleep_for(std::chrono::microseconds(300 + t % 7));
             if (mode == "pack")
               throw akx::Error(AKX_ERR_HIP, "launch");
             fake::records_to_fail = 1;
           } else if (fails && ++calls > 4) {
             // one chunk is the helper's (which may take its time to come)
             for (int k = 0; !taken.load() && k < 200; ++k)
               std::this_thread::sleep_for(std::chrono::microseconds(100));
           }
           for (int64_t i = 0; i < count; ++i)
             ((unsigned char *)p)[i] = (unsigned char)(1 + ((first + i) >> 12) % 251);
           packed += count;
         }}};
    bool threw = false;
    try {
      down.get(0, nullptr, f);
    } catch (const akx::Error &) {
      threw = true;
    }
    bool whole = true;
    for (int64_t i = 0; i < n; i += 4096)
      whole = whole && host[i] == 1 + (i >> 12) % 251 && copy[i] == 1 + (i >> 12) % 251;
    errors += threw;
    silent += !threw && !whole;
    helped += taken;
    unwaited += threw && fake::stream_waits.load() == 0;
  }
  std::printf("%d %d %d %d %d\n", trials, helped, errors, silent, unwaited);
}
