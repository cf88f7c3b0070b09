// Downloads of 16 chunks on two threads (akx_download.hpp over the host
// stand-in of HIP) whose helper thread fails on its last chunk, while the
// calling thread has nothing left but to wait for it: the call has to end in
// the error, every time, and to have waited for the stream (the failed chunk's
// kernel may be running).  argv[1]: "pack" (the launch throws) or "record" (the
// event cannot be recorded after the launch) or "none".  Prints the trials, the
// errors seen and the calls that returned without one although rows are missing.
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
  int errors = 0, silent = 0, wrong = 0, unwaited = 0;
  const int trials = mode == "none" ? 20 : 400;
  for (int t = 0; t < trials; ++t) {
    std::memset(host.data(), 0, n);
    std::memset(copy.data(), 0, n);
    std::atomic<int> packed{0}, taken{0};
    fake::stream_waits = 0;
    fake::records_to_fail = 0;
    std::vector<akx::Downloader::Field> f{
        {n, 1, host.data(), copy.data(), [&](void *p, int64_t first, int64_t count) {
           if (fake::helper && mode != "none") {
             taken = 1;
             // the calling thread does the others and waits
             while (packed.load() < 15)
               std::this_thread::yield();
             std::this_thread::sleep_for(std::chrono::microseconds(300 + t % 7));
             if (mode == "pack")
               throw akx::Error(AKX_ERR_HIP, "launch");
             fake::records_to_fail = 1;
           } else if (mode != "none") {
             // one chunk is the helper's (which may take its time to come)
             for (int k = 0; !taken.load() && k < 5000; ++k)
               std::this_thread::sleep_for(std::chrono::microseconds(100));
           }
           std::memset(p, 1 + (int)(first >> 20), count);
           ++packed;
         }}};
    bool threw = false;
    try {
      down.get(0, nullptr, f);
    } catch (const akx::Error &) {
      threw = true;
    }
    bool whole = true;
    for (int64_t i = 0; i < n; i += 4096)
      whole = whole && host[i] == 1 + (i >> 20) && copy[i] == 1 + (i >> 20);
    errors += threw;
    silent += !threw && !whole;
    wrong += mode == "none" && !whole;
    unwaited += threw && fake::stream_waits.load() == 0;
  }
  std::printf("%d %d %d %d %d\n", trials, errors, silent, wrong, unwaited);
}
