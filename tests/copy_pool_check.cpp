// CPU check of the copy threads (csrc/copy_pool.h), without a device: chunks
// through the ring of slots as copy_to_host drives it.
//   copy <bytes> <chunk> <use>: prints 1 if every byte arrived; the target
//       starts unaligned, the last chunk is a remainder
//   idle <ms>: a copy whose first chunk comes after <ms>, and a second part
//       after <ms> more; prints the CPU time of the process in ms
//   abandon: a copy given up after two of five chunks, then a whole one
#include "copy_pool.h"

#include <sys/resource.h>

#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

using llfem::CopyPool;

static double cpu_ms() {
  rusage r;
  getrusage(RUSAGE_SELF, &r);
  return 1e3 * (r.ru_utime.tv_sec + r.ru_stime.tv_sec) + 1e-3 * (r.ru_utime.tv_usec + r.ru_stime.tv_usec);
}

// chunks `given` of the copy; stage: kSlots * chunk bytes
static void copy(CopyPool& pool, std::vector<char>& stage, const std::vector<char>& from, char* to, size_t chunk, int use,
                 size_t given, bool abandon, int pause_ms) {
  const size_t n = (from.size() + chunk - 1) / chunk;
  pool.begin(n, use);
  for (size_t i = 0; i < given; ++i) {
    const size_t s = i % CopyPool::kSlots, off = i * chunk, len = std::min(chunk, from.size() - off);
    if (pause_ms && (i == 0 || i == n / 2)) std::this_thread::sleep_for(std::chrono::milliseconds(pause_ms));
    pool.wait_free(s);
    std::memcpy(&stage[s * chunk], &from[off], len);   // the device's part
    pool.arrived(i, to + off, &stage[s * chunk], len);
  }
  pool.finish(abandon);
}

int main(int argc, char** argv) {
  const std::string what = argv[1];
  CopyPool pool;
  const size_t bytes = what == "copy" ? std::strtoull(argv[2], nullptr, 10) : size_t(5) << 20;
  const size_t chunk = what == "copy" ? std::strtoull(argv[3], nullptr, 10) : size_t(1) << 20;
  const int use = what == "copy" ? std::atoi(argv[4]) : CopyPool::kThreads;
  const size_t n = (bytes + chunk - 1) / chunk;
  std::vector<char> from(bytes), to(bytes + 3, 0), stage(CopyPool::kSlots * chunk);
  for (size_t i = 0; i < bytes; ++i) from[i] = (char)(1 + i * 2654435761u % 255);
  if (what == "idle") {
    const double c0 = cpu_ms();
    copy(pool, stage, from, to.data() + 3, chunk, use, n, false, std::atoi(argv[2]));
    std::printf("%.1f\n", cpu_ms() - c0);
  } else if (what == "abandon") {
    copy(pool, stage, from, to.data() + 3, chunk, use, 2, true, 0);
    std::fill(to.begin(), to.end(), 0);
  }
  for (int rep = 0; rep < (what == "copy" ? 20 : 1); ++rep) {
    std::fill(to.begin(), to.end(), 0);
    copy(pool, stage, from, to.data() + 3, chunk, use, n, false, 0);
    if (std::memcmp(from.data(), to.data() + 3, bytes) != 0 || to[0] || to[1] || to[2]) {
      std::printf("0\n");
      return 1;
    }
  }
  if (what != "idle") std::printf("1\n");
  return 0;
}
