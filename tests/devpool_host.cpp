// The device-memory pool (csrc/devpool.cpp) on the CPU: the HIP calls it makes
// are stand-ins over a simulated device of limited size, whose addresses are
// never touched.  Runs the scenario named on the command line; exits with 0,
// or prints the check that failed.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"

namespace {
std::mutex g_mu;
std::map<char*, size_t> g_live;
size_t g_used = 0, g_limit = (size_t)64 << 30;
int g_mallocs = 0, g_frees = 0;
constexpr size_t kGiB = (size_t)1 << 30;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_used + bytes > g_limit) return hipErrorOutOfMemory;
  char* at = reinterpret_cast<char*>((uintptr_t)1 << 40);  // the first gap, so that addresses come again
  for (auto& kv : g_live) {
    if (at + bytes <= kv.first) break;
    at = kv.first + kv.second;
  }
  g_live[at] = bytes;
  g_used += bytes;
  ++g_mallocs;
  *p = at;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_live.find(static_cast<char*>(p));
  if (it == g_live.end()) {
    std::printf("free of an address that is not allocated\n");
    std::_Exit(1);
  }
  g_used -= it->second;
  g_live.erase(it);
  ++g_frees;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "simulated"; }
hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return hipErrorNotSupported; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipErrorNotSupported; }
}

#define CHECK(c)                                     \
  do {                                               \
    if (!(c)) {                                      \
      std::printf("line %d: %s\n", __LINE__, #c);    \
      std::exit(1);                                  \
    }                                                \
  } while (0)

using fem::DevBuf;
using fem::DevPoolScope;

namespace {

// a block that a scope's owner keeps (a handle's buffer)
DevBuf<char> kept_block(size_t bytes) {
  DevPoolScope s(nullptr);
  return DevBuf<char>(bytes);
}

// work captured by a caller may run on any stream: what its handle releases
// goes through hipFree, which waits for the device, and is not handed on
void foreign_work() {
  DevBuf<char> old = kept_block(kGiB);
  {
    DevPoolScope s(nullptr, /*adopt=*/false);
    old.release();
    CHECK(g_frees == 1);
    DevBuf<char> next(kGiB);
    CHECK(g_mallocs == 2);
  }
  old = kept_block(2 * kGiB);
  {
    DevPoolScope s(nullptr);
    old.release();
    const int m = g_mallocs;
    DevBuf<char> next(2 * kGiB);
    CHECK(g_mallocs == m);  // reused in stream order
  }
}

// a setup that replaces a hierarchy by one of other sizes, near the limit of
// the device: the old blocks make room
void failed_allocation() {
  g_limit = 10 * kGiB;
  DevBuf<char> old = kept_block(7 * kGiB);
  DevBuf<char> other = kept_block(kGiB);
  {
    DevPoolScope outer(nullptr);
    other.release();
    DevPoolScope s(nullptr);
    old.release();
    DevBuf<char> next(9 * kGiB);  // fits without the two
    CHECK(g_used == 9 * kGiB);
    // the freed addresses are new blocks now, of their own sizes
    next.release();
    DevBuf<char> a(4 * kGiB), b(4 * kGiB);
    CHECK(a.get() != b.get() && g_live.at(a.get()) == 4 * kGiB && g_live.at(b.get()) == 4 * kGiB);
    a.release();
    DevBuf<char> c(4 * kGiB);
    CHECK(g_live.at(c.get()) == 4 * kGiB);
  }
  bool failed = false;
  try {
    DevBuf<char> more(11 * kGiB);
  } catch (const fem::FemError& e) {
    failed = e.status == 3;
  }
  CHECK(failed);
}

// the reserve keeps the newest blocks: a process that goes from one size to
// another finds the blocks of its present size there
void reserve_ages() {
  for (int size = 1; size <= 4; ++size) {  // 10 GiB of each
    for (int round = 0; round < 2; ++round) {
      DevPoolScope s(nullptr);
      const int m = g_mallocs;
      std::vector<DevBuf<char>> v;
      for (int i = 0; i < 10 * 4 / size; ++i) v.emplace_back((size_t)size * kGiB / 4);
      CHECK(g_mallocs - m == (round == 0 ? 10 * 4 / size : 0));
    }
    CHECK(g_used <= 16 * kGiB);
  }
  // a block larger than the reserve leaves it as it is
  const size_t held = g_used;
  { DevPoolScope s(nullptr); DevBuf<char> big(17 * kGiB); }
  CHECK(g_used == held);
  fem::pool_flush_reserve();
  CHECK(g_used == 0 && g_live.empty());
}

// fem_release_cached_memory beside setups, solves and destroys of other
// threads: no block is ever with two owners, and none is lost
void flush_beside_work() {
  std::mutex mu;
  std::map<void*, int> owner;
  std::atomic<bool> stop{false};
  std::thread flusher([&] {
    while (!stop) fem::pool_flush_reserve();
  });
  auto work = [&](int id) {
    unsigned x = 12345u + (unsigned)id;
    auto next = [&] { return (x = x * 1664525u + 1013904223u) >> 8; };
    for (int round = 0; round < 300; ++round) {
      std::vector<DevBuf<char>> kept;
      {
        DevPoolScope s(nullptr);
        for (int i = 0; i < 20; ++i) {
          DevBuf<char> b(((size_t)1 << (8 + next() % 4)) * 3);
          {
            std::lock_guard<std::mutex> lk(mu);
            CHECK(owner.emplace(b.get(), id).second);
          }
          if (next() % 2) {
            kept.push_back(std::move(b));
          } else {
            std::lock_guard<std::mutex> lk(mu);
            owner.erase(b.get());
            b.release();
          }
        }
      }
      fem::DevRetireScope r(0);
      std::lock_guard<std::mutex> lk(mu);
      for (auto& b : kept) owner.erase(b.get());
      kept.clear();
    }
  };
  std::vector<std::thread> th;
  for (int id = 0; id < 4; ++id) th.emplace_back(work, id);
  for (auto& t : th) t.join();
  stop = true;
  flusher.join();
  fem::pool_flush_reserve();
  CHECK(g_used == 0 && g_live.empty());
}

}  // namespace

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "foreign_work")) foreign_work();
  else if (!std::strcmp(what, "failed_allocation")) failed_allocation();
  else if (!std::strcmp(what, "reserve_ages")) reserve_ages();
  else if (!std::strcmp(what, "flush_beside_work")) flush_beside_work();
  else { std::printf("unknown scenario\n"); return 2; }
  return 0;
}
