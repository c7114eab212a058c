// Setup-phase device allocation pool (see DevPoolScope in common.hpp) and
// the threaded host -> device upload.

#include <algorithm>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <unordered_set>

#include "../../include/fem_mi355x.h"
#include "common.hpp"

namespace fem {

namespace {

struct Pool {
  std::unordered_set<void*> own;       // blocks handed out by this pool
  std::multimap<size_t, void*> free_;  // released blocks by size class
  int device = 0;
  bool adopt = true;                   // takes blocks of earlier scopes
  hipStream_t stream = nullptr;        // of all the scope's work
  Pool* prev = nullptr;                // the enclosing scope
};

thread_local Pool* g_pool = nullptr;
thread_local int g_retire = -1;  // device whose idle blocks this thread's releases go to the reserve of

// size classes: 256 B, then 2^k (1 + j / 8): at most 12.5 % above the request
size_t size_class(size_t bytes) {
  if (bytes <= 256) return 256;
  size_t p = 256;
  while (p * 2 <= bytes) p *= 2;
  const size_t step = p / 8;
  return (bytes + step - 1) / step * step;
}

// free blocks of ended scopes and destroyed handles, per device, by size
// class; and every live block that came from a pool, so that it can return
// to one (process-lifetime objects: handles may be destroyed at exit)
constexpr size_t kReserveCap = (size_t)16 << 30;  // a 161^3 handle and its temporaries: about 12 GiB
struct Reserve {
  struct Idle {
    void* p;
    uint64_t age;
  };
  typedef std::multimap<size_t, Idle> Blocks;
  Blocks blocks;  // by size class
  size_t bytes = 0;
  uint64_t next = 0;

  void put(size_t cls, void* p) {
    blocks.emplace(cls, Idle{p, next++});
    bytes += cls;
  }
  void* take(Blocks::iterator it) {
    void* p = it->second.p;
    bytes -= it->first;
    blocks.erase(it);
    return p;
  }
  Blocks::iterator oldest() {  // only a full reserve asks, before a hipFree
    return std::min_element(blocks.begin(), blocks.end(), [](const Blocks::value_type& a, const Blocks::value_type& b) {
      return a.second.age < b.second.age;
    });
  }
};
struct Block {
  size_t cls;
  int device;
};
std::mutex g_res_mu;
std::unordered_map<int, Reserve>& reserves() {
  static auto* r = new std::unordered_map<int, Reserve>();
  return *r;
}
std::unordered_map<void*, Block>& blocks() {
  static auto* b = new std::unordered_map<void*, Block>();
  return *b;
}

void free_block(void* p) {
  blocks().erase(p);
  (void)hipFree(p);
}

// an idle block into its device's reserve, whose oldest blocks make room: what
// a process works on now has the sizes of the newest ones (the caller holds
// g_res_mu)
void retire_locked(void* p, size_t cls, int device) {
  Reserve& r = reserves()[device];
  if (cls > kReserveCap) {
    free_block(p);
    return;
  }
  while (r.bytes + cls > kReserveCap) free_block(r.take(r.oldest()));
  r.put(cls, p);
}

}  // namespace

void pool_flush_reserve() {
  std::lock_guard<std::mutex> lk(g_res_mu);
  for (auto& dr : reserves())
    while (!dr.second.blocks.empty()) free_block(dr.second.take(dr.second.blocks.begin()));
}

namespace {
// frees the released blocks that this thread's scopes hold (a setup that
// replaces a hierarchy of other sizes holds all of the old one)
void free_released() {
  for (Pool* pl = g_pool; pl; pl = pl->prev) {
    if (pl->free_.empty() || hipStreamSynchronize(pl->stream) != hipSuccess) continue;
    std::lock_guard<std::mutex> lk(g_res_mu);
    for (auto& kv : pl->free_) {
      for (Pool* q = g_pool; q; q = q->prev) q->own.erase(kv.second);
      free_block(kv.second);
    }
    pl->free_.clear();
  }
}
}  // namespace

void* dev_malloc(size_t bytes) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    free_released();
    pool_flush_reserve();
    HIP_CHECK(hipMalloc(&p, bytes));
  }
  return p;
}

void* pool_alloc(size_t bytes) {
  Pool* pl = g_pool;
  if (!pl || bytes == 0) return nullptr;
  const size_t c = size_class(bytes);
  auto it = pl->free_.find(c);
  if (it != pl->free_.end()) {
    void* p = it->second;
    pl->free_.erase(it);
    return p;
  }
  void* p = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_res_mu);
    auto rt = reserves().find(pl->device);
    if (rt != reserves().end()) {
      auto jt = rt->second.blocks.find(c);
      if (jt != rt->second.blocks.end()) p = rt->second.take(jt);
    }
  }
  if (!p) {
    p = dev_malloc(c);
    std::lock_guard<std::mutex> lk(g_res_mu);
    blocks()[p] = Block{c, pl->device};
  }
  pl->own.insert(p);
  return p;
}

bool pool_release(void* p) {
  Pool* pl = g_pool;
  std::lock_guard<std::mutex> lk(g_res_mu);
  auto bt = blocks().find(p);
  if (bt == blocks().end()) return false;
  const Block b = bt->second;
  if (pl && b.device == pl->device && (pl->adopt || pl->own.count(p))) {
    // also a block of an earlier scope (the hierarchy that a setup replaces):
    // its uses are on this scope's stream, before whatever it serves next
    pl->free_.emplace(b.cls, p);
    return true;
  }
  if (g_retire == b.device) {
    retire_locked(p, b.cls, b.device);
    return true;
  }
  blocks().erase(bt);
  return false;
}

DevPoolScope::DevPoolScope(hipStream_t stream, bool adopt) {
  Pool* pl = new Pool();
  (void)hipGetDevice(&pl->device);
  pl->adopt = adopt;
  pl->stream = stream;
  pl->prev = g_pool;
  g_pool = pl;
}

DevPoolScope::~DevPoolScope() {
  Pool* pl = g_pool;
  if (!pl->free_.empty()) {
    // queued work may still use the blocks: they are handed on once the
    // scope's stream has drained (a device synchronization would also end
    // another thread's stream capture)
    const bool idle = hipStreamSynchronize(pl->stream) == hipSuccess;
    std::lock_guard<std::mutex> lk(g_res_mu);
    for (auto& kv : pl->free_) {
      if (idle) {
        retire_locked(kv.second, kv.first, pl->device);
      } else {
        free_block(kv.second);
      }
    }
  }
  g_pool = pl->prev;
  delete pl;
}

DevRetireScope::DevRetireScope(int device) : prev_(g_retire) { g_retire = device; }
DevRetireScope::~DevRetireScope() { g_retire = prev_; }

namespace {

constexpr int kUploadThreads = 4;
constexpr size_t kUploadSplit = (size_t)8 << 20;  // smaller copies stay one async copy on s
constexpr int kMaxDevices = 64;
std::mutex g_up_mu;
hipStream_t g_up[kMaxDevices][kUploadThreads];  // per device, created on first use, kept

// bytes [a, b) of the pieces taken end to end, copied on st
hipError_t upload_range(const HostPiece* pc, int np, size_t a, size_t b, hipStream_t st) {
  size_t base = 0;
  for (int i = 0; i < np; ++i) {
    const size_t lo = std::max(a, base), hi = std::min(b, base + pc[i].bytes);
    if (lo < hi) {
      const hipError_t e = hipMemcpyAsync(static_cast<char*>(pc[i].dst) + (lo - base),
                                          static_cast<const char*>(pc[i].src) + (lo - base), hi - lo,
                                          hipMemcpyHostToDevice, st);
      if (e != hipSuccess) return e;
    }
    base += pc[i].bytes;
  }
  return hipStreamSynchronize(st);
}

}  // namespace

void upload_pieces(const HostPiece* pc, int np, hipStream_t s) {
  size_t total = 0;
  for (int i = 0; i < np; ++i) total += pc[i].bytes;
  // the destinations may be blocks that earlier work on s still uses
  HIP_CHECK(hipStreamSynchronize(s));
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) fail(FEM_ERR_CAPACITY, "device index beyond the upload stream table");
  hipStream_t st[kUploadThreads];
  {
    // the streams are created, and each takes a first small copy (a prefix
    // of the first piece, so what lands there is the data itself), on the
    // first upload of the process, whatever its size: a stream's first copy
    // costs milliseconds more than the later ones
    std::lock_guard<std::mutex> lk(g_up_mu);
    for (int k = 0; k < kUploadThreads; ++k) {
      if (!g_up[dev][k]) {
        HIP_CHECK(hipStreamCreateWithFlags(&g_up[dev][k], hipStreamNonBlocking));
        const HostPiece* first = nullptr;
        for (int i = 0; i < np && !first; ++i)
          if (pc[i].bytes) first = &pc[i];
        if (first) {
          HIP_CHECK(hipMemcpyAsync(first->dst, first->src, std::min<size_t>(first->bytes, 4096),
                                   hipMemcpyHostToDevice, g_up[dev][k]));
          HIP_CHECK(hipStreamSynchronize(g_up[dev][k]));
        }
      }
      st[k] = g_up[dev][k];
    }
  }
  if (total < kUploadSplit) {
    for (int i = 0; i < np; ++i)
      if (pc[i].bytes) HIP_CHECK(hipMemcpyAsync(pc[i].dst, pc[i].src, pc[i].bytes, hipMemcpyHostToDevice, s));
    return;
  }
  hipError_t err[kUploadThreads];
  std::vector<std::thread> th;
  for (int k = 0; k < kUploadThreads; ++k) {
    const size_t a = total * k / kUploadThreads, b = total * (k + 1) / kUploadThreads;
    auto work = [&err, pc, np, a, b, dev, k, &st]() {
      hipError_t e = hipSetDevice(dev);  // the current device is per thread
      err[k] = e == hipSuccess ? upload_range(pc, np, a, b, st[k]) : e;
    };
    try {
      th.emplace_back(work);
    } catch (...) {
      work();  // no thread: copy this share here
    }
  }
  for (auto& t : th) t.join();
  for (int k = 0; k < kUploadThreads; ++k) HIP_CHECK(err[k]);
}

}  // namespace fem
