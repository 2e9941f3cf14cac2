// Context, error reporting and device-memory accounting.
#include <mutex>

#include "common.h"
#include "copy_pool.h"

#include <algorithm>
#include <cstring>
#include <thread>
#include <utility>
#include <vector>

namespace llfem {

static thread_local std::string g_error;

void set_error(const std::string& msg) { g_error = msg; }

int dmalloc(llfem_ctx* ctx, void** p, size_t bytes) {
  *p = nullptr;
  if (bytes == 0) return LLFEM_OK;
  if (ctx->budget && ctx->in_use + bytes > ctx->budget) ws_release(ctx);
  if (ctx->budget && ctx->in_use + bytes > ctx->budget)
    return fail(LLFEM_ENOMEM, "HBM budget exceeded: need " + std::to_string(bytes) +
                                  " more bytes, " + std::to_string(ctx->in_use) + " of " +
                                  std::to_string(ctx->budget) + " in use");
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess && ctx->ws && !ctx->ws_busy) {
    (void)hipGetLastError();
    ws_release(ctx);
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(LLFEM_ENOMEM, std::string("hipMalloc(") + std::to_string(bytes) +
                                  ") failed: " + hipGetErrorString(e));
  }
  ctx->in_use += bytes;
  return LLFEM_OK;
}

void dfree(llfem_ctx* ctx, void* p, size_t bytes) {
  if (!p) return;
  (void)hipFree(p);
  ctx->in_use -= bytes;
}

void ws_release(llfem_ctx* ctx) {
  if (!ctx->ws || ctx->ws_busy) return;
  dfree(ctx, ctx->ws, ctx->ws_bytes);
  ctx->ws = nullptr;
  ctx->ws_bytes = 0;
}

int WsGuard::get(size_t bytes) {
  if (c_->ws_bytes < bytes) {
    ws_release(c_);
    LLFEM_TRY(dmalloc(c_, &c_->ws, bytes));
    c_->ws_bytes = bytes;
  }
  c_->ws_busy = held_ = true;
  return LLFEM_OK;
}

WsGuard::~WsGuard() {
  if (!held_) return;
  c_->ws_busy = false;
  if (c_->ws_bytes > kWsKeep) ws_release(c_);
}

// Device memory to the caller's pageable memory through pinned staging.  Up
// to kOneCopy bytes: one copy, emptied by this thread.  Above: chunks through
// a ring of slots, the device filling some while the pool's threads empty
// others; large chunks first (each costs the device about 15 us besides its
// transfer), small ones last (what is left for the threads after the last has
// arrived).  PCIe bound, 57 GB/s.  HIP's own pageable path takes 18 GB/s:
//   64 KB 39 -> 11 us, 4 MB 236 -> 120, 50 MB 2.97 -> 1.06 ms, 124 MB 7.4 -> 2.5.
// Only as many threads take part as the largest chunk has kSlice: 1.1 MB takes
// 47 us with 64, 128 and 256 KB a thread and 50 with 512, and 0.28, 0.28, 0.17
// and 0.13 ms of CPU time (always eight threads: 47 us and 0.23 to 0.28 ms).
// gates (ascending, the last one covers all): chunks end where a gate does, and
// the first chunk behind a gate's predecessor waits for the gate.
int copy_to_host(llfem_ctx* ctx, double* dst_, const double* src_, size_t n, const CopyGate* gates, int ngates) {
  constexpr size_t kOneCopy = size_t(512) << 10, kSmall = size_t(4) << 20, kSlot = size_t(16) << 20;
  constexpr size_t kSlice = size_t(256) << 10;   // of the largest chunk, per thread
  constexpr size_t kSlots = CopyPool::kSlots;
  const size_t bytes = n * sizeof(double);
  if (bytes == 0) {
    LLFEM_HIP(hipStreamSynchronize(ctx->stream));
    return LLFEM_OK;
  }
  hipStream_t st = ctx->stream;
  char* dst = reinterpret_cast<char*>(dst_);
  const char* src = reinterpret_cast<const char*>(src_);
  auto slot = [&](size_t s) -> int {
    if (ctx->h_stage[s]) return LLFEM_OK;
    if (!ctx->stage_ev[s]) LLFEM_HIP(hipEventCreateWithFlags(&ctx->stage_ev[s], hipEventDisableTiming));
    LLFEM_HIP(hipHostMalloc(&ctx->h_stage[s], kSlot, hipHostMallocDefault));
    return LLFEM_OK;
  };
  LLFEM_TRY(slot(0));
  if (bytes <= kOneCopy) {
    for (int g = 0; g < ngates; ++g)
      for (hipEvent_t e : gates[g].ev)
        if (e) LLFEM_HIP(hipStreamWaitEvent(st, e, 0));
    LLFEM_HIP(hipMemcpyAsync(ctx->h_stage[0], src, bytes, hipMemcpyDeviceToHost, st));
    LLFEM_HIP(hipStreamSynchronize(st));
    std::memcpy(dst, ctx->h_stage[0], bytes);
    return LLFEM_OK;
  }
  std::vector<std::pair<size_t, size_t>> chunk;   // offset, length
  int g = 0;
  for (size_t off = 0; off < bytes;) {
    while (g < ngates && gates[g].end * sizeof(double) <= off) ++g;
    const size_t left = bytes - off;
    size_t len = std::min(left, std::min(kSlot, std::max(kSmall, left / 4 / kSmall * kSmall)));
    if (g < ngates) len = std::min(len, gates[g].end * sizeof(double) - off);
    chunk.push_back({off, len});
    off += len;
  }
  int opened = 0;   // gates waited for
  auto issue = [&](size_t i) -> int {
    const size_t s = i % kSlots;
    LLFEM_TRY(slot(s));
    const size_t end = (chunk[i].first + chunk[i].second) / sizeof(double);
    for (; opened < ngates && (opened == 0 || gates[opened - 1].end < end); ++opened)
      for (hipEvent_t e : gates[opened].ev)
        if (e) LLFEM_HIP(hipStreamWaitEvent(st, e, 0));
    LLFEM_HIP(hipMemcpyAsync(ctx->h_stage[s], src + chunk[i].first, chunk[i].second, hipMemcpyDeviceToHost, st));
    LLFEM_HIP(hipEventRecord(ctx->stage_ev[s], st));
    return LLFEM_OK;
  };
  size_t issued = 0;
  for (; issued < chunk.size() && issued < kSlots; ++issued) LLFEM_TRY(issue(issued));
  if (!ctx->pool) ctx->pool = new CopyPool();
  CopyPool& pool = *ctx->pool;
  const bool threads = pool.threads() > 0;
  size_t largest = 0;
  for (const auto& c : chunk) largest = std::max(largest, c.second);
  if (threads) pool.begin(chunk.size(), (int)((largest + kSlice - 1) / kSlice));
  auto drain = [&]() -> int {
    for (size_t i = 0; i < chunk.size(); ++i) {
      const size_t s = i % kSlots;
      LLFEM_HIP(hipEventSynchronize(ctx->stage_ev[s]));
      if (threads) pool.arrived(i, dst + chunk[i].first, static_cast<const char*>(ctx->h_stage[s]), chunk[i].second);
      else std::memcpy(dst + chunk[i].first, ctx->h_stage[s], chunk[i].second);
      // refill the slots emptied meanwhile: the one of the chunk before this one
      if (i >= 1 && issued < chunk.size()) {
        if (threads) pool.wait_free(issued % kSlots);
        LLFEM_TRY(issue(issued));
        ++issued;
      }
    }
    return LLFEM_OK;
  };
  const int rc = drain();
  if (threads) pool.finish(rc != LLFEM_OK);
  return rc;
}

// Content hash for cache keys (not cryptographic): four independent 64-bit
// multiply-rotate lanes over 32-byte strides, byte-wise FNV-1a on the tail,
// then a final avalanche.  Several GB/s, so hashing a request's mesh arrays
// costs milliseconds.
uint64_t hash_bytes(const void* p, size_t n, uint64_t h) {
  constexpr uint64_t kA = 0x9E3779B97F4A7C15ull, kB = 0xBF58476D1CE4E5B9ull, kC = 0x94D049BB133111EBull;
  auto rotl = [](uint64_t x, int r) { return (x << r) | (x >> (64 - r)); };
  const unsigned char* c = static_cast<const unsigned char*>(p);
  uint64_t lane[4] = {h ^ kA, h + kB, rotl(h, 21) ^ kC, h - kA};
  size_t i = 0;
  for (; i + 32 <= n; i += 32)
    for (int k = 0; k < 4; ++k) {
      uint64_t w;
      std::memcpy(&w, c + i + 8 * k, 8);
      lane[k] = rotl(lane[k] + w * kB, 31) * kA;
    }
  uint64_t r = h ^ ((uint64_t)n * kC);
  for (int k = 0; k < 4; ++k) r = (r ^ rotl(lane[k], 17 + 8 * k)) * kB;
  for (; i < n; ++i) r = (r ^ c[i]) * 1099511628211ull;
  r ^= r >> 31;
  r *= kC;
  r ^= r >> 29;
  return r;
}

}  // namespace llfem

// ---- workspace of the allocation-free solve ------------------------------
// One array per GPU, part of this library's device image: the runtime places
// it when the image is loaded on a device and it stays until the process
// ends.  In host code `scratch` names a host-side stand-in, never the device
// memory: host code uses only the address hipGetSymbolAddress returns for
// the current device, kept per device in g_scratch.
static __device__ __align__(256) unsigned char scratch[llfem::kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
struct ScratchSlot {
  std::mutex call;          // one allocation-free solve at a time on the device
  void* ptr = nullptr;      // device address of `scratch` on this device
};
ScratchSlot g_scratch[kMaxDevices];
std::mutex g_scratch_setup;
}  // namespace

namespace llfem {

int noalloc_scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices)
    return fail(LLFEM_EUNSUP, "device ordinal " + std::to_string(device) + " above the supported maximum");
  std::lock_guard<std::mutex> lk(g_scratch_setup);
  if (g_scratch[device].ptr) return LLFEM_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    return fail(LLFEM_EHIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
  g_scratch[device].ptr = p;
  return LLFEM_OK;
}

bool noalloc_scratch(int device, void** ptr, std::mutex** lock) {
  if (device < 0 || device >= kMaxDevices) return false;
  {
    std::lock_guard<std::mutex> lk(g_scratch_setup);
    if (!g_scratch[device].ptr) return false;
    *ptr = g_scratch[device].ptr;
  }
  *lock = &g_scratch[device].call;
  return true;
}

}  // namespace llfem

using namespace llfem;

extern "C" {

const char* llfem_last_error(void) { return g_error.c_str(); }

int llfem_ctx_create(int device, size_t hbm_budget_bytes, llfem_ctx** out) {
  if (!out) return fail(LLFEM_EINVAL, "llfem_ctx_create: out is NULL");
  *out = nullptr;
  int ndev = 0;
  LLFEM_HIP(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev)
    return fail(LLFEM_EINVAL, "llfem_ctx_create: device " + std::to_string(device) +
                                  " out of range (" + std::to_string(ndev) + " devices)");
  LLFEM_HIP(hipSetDevice(device));
  hipDeviceProp_t prop;
  LLFEM_HIP(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(LLFEM_EUNSUP, std::string("libllfem is built for gfx950; device is ") +
                                  prop.gcnArchName);
  // device address of the allocation-free solve's workspace, once per device
  LLFEM_TRY(llfem::noalloc_scratch_setup(device));
  llfem_ctx* c = new llfem_ctx();
  c->device = device;
  c->budget = hbm_budget_bytes;
  c->num_cus = prop.multiProcessorCount;
  // default-priority stream (never a priority stream)
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return fail(LLFEM_EHIP, "hipStreamCreate failed");
  }
  for (auto& e : c->ev) (void)hipEventCreate(&e);
  // side streams for concurrent panel launches, created here so the first
  // assembly does not pay for them
  for (int k = 0; k < 2; ++k) {
    if (hipStreamCreateWithFlags(&c->side[k], hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c->join_ev[k], hipEventDisableTiming) != hipSuccess) {
      llfem_ctx_destroy(c);
      return fail(LLFEM_EHIP, "hipStreamCreate failed");
    }
  }
  if (hipEventCreateWithFlags(&c->fork_ev, hipEventDisableTiming) != hipSuccess) {
    llfem_ctx_destroy(c);
    return fail(LLFEM_EHIP, "hipEventCreate failed");
  }
  if (hipHostMalloc((void**)&c->h_poll, 64, hipHostMallocDefault) != hipSuccess ||
      hipEventCreateWithFlags(&c->poll_ev[0], hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->poll_ev[1], hipEventDisableTiming) != hipSuccess) {
    llfem_ctx_destroy(c);
    return fail(LLFEM_EHIP, "llfem_ctx_create: pinned memory or events failed");
  }
  *out = c;
  return LLFEM_OK;
}

int llfem_ctx_destroy(llfem_ctx* ctx) {
  if (!ctx) return LLFEM_OK;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  for (auto& e : ctx->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto& kv : ctx->tables) llfem::dfree(ctx, kv.second.ptr, kv.second.bytes);
  ctx->tables.clear();
  if (ctx->d_scratch) llfem::dfree(ctx, ctx->d_scratch, ctx->scratch_bytes);
  llfem::ws_release(ctx);
  if (ctx->d_sink) llfem::dfree(ctx, ctx->d_sink, 64 * sizeof(double));
  for (int k = 0; k < 2; ++k) {
    if (ctx->side[k]) {
      (void)hipStreamSynchronize(ctx->side[k]);
      (void)hipStreamDestroy(ctx->side[k]);
    }
    if (ctx->join_ev[k]) (void)hipEventDestroy(ctx->join_ev[k]);
  }
  if (ctx->fork_ev) (void)hipEventDestroy(ctx->fork_ev);
  if (ctx->h_poll) (void)hipHostFree(ctx->h_poll);
  for (auto& e : ctx->poll_ev)
    if (e) (void)hipEventDestroy(e);
  for (auto& part : ctx->gate_ev)
    for (auto& e : part)
      if (e) (void)hipEventDestroy(e);
  delete ctx->pool;
  for (size_t b = 0; b < sizeof(ctx->h_stage) / sizeof(ctx->h_stage[0]); ++b) {
    if (ctx->h_stage[b]) (void)hipHostFree(ctx->h_stage[b]);
    if (ctx->stage_ev[b]) (void)hipEventDestroy(ctx->stage_ev[b]);
  }
  (void)hipStreamDestroy(ctx->stream);
  delete ctx;
  return LLFEM_OK;
}

int llfem_ctx_synchronize(llfem_ctx* ctx) {
  if (!ctx) return fail(LLFEM_EINVAL, "llfem_ctx_synchronize: NULL context");
  LLFEM_HIP(hipStreamSynchronize(ctx->stream));
  return LLFEM_OK;
}

size_t llfem_ctx_bytes_in_use(const llfem_ctx* ctx) { return ctx ? ctx->in_use : 0; }

}  // extern "C"
