// spk_runtime.hip -- device selection, the library stream, device memory,
// timers, the workspace pool and the reduction scratch.
#include "spk_link.hpp"
#include "spk_tri.hpp"

#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <unordered_map>

namespace spk {

// Device scratch for the entry points that allocate nothing
// (spk_cg_solve_noalloc).  In host code `scratch` names a host-side stand-in,
// not device memory: every host use goes through the address
// hipGetSymbolAddress returned for the current device (g_scratch_dev).
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
void* g_scratch_dev[kMaxDevices] = {};

struct Arena {
  char* base = nullptr;
  size_t cap = 0, used = 0;
  void* slot_ptr[kArenaSlots] = {};
  size_t slot_bytes[kArenaSlots] = {};
  double* partials = nullptr;
  size_t partials_count = 0;
};
Arena* g_arena = nullptr;

void* arena_carve(Arena& a, size_t bytes) {
  const size_t need = arena_round(bytes > 0 ? bytes : 1);
  if (need > a.cap - a.used)
    throw Error{SPK_INVALID_ARGUMENT,
                "no-allocation scratch exhausted: " + std::to_string(a.used) +
                    " + " + std::to_string(need) + " bytes > " +
                    std::to_string(a.cap)};
  void* p = a.base + a.used;
  a.used += need;
  return p;
}

thread_local std::string g_last_error;
Context g_ctx;
std::mutex g_init_mutex;
hipStream_t g_user_stream = nullptr;
hipEvent_t g_ev0 = nullptr, g_ev1 = nullptr;
std::unique_ptr<Workspace> g_ws;
DevBuf<double>* g_partials = nullptr;
DevBuf<unsigned long long>* g_link = nullptr;

__global__ void link_clear_kernel(unsigned long long* w, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) w[k] = 0;
}

unsigned g_link_polls = kLinkPolls;

bool g_own_all_cus = true;  // of g_ctx.stream, which does not change

// Whether a stream may use every CU: one made with a CU mask may not.
bool stream_has_all_cus(hipStream_t s) {
  uint32_t mask[64] = {};
  if (hipExtStreamGetCUMask(s, 64, mask) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  int cus = 0;
  for (uint32_t w : mask) cus += __builtin_popcount(w);
  return cus >= g_ctx.num_cus;
}

// the link's words: slots, tag and flag
void clear_link(unsigned long long* w, hipStream_t s) {
  const int n = (int)kLinkWords;
  hipLaunchKernelGGL(link_clear_kernel, dim3((n + 255) / 256), dim3(256), 0, s, w, n);
  SPK_HIP_TRY(hipGetLastError());
}

// ---- the device memory pool
//
// A block freed waits in `idle` of its size until something of that size is
// wanted and no block is `ready`; then the device is waited for once, and
// every block that was idle by then is ready.  So a block's next owner starts
// after all work queued before the free, on any stream of any thread, as with
// hipFree (which waits too, each time).  Small sizes keep several blocks, so
// that a loop that makes and drops a vector waits once in many rounds.
// Measured on y = multiply(A, x), 4,096 rows: hipMalloc and hipFree took 13
// of the call's 16.5 us.
class Pool {
 public:
  hipError_t get(void** p, size_t bytes) {
    const size_t size = rounded(bytes);
    std::lock_guard<std::mutex> lk(m_);
    if (!open()) {
      const hipError_t e = hipMalloc(p, bytes);
      if (e == hipSuccess) owned_.erase(*p);
      return e;
    }
    Size& c = sizes_[size];
    c.used = ++uses_;
    if (c.ready.empty() && c.idle.size() >= idle_limit(size)) {
      if (hipDeviceSynchronize() == hipSuccess) {
        for (auto& s : sizes_) {
          s.second.ready.insert(s.second.ready.end(), s.second.idle.begin(),
                                s.second.idle.end());
          s.second.idle.clear();
        }
      } else {
        (void)hipGetLastError();
      }
    }
    if (!c.ready.empty()) {
      *p = c.ready.back();
      c.ready.pop_back();
      kept_ -= size;
      --blocks_;
      own(*p, size);
      return hipSuccess;
    }
    hipError_t e = hipMalloc(p, size);
    if (e != hipSuccess && kept_ > 0) {
      (void)hipGetLastError();
      give_back();
      e = hipMalloc(p, size);
    }
    if (e == hipSuccess) own(*p, size);
    return e;
  }
  enum Put { kTaken, kForeign, kFreed };  // kFreed: it has been freed before
  Put put(void* p) {
    std::lock_guard<std::mutex> lk(m_);
    auto it = owned_.find(p);
    if (it == owned_.end()) return kForeign;
    if (it->second.kept) return kFreed;
    const size_t size = it->second.size;
    if (!open() || !still_ours(p, size)) {
      owned_.erase(it);
      return kForeign;
    }
    if (size > kLargest) {
      owned_.erase(it);
      (void)hipFree(p);
      return kTaken;
    }
    Size& c = sizes_[size];
    c.idle.push_back(p);
    c.used = ++uses_;
    it->second.kept = true;
    kept_ += size;
    ++blocks_;
    while (kept_ > kMost || blocks_ > kMostBlocks) evict();
    return kTaken;
  }
  void drain() {
    std::lock_guard<std::mutex> lk(m_);
    give_back();
  }

 private:
  struct Block {
    size_t size;
    bool kept;
  };
  struct Size {
    std::vector<void*> ready, idle;
    unsigned long long used = 0;  // when it was last asked for or freed into
  };
  static constexpr size_t kMost = size_t(2) << 30;      // bytes kept, at most
  static constexpr size_t kLargest = size_t(256) << 20;  // a kept block's size
  static constexpr size_t kMostBlocks = 512;
  // sizes an eighth of a power of two apart, few enough to meet again; what
  // is never kept is not rounded
  static size_t rounded(size_t bytes) {
    if (bytes > kLargest) return bytes;
    size_t step = 512;
    while (bytes > 8 * step) step *= 2;
    return bytes == 0 ? step : (bytes + step - 1) / step * step;
  }
  static size_t idle_limit(size_t size) {
    return size <= (64 << 10) ? 16 : size <= (1 << 20) ? 4 : 1;
  }
  // The pool keeps out of captures, of other devices and of the time after
  // spk_finalize: hipMalloc and hipFree then decide, as without a pool.
  static bool open() {
    int dev = -1;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (g_ctx.device < 0) return false;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipStreamIsCapturing(g_user_stream ? g_user_stream : g_ctx.stream, &st) !=
            hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return dev == g_ctx.device && st == hipStreamCaptureStatusNone;
  }
  // A caller may have given a block of the pool back by hipFree; its address is
  // then whatever was allocated there since.
  static bool still_ours(void* p, size_t size) {
    hipDeviceptr_t base = nullptr;
    size_t bytes = 0;
    if (hipMemGetAddressRange(&base, &bytes, (hipDeviceptr_t)p) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return base == (hipDeviceptr_t)p && bytes == size;
  }
  void drop(void* p) {
    owned_.erase(p);
    (void)hipFree(p);
  }
  void own(void* p, size_t size) {
    try {
      owned_[p] = Block{size, false};
    } catch (const std::bad_alloc&) {  // then it goes back by hipFree
    }
  }
  // a block of the size that has lain longest goes back
  void evict() {
    auto old = sizes_.end();
    for (auto it = sizes_.begin(); it != sizes_.end(); ++it)
      if ((!it->second.ready.empty() || !it->second.idle.empty()) &&
          (old == sizes_.end() || it->second.used < old->second.used))
        old = it;
    std::vector<void*>& v = old->second.ready.empty() ? old->second.idle : old->second.ready;
    drop(v.back());
    v.pop_back();
    kept_ -= old->first;
    --blocks_;
  }
  void give_back() {  // hipFree waits for the device itself
    for (auto& s : sizes_) {
      for (void* p : s.second.ready) drop(p);
      for (void* p : s.second.idle) drop(p);
    }
    sizes_.clear();
    kept_ = blocks_ = 0;
  }
  std::mutex m_;
  std::map<size_t, Size> sizes_;
  std::unordered_map<void*, Block> owned_;  // handed out or kept
  size_t kept_ = 0, blocks_ = 0;
  unsigned long long uses_ = 0;
};
Pool& pool() {
  static Pool* p = new Pool();  // outlives the objects that free into it
  return *p;
}

void init_device(int device) {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
    throw Error{SPK_NO_DEVICE, "no HIP device available"};
  SPK_REQUIRE(device >= 0 && device < count, SPK_INVALID_ARGUMENT,
              "device index out of range");
  SPK_HIP_TRY(hipSetDevice(device));
  SPK_REQUIRE(device < kMaxDevices, SPK_INVALID_ARGUMENT, "device index too large");
  if (!g_scratch_dev[device]) {
    void* p = nullptr;
    SPK_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_dev[device] = p;
  }
  hipDeviceProp_t prop;
  SPK_HIP_TRY(hipGetDeviceProperties(&prop, device));
  g_ctx.device = device;
  g_ctx.num_cus = prop.multiProcessorCount;
  SPK_HIP_TRY(hipStreamCreateWithFlags(&g_ctx.stream, hipStreamNonBlocking));
  SPK_HIP_TRY(hipEventCreate(&g_ev0));
  SPK_HIP_TRY(hipEventCreate(&g_ev1));
  g_partials = new DevBuf<double>(1 << 16);
  g_ws.reset(new Workspace());
  g_own_all_cus = stream_has_all_cus(g_ctx.stream);
  // made here, so that a solve which may not allocate has it too
  g_link = new DevBuf<unsigned long long>(kLinkWords);
  clear_link(g_link->p, g_ctx.stream);
  SPK_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
}
}  // namespace

void set_error(const std::string& msg) { g_last_error = msg; }

hipError_t pool_malloc(void** p, size_t bytes) { return pool().get(p, bytes); }
void pool_free(void* p) {
  Pool::Put r = Pool::kForeign;
  try {
    r = pool().put(p);
  } catch (const std::bad_alloc&) {  // called by destructors
  }
  if (r == Pool::kForeign) (void)hipFree(p);
}

Context& ctx() {
  if (g_ctx.device < 0) {
    std::lock_guard<std::mutex> lk(g_init_mutex);
    if (g_ctx.device < 0) init_device(0);
  }
  return g_ctx;
}

hipStream_t stream() {
  Context& c = ctx();
  return g_user_stream ? g_user_stream : c.stream;
}

void* scratch_ptr() {
  Context& c = ctx();
  void* p = g_scratch_dev[c.device];
  SPK_REQUIRE(p, SPK_HIP_ERROR, "scratch address unknown for this device");
  return p;
}

size_t scratch_bytes() { return kScratchBytes; }

ArenaScope::ArenaScope(void* base, size_t bytes, size_t partials) {
  SPK_REQUIRE(!g_arena, SPK_INVALID_ARGUMENT, "nested no-allocation calls");
  static Arena arena;  // fixed host bookkeeping, reset per scope
  arena = Arena{};
  arena.base = (char*)base;
  arena.cap = bytes;
  arena.partials = (double*)arena_carve(arena, partials * sizeof(double));
  arena.partials_count = partials;
  g_arena = &arena;
}

ArenaScope::~ArenaScope() { g_arena = nullptr; }

void* Workspace::get(int slot, size_t bytes) {
  if (g_arena) {
    Arena& a = *g_arena;
    SPK_REQUIRE(slot >= 0 && slot < kArenaSlots, SPK_INVALID_ARGUMENT,
                "workspace slot out of range");
    if (!a.slot_ptr[slot] || a.slot_bytes[slot] < bytes) {
      a.slot_ptr[slot] = arena_carve(a, bytes);
      a.slot_bytes[slot] = bytes;
    }
    return a.slot_ptr[slot];
  }
  if ((size_t)slot >= bufs.size()) bufs.resize(slot + 1);
  bufs[slot].reserve(bytes);
  return bufs[slot].p;
}

Workspace& workspace() {
  ctx();
  return *g_ws;
}

double* reduce_partials(size_t count) {
  ctx();
  if (g_arena) {
    SPK_REQUIRE(count <= g_arena->partials_count, SPK_INVALID_ARGUMENT,
                "no-allocation scratch: reduction partials exceed the reserve");
    return g_arena->partials;
  }
  if (count > g_partials->n) {
    // the old array may still be read by queued kernels
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    g_partials->alloc(count + count / 4);
  }
  return g_partials->p;
}

GridLink grid_link() {
  unsigned long long* w = (ctx(), g_link->p);
  return GridLink{w, (unsigned*)(w + kLinkSlotWords), (int*)(w + kLinkSlotWords + 1),
                  (g_user_stream ? stream_has_all_cus(g_user_stream) : g_own_all_cus)
                      ? std::min(kLinkBlocks, g_ctx.num_cus)
                      : 1,
                  g_link_polls};
}

void renew_link(const GridLink& l) { clear_link(l.slots, stream()); }

}  // namespace spk

using namespace spk;

extern "C" {

const char* spk_last_error(void) { return g_last_error.c_str(); }

spk_status spk_init(int device) {
  return guarded([&] {
    std::lock_guard<std::mutex> lk(g_init_mutex);
    if (g_ctx.device < 0) init_device(device);
    else SPK_REQUIRE(g_ctx.device == device, SPK_INVALID_ARGUMENT,
                     "library already initialised on another device");
  });
}

spk_status spk_finalize(void) {
  return guarded([&] {
    if (g_ctx.device < 0) return;
    SPK_HIP_TRY(hipDeviceSynchronize());
    g_ws.reset();
    delete g_partials;
    g_partials = nullptr;
    delete g_link;
    g_link = nullptr;
    pool().drain();
    (void)hipEventDestroy(g_ev0);
    (void)hipEventDestroy(g_ev1);
    (void)hipStreamDestroy(g_ctx.stream);
    g_ctx = Context{};
  });
}

spk_status spk_set_stream(void* s) {
  return guarded([&] {
    ctx();
    g_user_stream = (hipStream_t)s;
  });
}

void* spk_get_stream(void) {
  void* s = nullptr;
  guarded([&] { s = (void*)stream(); });
  return s;
}

spk_status spk_synchronize(void) {
  return guarded([&] { SPK_HIP_TRY(hipStreamSynchronize(stream())); });
}

spk_status spk_device_info(int* num_cus, char* name, size_t name_len) {
  return guarded([&] {
    Context& c = ctx();
    if (num_cus) *num_cus = c.num_cus;
    if (name && name_len) {
      hipDeviceProp_t prop;
      SPK_HIP_TRY(hipGetDeviceProperties(&prop, c.device));
      std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
  });
}

spk_status spk_set_exchange_polls(uint32_t polls) {
  return guarded([&] { g_link_polls = polls ? polls : kLinkPolls; });
}

spk_status spk_set_sweep_wait(uint64_t ticks) {
  return guarded([&] { set_tri_wait(ticks); });
}

spk_status spk_malloc(void** dptr, size_t bytes) {
  return guarded([&] {
    ctx();
    SPK_REQUIRE(dptr, SPK_INVALID_ARGUMENT, "null output pointer");
    hipError_t e = pool_malloc(dptr, bytes ? bytes : 1);
    if (e != hipSuccess)
      throw Error{SPK_OUT_OF_MEMORY, "hipMalloc failed: " +
                  std::string(hipGetErrorString(e))};
  });
}

spk_status spk_free(void* dptr) {
  return guarded([&] {
    ctx();
    if (!dptr) return;
    const Pool::Put r = pool().put(dptr);
    if (r == Pool::kTaken) return;
    if (r == Pool::kFreed) SPK_HIP_TRY(hipErrorInvalidValue);  // as hipFree says
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    SPK_HIP_TRY(hipFree(dptr));
  });
}

spk_status spk_release_memory(void) {
  return guarded([&] {
    ctx();
    pool().drain();
  });
}

spk_status spk_memcpy_htod(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    SPK_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream()));
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
  });
}

spk_status spk_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    SPK_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream()));
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
  });
}

spk_status spk_memcpy_dtod(void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    SPK_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream()));
  });
}

spk_status spk_memset(void* dst, int value, size_t bytes) {
  return guarded([&] { SPK_HIP_TRY(hipMemsetAsync(dst, value, bytes, stream())); });
}

spk_status spk_timer_start(void) {
  return guarded([&] {
    ctx();
    SPK_HIP_TRY(hipEventRecord(g_ev0, stream()));
  });
}

spk_status spk_timer_stop(float* ms) {
  return guarded([&] {
    ctx();
    SPK_HIP_TRY(hipEventRecord(g_ev1, stream()));
    SPK_HIP_TRY(hipEventSynchronize(g_ev1));
    SPK_HIP_TRY(hipEventElapsedTime(ms, g_ev0, g_ev1));
  });
}

}  // extern "C"
