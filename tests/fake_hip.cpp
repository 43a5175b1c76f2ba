// fake_hip.cpp -- the HIP calls that liblcr.so makes, over host memory and without
// kernels, for CPU tests of its host code: what is allocated, kept and given back,
// what is in flight when, and what a failing call leaves.  Loaded before liblcr.so
// (preloaded), so that liblcr.so's calls bind here.
//
// Device blocks come from slots of address space, the lowest free one first: a block
// freed and one allocated next share an address, whatever their sizes.  Every new
// block is filled with kPoison.  Copies are done at once and checked against the
// blocks' bounds; work on a stream counts as pending until something waits for it.
// A few kernels leave what the host needs to go on (see launch()).
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <chrono>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

constexpr size_t kSlot = (size_t)1 << 31;
constexpr int kSlots = 2048;
constexpr int kPoison = 0xA5;

struct Stream {
  int pending = 0;
};
struct Config {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
};

std::mutex mu;
char* arena = nullptr;
size_t used[kSlots];                 // bytes of the block in each slot, 0: free
std::map<char*, size_t> pinned;      // pinned blocks
std::map<const void*, std::string> names;
std::map<std::string, int64_t> launches;  // by mangled kernel name
thread_local std::vector<Config> configs;
std::map<Stream*, int> streams;
int* compact_host = nullptr;         // where the last k_compact reports to
std::string faults;                  // what a check found, a line each
int64_t opt[8];                      // see fake_set
int64_t stat[8];                     // see fake_get
enum Opt { kPoints, kDeviceLimit, kPinnedLimit, kFailMallocFrom, kNoCompact, kClockNs, kPrevAt, kFitListAt };
enum Stat { kDeviceBytes, kDevicePeak, kPinnedBytes, kPinnedPeak, kMallocs, kLargestPinned, kPageable, kFitnessOld };

void fault(const std::string& what) { faults += what + "\n"; }

int slot_of(const void* p) {
  const char* c = static_cast<const char*>(p);
  if (!arena || c < arena || c >= arena + kSlots * kSlot) return -1;
  return (int)((c - arena) / kSlot);
}

// The block that holds [p, p + n), or a fault when it leaves one.
bool in_bounds(const void* p, size_t n, const char* what) {
  if (n == 0) return true;
  if (!p) {
    fault(std::string(what) + ": null pointer");
    return false;
  }
  const int s = slot_of(p);
  if (s < 0) return true;  // the program's own memory
  const size_t at = (size_t)(static_cast<const char*>(p) - (arena + s * kSlot));
  if (at + n <= used[s]) return true;
  fault(std::string(what) + ": outside its block");
  return false;
}

bool on_device(const void* p) { return slot_of(p) >= 0; }
bool is_pinned(const void* p) {
  auto it = pinned.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
  if (it == pinned.begin()) return false;
  --it;
  return p < it->first + it->second;
}

void work(hipStream_t s) {
  auto* q = reinterpret_cast<Stream*>(s);
  if (streams.count(q)) q->pending += 1;
}
void wait(hipStream_t s) {
  auto* q = reinterpret_cast<Stream*>(s);
  if (streams.count(q)) q->pending = 0;
}
void wait_all() {
  for (auto& s : streams) s.first->pending = 0;
}

hipError_t copy(void* dst, const void* src, size_t n) {
  if (!in_bounds(dst, n, "copy to") || !in_bounds(src, n, "copy from")) return hipErrorInvalidValue;
  // a copy to or from memory that is not pinned
  for (const void* p : {(const void*)dst, src})
    if (n && !on_device(p) && !is_pinned(p)) stat[kPageable] += (int64_t)n;
  memcpy(dst, src, n);
  return hipSuccess;
}

// No instance is active any more.
void compact() {
  if (!compact_host || opt[kNoCompact]) return;
  compact_host[0] = compact_host[1] = 0;
  compact_host[2] = 1;
}

template <class T>
T arg(void** args, int i) {
  return *static_cast<T*>(args[i]);
}

void launch(const std::string& name, dim3 grid, void** args) {
  auto is = [&](const char* k) { return name.find(k) != std::string::npos; };
  if (is("k_fill_i32")) {
    int* p = arg<int*>(args, 0);
    const int64_t n = arg<int64_t>(args, 1);
    if (in_bounds(p, (size_t)n * 4, "k_fill_i32"))
      for (int64_t i = 0; i < n; ++i) p[i] = arg<int>(args, 2);
  } else if (is("k_bbox_final")) {
    // unit boxes of opt[kPoints] points, a quarter of as many probe cells occupied
    float* g = arg<float*>(args, 1);
    for (unsigned c = 0; c < grid.x; ++c) {
      const float box[7] = {0, 0, 0, 1, 1, 1, (float)opt[kPoints]};
      memcpy(g + 8 * c, box, sizeof box);
      const int occ = (int)(opt[kPoints] / 4);
      memcpy(g + 8 * c + 7, &occ, 4);
    }
  } else if (is("k_cell_count")) {
    // the counters have to be zero over their whole block
    const char* p = reinterpret_cast<const char*>(arg<int*>(args, 5));
    const int s = slot_of(p);
    if (s < 0) {
      fault("k_cell_count: no counters");
    } else {
      for (size_t i = 0; i < used[s]; ++i)
        if (p[i]) {
          fault("k_cell_count: counters not zero");
          break;
        }
    }
  } else if (is("k_fitness") && !is("fold") && opt[kPrevAt]) {
    // whether the last fitness pass was given previous matches or a list of tiles
    const char* b = static_cast<const char*>(args[0]);
    void *prev, *list;
    memcpy(&prev, b + opt[kPrevAt], sizeof prev);
    memcpy(&list, b + opt[kFitListAt], sizeof list);
    stat[kFitnessOld] = (prev ? 1 : 0) + (list ? 2 : 0);
  } else if (is("k_icp_iter") && opt[kPrevAt]) {
    // every buffer up to prev is there (normals: not point-to-point)
    const char* b = static_cast<const char*>(args[0]);
    for (int64_t at = 0; at <= opt[kPrevAt]; at += 8) {
      void* p;
      memcpy(&p, b + at, sizeof p);
      if (!p && at != 24) return fault("k_icp_iter: null buffer");
    }
  } else if (is("k_enc_bf16_weights")) {
    memset(arg<char*>(args, 1), 0, 64 * 128 * 2);
    memset(arg<char*>(args, 2), 0, 128 * 256 * 2);
  } else if (is("k_enc_points")) {
    // every buffer is there and both layers' BF16 weights were written
    for (int i : {0, 4, 5, 6, 7, 8})
      if (!arg<char*>(args, i)) return fault("k_enc_points: null buffer");
    for (int i : {5, 6})
      if (*arg<unsigned char*>(args, i) == kPoison) fault("k_enc_points: weights not written");
  } else if (is("9k_compact")) {
    if (arg<int*>(args, 5)) {
      compact_host = arg<int*>(args, 5);
      compact();
    }
  }
}

}  // namespace

// Time stands still unless a test moves it.
std::chrono::steady_clock::time_point std::chrono::_V2::steady_clock::now() noexcept {
  return time_point(duration(1000000000ll + opt[kClockNs]));
}

extern "C" {

// ------------------------------------------------------------- for the tests
void fake_set(int what, int64_t v) { opt[what] = v; }
int64_t fake_get(int what) { return stat[what]; }
void fake_reset_peaks() {
  stat[kDevicePeak] = stat[kDeviceBytes];
  stat[kPinnedPeak] = stat[kPinnedBytes];
  stat[kLargestPinned] = stat[kPageable] = 0;
}
int64_t fake_pending() {
  int64_t n = 0;
  for (auto& s : streams) n += s.first->pending;
  return n;
}
int64_t fake_streams() { return (int64_t)streams.size(); }
int64_t fake_launches(const char* part) {
  int64_t n = 0;
  for (auto& l : launches)
    if (l.first.find(part) != std::string::npos) n += l.second;
  return n;
}
const char* fake_faults() { return faults.c_str(); }

// --------------------------------------------------------------- memory
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> g(mu);
  stat[kMallocs] += 1;
  *p = nullptr;
  if ((opt[kFailMallocFrom] && stat[kMallocs] >= opt[kFailMallocFrom]) ||
      (opt[kDeviceLimit] && stat[kDeviceBytes] + (int64_t)n > opt[kDeviceLimit]) || n > kSlot)
    return hipErrorOutOfMemory;
  if (!arena)
    arena = static_cast<char*>(mmap(nullptr, kSlots * kSlot, PROT_READ | PROT_WRITE,
                                    MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0));
  for (int s = 0; s < kSlots; ++s) {
    if (used[s]) continue;
    used[s] = n;
    *p = arena + s * kSlot;
    if (n <= ((size_t)256 << 20)) memset(*p, kPoison, n);
    stat[kDeviceBytes] += (int64_t)n;
    if (stat[kDeviceBytes] > stat[kDevicePeak]) stat[kDevicePeak] = stat[kDeviceBytes];
    return hipSuccess;
  }
  return hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> g(mu);
  wait_all();
  const int s = slot_of(p);
  if (s < 0 || !used[s]) {
    fault("hipFree: not a block");
    return hipErrorInvalidValue;
  }
  stat[kDeviceBytes] -= (int64_t)used[s];
  (void)madvise(arena + s * kSlot, used[s], MADV_DONTNEED);
  used[s] = 0;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> g(mu);
  *p = nullptr;
  if (opt[kPinnedLimit] && stat[kPinnedBytes] + (int64_t)n > opt[kPinnedLimit]) return hipErrorOutOfMemory;
  char* c = static_cast<char*>(mmap(nullptr, n, PROT_READ | PROT_WRITE,
                                    MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0));
  pinned[c] = n;
  *p = c;
  stat[kPinnedBytes] += (int64_t)n;
  if (stat[kPinnedBytes] > stat[kPinnedPeak]) stat[kPinnedPeak] = stat[kPinnedBytes];
  if ((int64_t)n > stat[kLargestPinned]) stat[kLargestPinned] = (int64_t)n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> g(mu);
  wait_all();
  auto it = pinned.find(static_cast<char*>(p));
  if (it == pinned.end()) {
    fault("hipHostFree: not a block");
    return hipErrorInvalidValue;
  }
  stat[kPinnedBytes] -= (int64_t)it->second;
  munmap(p, it->second);
  pinned.erase(it);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::lock_guard<std::mutex> g(mu);
  return copy(d, s, n);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  std::lock_guard<std::mutex> g(mu);
  work(q);
  return copy(d, s, n);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t q) {
  std::lock_guard<std::mutex> g(mu);
  work(q);
  if (!in_bounds(d, n, "memset")) return hipErrorInvalidValue;
  memset(d, v, n);
  return hipSuccess;
}

// ------------------------------------------------------- streams and events
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  std::lock_guard<std::mutex> g(mu);
  auto* q = new Stream;
  streams[q] = 1;
  *s = reinterpret_cast<hipStream_t>(q);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> g(mu);
  streams.erase(reinterpret_cast<Stream*>(s));
  delete reinterpret_cast<Stream*>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> g(mu);
  wait(s);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(new hipStream_t());
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<hipStream_t*>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  *reinterpret_cast<hipStream_t*>(e) = s;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}

// ------------------------------------------------------------------ devices
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char symbol[1 << 16];
  *p = symbol;
  return hipSuccess;
}

// ------------------------------------------------------------------ kernels
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
  configs.push_back(Config{grid, block, shmem, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
  const Config c = configs.back();
  configs.pop_back();
  *grid = c.grid;
  *block = c.block;
  *shmem = c.shmem;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
  std::lock_guard<std::mutex> g(mu);
  work(s);
  launches[names[f]] += 1;
  launch(names[f], grid, args);
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(1);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  opt[kClockNs] += 1000000;  // the only call that takes time: a millisecond
  *e = reinterpret_cast<hipGraphExec_t>(1);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  std::lock_guard<std::mutex> g(mu);
  work(s);
  compact();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
