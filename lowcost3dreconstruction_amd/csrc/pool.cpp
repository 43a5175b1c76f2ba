// pool.cpp -- see pool.hpp.
#include "pool.hpp"

#include <string>

#include "runtime.hpp"

namespace lcr {

Pool& Pool::get() {
  static Pool* p = new Pool();
  return *p;
}

size_t Pool::size_class(size_t n) {
  constexpr size_t kLeast = 4096;
  if (n <= kLeast) return kLeast;
  size_t top = kLeast;
  while (top <= (n - 1) / 2) top *= 2;  // top < n <= 2 top
  constexpr size_t kMostStep = (size_t)16 << 20;
  const size_t step = top / 4 < kMostStep ? top / 4 : kMostStep;
  return (n + step - 1) / step * step;
}

void* Pool::take(const Key& k) {
  std::vector<std::pair<int, void*>> old;
  void* p = nullptr;
  {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = blocks_.find(k);
    if (it != blocks_.end()) {
      p = it->second.back().p;
      it->second.pop_back();
      if (it->second.empty()) blocks_.erase(it);
      kept_[k.first] -= k.second;
    }
    trim(&old);
  }
  release(old);
  return p;
}

void Pool::give(const Key& k, void* p) noexcept {
  std::vector<std::pair<int, void*>> old;
  try {
    std::lock_guard<std::mutex> lock(mu_);
    size_t& kept = kept_[k.first];
    std::vector<Block>& v = blocks_[k];
    try {
      v.push_back(Block{p, Clock::now()});
    } catch (...) {
      if (v.empty()) blocks_.erase(k);
      throw;
    }
    kept += k.second;
    p = nullptr;
    trim(&old);
  } catch (...) {  // no memory for the bookkeeping
  }
  if (p) free_block(k.first, p);
  release(old);
}

void Pool::trim(std::vector<std::pair<int, void*>>* out) noexcept {
  const Clock::time_point now = Clock::now();
  bool over = false;
  for (const auto& o : kept_) over = over || o.second > limit(o.first);
  // a walk over every class: when over a limit, else once a second
  if (!over && now - trimmed_ < std::chrono::seconds(1)) return;
  trimmed_ = now;
  const Clock::time_point stale = now - std::chrono::seconds(kIdleSeconds);
  try {
    for (auto& o : kept_) {
      for (;;) {
        // the block of this owner unused for longest (the first of its class's vector)
        auto oldest = blocks_.end();
        for (auto it = blocks_.lower_bound(Key(o.first, 0));
             it != blocks_.end() && it->first.first == o.first; ++it)
          if (oldest == blocks_.end() || it->second.front().since < oldest->second.front().since) oldest = it;
        if (oldest == blocks_.end()) break;
        if (o.second <= limit(o.first) && oldest->second.front().since > stale) break;
        out->emplace_back(o.first, oldest->second.front().p);
        o.second -= oldest->first.second;
        oldest->second.erase(oldest->second.begin());
        if (oldest->second.empty()) blocks_.erase(oldest);
      }
    }
  } catch (...) {  // no memory for the list: later
  }
}

void Pool::free_block(int owner, void* p) noexcept {
  if (owner == kPinned)
    (void)hipHostFree(p);
  else
    (void)hipFree(p);
}

void Pool::release(const std::vector<std::pair<int, void*>>& blocks) noexcept {
  for (const auto& b : blocks) free_block(b.first, b.second);
}

void Pool::release_all() {
  std::vector<int> owners;
  std::vector<hipStream_t> streams;
  {
    std::lock_guard<std::mutex> lock(mu_);
    for (const auto& o : kept_) owners.push_back(o.first);
    for (auto& v : streams_) {
      streams.insert(streams.end(), v.second.begin(), v.second.end());
      v.second.clear();
    }
  }
  for (hipStream_t s : streams) (void)hipStreamDestroy(s);
  for (int o : owners) (void)flush(o);
}

bool Pool::flush(int owner) {
  std::vector<std::pair<int, void*>> old;
  {
    std::lock_guard<std::mutex> lock(mu_);
    for (auto it = blocks_.lower_bound(Key(owner, 0));
         it != blocks_.end() && it->first.first == owner;) {
      for (const Block& b : it->second) old.emplace_back(owner, b.p);
      it = blocks_.erase(it);
    }
    kept_[owner] = 0;
  }
  release(old);
  return !old.empty();
}

// A block that was not kept.  Without room for its class: what is kept goes first,
// then the bytes asked for have to do.
template <class F>
void* Pool::allocate(int owner, size_t asked, size_t* bytes, const char* what, F&& alloc) {
  void* p = nullptr;
  hipError_t e = alloc(&p, *bytes);
  if (e == hipErrorOutOfMemory && flush(owner)) {
    (void)hipGetLastError();
    e = alloc(&p, *bytes);
  }
  const size_t least = (asked + 255) / 256 * 256;
  if (e == hipErrorOutOfMemory && least < *bytes) {
    (void)hipGetLastError();
    *bytes = least;
    e = alloc(&p, *bytes);
  }
  if (e != hipSuccess) throw Error{-2, std::string(what) + " failed: " + hipGetErrorString(e)};
  return p;
}

void* Pool::take_device(size_t* bytes, int* device) {
  LCR_HIP(hipGetDevice(device));
  const size_t asked = *bytes;
  *bytes = size_class(asked);
  void* p = take(Key(*device, *bytes));
  if (p) return p;
  return allocate(*device, asked, bytes, "hipMalloc", [](void** q, size_t n) { return hipMalloc(q, n); });
}

void* Pool::take_pinned(size_t* bytes) {
  const size_t asked = *bytes;
  *bytes = size_class(asked);
  void* p = take(Key(kPinned, *bytes));
  if (p) return p;
  // coherent: kernels leave flags there that the host waits for
  return allocate(kPinned, asked, bytes, "hipHostMalloc", [](void** q, size_t n) {
    return hipHostMalloc(q, n, hipHostMallocMapped | hipHostMallocCoherent);
  });
}

void Pool::give_device(void* p, size_t bytes, int device) noexcept { give(Key(device, bytes), p); }

void Pool::give_pinned(void* p, size_t bytes) noexcept { give(Key(kPinned, bytes), p); }

hipStream_t Pool::take_stream(int device) {
  {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<hipStream_t>& v = streams_[device];
    if (!v.empty()) {
      hipStream_t s = v.back();
      v.pop_back();
      return s;
    }
  }
  hipStream_t s = nullptr;
  LCR_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  return s;
}

void Pool::give_stream(hipStream_t s, int device) noexcept {
  try {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<hipStream_t>& v = streams_[device];
    if (v.size() < kStreamsKeep) {
      v.push_back(s);
      return;
    }
  } catch (...) {
  }
  (void)hipStreamDestroy(s);
}

}  // namespace lcr
