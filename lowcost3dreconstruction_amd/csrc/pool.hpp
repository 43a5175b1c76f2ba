// pool.hpp -- device memory, pinned host memory and streams kept between calls.
//
// Allocating and freeing them is what a call on a few thousand points mostly
// costs: a stream takes 200-500 us to create, a pinned buffer 30-100 us, and
// every hipFree waits for the device (54 of them took 7.7 ms of a 24-capture cycle
// made from its clouds).  What a call or a handle releases is kept, by size class,
// for the next one (with the copies through pinned memory: a voxel grid of 60k
// points 1882 -> 321 us, normals of 2003 points 460 -> 195, a point-to-plane pair
// of 70k points 9.1 -> 1.3 ms, 24 captures from clouds to poses 17.4 -> 7.8 ms):
//   * bounded: at most kDeviceKeep bytes per device, kPinnedKeep bytes of pinned
//     memory and kStreamsKeep streams per device; the blocks unused for longest
//     are freed first;
//   * given back: everything by release_all (lcr_release_memory); a block unused for
//     kIdleSeconds at the next use of the pool (nothing runs between calls: after its
//     last one a process keeps what the limits allow); everything kept on a device
//     when an allocation there fails;
//   * only idle memory enters: an owner synchronises the stream that used its
//     buffers before it releases them (Stream's release does, and every handle's
//     destructor and every call's normal end come after such a wait), and buffers
//     released while an exception unwinds are freed, not kept (hipFree waits for
//     the work that may still use them).  A kept block can therefore go to any
//     thread and stream.
#pragma once
#include <hip/hip_runtime.h>

#include <stddef.h>

#include <chrono>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace lcr {

class Pool {
 public:
  static Pool& get();  // never destroyed: buffers may be released at process exit
  // bytes is rounded up to the block's size; throws Error when out of memory
  void* take_device(size_t* bytes, int* device);
  void* take_pinned(size_t* bytes);
  hipStream_t take_stream(int device);  // `device` must be current
  void give_device(void* p, size_t bytes, int device) noexcept;
  void give_pinned(void* p, size_t bytes) noexcept;
  void give_stream(hipStream_t s, int device) noexcept;  // synchronised by the caller
  void release_all();

  // Size classes: four per power of two, so a block is at most a quarter larger
  // than asked for and a slightly different cloud finds the last one's blocks; above
  // 64 MiB steps of 16 MiB, so that a large call takes little more than it asks for.
  // Where that does not fit either, a block has the size asked for.
  static size_t size_class(size_t n);

 private:
  using Clock = std::chrono::steady_clock;
  struct Block {
    void* p;
    Clock::time_point since;
  };
  // (device, class) -> blocks, the last released last; device kPinned: pinned memory
  using Key = std::pair<int, size_t>;
  static constexpr int kPinned = -1;
  // The device limit is about what a cycle of 2.5 M points takes (420 bytes a point),
  // so that cycles up to that size made from their clouds again find their blocks: of
  // 36 captures with that many, 7.7 ms from clouds to poses, about 1 ms goes to the
  // 25 blocks that do not fit.  Pinned memory: the staging of an upload of 8 M points
  // with normals.
  static constexpr size_t kDeviceKeep = (size_t)1 << 30;
  static constexpr size_t kPinnedKeep = (size_t)256 << 20;
  static constexpr size_t kStreamsKeep = 8;
  static constexpr int kIdleSeconds = 20;

  static size_t limit(int owner) { return owner == kPinned ? kPinnedKeep : kDeviceKeep; }
  void* take(const Key& k);
  void give(const Key& k, void* p) noexcept;
  // Moves to `out` what is over an owner's limit or idle for too long.
  void trim(std::vector<std::pair<int, void*>>* out) noexcept;
  static void free_block(int owner, void* p) noexcept;
  static void release(const std::vector<std::pair<int, void*>>& blocks) noexcept;
  bool flush(int owner);
  template <class F>
  void* allocate(int owner, size_t asked, size_t* bytes, const char* what, F&& alloc);

  std::mutex mu_;
  std::map<Key, std::vector<Block>> blocks_;
  std::map<int, size_t> kept_;
  Clock::time_point trimmed_{};
  std::map<int, std::vector<hipStream_t>> streams_;
};

}  // namespace lcr
