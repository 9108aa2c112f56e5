// omhd_slot.h -- the result slots of the separate routines.
#pragma once
#include <condition_variable>
#include <mutex>
#include <vector>

#include "omhd_host.h"

namespace omhd {

// What u2v and set_dt hand back besides arrays, without an allocation, a fill
// and a copy per call (those and a second wait were 35 of the 50 us a call
// took on 202^2 cells): `out`, two words of pinned host memory that the kernel
// writes and the call reads after its one wait, and `red`, two device words
// that every call leaves zero.  CALL_SLOTS calls may be under way at once, in
// any threads; a further one waits for a slot to be given back.
//
// A call that has waited for its kernels says so (finished()).  One that ends
// before that may leave a kernel that still writes to `out`, or `red` as its
// first kernel left it: the slot then waits for the stream and clears `red`
// before it is given back, and is given up if that fails.
constexpr int CALL_SLOTS = 64;
struct CallSlot {
  unsigned long long *out = nullptr, *red = nullptr;
  int id = -1;
  CallSlot() = default;
  CallSlot(const CallSlot &) = delete;
  CallSlot &operator=(const CallSlot &) = delete;
  ~CallSlot() {
    if (id < 0) return;
    if (!clean)
      clean = hipStreamSynchronize(stream) == hipSuccess &&
              hipMemsetAsync(red, 0, 2 * sizeof *red, stream) == hipSuccess &&
              hipStreamSynchronize(stream) == hipSuccess;
    std::lock_guard<std::mutex> lock(pool().mu);
    if (clean) {
      pool().free_ids.push_back(id);  // the capacity is there: nothing is thrown
      pool().given_back.notify_one();
    } else if (--pool().usable == 0) {
      pool().given_back.notify_all();
    }
  }
  int acquire(hipStream_t s) {
    Pool &p = pool();
    std::unique_lock<std::mutex> lock(p.mu);
    if (!p.red) {
      unsigned long long *d = nullptr;
      p.free_ids.reserve(CALL_SLOTS);
      if (!p.out)
        OMHD_HIP(hipHostMalloc((void **)&p.out, 2 * CALL_SLOTS * sizeof *p.out, hipHostMallocMapped | hipHostMallocCoherent));
      OMHD_HIP(hipMallocAsync((void **)&d, 2 * CALL_SLOTS * sizeof *d, s));
      OMHD_HIP(hipMemsetAsync(d, 0, 2 * CALL_SLOTS * sizeof *d, s));
      OMHD_HIP(hipStreamSynchronize(s));
      p.red = d;
      p.usable = CALL_SLOTS;
      for (int i = 0; i < CALL_SLOTS; i++) p.free_ids.push_back(i);
    }
    p.given_back.wait(lock, [&] { return !p.free_ids.empty() || p.usable == 0; });
    if (p.free_ids.empty()) return set_error(OMHD_ERR_HIP, "every result slot was given up after a failed wait");
    id = p.free_ids.back();
    p.free_ids.pop_back();
    stream = s;
    out = p.out + 2 * id;
    red = p.red + 2 * id;
    out[0] = out[1] = 0;
    return OMHD_OK;
  }
  // the call's kernels have run (its wait succeeded), and left `red` zero
  void finished() { clean = true; }

 private:
  hipStream_t stream = nullptr;
  bool clean = false;
  struct Pool {
    std::mutex mu;
    std::condition_variable given_back;
    std::vector<int> free_ids;
    int usable = 0;
    unsigned long long *out = nullptr, *red = nullptr;
  };
  static Pool &pool() {
    static Pool *p = new Pool;  // outlives every thread that may still hold a slot
    return *p;
  }
};

}  // namespace omhd
