// The result slots of the separate routines (openmhd_amd/csrc/omhd_slot.h) over
// a stand-in for the HIP calls they make: device work queued on the one stream
// runs when that stream is waited for, and a wait can be told to fail.
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <functional>
#include <memory>
#include <thread>
#include <vector>

#include "../../openmhd_amd/csrc/omhd_slot.h"

namespace {
std::mutex mu;
std::vector<std::function<void()>> queue;
int failing_waits = 0;

void launch(std::function<void()> f) {
  std::lock_guard<std::mutex> lock(mu);
  queue.push_back(std::move(f));
}
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) {
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
  launch([=] { memset(p, v, n); });
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> lock(mu);
  if (failing_waits > 0) {
    failing_waits--;
    return hipErrorUnknown;
  }
  for (auto &f : queue) f();
  queue.clear();
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
}

namespace omhd {
omhd_error_info &tls_error() {
  static thread_local omhd_error_info e{};
  return e;
}
}  // namespace omhd

using omhd::CallSlot;
using omhd::CALL_SLOTS;

// a call that queues a kernel and ends on an error before its wait
static void broken_call() {
  CallSlot s;
  if (s.acquire(nullptr)) return;
  unsigned long long *red = s.red, *out = s.out;
  launch([=] {
    red[0] = 7;
    out[1] = 1;
  });
}

extern "C" {
// Takes every slot that can be taken (CALL_SLOTS + 1 at most, without waiting
// for more than `expect`) and runs what is still queued; the number taken, or
// -1 if one of them holds anything but zeros then.
int slotc_take_all(int expect) {
  std::vector<std::unique_ptr<CallSlot>> held;
  for (int i = 0; i < expect; i++) {
    held.emplace_back(new CallSlot);
    if (held.back()->acquire(nullptr)) {
      held.pop_back();
      break;
    }
  }
  (void)hipStreamSynchronize(nullptr);
  int n = (int)held.size();
  for (auto &s : held) {
    if (s->out[0] || s->out[1] || s->red[0] || s->red[1]) n = -1;
    s->finished();
  }
  return n;
}
// `n` broken calls one after the other, the next `waits` waits failing
void slotc_break(int n, int waits) {
  {
    CallSlot first;  // the pool is there
    (void)first.acquire(nullptr);
    first.finished();
  }
  failing_waits = waits;
  for (int i = 0; i < n; i++) broken_call();
  failing_waits = 0;
}
// More threads than slots, half of their calls broken: whether every unbroken
// one found its slot clear and got its own result back.
int slotc_threads(int threads, int calls) {
  std::atomic<int> bad{0};
  std::vector<std::thread> t;
  for (int k = 0; k < threads; k++)
    t.emplace_back([&, k] {
      for (int i = 0; i < calls; i++) {
        if ((i + k) % 2) {
          broken_call();
          continue;
        }
        CallSlot s;
        if (s.acquire(nullptr)) {
          bad++;
          continue;
        }
        unsigned long long *red = s.red, *out = s.out, mine = (unsigned long long)(k * calls + i + 1);
        launch([=] {
          red[0] += mine;
          out[0] = red[0];
          red[0] = 0;
        });
        (void)hipStreamSynchronize(nullptr);
        s.finished();
        if (s.out[0] != mine || s.out[1]) bad++;
      }
    });
  for (auto &x : t) x.join();
  return bad;
}
int slotc_acquire() {  // the error code of one more call
  CallSlot s;
  const int rc = s.acquire(nullptr);
  s.finished();
  return rc;
}
}
