// Mailboxes: one word a kernel answers a waiting host thread with (pk_mailbox_create / _wait).
//
// Where a call needs a value from the GPU before it may return -- a range check that raises, a
// scale that is handed back -- a copy to the host and a stream synchronisation cost a blit
// kernel, a signal and a wake-up after everything queued behind the producer as well (measured
// on MI355X: about 25 us of a call). Here the kernel's last workgroup stores the word, with the
// call's sequence number, into pinned host memory that the host polls: the call waits for that
// kernel only, and what was launched behind it runs on meanwhile.
#include "pk_internal.h"

#include <time.h>

using namespace pk;

static_assert(kPostCounterBytes == PK_POST_COUNTER_BYTES, "header");

extern "C" void* pk_mailbox_create(void) {
  void* box = nullptr;
  const hipError_t e = hipHostMalloc(&box, 64, hipHostMallocCoherent | hipHostMallocMapped | hipHostMallocPortable);
  if (e != hipSuccess) {
    hip_status(e, "pk_mailbox_create: hipHostMalloc");
    return nullptr;
  }
  __atomic_store_n(static_cast<uint64_t*>(box), 0, __ATOMIC_RELEASE);
  return box;
}

extern "C" void pk_mailbox_destroy(void* box) {
  if (box != nullptr && hipHostFree(box) != hipSuccess) (void)hipGetLastError();
}

extern "C" int pk_mailbox_wait(const void* box, uint32_t seq, uint32_t* value, void* stream) {
  PK_REQUIRE(box != nullptr && value != nullptr, "pk_mailbox_wait: null pointer");
  const uint64_t* word = static_cast<const uint64_t*>(box);
  auto arrived = [&]() {
    const uint64_t v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
    if ((uint32_t)(v >> 32) != seq) return false;
    *value = (uint32_t)v;
    return true;
  };
  // Poll for as long as a short queue takes; behind a longer one (or where a device's stores
  // are not seen before its kernel ends) the stream's own wait does not burn the core.
  constexpr int64_t kPollNs = 300 * 1000;
  timespec t0, t;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  for (;;) {
    for (int i = 0; i < 64; ++i) {
      if (arrived()) return PK_OK;
      __builtin_ia32_pause();
    }
    clock_gettime(CLOCK_MONOTONIC, &t);
    if ((t.tv_sec - t0.tv_sec) * 1000000000ll + (t.tv_nsec - t0.tv_nsec) > kPollNs) break;
  }
  const hipError_t e = hipStreamSynchronize((hipStream_t)stream);
  if (e != hipSuccess) return hip_status(e, "pk_mailbox_wait: hipStreamSynchronize");
  if (arrived()) return PK_OK;
  set_error("pk_mailbox_wait: the stream is done and message %u has not come", seq);
  return PK_EHIP;
}
