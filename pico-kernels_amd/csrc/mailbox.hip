// Mailboxes: one word a kernel answers a waiting host thread with (pk_mailbox_create / _wait).
//
// Where a call needs a value from the GPU before it may return -- a range check that raises, a
// scale that is handed back -- a copy to the host and a stream synchronisation cost a blit
// kernel, a signal and a wake-up after everything queued behind the producer as well (measured
// on MI355X: about 25 us of a call). Here the kernel's last workgroup stores the word, with the
// call's sequence number, into pinned host memory that the host polls: the call waits for that
// kernel only, and what was launched behind it runs on meanwhile.
#include "pk_internal.h"

#include <sched.h>
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
  // Poll, for as long as a short queue takes without pause, behind a longer one with the core
  // given up between polls: the stream's own wait would take in what was launched behind the
  // post as well. A sleep lasts about 0.1 ms (the timer's slack), a small part of the wait by
  // then. The stream is asked now and then, so that an error, or a message that never comes,
  // ends the wait.
  constexpr int64_t kSpinNs = 300 * 1000, kYieldNs = 3000 * 1000;
  const timespec nap = {0, 50 * 1000};
  timespec t0, t;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  for (unsigned turn = 1;; ++turn) {
    for (int i = 0; i < 64; ++i) {
      if (arrived()) return PK_OK;
      __builtin_ia32_pause();
    }
    clock_gettime(CLOCK_MONOTONIC, &t);
    const int64_t waited = (t.tv_sec - t0.tv_sec) * 1000000000ll + (t.tv_nsec - t0.tv_nsec);
    if (waited <= kSpinNs) continue;
    if (waited <= kYieldNs) sched_yield();
    else nanosleep(&nap, nullptr);
    if (turn % 16 != 0) continue;
    const hipError_t e = hipStreamQuery((hipStream_t)stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();  // no error: the next launch must not find it
      continue;
    }
    if (e != hipSuccess) return hip_status(e, "pk_mailbox_wait: hipStreamQuery");
    if (arrived()) return PK_OK;
    set_error("pk_mailbox_wait: the stream is done and message %u has not come", seq);
    return PK_EHIP;
  }
}
