// Results that a call hands to its host thread before it returns (whether an index is well formed,
// how large a product will be).
//
// Reading them with a copy costs the copy's own launch and a wait for the stream to drain, 15 to
// 20 us together.  Here the last kernel writes them into host memory that the GPU can address,
// followed by the call's sequence number, and the host thread watches for that number: 3 to 5 us
// after the kernel's last store.  A SyncSlot is one thread's on one device while the call lasts
// (slots are kept in a list and handed out again); calls that use one end before the thread makes
// another, so a slot's device memory is never used twice at a time.
#pragma once

#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace scorch {

constexpr int kSyncWords = 16;             // 64-bit words a call can hand over
constexpr int kSyncDeviceInts = 16 + 4096; // [0]: tickets taken so far; from [16]: partial results

struct SyncSlot {
  int device;
  volatile int64_t *host;   // [0]: sequence number of the last call answered; [1 ..]: its results
  int64_t *host_on_device;
  int *scratch;             // device memory, kSyncDeviceInts ints
  int64_t sequence;
  unsigned tickets;         // taken by all calls so far (as scratch[0] counts them)
};

// Device side: thread 0 of the last workgroup hands over `n` words.
__device__ __forceinline__ void sync_publish(int64_t *__restrict__ to, int64_t sequence, const int64_t *words, int n) {
  for (int i = 0; i < n; ++i) __hip_atomic_store(to + 1 + i, words[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(to, sequence, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

class SyncCall {
 public:
  // Takes a slot for the current device; null() if there is no memory for one.
  SyncCall();
  ~SyncCall();
  SyncCall(const SyncCall &) = delete;
  SyncCall &operator=(const SyncCall &) = delete;
  bool null() const { return slot_ == nullptr; }
  int64_t *target() const { return slot_->host_on_device; }
  int64_t sequence() const { return slot_->sequence; }
  int *scratch() const { return slot_->scratch; }
  // The ticket count before this call's workgroups take theirs, of which there will be n.
  unsigned tickets_before(unsigned n) {
    const unsigned before = slot_->tickets;
    slot_->tickets += n;
    return before;
  }
  // Waits for the answer; SCORCH_HIP_OK, or an error if the stream ends without one.
  int wait(const char *fn, hipStream_t stream, int64_t *words, int n);

 private:
  SyncSlot *slot_;
};

// Whether columns handed over for the first time lie in range: what workgroups find, and the call that waits for it.
struct ColumnsSync {
  int *tickets;      // [0]: see SyncSlot; [16]: whether a column lies outside, left 0
  unsigned tickets_before;
  int64_t *to;
  int64_t sequence;
};
// One thread of each of `workgroups` workgroups, once; the last of them hands the verdict over.  Nothing but these few words is
// handed over, and a wait for each before the next orders them: a release would write the L2 back, for every workgroup, which a
// kernel that goes on does not want (the decoder's product 142 -> 180 us).
__device__ __forceinline__ void columns_checked(const ColumnsSync &sync, int bad, unsigned workgroups) {
  const auto arrived = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  if (bad) (void)__hip_atomic_fetch_or(sync.tickets + 16, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  arrived();
  const unsigned ticket = __hip_atomic_fetch_add(reinterpret_cast<unsigned *>(sync.tickets), 1u, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  if (ticket - sync.tickets_before != workgroups - 1) return;  // not the last workgroup
  const int64_t verdict = __hip_atomic_exchange(sync.tickets + 16, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(sync.to + 1, verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  arrived();
  __hip_atomic_store(sync.to, sync.sequence, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// A check whose verdict has not been read yet.
struct ColumnsPending {
  SyncCall sync;
  hipStream_t stream;
};

}  // namespace scorch
