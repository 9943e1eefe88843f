// The slots of sync.hpp.
#include "sync.hpp"

#include <immintrin.h>

#include <atomic>

namespace scorch {
namespace {
std::mutex g_mutex;
std::vector<SyncSlot *> g_free;  // as many as threads have waited at the same time
}  // namespace

__global__ void sync_clear_kernel(int *scratch) {
  for (int i = threadIdx.x; i < kSyncDeviceInts; i += kBlockThreads) scratch[i] = 0;
}

SyncCall::SyncCall() : slot_(nullptr) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return;
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    for (size_t i = 0; i < g_free.size(); ++i)
      if (g_free[i]->device == device) {
        slot_ = g_free[i];
        g_free.erase(g_free.begin() + i);
        break;
      }
  }
  if (!slot_) {
    SyncSlot s = {};
    s.device = device;
    void *host = nullptr, *mapped = nullptr, *scratch = nullptr;
    if (hipHostMalloc(&host, (kSyncWords + 1) * sizeof(int64_t), hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) return;
    std::memset(host, 0, (kSyncWords + 1) * sizeof(int64_t));
    if (hipHostGetDevicePointer(&mapped, host, 0) != hipSuccess || hipMalloc(&scratch, kSyncDeviceInts * sizeof(int)) != hipSuccess) {
      (void)hipHostFree(host);
      return;
    }
    s.host = static_cast<volatile int64_t *>(host);
    s.host_on_device = static_cast<int64_t *>(mapped);
    s.scratch = static_cast<int *>(scratch);
    sync_clear_kernel<<<1, kBlockThreads, 0, nullptr>>>(s.scratch);
    if (hipStreamSynchronize(nullptr) != hipSuccess) {
      (void)hipHostFree(host);
      (void)hipFree(scratch);
      return;
    }
    slot_ = new SyncSlot(s);
  }
  ++slot_->sequence;
}

SyncCall::~SyncCall() {
  if (!slot_) return;
  std::lock_guard<std::mutex> lock(g_mutex);
  g_free.push_back(slot_);
}

int SyncCall::wait(const char *fn, hipStream_t stream, int64_t *words, int n) {
  using clock = std::chrono::steady_clock;
  const auto begin = clock::now();
  bool answered = false;
  for (int spins = 0; !(answered = slot_->host[0] == slot_->sequence); ++spins) {
    _mm_pause();
    // a long queue in front of the call: stop burning the core and let the runtime wait
    if ((spins & 1023) == 1023 && clock::now() - begin > std::chrono::milliseconds(2)) break;
  }
  if (!answered) {
    const hipError_t err = hipStreamSynchronize(stream);
    if (err != hipSuccess || slot_->host[0] != slot_->sequence) {
      slot_ = nullptr;  // its state is unknown: not handed out again
      return fail(SCORCH_HIP_ERUNTIME, "%s: no answer from the device (%s)", fn, hipGetErrorString(err));
    }
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  for (int i = 0; i < n; ++i) words[i] = slot_->host[1 + i];
  return SCORCH_HIP_OK;
}

}  // namespace scorch

SCORCH_DEFINE_PRELOAD(sync)
