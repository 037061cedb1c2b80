// Staged transfers (mithra_amd/csrc/gpu/stage.h) on a runtime of the host's own that refuses memory on demand
// and, as HIP does, keeps a refusal as the last error until it is asked for.  Each line printed: what ran, status,
// whether the items came through, calls of `put`, bytes held pinned, bytes held on the device.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "hip/hip_runtime.h"

size_t pinned_most = ~(size_t)0, device_most = ~(size_t)0;  // refused above
hipError_t last = hipSuccess;
struct Memory {
  std::map<void*, size_t> held;
  hipError_t grant(void** p, size_t n, size_t most) {
    if (n > most) return last = hipErrorOutOfMemory;
    held[*p = std::malloc(n)] = n;
    return hipSuccess;
  }
  hipError_t give_back(void* p) {
    held.erase(p);
    std::free(p);
    return hipSuccess;
  }
  size_t bytes() const {
    size_t sum = 0;
    for (auto& a : held) sum += a.second;
    return sum;
  }
} pinned, device;
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return pinned.grant(p, n, pinned_most); }
hipError_t hipHostFree(void* p) { return pinned.give_back(p); }
hipError_t hipMalloc(void** p, size_t n) { return device.grant(p, n, device_most); }
hipError_t hipFree(void* p) { return device.give_back(p); }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = 1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

#include "stage.h"

static void transfer(const char* name, mithra::HostStage* h, long n, size_t fail_at = ~(size_t)0,
                     long most = 1l << 62) {
  struct Item { long in; double out[10]; };  // 88 bytes, as a particle's record
  std::vector<Item> got(n);
  size_t puts = 0;
  auto put = [&](long first, long m, char* slot) {
    if (puts++ == fail_at) return hipErrorUnknown;
    Item* it = (Item*)slot;
    for (long i = 0; i < m; ++i) {
      it[i].in = first + i;
      for (double& v : it[i].out) v = 3.0 * (double)(first + i);
    }
    return hipGetLastError();  // as after a launch
  };
  auto take = [&](long first, long m, const char* slot) { std::memcpy(got.data() + first, slot, sizeof(Item) * m); };
  const int rc = mithra::stage_chunks(h, 0, n, sizeof(Item), put, take, most);
  bool good = true;
  for (long i = 0; i < n; ++i) good = good && got[i].in == i && got[i].out[9] == 3.0 * (double)i;
  std::printf("%s %ld %d %d %zu %zu %zu\n", name, n, rc, (int)good, puts, pinned.bytes(), device.bytes());
}

int main() {
  for (long n : {0L, 1L, 744L, 745L, 5957L, 5958L, 100001L}) {
    mithra::HostStage h = {};
    transfer("first", &h, n);
    transfer("pinned", &h, n);
    transfer("failing", &h, n, 0);
    mithra::stage_free(&h);
    transfer("three", &h, n, ~(size_t)0, 3);
    mithra::stage_free(&h);
    pinned_most = 0;
    transfer("three", &h, n, ~(size_t)0, 3);
    mithra::stage_free(&h);
    transfer("refused", &h, n);
    transfer("refused", &h, n);
    pinned_most = ~(size_t)0;
    transfer("granted", &h, n);
    mithra::stage_free(&h);
    pinned_most = 0;
    device_most = 50000;
    transfer("little", &h, n);
    transfer("little", &h, n);
    mithra::stage_free(&h);
    device_most = 0;
    pinned_most = ~(size_t)0;
    transfer("full", &h, n);
    mithra::stage_free(&h);
    pinned_most = 0;
    transfer("none", &h, n);
    mithra::stage_free(&h);
    device_most = pinned_most = ~(size_t)0;
    std::printf("left %ld 0 0 0 %zu %zu\n", n, pinned.bytes(), device.bytes());
  }
}
