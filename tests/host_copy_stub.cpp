// host_copy.h on the CPU: the HIP runtime calls it makes, done at once on host
// memory, each of which can be told to fail.
#include "../amdkiit_amd/csrc/host_copy.h"

#include <cstdio>
#include <cstdlib>

static std::atomic<int> n_alloc{0}, n_event{0}, n_live{0}, n_async{0}, n_plain{0}, n_sync{0};
static int fail_alloc, fail_event, fail_async;  // the call (from 1) that fails, 0: none
static std::atomic<int> last{(int)hipSuccess};
static thread_local int current = 3;  // the thread's device
static const std::thread::id caller = std::this_thread::get_id();
static std::atomic<int> n_other{0};   // copies by threads whose device is neither the context's (0) nor the caller's

static hipError_t told(bool fail, hipError_t e) {
  if (fail) last = (int)e;
  return fail ? e : hipSuccess;
}
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (++n_alloc == fail_alloc) return told(true, hipErrorOutOfMemory);
  *p = std::malloc(n);
  ++n_live;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  --n_live;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (++n_event == fail_event) return told(true, hipErrorOutOfMemory);
  *e = (hipEvent_t)std::malloc(1);
  ++n_live;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void*)e);
  --n_live;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipSetDevice(int d) {
  current = d;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  ++n_sync;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  n_other += current != 0 && std::this_thread::get_id() != caller;
  if (++n_async == fail_async) return told(true, hipErrorInvalidValue);
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  ++n_plain;
  for (size_t i = 0; i < h; ++i) std::memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return (hipError_t)last.exchange((int)hipSuccess); }
}

// stub rows row_bytes pitch calls fail_alloc fail_event fail_async: prints the
// return code of each call, whether the arrays agree, and what was called
int main(int, char** a) {
  const size_t rows = std::atoll(a[1]), rb = std::atoll(a[2]), pitch = std::atoll(a[3]);
  const int calls = std::atoi(a[4]);
  fail_alloc = std::atoi(a[5]);
  fail_event = std::atoi(a[6]);
  fail_async = std::atoi(a[7]);
  std::vector<unsigned char> dev(rows * rb), host(rows * pitch);
  amdk::CopySlots slots;
  for (int k = 0; k < calls; ++k) {
    for (size_t i = 0; i < dev.size(); ++i) dev[i] = (unsigned char)((i * 2654435761u + k) >> 13);
    std::fill(host.begin(), host.end(), 0x5a);
    const hipError_t e = amdk::copy_out(slots, 0, nullptr, dev.data(), host.data(), rows, rb, pitch);
    bool same = true, pad = true;
    for (size_t r = 0; r < rows; ++r) {
      same &= std::memcmp(&host[r * pitch], &dev[r * rb], rb) == 0;
      for (size_t i = rb; i < pitch; ++i) pad &= host[r * pitch + i] == 0x5a;
    }
    std::printf("%d %d %d\n", (int)e, same, pad);
  }
  const int workers = slots.workers;
  slots.release();
  std::printf("%d %d %d %d %d %d %d %d %d\n", n_alloc.load(), n_async.load(), n_plain.load(), n_sync.load(), workers,
              n_live.load(), (int)hipGetLastError(), current, n_other.load());
}
