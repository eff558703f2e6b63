// Copies of large results from the device into a caller's (pageable) host
// array by several threads.  Host code only.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace amdk {

// The runtime's copy out of the device is one thread's (15-18 GB/s, first
// touch of the caller's pages included), so workers take 2 MiB chunks through
// two pinned slots each, one moved to the caller's array while the DMA fills
// the other: 64 H2O bands (320 MB) into new memory 31.5 -> 10.7 ms, 32 H2O
// (65 MB) 6.0 -> 2.1 ms.
//
// Beside the spinning threads of a caller's parallel region a worker may lose its
// CPU in the middle of a chunk, and the copy waits for it, some milliseconds, whatever
// its size: the fewer workers, the rarer.  So there are only as many as have COPY_SHARE each, which
// is two at COPY_MIN, and they sleep for the DMA instead of spinning.  34 MB into
// touched memory, alone / beside such threads: plain copy 2.3-2.5 / 2.3 ms, eight
// spinning workers 1.0 / 3.5-4.0, two sleeping ones 1.0 / 1.4-1.9; 66 MB 4.4 / 4.5,
// 1.8 / 2.7-3.8, five 1.8 / 2.4-3.1.  Only where the threads of two such regions
// outnumber the CPUs is the plain copy faster, up to 50 MB (34 MB 2.4 against 4.1 ms; eight
// workers 8.1).  Below COPY_MIN the plain copy stays: there is at most a millisecond to
// save.
constexpr size_t COPY_SLOT = 2u << 20, COPY_MIN = 32u << 20, COPY_SHARE = 12u << 20;
constexpr int COPY_WORKERS = 8;
static_assert(COPY_MIN / COPY_SHARE >= 2 && COPY_SHARE >= 2 * COPY_SLOT, "work for two, and two slots each");

// Pinned slots (two per worker) of one context, made at the first copy that
// uses them.  Without them (no pinned memory left, one CPU) the plain copy does
// the same, so this is never an error and is tried once.
struct CopySlots {
  char* mem = nullptr;
  std::vector<hipEvent_t> ev;
  int workers = 0;
  bool tried = false;

  bool ready() noexcept {
    if (!tried) {
      tried = true;
      const int n = std::min(COPY_WORKERS, (int)std::thread::hardware_concurrency() / 2);
      if (n >= 2 && !make(n)) {
        release();
        (void)hipGetLastError();  // not for the next launch check to find
      }
    }
    return workers >= 2;
  }
  bool make(int n) noexcept {
    try {
      ev.assign(2 * n, nullptr);
    } catch (const std::exception&) {
      return false;
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * COPY_SLOT * n, hipHostMallocDefault) != hipSuccess) return false;
    mem = (char*)p;
    for (hipEvent_t& e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventBlockingSync) != hipSuccess) {
        e = nullptr;
        return false;
      }
    workers = n;
    return true;
  }
  void release() noexcept {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    ev.clear();
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    workers = 0;
  }
};

// `rows` rows of row_bytes, packed on the device, `pitch` bytes apart in the
// host array.  The workers live for the call; the calling thread is one of them
// and does all the work if no other can be started.  Returns with the data in
// the caller's array and no slot in use, or with the first error.
inline hipError_t copy_out(CopySlots& slots, int device, hipStream_t stream, const void* dev, void* host, size_t rows,
                           size_t row_bytes, size_t pitch) noexcept {
  const size_t total = rows * row_bytes;
  if (total < COPY_MIN || !slots.ready()) {
    const hipError_t e = hipMemcpy2DAsync(host, pitch, dev, row_bytes, row_bytes, rows, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }
  if (pitch == row_bytes) {  // one run
    row_bytes = total;
    rows = 1;
  }
  const size_t per_row = (row_bytes + COPY_SLOT - 1) / COPY_SLOT, nchunk = rows * per_row;
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  const int nw = (int)std::min<size_t>(slots.workers, total / COPY_SHARE);  // 2 at least
  struct Piece { char* h; const char* d; size_t n; };
  auto work = [&](int w) noexcept {
    auto ok = [&](hipError_t e) {
      int none = (int)hipSuccess;
      if (e != hipSuccess) err.compare_exchange_strong(none, (int)e);
      return e == hipSuccess;
    };
    if (w > 0 && !ok(hipSetDevice(device))) return;  // the calling thread keeps its own
    char* slot[2] = {slots.mem + 2 * COPY_SLOT * w, slots.mem + 2 * COPY_SLOT * w + COPY_SLOT};
    const hipEvent_t ev[2] = {slots.ev[2 * w], slots.ev[2 * w + 1]};
    auto fetch = [&](Piece& p, int s) {  // the next chunk into slot s; false: none left, or an error
      if (err != (int)hipSuccess) return false;
      const size_t k = next++;
      if (k >= nchunk) return false;
      const size_t r = k / per_row, o = (k % per_row) * COPY_SLOT;
      p = {(char*)host + r * pitch + o, (const char*)dev + r * row_bytes + o, std::min(COPY_SLOT, row_bytes - o)};
      return ok(hipMemcpyAsync(slot[s], p.d, p.n, hipMemcpyDeviceToHost, stream)) && ok(hipEventRecord(ev[s], stream));
    };
    Piece p[2];
    bool have = fetch(p[0], 0);
    for (int i = 0; have; ++i) {
      const int s = i & 1;
      have = fetch(p[s ^ 1], s ^ 1);
      if (!ok(hipEventSynchronize(ev[s]))) return;
      std::memcpy(p[s].h, slot[s], p[s].n);
    }
  };
  {
    struct Team {
      std::vector<std::thread> t;
      ~Team() {
        for (auto& x : t) x.join();
      }
    } team;
    try {
      team.t.reserve(nw - 1);
      for (int w = 1; w < nw; ++w) team.t.emplace_back(work, w);
    } catch (const std::exception&) {
      // fewer workers: the ones that run take all the chunks
    }
    work(0);
  }
  const hipError_t fin = hipStreamSynchronize(stream);
  return err != (int)hipSuccess ? (hipError_t)err.load() : fin;
}

}  // namespace amdk
