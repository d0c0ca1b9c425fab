// Field copies between the caller's pageable memory and the device, through pinned slots that a
// context owns (allocated on first use, freed with it).  Copies of one context from several threads
// take turns: the slots are shared.
//
// A pageable copy goes through the runtime's own path, which pins or stages the caller's pages on
// one thread: 2.6 ms down for a 26.7 MB field into fresh memory (10 GB/s), 0.17 ms for 0.3 MB.
// Down, large fields are cut into chunks that cross the bus into a ring of slots while a few
// threads copy the arrived ones out (their page faults are most of the cost): 0.93 ms, 29 GB/s;
// 206 MB 18.9 -> 5.3 ms; fields below 2 MB take one slot: 0.3 MB 0.17 -> 0.09 ms.  Up, fields below
// 2 MB are copied to a slot and the call returns while the slot crosses the bus, in stream order
// (0.3 MB 0.13 -> 0.04 ms); larger ones go the runtime's way (32 GB/s, as fast as the ring).
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

struct HostIo {
  static constexpr int kSlots = 8;                  // ring of a context with large fields
  static constexpr int kSmall = 3;                  // slots of one whose fields all fit a slot
  static constexpr size_t kChunk = size_t(2) << 20;  // largest slot, and one-slot field
  static constexpr int kThreads = 4;
  size_t field = 0;        // bytes of the context's largest field
  char* block = nullptr;   // the slots, one allocation on first use
  int slots = 0;           // 0: none yet, -1: none to be had (plain copies)
  size_t size = 0;         // bytes per slot
  hipEvent_t ev[kSlots] = {};
  bool busy[kSlots] = {};  // an upload from the slot may still be running (its event tells)
  int next = 0;            // slot of the next small upload
  std::mutex turn;

  char* buf(int s) const { return block + s * size; }

  bool ready() {
    if (slots) return slots > 0;
    slots = -1;
    const int ns = field < kChunk ? kSmall : kSlots;
    size = std::min(kChunk, (std::max(field, size_t(1)) + 0xffff) & ~size_t(0xffff));
    if (hipHostMalloc((void**)&block, ns * size, hipHostMallocDefault) != hipSuccess) {
      block = nullptr;
      (void)hipGetLastError();
      return false;
    }
    for (int s = 0; s < ns; ++s)
      if (hipEventCreateWithFlags(&ev[s], hipEventDisableTiming) != hipSuccess) {
        ev[s] = nullptr;
        (void)hipGetLastError();
        return false;
      }
    slots = ns;
    return true;
  }

  // slot s free of earlier uploads
  hipError_t idle(int s) {
    if (!busy[s]) return hipSuccess;
    busy[s] = false;
    return hipEventSynchronize(ev[s]);
  }

  void release() {
    for (int s = 0; s < kSlots; ++s) {
      (void)idle(s);
      if (ev[s]) (void)hipEventDestroy(ev[s]);
      ev[s] = nullptr;
    }
    if (block) (void)hipHostFree(block);
    block = nullptr;
    slots = 0;
  }

  // n bytes to the device in stream order; src may be reused when the call returns
  hipError_t up(void* dev, const void* src, size_t n, hipStream_t st) {
    const std::lock_guard<std::mutex> lock(turn);
    if (n < kChunk && ready() && n <= size) {
      const int s = next;
      next = (next + 1) % slots;
      hipError_t e = idle(s);
      if (e != hipSuccess) return e;
      memcpy(buf(s), src, n);
      e = hipMemcpyAsync(dev, buf(s), n, hipMemcpyHostToDevice, st);
      if (e != hipSuccess) return e;
      busy[s] = true;
      return hipEventRecord(ev[s], st);
    }
    const hipError_t e = hipMemcpyAsync(dev, src, n, hipMemcpyHostToDevice, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }

  // n bytes from the device, complete when the call returns
  hipError_t down(void* dst, const void* dev, size_t n, hipStream_t st) {
    const std::lock_guard<std::mutex> lock(turn);
    if (n < kChunk && ready() && n <= size) {
      hipError_t e = idle(0);
      if (e == hipSuccess) e = hipMemcpyAsync(buf(0), dev, n, hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e == hipSuccess) memcpy(dst, buf(0), n);
      return e;
    }
    if (n >= kChunk && ready() && slots == kSlots) {
      for (int s = 0; s < kSlots; ++s) {
        const hipError_t e = idle(s);
        if (e != hipSuccess) return e;
      }
      // the copy of a few MB is over before eight 2 MB chunks are under way
      return ring(static_cast<char*>(dst), static_cast<const char*>(dev), n,
                  n < 4 * kChunk ? kChunk / 4 : kChunk, st);
    }
    const hipError_t e = hipMemcpyAsync(dst, dev, n, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }

 private:
  // Chunk c crosses into slot c % kSlots; the threads take the chunks in order, wait for their
  // events and copy them out.  The calling thread issues the transfers and, when all are issued,
  // copies too, so the copy ends with however many threads could be started.
  hipError_t ring(char* dst, const char* dev, size_t n, size_t ch, hipStream_t st) {
    const size_t nc = (n + ch - 1) / ch;
    std::atomic<size_t> issued{0}, take{0};
    std::atomic<size_t> freed[kSlots] = {};  // chunks copied out of the slot
    std::atomic<int> err{(int)hipSuccess};
    auto copy_one = [&](size_t c) {
      const int s = (int)(c % kSlots);
      for (;;) {
        const hipError_t e = hipEventQuery(ev[s]);
        if (e == hipSuccess) break;
        if (e != hipErrorNotReady) { err = (int)e; break; }
        std::this_thread::yield();
      }
      const size_t o = c * ch;
      if (err == (int)hipSuccess) memcpy(dst + o, buf(s), std::min(ch, n - o));
      freed[s].fetch_add(1, std::memory_order_release);
    };
    // a taken chunk is always issued: the calling thread issues every chunk or, after an error,
    // counts the rest as issued
    auto work = [&]() {
      for (size_t c; (c = take.fetch_add(1)) < nc;) {
        while (issued.load(std::memory_order_acquire) <= c) std::this_thread::yield();
        copy_one(c);
      }
    };
    std::thread pool[kThreads];
    int nt = 0;
    try {
      for (; nt < kThreads; ++nt) pool[nt] = std::thread(work);
    } catch (...) {  // fewer threads
    }
    for (size_t c = 0; c < nc; ++c) {
      const int s = (int)(c % kSlots);
      while (freed[s].load(std::memory_order_acquire) < c / kSlots) {
        if (nt > 0) { std::this_thread::yield(); continue; }
        const size_t q = take.fetch_add(1);  // no thread could be started: copy here
        if (q < c) copy_one(q);
      }
      if (err == (int)hipSuccess) {
        const size_t o = c * ch;
        hipError_t e = hipMemcpyAsync(buf(s), dev + o, std::min(ch, n - o),
                                      hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev[s], st);
        if (e != hipSuccess) err = (int)e;
      }
      issued.store(c + 1, std::memory_order_release);
    }
    work();
    for (int t = 0; t < nt; ++t) pool[t].join();
    return (hipError_t)err.load();
  }
};
