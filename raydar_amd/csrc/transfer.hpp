// Copies between a caller's ordinary host memory and the device, through
// pinned buffers that an engine keeps.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

namespace rdh {

// One stream's copies.  The runtime's own path for ordinary memory stages and
// waits per copy: 110 us for 256 KB from the device and 80 us for each MB of a
// larger image, where pinned memory takes 13 us and 20 us per MB and one thread
// copies on at 34 to 65 us per MB.  So the device writes a ring of pinned slots
// while up to four threads copy out of it, and uploads are gathered in pinned
// memory and not waited for.  Whole calls: 4K image of 8 spp 8.0 -> 6.9 ms, a
// progressive 1080p sample with its image 0.83 -> 0.60 ms, 256x256 of 16 spp
// 0.28 -> 0.25 ms, 16 scenes batched 7.5 -> 6.4 ms.  For one host thread at a
// time, as the engine that owns it.
class HostTransfer {
 public:
  struct Piece {  // `bytes` from `src` to `offset` bytes behind an upload's start
    const void *src;
    uint64_t offset, bytes;
  };
  struct Read {
    void *dst;  // host
    const void *src;
    uint64_t bytes;
  };

  ~HostTransfer() { release(); }

  // No copy of this object's may be in flight.
  void release() {
    if (up_) (void)hipHostFree(up_);
    if (ring_) (void)hipHostFree(ring_);
    for (hipEvent_t e : events_) (void)hipEventDestroy(e);
    up_ = ring_ = nullptr;
    up_cap_ = up_used_ = 0;
    events_.clear();
  }

  // Allocates the buffers of ordinary uploads and reads, which the first ones
  // do otherwise.
  hipError_t reserve() {
    while (events_.size() < kSlots) {
      hipEvent_t ev;
      const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (e != hipSuccess) return e;
      events_.push_back(ev);
    }
    if (!ring_) {
      const hipError_t e = hipHostMalloc((void **)&ring_, kSlots * kSlot, hipHostMallocDefault);
      if (e != hipSuccess) return e;
    }
    return up_ ? hipSuccess : grow_upload(kMinUpload);
  }

  // Copies the pieces to dst.. in stream order; their sources may change or go
  // once this returns.  The gaps between the pieces hold anything afterwards.
  hipError_t upload(void *dst, const Piece *pieces, int n, hipStream_t stream) {
    uint64_t total = 0;
    for (int k = 0; k < n; ++k)
      if (pieces[k].bytes) total = std::max(total, pieces[k].offset + pieces[k].bytes);
    if (total == 0) return hipSuccess;
    if (total > kMaxUpload) {
      for (int k = 0; k < n; ++k) {
        if (!pieces[k].bytes) continue;
        const hipError_t e = hipMemcpyAsync(static_cast<unsigned char *>(dst) + pieces[k].offset, pieces[k].src,
                                            pieces[k].bytes, hipMemcpyHostToDevice, stream);
        if (e != hipSuccess) return e;
      }
      return hipStreamSynchronize(stream);
    }
    const uint64_t room = (total + 255) & ~255ull;
    if (up_used_ + room > up_cap_) {
      // the earlier uploads have left the buffer
      hipError_t e = up_ ? hipStreamSynchronize(stream) : hipSuccess;
      if (e != hipSuccess) return e;
      up_used_ = 0;
      if (room > up_cap_ && (e = grow_upload(2 * room)) != hipSuccess) return e;
    }
    unsigned char *p = up_ + up_used_;
    for (int k = 0; k < n; ++k)
      if (pieces[k].bytes) std::memcpy(p + pieces[k].offset, pieces[k].src, pieces[k].bytes);
    up_used_ += room;
    return hipMemcpyAsync(dst, p, total, hipMemcpyHostToDevice, stream);
  }
  hipError_t upload(void *dst, const void *src, uint64_t bytes, hipStream_t stream) {
    const Piece p{src, 0, bytes};
    return upload(dst, &p, 1, stream);
  }
  // The same within the memory that reserve() allocated, whatever the size:
  // through the ring, which the reads behind it in the stream may use, with a
  // wait only where the upload fills it.
  hipError_t upload_reserved(void *dst, const Piece *pieces, int n, hipStream_t stream) {
    uint64_t total = 0;
    for (int k = 0; k < n; ++k)
      if (pieces[k].bytes) total = std::max(total, pieces[k].offset + pieces[k].bytes);
    for (uint64_t at = 0; at < total; at += kSlots * kSlot) {
      const uint64_t end = std::min<uint64_t>(total, at + kSlots * kSlot);
      hipError_t e = hipStreamSynchronize(stream);  // the ring's earlier contents have left it
      if (e != hipSuccess) return e;
      for (int k = 0; k < n; ++k) {
        const uint64_t lo = std::max(at, pieces[k].offset), hi = std::min(end, pieces[k].offset + pieces[k].bytes);
        if (lo < hi)
          std::memcpy(ring_ + (lo - at), static_cast<const unsigned char *>(pieces[k].src) + (lo - pieces[k].offset),
                      hi - lo);
      }
      e = hipMemcpyAsync(static_cast<unsigned char *>(dst) + at, ring_, end - at, hipMemcpyHostToDevice, stream);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }

  // Pinned memory of kDirect bytes for the device to write by itself: valid
  // until the next read.
  static constexpr uint64_t kDirect = 1u << 20;
  hipError_t direct(unsigned char **p) {
    const hipError_t e = reserve();
    *p = ring_;
    return e;
  }

  // Waits for the stream's work so far and copies the reads' bytes to the host.
  // `queued`, if there is one, is called once the first copies are queued.
  hipError_t read(const Read *reads, int n, hipStream_t stream, int device,
                  const std::function<hipError_t()> &queued = nullptr) {
    std::vector<Read> chunks;
    uint64_t total = 0;
    for (int k = 0; k < n; ++k) {
      total += reads[k].bytes;
      for (uint64_t at = 0; at < reads[k].bytes; at += kSlot)
        chunks.push_back({static_cast<unsigned char *>(reads[k].dst) + at,
                          static_cast<const unsigned char *>(reads[k].src) + at,
                          std::min<uint64_t>(kSlot, reads[k].bytes - at)});
    }
    const size_t count = chunks.size();
    if (count == 0) return hipStreamSynchronize(stream);
    hipError_t e = reserve();
    if (e != hipSuccess) return e;
    const size_t slots = std::min<size_t>(count, kSlots);
    if (count <= slots && total < kThreaded) {
      for (size_t i = 0; i < count && e == hipSuccess; ++i)
        e = hipMemcpyAsync(ring_ + i * kSlot, chunks[i].src, chunks[i].bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess && queued) e = queued();
      const hipError_t s = hipStreamSynchronize(stream);
      if (e != hipSuccess || s != hipSuccess) return e != hipSuccess ? e : s;
      for (size_t i = 0; i < count; ++i) std::memcpy(chunks[i].dst, ring_ + i * kSlot, chunks[i].bytes);
      return hipSuccess;
    }
    // Chunk i goes through slot i % slots, in parts that the threads take one
    // after another; who copies out its last part queues the slot's next chunk.
    // issued[slot] counts the chunks queued for it, each followed by the slot's
    // event, left[slot] the parts of its chunk still to copy.
    std::vector<uint32_t> first_part(count + 1, 0);
    for (size_t i = 0; i < count; ++i)
      first_part[i + 1] = first_part[i] + (uint32_t)((chunks[i].bytes + kPart - 1) / kPart);
    std::atomic<uint32_t> issued[kSlots], left[kSlots], next{0};
    for (size_t s = 0; s < kSlots; ++s) {
      issued[s].store(0, std::memory_order_relaxed);
      left[s].store(0, std::memory_order_relaxed);
    }
    std::atomic<int> failed{hipSuccess};
    auto issue = [&](size_t i) {
      const size_t s = i % slots;
      left[s].store(first_part[i + 1] - first_part[i], std::memory_order_relaxed);
      hipError_t r = hipMemcpyAsync(ring_ + s * kSlot, chunks[i].src, chunks[i].bytes,
                                    hipMemcpyDeviceToHost, stream);
      if (r == hipSuccess) r = hipEventRecord(events_[s], stream);
      if (r != hipSuccess) failed.store(r);
      issued[s].fetch_add(1, std::memory_order_release);
    };
    auto work = [&] {
      size_t i = 0, waited = count;  // the part's chunk, the last one waited for
      for (uint32_t part; failed.load() == hipSuccess && (part = next.fetch_add(1)) < first_part[count];) {
        while (part >= first_part[i + 1]) ++i;
        const size_t s = i % slots;
        if (waited != i) {
          while (issued[s].load(std::memory_order_acquire) <= i / slots) {
            if (failed.load() != hipSuccess) return;
            std::this_thread::yield();
          }
          const hipError_t r = hipEventSynchronize(events_[s]);
          if (r != hipSuccess) {
            failed.store(r);
            return;
          }
          waited = i;
        }
        const uint64_t at = (part - first_part[i]) * kPart;
        std::memcpy(static_cast<unsigned char *>(chunks[i].dst) + at, ring_ + s * kSlot + at,
                    std::min<uint64_t>(kPart, chunks[i].bytes - at));
        if (left[s].fetch_sub(1, std::memory_order_acq_rel) == 1 && i + slots < count) issue(i + slots);
      }
    };
    for (size_t i = 0; i < slots; ++i) issue(i);
    if (queued && (e = queued()) != hipSuccess) failed.store(e);
    std::vector<std::thread> helpers;
    try {
      helpers.reserve(kHelpers);
      for (uint64_t k = 0; k < std::min<uint64_t>(kHelpers, total / kThreaded); ++k)
        helpers.emplace_back([&] {
          if (hipSetDevice(device) == hipSuccess) work();
        });
    } catch (...) {  // no thread or no memory for one: fewer threads then
    }
    work();
    for (std::thread &t : helpers) t.join();
    // nothing is queued for the ring any more
    e = hipStreamSynchronize(stream);
    return failed.load() != hipSuccess ? (hipError_t)failed.load() : e;
  }
  hipError_t read(void *dst, const void *src, uint64_t bytes, hipStream_t stream, int device) {
    const Read r{dst, src, bytes};
    return read(&r, 1, stream, device);
  }

 private:
  static constexpr uint64_t kMinUpload = 256u << 10, kMaxUpload = 4u << 20;
  static constexpr uint64_t kSlot = 2u << 20;      // a copy of the ring
  static constexpr uint64_t kPart = 256u << 10;    // what a thread takes of it
  static constexpr uint64_t kThreaded = kDirect;  // reads of one thread, and bytes per further one
  static constexpr size_t kSlots = 4, kHelpers = 3;

  hipError_t grow_upload(uint64_t bytes) {
    uint64_t cap = kMinUpload;
    while (cap < bytes) cap *= 2;
    if (up_) (void)hipHostFree(up_);
    up_ = nullptr;
    up_cap_ = 0;
    const hipError_t e = hipHostMalloc((void **)&up_, cap, hipHostMallocDefault);
    if (e == hipSuccess) up_cap_ = cap;
    return e;
  }

  unsigned char *up_ = nullptr;  // pinned; [0, up_used_) may be in flight
  uint64_t up_cap_ = 0, up_used_ = 0;
  unsigned char *ring_ = nullptr;  // kSlots pinned slots of kSlot bytes
  std::vector<hipEvent_t> events_;
};

}  // namespace rdh
