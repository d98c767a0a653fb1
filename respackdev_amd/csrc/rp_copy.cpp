// Large copies between device memory and the caller's (pageable) host arrays.
//
// hipMemcpy on pageable memory stages through one host thread: 10 GB/s into a
// fresh array (whose pages are first touched by the copy), 30 GB/s out of a
// warm one, where the link carries 57 GB/s.  Here the array is dealt in chunks
// to a few threads, each with two pinned chunks of the handle: one is on the
// link while the other is copied on the host.  440 MB of eps^-1 of six q points
// leave in about 21 ms instead of 42; 108 MB in and 108 MB out with the Dyson
// step between 8.9 ms instead of 17.1.  Four threads of 2 MiB chunks: eight or
// twelve of 1 MiB are 1.5 ms slower on the latter (a chunk costs 20 us of runtime
// calls under its locks), 512 KiB 4.6 ms; 4 MiB gain nothing and pin more.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <string>
#include <thread>
#include <vector>

#include "rp_internal.h"

namespace rp {

namespace {

constexpr size_t kChunkBytes = size_t(2) << 20;
constexpr int kMaxThreads = 4;
constexpr size_t kPlainBytes = size_t(4) << 20;  // below: one hipMemcpyAsync

// The chunks t, t + nt, ... of thread t.
void copy_chunks(rp_ctx* h, char* host, char* dev, size_t bytes, bool to_host, int t, int nt) {
  RP_HIP(hipSetDevice(h->device));
  hipEvent_t ev[2] = {};
  struct Done {
    hipEvent_t* e;
    ~Done() {
      for (int i = 0; i < 2; ++i)
        if (e[i]) {
          (void)hipEventSynchronize(e[i]);  // nothing in flight uses the pinned chunks
          (void)hipEventDestroy(e[i]);
        }
    }
  } done{ev};
  for (auto& e : ev) RP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  char* pin[2] = {h->h_copy.p + (size_t)(2 * t) * kChunkBytes,
                  h->h_copy.p + (size_t)(2 * t + 1) * kChunkBytes};
  const size_t n = (bytes + kChunkBytes - 1) / kChunkBytes;
  auto size_of = [&](size_t c) { return std::min(kChunkBytes, bytes - c * kChunkBytes); };
  size_t last = n;  // chunk on the link (to the host), n: none
  int slot = 0;
  for (size_t c = (size_t)t; c < n; c += (size_t)nt, slot ^= 1) {
    const size_t off = c * kChunkBytes, m = size_of(c);
    if (to_host) {
      RP_HIP(hipMemcpyAsync(pin[slot], dev + off, m, hipMemcpyDeviceToHost, h->stream));
      RP_HIP(hipEventRecord(ev[slot], h->stream));
      if (last < n) {
        RP_HIP(hipEventSynchronize(ev[slot ^ 1]));
        std::memcpy(host + last * kChunkBytes, pin[slot ^ 1], size_of(last));
      }
      last = c;
    } else {
      if (c >= 2 * (size_t)nt) RP_HIP(hipEventSynchronize(ev[slot]));  // its last chunk has left
      std::memcpy(pin[slot], host + off, m);
      RP_HIP(hipMemcpyAsync(dev + off, pin[slot], m, hipMemcpyHostToDevice, h->stream));
      RP_HIP(hipEventRecord(ev[slot], h->stream));
    }
  }
  if (to_host && last < n) {
    RP_HIP(hipEventSynchronize(ev[slot ^ 1]));
    std::memcpy(host + last * kChunkBytes, pin[slot ^ 1], size_of(last));
  }
}

// Whether the runtime knows the caller's memory (pinned, managed): it then copies
// straight to or from it, at the rate of the link.
bool known_memory(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// Threads for a copy, with the handle's pinned chunks for them; 0: none of this, the
// copy is left to the runtime.
int copy_threads(rp_ctx* h, const void* host, size_t bytes) {
  if (bytes < kPlainBytes || known_memory(host)) return 0;
  const int nt = std::min(kMaxThreads, std::max(1, (int)std::thread::hardware_concurrency() / 2));
  try {
    h->h_copy.reserve(2 * (size_t)nt * kChunkBytes);
  } catch (const Error&) {  // no pinned memory to be had
    (void)hipGetLastError();
    return 0;
  }
  return nt;
}

void copy(rp_ctx* h, void* host, void* dev, size_t bytes, bool to_host) {
  const int nt = copy_threads(h, host, bytes);
  if (nt == 0) {
    if (to_host) RP_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, h->stream));
    else RP_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, h->stream));
    RP_HIP(hipStreamSynchronize(h->stream));
    return;
  }
  std::vector<std::exception_ptr> err(nt);
  auto work = [&](int t) {
    try {
      copy_chunks(h, (char*)host, (char*)dev, bytes, to_host, t, nt);
    } catch (...) {
      err[t] = std::current_exception();
    }
  };
  struct Join {
    std::vector<std::thread> th;
    ~Join() {
      for (auto& x : th) x.join();
    }
  };
  {
    Join join;
    join.th.reserve(nt - 1);
    for (int t = 1; t < nt; ++t) {
      try {
        join.th.emplace_back(work, t);
      } catch (...) {  // no thread to be had: its share is done here
        work(t);
      }
    }
    work(0);
  }
  for (const auto& e : err)
    if (e) std::rethrow_exception(e);
}

}  // namespace

void copy_to_host(rp_ctx* h, void* dst, const void* dev, size_t bytes) {
  copy(h, dst, const_cast<void*>(dev), bytes, true);
}

void copy_to_device(rp_ctx* h, void* dev, const void* src, size_t bytes) {
  copy(h, const_cast<void*>(src), dev, bytes, false);
}

}  // namespace rp
