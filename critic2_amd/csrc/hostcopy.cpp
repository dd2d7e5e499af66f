// Large transfers between pageable host memory (or a file) and the device.
//
// The runtime moves pageable memory through one staging thread (29 GB/s in,
// 18 GB/s out here, less where the destination's pages are touched for the
// first time) against 57 GB/s of the link.  Here the transfer is cut into
// chunks and STAGE_THREADS threads each carry theirs through a pinned slot of
// the context's own, so that the copies and page faults of several chunks run
// beside the link.  Measured: a 160 MB cube file read and parsed into HBM
// 41.6 -> 4.2 ms (two 64 MiB slots made per call before), 386 MB of cube text
// out of it 110 -> 10.4 ms.  Six threads: a warm destination takes 49 GB/s,
// and four already read the page cache at 40 GB/s.  The slots (24 MiB) are made
// on first use, kept by the context and given back with it; where pinned memory
// runs out the slots there are do the work, and with none the runtime's copy.
#include <fcntl.h>
#include <hip/hip_runtime.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cerrno>
#include <cstring>
#include <exception>
#include <mutex>
#include <optional>
#include <string>
#include <thread>
#include <vector>

#include "common.hpp"

namespace c2 {

namespace {

constexpr int STAGE_THREADS = c2gpu_ctx::STAGE_SLOTS;
constexpr size_t STAGE_CHUNK = (size_t)4 << 20;  // bytes of a slot
// Below these the runtime's copy is the faster: starting the threads takes 0.1
// ms.  From and to memory that no cache holds, runtime against staged, in us: in
// 2 MiB 109, 170; 8 MiB 320, 430; 16 MiB 603, 615; 24 MiB 885, 790; out 2 MiB
// 123, 175; 4 MiB 248, 285; 6 MiB 372, 385; 8 MiB 486, 426.
constexpr size_t STAGE_MIN_IN = (size_t)16 << 20, STAGE_MIN_OUT = (size_t)7 << 20;

// The number of slots to be had, the first of the context's: fewer than
// STAGE_THREADS, or none, where pinned memory runs out.  The missing ones are
// asked for again by the next transfer.
int stage_slots(c2gpu_ctx *ctx) {
  for (int i = 0; i < STAGE_THREADS; i++) {
    auto &s = ctx->stage[i];
    if (!s.ptr && hipHostMalloc(&s.ptr, STAGE_CHUNK, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      s.ptr = nullptr;
      return i;
    }
    if (!s.ev) C2_HIP(hipEventCreateWithFlags(&s.ev, hipEventDisableTiming));
  }
  return STAGE_THREADS;
}

// The slots a transfer may use: the context's own, or, for a batch's worker,
// those of the batch's context, as long as no other thread is using them.  So
// a batch starts no more staging threads and pins no more memory than one
// context does; a worker that finds them taken leaves its copy to the runtime.
// (Six threads and slots for each of 8 workers: 8 host cells of 160^3 280 ms
// against 285 with the runtime's copies, other batches within the noise.)
struct Slots {
  std::unique_lock<std::mutex> held;
  c2gpu_ctx::Stage *first = nullptr;
  int n = 0;
  explicit Slots(c2gpu_ctx *ctx) {
    c2gpu_ctx *owner = ctx->stage_of ? ctx->stage_of : ctx;
    held = std::unique_lock<std::mutex>(owner->stage_mu, std::try_to_lock);
    if (!held) return;
    first = owner->stage;
    n = stage_slots(owner);
  }
};

// A slot of ordinary memory, for files where no pinned slot is to be had.
struct PlainSlot {
  std::vector<char> mem;
  c2gpu_ctx::Stage slot;
  explicit PlainSlot(size_t bytes) : mem(bytes) {
    slot.ptr = mem.data();
    C2_HIP(hipEventCreateWithFlags(&slot.ev, hipEventDisableTiming));
  }
  ~PlainSlot() { (void)hipEventDestroy(slot.ev); }
};

// Runs carry(slot, offset, length) for every chunk of [0, bytes), chunks
// spread over a thread for each of the `slots`; the first error stops the rest
// and is rethrown once every thread has ended.
template <class F>
void run_chunks(c2gpu_ctx *ctx, c2gpu_ctx::Stage *stage, int slots, size_t bytes, F &&carry) {
  // at least two chunks a thread where the transfer allows it
  const size_t chunk = std::min(STAGE_CHUNK, std::max((size_t)1 << 19, bytes / (2 * slots) + 1));
  const size_t n = (bytes + chunk - 1) / chunk;
  const int nt = (int)std::min<size_t>(slots, n);
  std::atomic<size_t> next{0};
  std::atomic<bool> failed{false};
  std::exception_ptr first;  // written by the thread that sets failed
  auto work = [&](int t) {
    try {
      C2_HIP(hipSetDevice(ctx->device));
      for (;;) {
        const size_t c = next.fetch_add(1);
        if (c >= n || failed.load()) break;
        const size_t o = c * chunk;
        carry(stage[t], o, std::min(chunk, bytes - o));
      }
      C2_HIP(hipEventSynchronize(stage[t].ev));  // the slot is free again
    } catch (...) {  // nothing may leave a thread
      if (!failed.exchange(true)) first = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  try {
    pool.reserve(slots);
    for (int t = 1; t < nt; t++) pool.emplace_back(work, t);
  } catch (const std::exception &) {
    // fewer threads than asked for: the others take the chunks
  }
  work(0);
  for (auto &t : pool) t.join();
  if (failed.load()) {
    (void)hipStreamSynchronize(ctx->stream);
    try {
      std::rethrow_exception(first);
    } catch (const Error &) {
      throw;
    } catch (const std::exception &e) {  // callers on threads of their own catch Error alone
      fail(C2GPU_ERR_ALLOC, std::string("host transfer: ") + e.what());
    }
  }
}

// run_chunks with the context's slots, or one of ordinary memory.
template <class F>
void run_file(c2gpu_ctx *ctx, size_t bytes, F &&carry) {
  const Slots slots(ctx);
  if (slots.n) {
    run_chunks(ctx, slots.first, slots.n, bytes, carry);
  } else {
    PlainSlot plain(std::min(STAGE_CHUNK, bytes));
    run_chunks(ctx, &plain.slot, 1, bytes, carry);
  }
}

// Ordinary memory that the staging threads may read and write themselves.
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// Whether a copy is worth staging and its host side allows it.  One with a null
// pointer is left to the runtime, which turns it into an error.
bool staged(size_t bytes, size_t least, const void *dst, const void *src, const void *host) {
  return bytes >= least && dst && src && pageable(host);
}

}  // namespace

void copy_in(c2gpu_ctx *ctx, void *dst, const void *src, size_t bytes) {
  if (bytes == 0) return;
  std::optional<Slots> slots;
  if (staged(bytes, STAGE_MIN_IN, dst, src, src)) slots.emplace(ctx);
  if (!slots || !slots->n) {
    C2_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    return;
  }
  run_chunks(ctx, slots->first, slots->n, bytes, [&](c2gpu_ctx::Stage &s, size_t o, size_t n) {
    C2_HIP(hipEventSynchronize(s.ev));
    std::memcpy(s.ptr, static_cast<const char *>(src) + o, n);
    C2_HIP(hipMemcpyAsync(static_cast<char *>(dst) + o, s.ptr, n, hipMemcpyHostToDevice, ctx->stream));
    C2_HIP(hipEventRecord(s.ev, ctx->stream));
  });
}

void copy_out(c2gpu_ctx *ctx, void *dst, const void *src, size_t bytes) {
  if (bytes == 0) return;
  std::optional<Slots> slots;
  if (staged(bytes, STAGE_MIN_OUT, dst, src, dst)) slots.emplace(ctx);
  if (!slots || !slots->n) {
    C2_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    C2_HIP(hipStreamSynchronize(ctx->stream));
    return;
  }
  run_chunks(ctx, slots->first, slots->n, bytes, [&](c2gpu_ctx::Stage &s, size_t o, size_t n) {
    C2_HIP(hipMemcpyAsync(s.ptr, static_cast<const char *>(src) + o, n, hipMemcpyDeviceToHost, ctx->stream));
    C2_HIP(hipEventRecord(s.ev, ctx->stream));
    C2_HIP(hipEventSynchronize(s.ev));
    std::memcpy(static_cast<char *>(dst) + o, s.ptr, n);
  });
}

void file_in(c2gpu_ctx *ctx, void *dst, int fd, uint64_t from, uint64_t bytes, const char *ends) {
  run_file(ctx, bytes, [&](c2gpu_ctx::Stage &s, size_t o, size_t n) {
    C2_HIP(hipEventSynchronize(s.ev));
    for (size_t got = 0; got < n;) {
      const ssize_t r = pread(fd, static_cast<char *>(s.ptr) + got, n - got, (off_t)(from + o + got));
      if (r < 0 && errno == EINTR) continue;
      if (r <= 0) fail(C2GPU_ERR_FORMAT, ends);
      got += (size_t)r;
    }
    C2_HIP(hipMemcpyAsync(static_cast<char *>(dst) + o, s.ptr, n, hipMemcpyHostToDevice, ctx->stream));
    C2_HIP(hipEventRecord(s.ev, ctx->stream));
  });
}

void file_out(c2gpu_ctx *ctx, int fd, uint64_t to, const void *src, uint64_t bytes) {
  run_file(ctx, bytes, [&](c2gpu_ctx::Stage &s, size_t o, size_t n) {
    C2_HIP(hipMemcpyAsync(s.ptr, static_cast<const char *>(src) + o, n, hipMemcpyDeviceToHost, ctx->stream));
    C2_HIP(hipEventRecord(s.ev, ctx->stream));
    C2_HIP(hipEventSynchronize(s.ev));
    for (size_t done = 0; done < n;) {
      const ssize_t r = pwrite(fd, static_cast<const char *>(s.ptr) + done, n - done, (off_t)(to + o + done));
      if (r < 0 && errno == EINTR) continue;
      if (r <= 0) fail(C2GPU_ERR_FORMAT, "cube: write failed");
      done += (size_t)r;
    }
  });
}

void release_stage(c2gpu_ctx *ctx) {
  for (auto &s : ctx->stage) {
    if (s.ev) (void)hipEventDestroy(s.ev);
    if (s.ptr) (void)hipHostFree(s.ptr);
    s.ev = nullptr;
    s.ptr = nullptr;
  }
}

}  // namespace c2
