// Host arrays to device arrays in front of a step, without waiting for the step before
// (DLArrayFeed; no counterpart in the reference, whose executor copies with
// cudaMemcpy, src/c_runtime_api.cc:148-158).
//
// A synchronous copy from pageable memory waits for the device, copies, and leaves the queue
// empty for as long as the host then takes to fill it: 1.6 ms of a ResNet-50 step of batch 64, 0.27 of the
// 0.40 ms of an MLP step.  Here the call copies the host arrays into pinned memory of its own - the caller may
// reuse theirs on return - and enqueues the rest:
//   * up to kDirectBytes a kernel on the caller's stream reads the pinned memory itself;
//   * more than that goes through a copy stream into a device buffer, in chunks while the next chunk is copied on
//     the host, overlapping with what the caller's stream still runs, and a kernel behind it distributes the buffer.
//     More than that with nothing to overlap with, a plain copy.
// Two slots of pinned memory and buffer per stream: a call waits for the last but one before it, so the host is
// at most two steps ahead.  They belong to the stream and go with it, or before: when anything else finds no room on the
// device, or a budget is set (feed_give_back).  A stream whose room could not be had, or was taken back, copies its
// large feeds synchronously from then on: asking again at every step would empty the allocator's cache each time.
#include "internal.h"

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

using namespace tf;

namespace {

constexpr size_t kDirectBytes = (size_t)1 << 20;
constexpr size_t kChunkBytes = (size_t)4 << 20;
constexpr size_t kMaxFeedBytes = (size_t)1 << 30;  // a slot at most; more is copied synchronously
constexpr size_t kAlign = 256;
constexpr int kSegments = 8;

// ---- memcpy by several threads ------------------------------------------------------------
// One thread copies 38 MB that its caches hold at 32 GB/s, the link takes 56.  The threads are started once and sleep
// between calls.
class CopyThreads {
 public:
  void copy(char *dst, const char *src, size_t bytes) {
    if (bytes < kPiece * 2 || !start()) {
      memcpy(dst, src, bytes);
      return;
    }
    std::lock_guard<std::mutex> one_job(job_mu_);
    {
      std::lock_guard<std::mutex> g(mu_);
      dst_ = dst;
      src_ = src;
      bytes_ = bytes;
      next_.store(0);
      working_ = (int)threads_.size();
      ++generation_;
    }
    wake_.notify_all();
    pieces();
    std::unique_lock<std::mutex> g(mu_);
    done_.wait(g, [&] { return working_ == 0; });
  }

 private:
  static constexpr size_t kPiece = (size_t)256 << 10;
  bool start() {
    std::call_once(once_, [&] {
      const unsigned n = std::min(7u, std::max(1u, std::thread::hardware_concurrency()) - 1);
      try {
        for (unsigned i = 0; i < n; ++i) {
          threads_.emplace_back([this] { work(); });
          threads_.back().detach();
        }
      } catch (...) {  // as many as there are
      }
    });
    return !threads_.empty();
  }
  void pieces() {
    for (;;) {
      const size_t at = next_.fetch_add(kPiece);
      if (at >= bytes_) return;
      memcpy(dst_ + at, src_ + at, std::min(kPiece, bytes_ - at));
    }
  }
  void work() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> g(mu_);
        wake_.wait(g, [&] { return generation_ != seen; });
        seen = generation_;
      }
      pieces();
      std::lock_guard<std::mutex> g(mu_);
      if (--working_ == 0) done_.notify_one();
    }
  }
  std::once_flag once_;
  std::vector<std::thread> threads_;
  std::mutex job_mu_, mu_;
  std::condition_variable wake_, done_;
  char *dst_ = nullptr;
  const char *src_ = nullptr;
  size_t bytes_ = 0;
  std::atomic<size_t> next_{0};
  int working_ = 0;
  uint64_t generation_ = 0;
};
CopyThreads &copy_threads() {
  static CopyThreads *t = new CopyThreads();  // leaked on purpose: its threads outlive static destruction
  return *t;
}

// ---- the kernel ---------------------------------------------------------------------------
struct Segments {
  const float *src[kSegments];
  float *dst[kSegments];
  int64_t n[kSegments];
};
// Bound by where the sources are: 0.4 MB of pinned host memory in 12 us (33 GB/s, the link), a 38 MB buffer in 16 (4.8 TB/s
// read and written).
__global__ __launch_bounds__(256) void feed_kernel(Segments s, int count) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int k = 0; k < count; ++k) {
    int64_t done = 0;
    if ((reinterpret_cast<uintptr_t>(s.dst[k]) & 15u) == 0) {  // the sources are aligned
      const int64_t n4 = s.n[k] / 4;
      for (int64_t i = first; i < n4; i += step)
        reinterpret_cast<f32x4 *>(s.dst[k])[i] = reinterpret_cast<const f32x4 *>(s.src[k])[i];
      done = n4 * 4;
    }
    for (int64_t i = done + first; i < s.n[k]; i += step) s.dst[k][i] = s.src[k][i];
  }
}

// ---- slots ----------------------------------------------------------------------------------
struct Slot {
  char *host = nullptr, *dev = nullptr;
  hipEvent_t read = nullptr;  // behind the kernel that reads the slot
  bool pending = false;
};
struct Feed {
  std::mutex mu;
  hipEvent_t landed = nullptr;
  Slot slot[2];
  size_t host_bytes = 0, dev_bytes = 0;  // of a slot; both are halves of one block of the pools
  size_t refused = ~(size_t)0;           // feeds of this many bytes and more have no room
  int next = 0;
};
thread_local Feed *feed_in_hand = nullptr;  // whose mutex this thread holds
struct HoldFeed {
  explicit HoldFeed(Feed &f) : lock(f.mu) { feed_in_hand = &f; }
  ~HoldFeed() { feed_in_hand = nullptr; }
  std::lock_guard<std::mutex> lock;
};
std::mutex feeds_mu;
std::unordered_map<hipStream_t, std::unique_ptr<Feed>> *feeds = nullptr;  // leaked on purpose

Feed *feed_of(hipStream_t s) {
  std::lock_guard<std::mutex> g(feeds_mu);
  if (!feeds) feeds = new std::unordered_map<hipStream_t, std::unique_ptr<Feed>>();
  std::unique_ptr<Feed> &f = (*feeds)[s];
  if (!f) f.reset(new Feed());
  return f.get();
}

// One copy stream for all feeds; stays until the process ends.
hipStream_t copy_stream() {
  static const hipStream_t stream = [] {
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) {
      (void)hipGetLastError();
      return (hipStream_t) nullptr;
    }
    return s;
  }();
  return stream;
}

int wait_for_readers(Feed &f) {
  for (Slot &slot : f.slot) {
    if (slot.pending) TF_HIP(hipEventSynchronize(slot.read));
    slot.pending = false;
  }
  return 0;
}

// Behind wait_for_readers.
void drop_memory(Feed &f) {
  if (f.dev_bytes) (void)hipStreamSynchronize(copy_stream());  // a feed that failed part way leaves copies behind
  if (f.slot[0].host) pinned_free(f.slot[0].host);
  if (f.slot[0].dev) device_free(f.slot[0].dev);
  for (Slot &slot : f.slot) slot.host = slot.dev = nullptr;
  f.host_bytes = f.dev_bytes = 0;
}

// Room for `bytes` in both slots: 0 there is, 1 it cannot be had, -1 error.
int make_room(Feed &f, size_t bytes) {
  const bool direct = bytes <= kDirectBytes;
  for (Slot &slot : f.slot)
    if (!slot.read) TF_HIP(hipEventCreateWithFlags(&slot.read, hipEventDisableTiming));
  if (!direct && !f.landed) TF_HIP(hipEventCreateWithFlags(&f.landed, hipEventDisableTiming));
  if (!direct && !copy_stream()) return 1;
  if (f.host_bytes >= bytes && (direct || f.dev_bytes >= bytes)) return 0;
  if (bytes >= f.refused) return 1;
  if (wait_for_readers(f) != 0) return -1;
  drop_memory(f);
  f.refused = bytes;  // until there is room
  char *host = (char *)pinned_alloc(2 * bytes);
  if (!host) return 1;
  char *dev = direct ? nullptr : (char *)device_alloc(2 * bytes);
  if (!direct && !dev) {
    pinned_free(host);
    return 1;
  }
  f.refused = ~(size_t)0;
  f.slot[0].host = host;
  f.slot[1].host = host + bytes;
  f.host_bytes = bytes;
  if (direct) return 0;
  f.slot[0].dev = dev;
  f.slot[1].dev = dev + bytes;
  f.dev_bytes = bytes;
  // kernels of the block's previous life may still run, and the copy stream is not ordered behind them
  TF_HIP(hipDeviceSynchronize());
  return 0;
}

int launch_feed(DLArrayHandle *to, const size_t *offset, int n, const char *base, hipStream_t s) {
  for (int first = 0; first < n; first += kSegments) {
    Segments seg = {};
    const int count = std::min(kSegments, n - first);
    int64_t most = 0;
    for (int k = 0; k < count; ++k) {
      seg.src[k] = reinterpret_cast<const float *>(base + offset[first + k]);
      seg.dst[k] = (float *)to[first + k]->data;
      seg.n[k] = numel(to[first + k]);
      most = std::max(most, seg.n[k]);
    }
    const int blocks = (int)std::min<int64_t>((most / 4 + 255) / 256 + 1, (int64_t)num_cus() * 8);
    hipLaunchKernelGGL(feed_kernel, dim3(blocks), dim3(256), 0, s, seg, count);
  }
  TF_HIP(hipGetLastError());
  return 0;
}

// Feeds that went each way, for tests: kernels reading pinned memory, the copy stream, plain copies.
std::atomic<long long> feeds_direct{0}, feeds_overlapped{0}, feeds_synchronous{0};

int copy_synchronously(DLArrayHandle *from, DLArrayHandle *to, int n) {
  feeds_synchronous.fetch_add(1);
  for (int i = 0; i < n; ++i)
    if (DLArrayCopyFromTo(from[i], to[i], nullptr) != 0) return -1;
  return 0;
}

}  // namespace

namespace tf {

void feed_forget_stream(hipStream_t s) {
  std::unique_ptr<Feed> f;
  {
    std::lock_guard<std::mutex> g(feeds_mu);
    if (!feeds) return;
    auto it = feeds->find(s);
    if (it == feeds->end()) return;
    f = std::move(it->second);
    feeds->erase(it);
  }
  (void)hipStreamSynchronize(s);
  drop_memory(*f);
  for (Slot &slot : f->slot) {
    if (slot.read) (void)hipEventDestroy(slot.read);
  }
  if (f->landed) (void)hipEventDestroy(f->landed);
}

// Returns whether any device memory was given back.  A feed that is under way on another thread keeps its own.
bool feed_give_back(bool for_good) {
  bool any = false;
  std::lock_guard<std::mutex> g(feeds_mu);
  if (!feeds) return false;
  for (auto &entry : *feeds) {
    Feed &f = *entry.second;
    if (&f == feed_in_hand || !f.mu.try_lock()) continue;
    std::lock_guard<std::mutex> held(f.mu, std::adopt_lock);
    if (f.dev_bytes == 0 || wait_for_readers(f) != 0) continue;
    drop_memory(f);
    if (for_good) f.refused = std::min(f.refused, kDirectBytes + 1);
    any = true;
  }
  return any;
}

}  // namespace tf

namespace {

// Whether feeds of this size go the asynchronous way at all.
bool asynchronous(size_t total, DLStreamHandle stream) {
  return stream && !sync_every_op() && !device_budget_active() && total <= kMaxFeedBytes;
}

size_t padded(int64_t elements) { return ((size_t)elements * sizeof(float) + kAlign - 1) / kAlign * kAlign; }

int feed(DLArrayHandle *from, DLArrayHandle *to, int n, DLStreamHandle stream) {
  size_t total = 0;
  std::vector<size_t> offset((size_t)n);
  for (int i = 0; i < n; ++i) {
    offset[i] = total;
    total += padded(numel(to[i]));
  }
  if (total == 0) return 0;
  if (!asynchronous(total, stream)) return copy_synchronously(from, to, n);
  hipStream_t s = reinterpret_cast<hipStream_t>(*reinterpret_cast<void **>(stream));
  Feed *f = feed_of(s);
  HoldFeed hold(*f);
  // nothing to overlap with: a plain copy is through sooner
  if (total > kDirectBytes && idle(s) && !other_streams_busy(s)) return copy_synchronously(from, to, n);
  if (const int rc = make_room(*f, total)) return rc > 0 ? copy_synchronously(from, to, n) : -1;
  Slot &slot = f->slot[f->next];
  f->next ^= 1;
  if (slot.pending) TF_HIP(hipEventSynchronize(slot.read));
  slot.pending = false;
  const bool direct = total <= kDirectBytes;
  if (direct) {
    for (int i = 0; i < n; ++i) memcpy(slot.host + offset[i], from[i]->data, (size_t)numel(from[i]) * sizeof(float));
  } else {
    for (int i = 0; i < n; ++i) {
      const size_t bytes = (size_t)numel(from[i]) * sizeof(float);
      for (size_t at = 0; at < bytes; at += kChunkBytes) {
        const size_t len = std::min(kChunkBytes, bytes - at);
        copy_threads().copy(slot.host + offset[i] + at, (const char *)from[i]->data + at, len);
        TF_HIP(hipMemcpyAsync(slot.dev + offset[i] + at, slot.host + offset[i] + at, len, hipMemcpyHostToDevice, copy_stream()));
      }
    }
  }
  // Kernels of other streams may still read the destinations, and blocks of the allocator go from one stream's step to
  // the next one's: what runs there ends first.  The host waits for it, as a synchronous copy would; a queue that waits
  // for another's event slows that one's launches down (ResNet-50 spatial at batch 8, three executors in turn: 4.55 ms a step
  // so, 3.97 with one executor, 4.25 with synchronous copies).
  if (host_waits_for_other_streams(s) != 0) return -1;
  if (direct) {
    if (launch_feed(to, offset.data(), n, slot.host, s) != 0) return -1;
  } else {
    TF_HIP(hipEventRecord(f->landed, copy_stream()));
    TF_HIP(hipStreamWaitEvent(s, f->landed, 0));
    if (launch_feed(to, offset.data(), n, slot.dev, s) != 0) return -1;
  }
  TF_HIP(hipEventRecord(slot.read, s));
  slot.pending = true;
  (direct ? feeds_direct : feeds_overlapped).fetch_add(1);
  return 0;
}

}  // namespace

extern "C" int DLArrayFeed(DLArrayHandle *from, DLArrayHandle *to, int n, DLStreamHandle stream) {
  TF_REQUIRE(n >= 0 && (n == 0 || (from && to)), "bad arguments");
  for (int i = 0; i < n; ++i) {
    announce_write(to[i]);
    TF_REQUIRE(from[i] && to[i] && from[i]->data && to[i]->data, "null array");
    TF_REQUIRE(from[i]->ctx.device_type == kCPU && to[i]->ctx.device_type == kGPU, "host to device only");
    TF_REQUIRE(numel(from[i]) == numel(to[i]), "size mismatch (%lld vs %lld elements)", (long long)numel(from[i]),
               (long long)numel(to[i]));
  }
  try {
    return feed(from, to, n, stream);
  } catch (const std::exception &e) {  // no host memory
    TF_REQUIRE(false, "%s", e.what());
  }
}

extern "C" int DLArrayFeedReserve(DLArrayHandle *to, int n, DLStreamHandle stream) {
  TF_REQUIRE(n >= 0 && (n == 0 || to), "bad arguments");
  size_t total = 0;
  for (int i = 0; i < n; ++i) {
    TF_REQUIRE(to[i], "null array");
    total += padded(numel(to[i]));
  }
  if (total == 0 || !asynchronous(total, stream)) return 0;
  try {
    Feed *f = feed_of(stream_of(reinterpret_cast<void **>(stream)));
    HoldFeed hold(*f);
    return make_room(*f, total) < 0 ? -1 : 0;  // without room the feeds are synchronous
  } catch (const std::exception &e) {
    TF_REQUIRE(false, "%s", e.what());
  }
}

extern "C" int DLArrayFeedCounts(long long *direct, long long *overlapped, long long *synchronous) {
  if (direct) *direct = feeds_direct.load();
  if (overlapped) *overlapped = feeds_overlapped.load();
  if (synchronous) *synchronous = feeds_synchronous.load();
  return 0;
}
