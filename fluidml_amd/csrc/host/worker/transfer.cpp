#include "worker/transfer.h"

#include <emmintrin.h>
#include <sched.h>

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>

#include "fluidml_hip.h"

namespace fluidml {
namespace worker {
namespace {

void Check(int rc, const char *what) {
  if (rc != 0) throw std::runtime_error(std::string(what) + ": " + fluidml_hip_error_string(rc));
}

constexpr size_t kAlign = 256;
constexpr size_t kFlagBase = 64;
size_t Padded(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

// From here on one thread no longer keeps up with the link (a core copies 23-30 GB/s of memory that the link has just
// written, the link moves 55) and the helpers, which take tens of microseconds to wake, are called; and the copies
// bypass the caches (51.5 MB: 1.65 ms with plain stores, 1.1 ms without, on one core).
constexpr size_t kLargeBytes = size_t{1} << 20;
constexpr double kWakeNs = 1.0e5;
constexpr size_t kSmallSlice = 16 << 10, kLargeSlice = 512 << 10;
// Slice of the way out, whole pieces of 16 KiB: as large as leaves about two hundred of them.
size_t OutSlice(size_t bytes) {
  size_t slice = kSmallSlice;
  while (slice < kLargeSlice && bytes / (2 * slice) >= 192) slice *= 2;
  return slice;
}
// The way in is staged and launched piece by piece: the first one small, so that the link starts early.
constexpr size_t kInSlice = 64 << 10, kInFirstPiece = 256 << 10, kInPiece = size_t{1} << 20;

void CopyStreaming(char *dst, const char *src, size_t bytes) {
  const size_t head = std::min(bytes, (16 - reinterpret_cast<uintptr_t>(dst) % 16) % 16);
  std::memcpy(dst, src, head);
  size_t i = head;
  for (; i + 64 <= bytes; i += 64) {
    const __m128i *s = reinterpret_cast<const __m128i *>(src + i);
    __m128i *d = reinterpret_cast<__m128i *>(dst + i);
    const __m128i a = _mm_loadu_si128(s), b = _mm_loadu_si128(s + 1), c = _mm_loadu_si128(s + 2), e = _mm_loadu_si128(s + 3);
    _mm_stream_si128(d, a);
    _mm_stream_si128(d + 1, b);
    _mm_stream_si128(d + 2, c);
    _mm_stream_si128(d + 3, e);
  }
  _mm_sfence();
  std::memcpy(dst + i, src + i, bytes - i);
}

// Work that several threads take piece by piece until none is left.
class Job {
 public:
  virtual ~Job() = default;
  virtual void Work(bool caller) = 0;
};

// A few threads of the process that help one large transfer at a time; they sleep in between.  A run that finds them
// busy with another plan's transfer does without.
class Helpers {
 public:
  static Helpers &Get() {
    static Helpers helpers;
    return helpers;
  }
  bool Call(Job *job) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (job_ != nullptr || count_ == 0) return false;
    if (threads_.empty()) {
      for (size_t i = 0; i < count_; ++i) threads_.emplace_back([this] { Loop(); });
    }
    job_ = job;
    ++round_;
    wake_.notify_all();
    return true;
  }
  // No helper touches the job once this has returned.  `poll` runs while it waits.
  template <typename F>
  void Dismiss(F poll) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      job_ = nullptr;
    }
    while (inside_.load(std::memory_order_acquire) != 0) poll();
  }

 private:
  Helpers() {
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    // (51.5 MB out: 2.25 ms with the caller alone, 1.35 with three helpers, 1.15 with seven, 1.16 with eleven)
    count_ = static_cast<size_t>(std::clamp(cpus / 2 - 1, 0, 7));
  }
  ~Helpers() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    wake_.notify_all();
    for (std::thread &t : threads_) t.join();
  }
  void Loop() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
      wake_.wait(lock, [&] { return stop_ || (job_ != nullptr && round_ != seen); });
      if (stop_) return;
      seen = round_;
      Job *job = job_;
      inside_.fetch_add(1, std::memory_order_relaxed);
      lock.unlock();
      job->Work(false);
      inside_.fetch_sub(1, std::memory_order_release);
      lock.lock();
    }
  }

  std::mutex mutex_;
  std::condition_variable wake_;
  std::vector<std::thread> threads_;
  size_t count_ = 0;
  Job *job_ = nullptr;
  uint64_t round_ = 0;
  bool stop_ = false;
  std::atomic<int> inside_{0};
};

}  // namespace

// Stages the inputs in slices; the caller launches the copies of what lies staged in one run from the front.
class Transfer::InJob : public Job {
 public:
  struct Slice {
    size_t slot, begin, bytes;
  };
  InJob(const Transfer &t, const std::vector<const void *> &host) : t_(t), host_(host) {
    for (size_t i = 0; i < t.inputs_.size(); ++i) {
      for (size_t at = 0; at < t.inputs_[i].bytes; at += kInSlice) {
        slices_.push_back({i, at, std::min(kInSlice, t.inputs_[i].bytes - at)});
      }
    }
    done_ = std::vector<std::atomic<bool>>(slices_.size());
  }
  const std::vector<Slice> &Slices() const { return slices_; }
  bool Done(size_t i) const { return done_[i].load(std::memory_order_acquire); }
  bool One() {
    const size_t i = next_.fetch_add(1, std::memory_order_relaxed);
    if (i >= slices_.size()) return false;
    const Slice &s = slices_[i];
    std::memcpy(t_.in_ + t_.inputs_[s.slot].offset + s.begin, static_cast<const char *>(host_[s.slot]) + s.begin, s.bytes);
    done_[i].store(true, std::memory_order_release);
    return true;
  }
  void Work(bool) override {
    while (One()) {
    }
  }

 private:
  const Transfer &t_;
  const std::vector<const void *> &host_;
  std::vector<Slice> slices_;
  std::vector<std::atomic<bool>> done_;
  std::atomic<size_t> next_{0};
};

// Takes the outbound slices over as their flags appear.
class Transfer::OutJob : public Job {
 public:
  struct Slice {
    size_t slot, begin, bytes;
  };
  OutJob(const Transfer &t, const std::vector<void *> &host, void *stream, bool streaming)
      : t_(t), host_(host), stream_(stream), streaming_(streaming) {
    for (size_t i = 0; i < t.outputs_.size(); ++i) {
      for (size_t at = 0; at < t.outputs_[i].bytes; at += t.out_slice_) {
        slices_.push_back({i, at, std::min(t.out_slice_, t.outputs_[i].bytes - at)});
      }
    }
  }
  void Work(bool caller) override {
    for (;;) {
      const size_t i = next_.fetch_add(1, std::memory_order_relaxed);
      if (i >= slices_.size() || !Wait(i, caller, [] {})) return;
      const Slice &s = slices_[i];
      char *dst = static_cast<char *>(host_[s.slot]) + s.begin;
      const char *src = t_.out_ + t_.outputs_[s.slot].offset + s.begin;
      if (streaming_) {
        CopyStreaming(dst, src, s.bytes);
      } else {
        std::memcpy(dst, src, s.bytes);
      }
    }
  }
  // The stream has failed, or is idle although a flag is missing: no flag will come any more.
  void Poll() {
    if (failed_.load(std::memory_order_relaxed)) return;
    int idle = 0;
    const int rc = fluidml_hip_stream_query(stream_, &idle);
    if (rc != 0) {
      rc_ = rc;
      failed_.store(true, std::memory_order_release);
    } else if (idle != 0 && ++idle_polls_ > 1000) {
      failed_.store(true, std::memory_order_release);
    }
  }
  template <typename F>
  bool Wait(size_t flag, bool caller, F between) {
    const auto *f = reinterpret_cast<const uint32_t *>(t_.mailbox_ + kFlagBase) + flag;
    for (uint32_t spins = 1; __atomic_load_n(f, __ATOMIC_ACQUIRE) != t_.value_; ++spins) {
      for (int i = 0; i < 16; ++i) _mm_pause();  // (a poll takes the flag's line away from the link)
      between();
      if (failed_.load(std::memory_order_relaxed)) return false;
      if (caller && spins % (1u << 12) == 0) Poll();
    }
    return true;
  }
  void Finish() const {
    if (!failed_.load(std::memory_order_acquire)) return;
    Check(rc_, "waiting for the outputs");
    throw std::runtime_error("waiting for the outputs: the stream is idle but they did not arrive");
  }

 private:
  const Transfer &t_;
  const std::vector<void *> &host_;
  void *stream_;
  bool streaming_;
  std::vector<Slice> slices_;
  std::atomic<size_t> next_{0};
  std::atomic<bool> failed_{false};
  int rc_ = 0;
  uint32_t idle_polls_ = 0;
};

Transfer::Transfer(std::vector<Slot> &&inputs, std::vector<Slot> &&outputs) {
  for (Slot &s : inputs) {
    if (s.bytes == 0) continue;
    s.offset = in_bytes_;
    in_bytes_ += Padded(s.bytes);
  }
  for (Slot &s : outputs) {
    if (s.bytes == 0) continue;
    s.offset = out_bytes_;
    out_bytes_ += Padded(s.bytes);
  }
  inputs_ = std::move(inputs);
  outputs_ = std::move(outputs);
  out_slice_ = OutSlice(out_bytes_);
  size_t flags = 1;
  for (const Slot &s : outputs_) flags += (s.bytes + out_slice_ - 1) / out_slice_;
  int khz = 0;
  Check(fluidml_hip_clock_khz(&khz), "reading the device clock's rate");
  if (khz > 0) ns_per_tick_ = 1.0e6 / khz;
  try {
    void *p = nullptr;
    Check(fluidml_hip_arena_create(sizeof(uint64_t), &p), "allocating the transfer clock");  // zero-filled
    clock_ = static_cast<uint64_t *>(p);
    Check(fluidml_hip_arena_create((flags + outputs_.size() + 1) * sizeof(uint32_t), &p), "allocating the transfer counters");
    counters_ = static_cast<uint32_t *>(p);
    Check(fluidml_hip_stream_synchronize(nullptr), "waiting for the cleared counters");
    Check(fluidml_hip_host_alloc(in_bytes_, &p), "allocating pinned memory for the inputs");
    in_ = static_cast<char *>(p);
    Check(fluidml_hip_host_alloc(out_bytes_, &p), "allocating pinned memory for the outputs");
    out_ = static_cast<char *>(p);
    Check(fluidml_hip_host_alloc(kFlagBase + flags * sizeof(uint32_t), &p), "allocating the transfer flags");
    mailbox_ = static_cast<char *>(p);
  } catch (...) {
    Release();
    throw;
  }
  std::memset(in_, 0, in_bytes_);  // (the padding is copied along)
  std::memset(mailbox_, 0, kFlagBase + flags * sizeof(uint32_t));
}

Transfer::~Transfer() { Release(); }

void Transfer::Release() {
  fluidml_hip_host_free(in_);
  fluidml_hip_host_free(out_);
  fluidml_hip_host_free(mailbox_);
  fluidml_hip_arena_destroy(clock_);
  fluidml_hip_arena_destroy(counters_);
}

void Transfer::In(const std::vector<const void *> &host, void *stream) {
  InJob job(*this, host);
  const std::vector<InJob::Slice> &slices = job.Slices();
  Helpers &helpers = Helpers::Get();
  const bool helped = in_bytes_ >= kLargeBytes && helpers.Call(&job);
  int rc = 0;
  void *dst[FL_MAX_TRANSFER_SEGMENTS];
  const void *src[FL_MAX_TRANSFER_SEGMENTS];
  size_t bytes[FL_MAX_TRANSFER_SEGMENTS];
  size_t launched = 0;  // slices
  size_t piece = in_bytes_ < kLargeBytes ? in_bytes_ : kInFirstPiece;
  do {
    // the next piece: whole slices from the front, neighbours of one argument as one segment
    int32_t n = 0;
    size_t taken = 0, end = launched;
    for (; end < slices.size() && taken < piece; ++end) {
      const InJob::Slice &s = slices[end];
      const Slot &slot = inputs_[s.slot];
      const bool extends = end > launched && slices[end - 1].slot == s.slot;
      if (!extends && n == FL_MAX_TRANSFER_SEGMENTS) break;
      if (extends) {
        bytes[n - 1] += s.bytes;
      } else {
        dst[n] = static_cast<char *>(slot.device) + s.begin;
        src[n] = in_ + slot.offset + s.begin;
        bytes[n++] = s.bytes;
      }
      taken += s.bytes;
    }
    for (size_t i = launched; i < end; ++i) {
      while (!job.Done(i)) {
        if (!job.One()) _mm_pause();
      }
    }
    rc = fluidml_hip_transfer_in(n, dst, src, bytes, clock_, stream);
    launched = end;
    piece = kInPiece;
  } while (rc == 0 && launched < slices.size());
  if (helped) helpers.Dismiss([] { _mm_pause(); });
  Check(rc, "copying the inputs to HBM");
}

double Transfer::Out(const std::vector<void *> &host, void *stream) {
  const bool large = out_bytes_ >= kLargeBytes;
  ++value_;
  OutJob job(*this, host, stream, large);
  uint64_t *elapsed = reinterpret_cast<uint64_t *>(mailbox_);
  uint32_t *flags = reinterpret_cast<uint32_t *>(mailbox_ + kFlagBase);
  void *dst[FL_MAX_TRANSFER_SEGMENTS];
  const void *src[FL_MAX_TRANSFER_SEGMENTS];
  size_t bytes[FL_MAX_TRANSFER_SEGMENTS];
  size_t at = 0, flag = 0, launches = 0;
  do {
    int32_t n = 0;
    const size_t first_flag = flag, first_counter = flag + launches++;  // (each launch has a counter of its own besides)
    for (; at < outputs_.size() && n < FL_MAX_TRANSFER_SEGMENTS; ++at) {
      const Slot &s = outputs_[at];
      if (s.bytes == 0) continue;
      dst[n] = out_ + s.offset;
      src[n] = s.device;
      bytes[n++] = s.bytes;
      flag += (s.bytes + out_slice_ - 1) / out_slice_;
    }
    Check(fluidml_hip_transfer_out(n, dst, src, bytes, out_slice_, clock_, first_flag == 0 ? elapsed : nullptr, flags + first_flag,
                                   counters_ + first_counter, value_, stream),
          "copying the outputs to the host");
  } while (at < outputs_.size());
  // Not at once: what is queued in front of the launch may take any time, and the helpers would poll through all of it.  But
  // a little before the first slice is due, by the previous run's wait, since they take tens of microseconds to wake
  // (1.6 MB of BERT-base at 512 tokens: called with the first flag 1547 us a pass, this way 1506).
  Helpers &helpers = Helpers::Get();
  const auto queued = std::chrono::steady_clock::now();
  auto waited = [&] { return std::chrono::duration<double, std::nano>(std::chrono::steady_clock::now() - queued).count(); };
  bool called = !large, helped = false;
  auto call = [&] {
    called = true;
    helped = helpers.Call(&job);
  };
  // (also without an output: the launch leaves one flag)
  job.Wait(0, true, [&] {
    if (!called && wait_ns_ > 0 && waited() > wait_ns_ - kWakeNs) call();
  });
  wait_ns_ = waited();
  if (!called) call();
  job.Work(true);
  if (helped) {
    uint32_t spins = 0;
    helpers.Dismiss([&] {
      _mm_pause();
      if (++spins % (1u << 14) == 0) job.Poll();
    });
  }
  job.Finish();
  return static_cast<double>(__atomic_load_n(elapsed, __ATOMIC_ACQUIRE)) * ns_per_tick_;
}

}  // namespace worker
}  // namespace fluidml
