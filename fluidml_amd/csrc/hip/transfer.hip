// Copies between pinned host memory and HBM for the arguments of one run: several arguments per launch, and on the
// way out a flag in host memory per slice, so that the host can take a slice over while later ones still travel.
#include "fl_common.h"

using namespace fl;

namespace {

constexpr uint32_t kThreads = 256;

struct Segment {
  const uint4 *src;
  uint4 *dst;
  uint32_t n16;          // 16-byte items; both sides are padded to whole items
  uint32_t first_block;  // block that copies the segment's first slice
};

struct TransferArgs {
  uint32_t n_segments;
  uint32_t slice16;  // 16-byte items of a slice; a block copies one slice
  uint64_t *clock;   // device: latest end of an inbound launch since the last outbound one
  uint32_t *flags;   // host: one per block (outbound only)
  uint64_t *elapsed;  // host: ticks between *clock and the start of the outbound launch
  uint32_t value;
  Segment segments[FL_MAX_TRANSFER_SEGMENTS];
};

// Bound by the link (about 55 GB/s each way: 51.5 MB take 0.93 ms, the copy engine needs 0.91) and, for the few
// kilobytes of a text request, by the launch (an asynchronous copy of pageable memory costs 13 us in and 21 us out per
// argument and a stream wait 11 us; one launch plus a polled flag 6 us).  Four 16-byte loads are in flight per lane.
template <bool OUTBOUND>
__global__ __launch_bounds__(kThreads) void TransferKernel(TransferArgs args) {
  if (OUTBOUND && blockIdx.x == 0 && threadIdx.x == 0 && args.elapsed != nullptr) {
    const uint64_t now = wall_clock64();
    const uint64_t since = *args.clock;
    *args.clock = 0;
    *args.elapsed = since != 0 && now > since ? now - since : 0;
  }
  uint32_t s = 0;
  while (s + 1 < args.n_segments && blockIdx.x >= args.segments[s + 1].first_block) ++s;
  if (args.n_segments != 0) {
    const Segment g = args.segments[s];
    const uint32_t begin = (blockIdx.x - g.first_block) * args.slice16;
    const uint32_t end = begin + args.slice16 < g.n16 ? begin + args.slice16 : g.n16;
    for (uint32_t i = begin + threadIdx.x; i < end; i += 4 * kThreads) {
      uint4 v[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        if (i + j * kThreads < end) v[j] = g.src[i + j * kThreads];
      }
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        if (i + j * kThreads < end) g.dst[i + j * kThreads] = v[j];
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores have been acknowledged
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (OUTBOUND) {
    __hip_atomic_store(args.flags + blockIdx.x, args.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  } else {
    atomicMax(reinterpret_cast<unsigned long long *>(args.clock), static_cast<unsigned long long>(wall_clock64()));
  }
}

int FillSegments(TransferArgs &a, uint32_t &blocks, int32_t n, void *const *dst, const void *const *src, const size_t *bytes,
                 size_t slice_bytes) {
  if (n < 0 || n > FL_MAX_TRANSFER_SEGMENTS) return FL_ERR_ATTR;
  if (slice_bytes == 0 || slice_bytes % 16 != 0) return FL_ERR_ATTR;
  std::memset(&a, 0, sizeof(a));
  a.slice16 = static_cast<uint32_t>(slice_bytes / 16);
  uint64_t at = 0;
  for (int32_t i = 0; i < n; ++i) {
    if (dst[i] == nullptr || src[i] == nullptr) return FL_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(dst[i]) | reinterpret_cast<uintptr_t>(src[i])) % 16 != 0) return FL_ERR_ATTR;
    if (bytes[i] == 0) return FL_ERR_SHAPE;
    if ((bytes[i] + 15) / 16 > 0x7fffffffu) return FL_ERR_TOO_LARGE;
    Segment &g = a.segments[a.n_segments++];
    g.src = static_cast<const uint4 *>(src[i]);
    g.dst = static_cast<uint4 *>(dst[i]);
    g.n16 = static_cast<uint32_t>((bytes[i] + 15) / 16);
    g.first_block = static_cast<uint32_t>(at);
    at += (g.n16 + a.slice16 - 1) / a.slice16;
    if (at > 0x7fffffffu) return FL_ERR_TOO_LARGE;
  }
  blocks = static_cast<uint32_t>(at == 0 ? 1 : at);
  return FL_OK;
}

}  // namespace

extern "C" {

int fluidml_hip_host_alloc(size_t bytes, void **host) {
  if (host == nullptr) return FL_ERR_NULL;
  *host = nullptr;
  void *p = nullptr;
  const hipError_t err = hipHostMalloc(&p, bytes == 0 ? 1 : bytes, hipHostMallocDefault);
  if (err != hipSuccess) {
    (void)hipGetLastError();
    return static_cast<int>(err);
  }
  *host = p;
  return FL_OK;
}

int fluidml_hip_host_free(void *host) {
  if (host == nullptr) return FL_OK;
  FL_HIP_CHECK(hipHostFree(host));
  return FL_OK;
}

int fluidml_hip_stream_query(void *stream, int *idle) {
  if (idle == nullptr) return FL_ERR_NULL;
  const hipError_t err = hipStreamQuery(AsStream(stream));
  if (err != hipSuccess && err != hipErrorNotReady) return static_cast<int>(err);
  if (err == hipErrorNotReady) (void)hipGetLastError();
  *idle = err == hipSuccess ? 1 : 0;
  return FL_OK;
}

int fluidml_hip_clock_khz(int *khz) {
  if (khz == nullptr) return FL_ERR_NULL;
  int dev = 0;
  FL_HIP_CHECK(hipGetDevice(&dev));
  FL_HIP_CHECK(hipDeviceGetAttribute(khz, hipDeviceAttributeWallClockRate, dev));
  return FL_OK;
}

int fluidml_hip_transfer_in(int32_t n, void *const *device, const void *const *host, const size_t *bytes, size_t slice_bytes,
                            uint64_t *clock, void *stream) {
  if (clock == nullptr || (n > 0 && (device == nullptr || host == nullptr || bytes == nullptr))) return FL_ERR_NULL;
  TransferArgs a;
  uint32_t blocks = 1;
  if (const int rc = FillSegments(a, blocks, n, device, host, bytes, slice_bytes)) return rc;
  a.clock = clock;
  FL_LAUNCH(TransferKernel<false>, dim3(blocks), dim3(kThreads), 0, AsStream(stream), a);
  return LaunchStatus();
}

int fluidml_hip_transfer_out(int32_t n, void *const *host, const void *const *device, const size_t *bytes, size_t slice_bytes,
                             uint64_t *clock, uint64_t *elapsed, uint32_t *flags, uint32_t value, void *stream) {
  if (flags == nullptr || (elapsed != nullptr && clock == nullptr)) return FL_ERR_NULL;
  if (n > 0 && (device == nullptr || host == nullptr || bytes == nullptr)) return FL_ERR_NULL;
  TransferArgs a;
  uint32_t blocks = 1;
  if (const int rc = FillSegments(a, blocks, n, host, device, bytes, slice_bytes)) return rc;
  a.clock = clock;
  a.elapsed = elapsed;
  a.flags = flags;
  a.value = value;
  FL_LAUNCH(TransferKernel<true>, dim3(blocks), dim3(kThreads), 0, AsStream(stream), a);
  return LaunchStatus();
}

}  // extern "C"
