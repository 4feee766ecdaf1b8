// Copies between pinned host memory and HBM for the arguments of one run: several arguments per launch, and on the
// way out a flag in host memory per slice, so that the host can take a slice over while later ones still travel.
#include <algorithm>

#include "fl_common.h"

using namespace fl;

namespace {

constexpr uint32_t kThreads = 256;

struct Segment {
  const uint4 *src;
  uint4 *dst;
  uint32_t n16;          // 16-byte items; both sides are padded to whole items
  uint32_t first_piece;
  uint32_t first_slice;
};

constexpr uint32_t kPiece16 = 4 * kThreads;  // 16-byte items of a piece: what a block has in flight at a time (16 KiB)
// Blocks of the way out.  They take the pieces in order, so that the slices are complete one after the other and the host
// takes one over while the next ones travel.  With a block per slice all of them were complete only towards the end (51.5 MB
// out of GPT-NeoX: the link busy for 0.94 ms, the host done 0.26 ms after it), and dealing the pieces out beforehand leaves
// the slices waiting for the slowest block (the link does not serve them evenly: 0.1 ms).
constexpr uint32_t kOutBlocks = 64;

struct TransferArgs {
  uint32_t n_segments, n_pieces;
  uint32_t pieces_per_slice;
  uint64_t *clock;    // device: latest end of an inbound launch since the last outbound one
  uint32_t *flags;    // host: one per slice (outbound only)
  uint32_t *arrived;  // device: pieces of each slice that have been acknowledged, zero between launches (outbound only)
  uint32_t *next;     // device: the next piece nobody has taken, zero between launches (outbound only)
  uint64_t *elapsed;  // host: ticks between *clock and the start of the outbound launch
  uint32_t value;
  Segment segments[FL_MAX_TRANSFER_SEGMENTS];
};

// The time of the replays, for the host.  By the block that takes piece 0, before it counts that piece: the flag of the
// first slice says then that it has been written (a block that only carried the first index could start after all others
// had raised every flag, and the host would read the previous run's time).
__device__ __forceinline__ void LeaveElapsed(const TransferArgs &args) {
  if (threadIdx.x != 0 || args.elapsed == nullptr) return;
  const uint64_t now = wall_clock64();
  const uint64_t since = *args.clock;
  *args.clock = 0;
  *args.elapsed = since != 0 && now > since ? now - since : 0;
}

// Bound by the link (about 55 GB/s each way: 51.5 MB take 0.93 ms, the copy engine needs 0.91) and, for the few
// kilobytes of a text request, by the launch (an asynchronous copy of pageable memory costs 13 us in and 21 us out per
// argument and a stream wait 11 us; one launch plus a polled flag 6 us).  Four 16-byte loads are in flight per lane.
template <bool OUTBOUND>
__global__ __launch_bounds__(kThreads) void TransferKernel(TransferArgs args) {
  __shared__ uint32_t taken;
  const bool in_turn = OUTBOUND && args.n_pieces > gridDim.x;
  uint32_t s = 0, piece = blockIdx.x;
  for (;;) {
    if (in_turn) {
      if (threadIdx.x == 0) {
        taken = __hip_atomic_fetch_add(args.next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // every block asks once in vain, and the last one to do so puts the counter back
        if (taken == args.n_pieces + gridDim.x - 1) __hip_atomic_store(args.next, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      piece = taken;
    }
    if (piece >= args.n_pieces) break;
    if (OUTBOUND && piece == 0) LeaveElapsed(args);
    while (s + 1 < args.n_segments && piece >= args.segments[s + 1].first_piece) ++s;
    const Segment g = args.segments[s];
    const uint32_t local = piece - g.first_piece, i = local * kPiece16 + threadIdx.x;
    uint4 v[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      if (i + j * kThreads < g.n16) v[j] = g.src[i + j * kThreads];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      if (i + j * kThreads < g.n16) g.dst[i + j * kThreads] = v[j];
    }
    if (OUTBOUND) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores have been acknowledged
      __syncthreads();
      if (threadIdx.x == 0) {
        // the block that acknowledges a slice's last piece raises its flag: every other one has waited for its own
        const uint32_t slice = g.first_slice + local / args.pieces_per_slice;
        const uint32_t begin = local / args.pieces_per_slice * args.pieces_per_slice;
        const uint32_t pieces = min(args.pieces_per_slice, (g.n16 + kPiece16 - 1) / kPiece16 - begin);
        const uint32_t before = __hip_atomic_fetch_add(args.arrived + slice, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_SYSTEM);
        if (before == pieces - 1) {
          __hip_atomic_store(args.arrived + slice, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(args.flags + slice, args.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
      }
    }
    if (!in_turn) break;  // (a block per piece)
  }
  if (OUTBOUND) {
    if (args.n_pieces != 0) return;
    LeaveElapsed(args);  // (one block, nothing but the flag)
    if (threadIdx.x == 0) __hip_atomic_store(args.flags, args.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(reinterpret_cast<unsigned long long *>(args.clock), static_cast<unsigned long long>(wall_clock64()));
}

int FillSegments(TransferArgs &a, int32_t n, void *const *dst, const void *const *src, const size_t *bytes, size_t slice_bytes) {
  if (n < 0 || n > FL_MAX_TRANSFER_SEGMENTS) return FL_ERR_ATTR;
  if (slice_bytes == 0 || slice_bytes % (kPiece16 * 16) != 0) return FL_ERR_ATTR;
  std::memset(&a, 0, sizeof(a));
  a.pieces_per_slice = static_cast<uint32_t>(slice_bytes / (kPiece16 * 16));
  uint64_t pieces = 0, slices = 0;
  for (int32_t i = 0; i < n; ++i) {
    if (dst[i] == nullptr || src[i] == nullptr) return FL_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(dst[i]) | reinterpret_cast<uintptr_t>(src[i])) % 16 != 0) return FL_ERR_ATTR;
    if (bytes[i] == 0) return FL_ERR_SHAPE;
    if ((bytes[i] + 15) / 16 > 0x7fffffffu) return FL_ERR_TOO_LARGE;
    Segment &g = a.segments[a.n_segments++];
    g.src = static_cast<const uint4 *>(src[i]);
    g.dst = static_cast<uint4 *>(dst[i]);
    g.n16 = static_cast<uint32_t>((bytes[i] + 15) / 16);
    g.first_piece = static_cast<uint32_t>(pieces);
    g.first_slice = static_cast<uint32_t>(slices);
    pieces += (g.n16 + kPiece16 - 1) / kPiece16;
    slices += (bytes[i] + slice_bytes - 1) / slice_bytes;
    if (pieces > 0x7fffffffu) return FL_ERR_TOO_LARGE;
  }
  a.n_pieces = static_cast<uint32_t>(pieces);
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

int fluidml_hip_transfer_in(int32_t n, void *const *device, const void *const *host, const size_t *bytes, uint64_t *clock, void *stream) {
  if (clock == nullptr || (n > 0 && (device == nullptr || host == nullptr || bytes == nullptr))) return FL_ERR_NULL;
  TransferArgs a;
  if (const int rc = FillSegments(a, n, device, host, bytes, kPiece16 * 16)) return rc;
  a.clock = clock;
  FL_LAUNCH(TransferKernel<false>, dim3(std::max(a.n_pieces, 1u)), dim3(kThreads), 0, AsStream(stream), a);
  return LaunchStatus();
}

int fluidml_hip_transfer_out(int32_t n, void *const *host, const void *const *device, const size_t *bytes, size_t slice_bytes,
                             uint64_t *clock, uint64_t *elapsed, uint32_t *flags, uint32_t *counters, uint32_t value, void *stream) {
  if (flags == nullptr || counters == nullptr || (elapsed != nullptr && clock == nullptr)) return FL_ERR_NULL;
  if (n > 0 && (device == nullptr || host == nullptr || bytes == nullptr)) return FL_ERR_NULL;
  TransferArgs a;
  if (const int rc = FillSegments(a, n, host, device, bytes, slice_bytes)) return rc;
  a.clock = clock;
  a.elapsed = elapsed;
  a.flags = flags;
  a.next = counters;
  a.arrived = counters + 1;
  a.value = value;
  FL_LAUNCH(TransferKernel<true>, dim3(std::clamp(a.n_pieces, 1u, kOutBlocks)), dim3(kThreads), 0, AsStream(stream), a);
  return LaunchStatus();
}

}  // extern "C"
