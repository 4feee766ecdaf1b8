// 3x3 convolutions with unit stride and group 1 against weights laid out once for the matrix cores.
// Reference: src/structure/kernel/kernel/conv.cpp:27-201 (ConvKernel::run, group == 1 branch :55-102; padded variant
// :230-280), the same operation as conv_halo.hip, which takes the weights as they stand in the graph.
//
// Every fp32 value enters as its three bf16 parts and the products run on v_mfma_f32_32x32x16_bf16 (fl_common.h: as
// close to the exact result as the fp32 instruction, at 2.2 times its rate); with the opt-in bf16 precision it enters
// as the one rounded value.  What bounds the kernel is then the matrix pipe (three parts) or the staging of the
// activations (one part), provided nothing else stands in the inner loop:
//   * the weights are packed when the plan goes onto the device: [32 filters][16 channels][tap][part][lane][8], one KiB
//     per part that a wave reads straight into its A operand, 16 bytes per lane, no LDS, no conversion.  The waves of a
//     workgroup own different filters, so nothing is read twice; a tap's 3 KiB serve TN x 6 products (768 cycles at
//     TN = 4), and the next two taps' loads are in flight;
//   * the input patch of 16 channels is split into its parts once per workgroup, on its way into LDS, where it lies as
//     [part][channel half][pixel][8 channels]: a lane's B operand is one 128-bit read at a per-lane base plus a
//     compile-time offset, consecutive pixels in consecutive 16-byte places, and a row of the patch serves all the
//     taps (3.8 conflict cycles per LDS instruction, reads and writes of 16 bytes per lane together);
//   * per chunk of 16 channels one barrier, TN x 54 products per wave; LDS is double buffered and the next chunk's
//     loads are in flight across the products;
//   * the loads that run ahead are held in their place by scheduling barriers (the compiler moves them down to their use), those of
//     the patch one by one between the products: sixteen in a row hold up the wave at the address unit, and its products behind
//     them (one part, 8 x 512 x 28^2 -> 512: 51.5 -> 43.7 us, of 30 that the products alone take; three parts 160 -> 156);
//   * one part, where a chunk's products take 0.5 us and one or two workgroups of a few chunks share a compute unit: two chunks
//     of activations and 17 taps of weights in flight, the conversion of the next chunk between the products (8 x 512 x 14^2 ->
//     512: 27 -> 22 us before the loads were spread).  With more workgroups per compute unit those fill the waits, and the
//     registers and the longer start cost more (8 x 64 x 224^2 -> 64: 54 us with one chunk ahead, 60 with two);
//   * few tiles: the channels of a tile go to several workgroups, whose partial tiles meet in the stream's workspace and
//     are added in split order by the wave that arrives last.
// Measured against conv_halo.hip, bias and ReLU included (us; TFLOP/s of the convolution's own operations):
//   images x channels x size -> filters        fp32 before -> now            bf16 before -> now
//   8 x  64 x 224^2 ->  64                     289 -> 161 (184)               95 -> 59 (502)
//   8 x 128 x 112^2 -> 128                     286 -> 154 (192)               87 -> 49 (603)
//   8 x 256 x  56^2 -> 256                     290 -> 150 (197)              105 -> 43 (688)
//   8 x 512 x  28^2 -> 512                     324 -> 156 (190)              108 -> 43 (688)
//   8 x 512 x  14^2 -> 512                      92 ->  50 (147)               35 -> 21 (352)
//   1 x 256 x  56^2 -> 256                      52 ->  30 (123)               23 -> 15 (247)
//   4 x 256 x  37^2 -> 256                     156 ->  46 (142)              106 -> 17 (384)
// A 2 x 2 pool behind the chain is taken in the epilogue, where neighbouring lanes hold whole windows: a quarter of the result
// is written and nothing read back (us, convolution and pool): 8 x 64 x 224^2 fp32 166 + 18 -> 162, bf16 70 + 18 -> 53;
// 8 x 256 x 56^2 fp32 158 + 6 -> 153; the five pools of VGG-16 at batch 8 43 -> 0 altogether.
// (the tiles of 56^2 images are seven eighths full, those of 28^2 and 14^2 ones 77 %: at 56^2 and 28^2 the pipes do 225 and 248 of the 287
// TFLOP/s that the instructions reach alone)
#include <algorithm>

#include "fl_common.h"

namespace fl {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 16;   // input channels per chunk
constexpr int kCols = 16;    // output columns of a workgroup's tile
constexpr int kPatchCols = kCols + 2;
// Taps whose weights are in flight while DEPTH chunks of activations are: one fewer than there are places for them, and the places
// divide the taps of DEPTH chunks.
constexpr int Ahead(int depth) { return depth == 2 ? 17 : 2; }
constexpr int kMostAhead = Ahead(2);

struct PartsArgs {
  int32_t C, H, W, F, OH, OW;
  int32_t ph, pw;
  int32_t chunks, ftiles;  // 16-channel chunks, 32-filter tiles
  int32_t sXn, sXc, sXh, sXw;
  int32_t sOn, sOf, sOh, sOw;
  uint32_t tiles_h, tiles_w, groups_f, tiles_pix;  // groups_f: workgroups along the filters
  uint32_t n_splits;
  int32_t chunks_per_split;
  int32_t weight_major;  // consecutive workgroups share weights (else: the patch)
  int32_t pooled;        // the result is the maximum of each 2 x 2 pixels (the strides are the pooled tensor's)
  const float *bias;
  int32_t sB;
  float *partials;
  uint32_t *counters;
  fl_ew_program chain;
};

// WF waves along the filters (32 each), 4 / WF along the rows; a wave owns TN tiles of 2 rows x 16 columns.
// RAGGED: the channels do not come in sixteens; the missing ones read as zero (and are zero in the packed weights).
// POOLS: the launch may be a pooled one; see Launch.
// DEPTH: chunks of activations in flight; 2 with one part, up to two workgroups per compute unit (see above) and a few chunks each (see Launch).
// SPLITS: the launch may have its channels split.  With one part and more than two workgroups per compute unit none has, and the
// exchange's registers would leave two of those a compute unit for three, or spill (bf16, bias and ReLU, us, with the exchange and
// without it: 8 x 64 x 224^2 -> 64 61 and 59, pooled 56.5 and 53, 8 x 128 x 112^2 -> 128 50.2 and 49.4; without a chain 2 x 96 x 150^2 -> 256 34
// and 31, 3 x 64 x 112^2 -> 256 27 and 23, but 784 workgroups, of which three on each compute unit leave sixteen over, 1 to 3 % longer,
// 8 x 128 x 112^2 -> 128 44.6 and 46).
template <int PARTS, int WF, int TN, bool RAGGED, bool POOLS, int DEPTH, bool SPLITS>
__global__ __launch_bounds__(kThreads, 2) void ConvPartsKernel(float *out, const float *in, const u32x4 *packed, PartsArgs p) {
  // (no __restrict__: loads of memory known to be constant move freely, and the compiler sinks the ones that are
  // requested ahead of time down to their first use; these keep their place between the scheduling barriers below)
  constexpr int kRows = 2 * TN * (4 / WF);
  constexpr int kPix = (kRows + 2) * kPatchCols;
  constexpr int kItems = 2 * kPix;  // (channel half, pixel): eight channels each
  constexpr int kPer = (kItems + kThreads - 1) / kThreads;
  constexpr int kAhead = Ahead(DEPTH), kSlots = kAhead + 1;
  __shared__ u32x4 lds[2 * PARTS * kItems];
  __shared__ uint32_t tiny_inputs;  // (BadSum)
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int lrow = lane % 32, half = lane / 32;
  const int wf = wave % WF, wp = wave / WF;

  // Workgroups are dealt round-robin to the 8 XCDs: give each a contiguous run of ids.
  const uint32_t n = gridDim.x, q = n / 8, r = n % 8, xcd = blockIdx.x % 8;
  uint32_t id = xcd * q + min(xcd, r) + blockIdx.x / 8;
  uint32_t group, split, pix;
  if (p.weight_major) {
    pix = id % p.tiles_pix, id /= p.tiles_pix;
    group = id % p.groups_f, split = id / p.groups_f;
  } else {
    group = id % p.groups_f, id /= p.groups_f;
    split = id % p.n_splits, pix = id / p.n_splits;
  }
  const uint32_t tile_id = pix * p.groups_f + group;
  const int ow0 = static_cast<int>(pix % p.tiles_w) * kCols;
  const int oh0 = static_cast<int>(pix / p.tiles_w % p.tiles_h) * kRows;
  const uint32_t img = pix / p.tiles_w / p.tiles_h;
  const int ftile = static_cast<int>(group) * WF + wf;
  const int c_first = static_cast<int>(split) * p.chunks_per_split;
  const int c_end = min(p.chunks, c_first + p.chunks_per_split);

  // what this thread stages per chunk
  const float *image = in + static_cast<int64_t>(img) * p.sXn;
  uint32_t x_at[kPer];  // bytes
  bool x_ok[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int i = tid + t * kThreads;
    const int h = i / kPix, px = i % kPix;
    const int ih = oh0 - p.ph + px / kPatchCols, iw = ow0 - p.pw + px % kPatchCols;
    x_ok[t] = i < kItems && static_cast<uint32_t>(ih) < static_cast<uint32_t>(p.H) &&
              static_cast<uint32_t>(iw) < static_cast<uint32_t>(p.W);
    x_at[t] = x_ok[t] ? 4u * (ih * p.sXh + iw * p.sXw + (RAGGED ? 0 : 8 * h * p.sXc)) : 0u;
  }
  float xr[DEPTH][kPer][8];
  uint32_t tiny_key = 0xffffffffu;
  if (PARTS == 3 && tid == 0) tiny_inputs = 0;
  // value v of this thread's of chunk c: channel v % 8 of item v / 8
  auto load_value = [&](int c, auto set_c, auto value_c) {
    constexpr int S = decltype(set_c)::value, t = decltype(value_c)::value / 8, e = decltype(value_c)::value % 8;
    if constexpr (RAGGED) {
      const int c8 = c * kChunk + 8 * ((tid + t * kThreads) / kPix);
      xr[S][t][e] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(image) +
                                                     (4u * min(c8 + e, p.C - 1) * p.sXc + x_at[t]));
    } else {
      const char *plane = reinterpret_cast<const char *>(image + (static_cast<int64_t>(c) * kChunk + e) * p.sXc);
      xr[S][t][e] = *reinterpret_cast<const float *>(plane + x_at[t]);
    }
  };
  auto store_item = [&](int c, int buf, auto set_c, int t) {
    constexpr int S = decltype(set_c)::value;
    const int i = tid + t * kThreads;
    if (i < kItems) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool ok = x_ok[t] && (!RAGGED || c * kChunk + 8 * (i / kPix) + e < p.C);
        x[e] = ok ? xr[S][t][e] : 0.0f;
      }
      if constexpr (PARTS == 3) tiny_key = TinyKey(tiny_key, x);
      u32x4 parts[PARTS];
      SplitParts<PARTS>(x, parts);
#pragma unroll
      for (int s = 0; s < PARTS; ++s) lds[(buf * PARTS + s) * kItems + i] = parts[s];
    }
  };

  // the weights of this wave, a linear stream of one KiB per part and tap
  const u32x4 *a_src = packed + (static_cast<int64_t>(min(ftile, p.ftiles - 1)) * p.chunks + c_first) * (9 * PARTS * 64) + lane;
  u32x4 a[kSlots][PARTS];
  auto load_a = [&](int tap, auto slot_c) {
#pragma unroll
    for (int s = 0; s < PARTS; ++s) a[decltype(slot_c)::value][s] = a_src[(tap * PARTS + s) * 64];
  };

  // three parts: the leading products in acc, the others, a 256th of them at most, in low
  floatx16 acc[TN], low[PARTS == 3 ? TN : 1];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[j][e] = low[PARTS == 3 ? j : 0][e] = 0.0f;
  const int py = wp * 2 * TN + lrow / 16, px = lrow % 16;
  const int b_base = half * kPix + py * kPatchCols + px;

  // (without a condition, so that the compiler can count the loads in flight: past the end the last chunk again)
  StaticFor<DEPTH>([&](auto d) {
    StaticFor<8 * kPer>([&](auto v) { load_value(min(c_first + decltype(d)::value, c_end - 1), d, v); });
  });
  StaticFor<kAhead>([&](auto t) { load_a(decltype(t)::value, t); });
#pragma unroll
  for (int t = 0; t < kPer; ++t) store_item(c_first, 0, std::integral_constant<int, 0>{}, t);
  __syncthreads();
  // Chunk c: its patch lies in LDS buffer (c - c_first) % 2, the next one's is in the registers of set (c + 1 - c_first) % DEPTH.
  auto chunk = [&](int c, auto idx_c) __attribute__((always_inline)) {
    constexpr int I = decltype(idx_c)::value;
    const int buf = DEPTH == 1 ? (c - c_first) & 1 : I;
    const u32x4 *xs = lds + buf * PARTS * kItems + b_base;
    u32x4 b[2][PARTS];  // operand of the current tile and tap, and of the next
    auto load_b = [&](auto step_c) {
      constexpr int step = decltype(step_c)::value, tap = step / TN, j = step % TN;
#pragma unroll
      for (int s = 0; s < PARTS; ++s) b[step % 2][s] = xs[s * kItems + (2 * j + tap / 3) * kPatchCols + tap % 3];
    };
    load_b(std::integral_constant<int, 0>{});
    const int c_load = min(c + DEPTH, c_end - 1);
    StaticFor<9 * TN>([&](auto step_c) {
      constexpr int step = decltype(step_c)::value, tap = step / TN, j = step % TN, place = I * 9 + tap;
      // (runs kAhead taps past this wave's chunks at the end: other weights, or the padding behind the last ones)
      if constexpr (j == 0) load_a(tap + kAhead, std::integral_constant<int, (place + kAhead) % kSlots>{});
      if constexpr (step + 1 < 9 * TN) load_b(std::integral_constant<int, step + 1>{});
      // the loads of the patch one by one: a wave that issues them in a row waits for the address unit, and its products behind it
      constexpr int kLoadSteps = DEPTH == 1 ? 4 * TN : 9 * TN;
      StaticFor<8 * kPer>([&](auto v) {
        if constexpr (step == v * kLoadSteps / (8 * kPer)) load_value(c_load, std::integral_constant<int, I % DEPTH>{}, v);
      });
      // nothing moves across: the compiler otherwise sinks all kinds of loads down to their first use
      __builtin_amdgcn_sched_barrier(0);
      MfmaParts<PARTS>(a[place % kSlots], b[step % 2], acc[j], low[PARTS == 3 ? j : 0]);
      // the next chunk on its way into LDS between the products of the last third of the taps, where nobody else fills the pipe
      if constexpr (DEPTH == 2) {
        StaticFor<kPer>([&](auto t) {
          if constexpr (step == 6 * TN + t * 3 * TN / kPer) store_item(min(c + 1, c_end - 1), buf ^ 1, std::integral_constant<int, 1 - I>{}, t);
        });
      }
    });
    if constexpr (DEPTH == 1) {
      if (c + 1 < c_end) StaticFor<kPer>([&](auto t) { store_item(c + 1, buf ^ 1, std::integral_constant<int, 0>{}, t); });
    }
    a_src += 9 * PARTS * 64;
    // one barrier per chunk: the buffer written here was last read in the previous chunk, and every wave passed the
    // previous barrier only after finishing that read
    __syncthreads();
  };
  for (int c = c_first;;) {  // (every workgroup has a chunk)
    chunk(c, std::integral_constant<int, 0>{});
    if (++c >= c_end) break;
    if constexpr (DEPTH == 2) {
      chunk(c, std::integral_constant<int, 1>{});
      if (++c >= c_end) break;
    }
  }

  if constexpr (PARTS == 3) {
    if (tiny_key < kTinyKey) tiny_inputs = 1;
    __syncthreads();
    const bool tiny = tiny_inputs != 0;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] += low[j][e];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) bad |= BadSum(acc[j][e], tiny);
    if (__any(bad)) {
      // the same channels once more with the fp32 instruction, operands straight from memory (filters and channels that do
      // not exist are zero in the packed weights)
      const uint16_t *w_src = reinterpret_cast<const uint16_t *>(packed) +
                              static_cast<int64_t>(min(ftile, p.ftiles - 1)) * p.chunks * (9 * PARTS * 512) + lrow * 8;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
      for (int c0 = c_first * kChunk; c0 < min(p.C, c_end * kChunk); c0 += 2) {
        const int ch = c0 + half;
        for (int tap = 0; tap < 9; ++tap) {
          const float w = JoinParts(w_src + (ch / 16 * 9 + tap) * (PARTS * 512) + ch % 16 / 8 * 256 + ch % 8, 512);
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int ih = oh0 + py + 2 * j - p.ph + tap / 3, iw = ow0 + px - p.pw + tap % 3;
            const bool inside = ch < p.C && static_cast<uint32_t>(ih) < static_cast<uint32_t>(p.H) &&
                                static_cast<uint32_t>(iw) < static_cast<uint32_t>(p.W);
            const float x = inside ? image[static_cast<int64_t>(ch) * p.sXc + ih * p.sXh + iw * p.sXw] : 0.0f;
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w, x, acc[j], 0, 0, 0);
          }
        }
      }
    }
  }

  // ---- channels split over workgroups: combine the partial tiles ----------------------------------------------
  // The hand-off of conv_halo.hip: device-coherent stores, the explicit wait, one arrival per wave, loads behind the
  // branch on the returned count.  Sums in split order, so the result does not depend on who arrives last.
  if (SPLITS && p.n_splits > 1) {
    const uint32_t n_splits = p.n_splits, slot = tile_id * 4 + wave;
    float *all = p.partials + static_cast<size_t>(slot) * n_splits * (TN * 1024);
    float *mine = all + split * (TN * 1024);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        __hip_atomic_store(mine + j * 1024 + e * 64 + lane, acc[j][e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t arrived = 0;
    if (lane == 0) arrived = __hip_atomic_fetch_add(&p.counters[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    arrived = __shfl(arrived, 0);
    if (arrived != n_splits - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // compiler ordering only: no instruction on gfx9
    if (lane == 0) __hip_atomic_store(&p.counters[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
    constexpr uint32_t kTogether = TN == 2 ? 4 : 2;  // splits whose loads are in flight together
    for (uint32_t z0 = 0; z0 < n_splits; z0 += kTogether) {
      float part[kTogether][TN][16];
#pragma unroll
      for (uint32_t u = 0; u < kTogether; ++u) {
        const uint32_t z = z0 + u < n_splits ? z0 + u : z0;  // repeats a valid slot, ignored below
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            part[u][j][e] = __hip_atomic_load(all + static_cast<size_t>(z) * (TN * 1024) + j * 1024 + e * 64 + lane, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
          }
      }
#pragma unroll
      for (uint32_t u = 0; u < kTogether; ++u) {
        if (z0 + u < n_splits) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] += part[u][j][e];
        }
      }
    }
  }

  // ---- epilogue: bias, elementwise chain, stores -------------------------------------------------------------
  float bias_v[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int f = ftile * 32 + (e / 4) * 8 + half * 4 + (e % 4);
    bias_v[e] = p.bias != nullptr && f < p.F ? p.bias[f * p.sB] : 0.0f;
  }
  StaticFor<TN>([&](auto j_c) {
    constexpr int j = decltype(j_c)::value;
    const int oh = oh0 + py + 2 * j, ow = ow0 + px;
    float vals[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) vals[e] = acc[j][e] + bias_v[e];
    if (p.chain.n != 0) RunChainBlock<16>(p.chain, vals);
    if (POOLS && p.pooled != 0) {
      // The four pixels of a window are a lane's neighbour and the two in the next row of sixteen.  Each exchange halves the
      // filters a lane goes on with instead of computing every maximum twice, and all lanes store in the end: lane r of
      // the upper (0) and the lower row (1), column parity c, has the filters e = 4 k + 2 r + c.
      float rows[8], four[4];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // (e = 4 (k / 2) + k % 2 stays with the upper row, the one two further with the lower)
        const int e = k / 2 * 4 + k % 2;
        const uint32_t a = __builtin_bit_cast(uint32_t, vals[e]), b = __builtin_bit_cast(uint32_t, vals[e + 2]);
        const auto both = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        const uint32_t first = both[0], second = both[1];
        rows[k] = MaximumF(__builtin_bit_cast(float, first), __builtin_bit_cast(float, second));
      }
      const bool odd = (lane & 1) != 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float keep = odd ? rows[2 * k + 1] : rows[2 * k], give = odd ? rows[2 * k] : rows[2 * k + 1];
        four[k] = MaximumF(keep, DppMove<0xB1>(give));
      }
      // (an odd last row or column belongs to no window)
      const int row = oh / 2, col = ow / 2;
      if (row < p.OH / 2 && col < p.OW / 2) {
        float *dst = out + static_cast<int64_t>(img) * p.sOn + static_cast<int64_t>(row) * p.sOh + static_cast<int64_t>(col) * p.sOw;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int f = ftile * 32 + k * 8 + half * 4 + lrow / 16 * 2 + (lane & 1);
          if (f < p.F) dst[static_cast<int64_t>(f) * p.sOf] = four[k];
        }
      }
      return;
    }
    if (oh < p.OH && ow < p.OW) {
      float *dst = out + static_cast<int64_t>(img) * p.sOn + static_cast<int64_t>(oh) * p.sOh + static_cast<int64_t>(ow) * p.sOw;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int f = ftile * 32 + (e / 4) * 8 + half * 4 + (e % 4);
        if (f < p.F) dst[static_cast<int64_t>(f) * p.sOf] = vals[e];
      }
    }
  });
}

// One thread per (filter tile, chunk, tap, lane): eight weights, their parts, 16 bytes per part.
template <int PARTS>
__global__ __launch_bounds__(kThreads) void ConvPackKernel(u32x4 *__restrict__ packed, const float *__restrict__ w, int F, int C,
                                                           int chunks, uint32_t items, int sWf, int sWc, int sWh, int sWw) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= items) return;
  const int lane = i % 64;
  const uint32_t block = i / 64, tap = block % 9, chunk = block / 9 % chunks, ftile = block / 9 / chunks;
  const int f = ftile * 32 + lane % 32, c0 = chunk * kChunk + 8 * (lane / 32);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool ok = f < F && c0 + e < C;
    x[e] = ok ? w[static_cast<int64_t>(f) * sWf + static_cast<int64_t>(c0 + e) * sWc + tap / 3 * sWh + tap % 3 * sWw] : 0.0f;
  }
  u32x4 parts[PARTS];
  SplitParts<PARTS>(x, parts);
#pragma unroll
  for (int s = 0; s < PARTS; ++s) packed[(static_cast<int64_t>(block) * PARTS + s) * 64 + lane] = parts[s];
}

int64_t Ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// How a convolution is cut up: WF, TN, splits.
struct Cut {
  int wf = 4, tn = 4;
  int64_t splits = 1;
  double cost = 0;
};
int64_t TilesPix(const PartsArgs &p, int64_t images, const Cut &c) {
  return images * Ceil(p.OH, 2 * c.tn * (4 / c.wf)) * Ceil(p.OW, kCols);
}
Cut ChooseCut(const PartsArgs &p, int64_t images, int parts) {
  // A workgroup's time goes with its chunks and TN (the matrix pipe is what it waits for), a launch's with the number
  // of workgroups a compute unit gets; a split adds the exchange of the partial tiles, which the wave that arrives last takes in,
  // eight tiles of 2 x 16 pixels at a time.  In microseconds.
  const double chunk_us = parts == 3 ? 0.9 : 0.3, fixed_us = 3.0;
  // Eight partial tiles cost 1 us where few workgroups exchange theirs, and with three parts 2 us from about 64 workgroups on (us,
  // TN = 2: 1 x 512 x 14^2 -> 512 in 16 splits, 256 workgroups, 24.7, in 11 21.4, in 8 21.2, in 4 25.9; 1 x 128 x 28^2 -> 256 in 8 18.6, in 4
  // 15.0; but 1 x 512 x 16^2 -> 64 in 16 splits, 32 workgroups, 17.9, in 8 19.4; 1 x 192 x 16^2 -> 64 in 12 14.2, in 4 15.7).  Ten are
  // taken for eight (8 x 384 x 10^2 -> 256 in five 24.0, in four 25.2).  The first eight cost 1 us with up to 64 filters, where a chunk's
  // patch has twice the rows and not splitting is dearer (1 x 48 x 56^2 -> 64 in three 12.3, in one 13.2; 4 x 48 x 14^2 -> 512 13.4, 11.9).
  // One part keeps 1 us throughout (1 x 256 x 28^2 -> 512 would take a sixth less with other cuts).
  auto exchange_us = [&](const Cut &c, int64_t workgroups) {
    const int64_t partials = c.splits * c.tn, rounds = partials <= 10 ? 1 : Ceil(partials, 8);
    if (parts == 1 || workgroups <= 64) return 2.0 + Ceil(partials, 8);
    return 2.0 + (rounds == 1 && c.wf == 2 ? 1.0 : 2.0 * rounds);
  };
  Cut best;
  best.cost = 1e30;
  for (int tn : {4, 2}) {
    Cut c;
    c.wf = p.F > 64 ? 4 : 2;
    c.tn = tn;
    const int64_t tiles = TilesPix(p, images, c) * Ceil(p.ftiles, c.wf);
    for (int64_t s = 1; s <= std::min<int64_t>(p.chunks, 16); ++s) {
      if (s > 1 && tiles * 4 * tn * s > static_cast<int64_t>(kWorkspaceTiles)) break;
      const int64_t per = Ceil(p.chunks, s);
      c.splits = Ceil(p.chunks, per);
      if (c.splits != s) continue;
      c.cost = Ceil(tiles * s, 256) * (fixed_us + per * tn * chunk_us) + (s > 1 ? exchange_us(c, tiles * s) : 0.0);
      if (c.cost < best.cost) best = c;
    }
  }
  return best;
}

// bf16 launches of more than two workgroups per compute unit have a kernel without the pooled epilogue, whose condition costs those
// without a pool up to 1 % (8 x 64 x 224^2 -> 64 58.9 us without it, 59.4 with it; 8 x 256 x 56^2 -> 512 84.3, 84.6).  The others share one,
// because a kernel that has not run just before starts with its instructions missing (VGG-16 of one image with two kernels throughout
// 438 us, with one 436; bf16 401, 398).
template <int PARTS, int WF, int TN>
void Launch(const PartsArgs &p, uint32_t grid, float *out, const float *in, const u32x4 *packed, hipStream_t s) {
#define FL_PARTS_AS(RAGGED_, POOLS_, DEPTH_, SPLITS_) \
  FL_LAUNCH((ConvPartsKernel<PARTS, WF, TN, RAGGED_, POOLS_, DEPTH_, SPLITS_>), dim3(grid), dim3(kThreads), 0, s, out, in, packed, p)
  if constexpr (PARTS == 1) {
    // (every launch that is split: its partial tiles fit the workspace)
    constexpr uint32_t kTwoPerUnit = 2 * 256;
    static_assert(kWorkspaceTiles <= kTwoPerUnit * 4 * TN, "a launch of more workgroups has no splits");
    if (grid <= kTwoPerUnit) {
      // Two chunks in flight from five chunks per workgroup on, from four where the channels are split and the weights take longer
      // to come: with fewer, the requests ahead are mostly for chunks that a workgroup does not have (bf16, us, one chunk ahead and two:
      // 1 chunk 3 x 16 x 79^2 -> 160 11.2, 13.1; 2 4 x 32 x 56^2 -> 128 7.6, 8.0; 4 8.7, 8.9; 5 9.4, 9.4; 6 10.1, 9.9; 8 11.4, 11.0; 16
      // 17.0, 15.5.  Split: 2 1 x 128 x 28^2 -> 512 13.9, 15.0; 3 3 x 192 x 14^2 -> 512 13.5, 14.3; 4 2 x 512 x 14^2 -> 512 19.3, 18.4, 1 x
      // 512 x 28^2 -> 256 19.0, 18.0, but 1 x 256 x 56^2 -> 128 12.0, 12.4; 6 1 x 384 x 28^2 -> 512 17.9, 16.6).
      const bool two = p.chunks_per_split >= (p.n_splits > 1 ? 4 : 5);
      if (p.C % kChunk != 0) {
        if (two) FL_PARTS_AS(true, true, 2, true);
        else FL_PARTS_AS(true, true, 1, true);
      } else {
        if (two) FL_PARTS_AS(false, true, 2, true);
        else FL_PARTS_AS(false, true, 1, true);
      }
      return;
    }
    if (p.C % kChunk != 0) {
      if (p.pooled) FL_PARTS_AS(true, true, 1, false);
      else FL_PARTS_AS(true, false, 1, false);
    } else {
      if (p.pooled) FL_PARTS_AS(false, true, 1, false);
      else FL_PARTS_AS(false, false, 1, false);
    }
  } else {
    if (p.C % kChunk != 0) FL_PARTS_AS(true, true, 1, true);
    else FL_PARTS_AS(false, true, 1, true);
  }
#undef FL_PARTS_AS
}

bool Fits(const fl_tensor *weights) {
  return weights->rank == 4 && weights->dtype == FL_FLOAT32 && weights->shape[2] == 3 && weights->shape[3] == 3 &&
         weights->shape[0] >= 32 && Numel(weights) <= 0x7fffffff;
}

}  // namespace
}  // namespace fl

extern "C" {

int fluidml_hip_conv3x3_packed_bytes(const fl_tensor *weights, int32_t parts, size_t *bytes) {
  using namespace fl;
  if (bytes == nullptr) return FL_ERR_NULL;
  *bytes = 0;
  FL_CHECK(CheckView(weights));
  if (parts != 1 && parts != 3) return FL_ERR_ATTR;
  if (!Fits(weights)) return FL_ERR_UNSUPPORTED;
  const int64_t taps = Ceil(weights->shape[0], 32) * Ceil(weights->shape[1], kChunk) * 9 + (parts == 1 ? kMostAhead : Ahead(1));
  *bytes = static_cast<size_t>(taps) * parts * 1024;
  return FL_OK;
}

int fluidml_hip_conv3x3_pack(const fl_tensor *weights, int32_t parts, void *packed, void *stream) {
  using namespace fl;
  if (packed == nullptr) return FL_ERR_NULL;
  size_t bytes = 0;
  FL_CHECK(fluidml_hip_conv3x3_packed_bytes(weights, parts, &bytes));
  if (!IsAligned(packed, 16)) return FL_ERR_ATTR;
  if (parts == 3) FL_CHECK(PartsCanCarry(weights, weights->shape[1] * 9, AsStream(stream)));
  const int F = static_cast<int>(weights->shape[0]), C = static_cast<int>(weights->shape[1]);
  const int chunks = static_cast<int>(Ceil(C, kChunk));
  const uint32_t items = static_cast<uint32_t>(Ceil(F, 32) * chunks * 9 * 64);
  const int s[4] = {static_cast<int>(weights->strides[0]), static_cast<int>(weights->strides[1]),
                    static_cast<int>(weights->strides[2]), static_cast<int>(weights->strides[3])};
  const dim3 grid((items + kThreads - 1) / kThreads);
  if (parts == 3) {
    FL_LAUNCH(ConvPackKernel<3>, grid, dim3(kThreads), 0, AsStream(stream), static_cast<u32x4 *>(packed),
              static_cast<const float *>(weights->base), F, C, chunks, items, s[0], s[1], s[2], s[3]);
  } else {
    FL_LAUNCH(ConvPackKernel<1>, grid, dim3(kThreads), 0, AsStream(stream), static_cast<u32x4 *>(packed),
              static_cast<const float *>(weights->base), F, C, chunks, items, s[0], s[1], s[2], s[3]);
  }
  return LaunchStatus();
}

static int PackedChain(const fl_tensor *in, const fl_tensor *weights, const void *packed, int32_t parts, const fl_tensor *bias,
                       const fl_tensor *out, const int64_t *pads, const fl_ew_program *chain, uint32_t flags, bool pooled,
                       void *stream) {
  using namespace fl;
  FL_CHECK(CheckChain(chain));
  FL_CHECK(CheckView(in));
  FL_CHECK(CheckView(weights));
  FL_CHECK(CheckView(out));
  if (packed == nullptr) return FL_ERR_NULL;
  if (!IsAligned(packed, 16)) return FL_ERR_ATTR;
  if (parts != 1 && parts != 3) return FL_ERR_ATTR;
  if (in->dtype != FL_FLOAT32 || weights->dtype != FL_FLOAT32 || out->dtype != FL_FLOAT32) return FL_ERR_DTYPE;
  if (in->rank != 4 || weights->rank != 4 || out->rank != 4) return FL_ERR_RANK;
  if (!Fits(weights)) return FL_ERR_UNSUPPORTED;
  const int64_t N = in->shape[0], C = in->shape[1], F = out->shape[1];
  if (out->shape[0] != N || weights->shape[0] != F || weights->shape[1] != C) return FL_ERR_SHAPE;
  int64_t extent[2];
  for (int d = 0; d < 2; ++d) {
    const int64_t before = pads ? pads[d] : 0, after = pads ? pads[d + 2] : 0;
    if (before < 0 || after < 0) return FL_ERR_ATTR;
    if (before > 0x3fffffff) return FL_ERR_TOO_LARGE;
    // (the whole output and nothing else: a smaller one would be a convolution with other strides or dilations, or a crop)
    extent[d] = in->shape[2 + d] + before + after - 2;
    if (out->shape[2 + d] != (pooled ? extent[d] / 2 : extent[d])) return FL_ERR_SHAPE;
  }
  if (Numel(in) > 0x7fffffff || N * F * extent[0] * extent[1] > 0x7fffffff) return FL_ERR_UNSUPPORTED;
  for (int d = 0; d < 4; ++d) {
    // (byte offsets inside an image are 32-bit)
    if (in->strides[d] < 0 || in->strides[d] * (in->shape[d] + kChunk) > 0x3fffffff || out->strides[d] > 0x7fffffff) return FL_ERR_UNSUPPORTED;
  }
  PartsArgs p;
  std::memset(&p, 0, sizeof(p));
  p.C = static_cast<int32_t>(C), p.H = static_cast<int32_t>(in->shape[2]), p.W = static_cast<int32_t>(in->shape[3]);
  p.F = static_cast<int32_t>(F), p.OH = static_cast<int32_t>(extent[0]), p.OW = static_cast<int32_t>(extent[1]);
  p.pooled = pooled ? 1 : 0;
  p.ph = pads ? static_cast<int32_t>(pads[0]) : 0, p.pw = pads ? static_cast<int32_t>(pads[1]) : 0;
  p.chunks = static_cast<int32_t>(Ceil(C, kChunk)), p.ftiles = static_cast<int32_t>(Ceil(F, 32));
  p.sXn = static_cast<int32_t>(in->strides[0]), p.sXc = static_cast<int32_t>(in->strides[1]);
  p.sXh = static_cast<int32_t>(in->strides[2]), p.sXw = static_cast<int32_t>(in->strides[3]);
  p.sOn = static_cast<int32_t>(out->strides[0]), p.sOf = static_cast<int32_t>(out->strides[1]);
  p.sOh = static_cast<int32_t>(out->strides[2]), p.sOw = static_cast<int32_t>(out->strides[3]);
  if (bias != nullptr) {
    FL_CHECK(CheckView(bias));
    if (bias->dtype != FL_FLOAT32) return FL_ERR_DTYPE;
    if (bias->rank != 1 || bias->shape[0] != F) return FL_ERR_SHAPE;
    p.bias = static_cast<const float *>(bias->base);
    p.sB = static_cast<int32_t>(bias->strides[0]);
  }
  if (chain != nullptr) p.chain = *chain;

  Cut cut = ChooseCut(p, N, parts);
  // the caller's own cut, as for the contractions: tile 1 = TN 2, 2 = TN 4, and the number of splits
  const uint32_t tile = (flags >> FL_CONTRACT_TILE_SHIFT) & 0xfu, forced = (flags >> FL_CONTRACT_SPLIT_SHIFT) & 0x3fu;
  if (tile > 2) return FL_ERR_ATTR;
  if (tile != 0) cut.tn = tile == 1 ? 2 : 4;
  if (forced != 0) cut.splits = std::min<int64_t>(forced, p.chunks);
  p.groups_f = static_cast<uint32_t>(Ceil(p.ftiles, cut.wf));
  p.tiles_h = static_cast<uint32_t>(Ceil(p.OH, 2 * cut.tn * (4 / cut.wf)));
  p.tiles_w = static_cast<uint32_t>(Ceil(p.OW, kCols));
  const int64_t tiles_pix = TilesPix(p, N, cut), tiles = tiles_pix * p.groups_f;
  if (cut.splits > 1 && tiles * 4 * cut.tn * cut.splits > static_cast<int64_t>(kWorkspaceTiles)) cut.splits = 1;
  StreamWorkspace *ws = cut.splits > 1 ? GetStreamWorkspace(AsStream(stream)) : nullptr;
  if (ws == nullptr) cut.splits = 1;
  if (tiles > 0x7fffffff) return FL_ERR_TOO_LARGE;
  p.tiles_pix = static_cast<uint32_t>(tiles_pix);
  p.chunks_per_split = static_cast<int32_t>(Ceil(p.chunks, cut.splits));
  p.n_splits = static_cast<uint32_t>(Ceil(p.chunks, p.chunks_per_split));
  if (ws != nullptr) p.partials = ws->partials, p.counters = ws->counters;
  p.weight_major = static_cast<int64_t>(p.ftiles) * p.chunks * 9 * parts * 1024 > Numel(in) * 4 ? 1 : 0;
  const uint32_t grid = static_cast<uint32_t>(tiles * p.n_splits);
  float *o = static_cast<float *>(out->base);
  const float *x = static_cast<const float *>(in->base);
  const u32x4 *w = static_cast<const u32x4 *>(packed);
  hipStream_t s = AsStream(stream);
#define FL_PARTS(PARTS_)                                            \
  do {                                                              \
    if (cut.wf == 4 && cut.tn == 4) Launch<PARTS_, 4, 4>(p, grid, o, x, w, s); \
    else if (cut.wf == 4) Launch<PARTS_, 4, 2>(p, grid, o, x, w, s);           \
    else if (cut.tn == 4) Launch<PARTS_, 2, 4>(p, grid, o, x, w, s);           \
    else Launch<PARTS_, 2, 2>(p, grid, o, x, w, s);                            \
  } while (0)
  if (parts == 3) FL_PARTS(3);
  else FL_PARTS(1);
#undef FL_PARTS
  NotePackedParts(parts);
  return LaunchStatus();
}

int fluidml_hip_conv3x3_packed_chain(const fl_tensor *in, const fl_tensor *weights, const void *packed, int32_t parts,
                                     const fl_tensor *bias, const fl_tensor *out, const int64_t *pads,
                                     const fl_ew_program *chain, uint32_t flags, void *stream) {
  return PackedChain(in, weights, packed, parts, bias, out, pads, chain, flags, false, stream);
}

int fluidml_hip_conv3x3_packed_chain_pool(const fl_tensor *in, const fl_tensor *weights, const void *packed, int32_t parts,
                                          const fl_tensor *bias, const fl_tensor *out, const int64_t *pads,
                                          const fl_ew_program *chain, uint32_t flags, void *stream) {
  return PackedChain(in, weights, packed, parts, bias, out, pads, chain, flags, true, stream);
}

}  // extern "C"
