// Contractions against constant weights laid out once for the matrix cores: MatMul and Gemm with every epilogue of the
// tiled kernel in matmul.hip (bias, elementwise chain, addends, deferred LayerNormalization, siblings, K split over
// workgroups).  Reference: src/structure/kernel/kernel/matmul.cpp:28-59, gemm.cpp:39-182.
//
// Every fp32 value enters as its three bf16 parts (fl_common.h: closer to the exact result than the fp32 instruction, 192
// instead of 512 matrix cycles per 32x32x16 products); with the opt-in bf16 precision it enters as the one rounded value.
//   * The weights are packed when the plan goes onto the device, [32 columns][16 k][part][lane][8]: one KiB per part that
//     a wave reads straight into its B operand, 16 bytes per lane, without LDS or conversion.  A wave owns 32 columns, so
//     nothing is read twice inside a workgroup.
//   * The rows of A are split into their parts once per workgroup, on their way from registers into LDS, where they lie
//     as [part][k / 8][row][8]: a lane's A operand is one 128-bit read, 32 consecutive places per half wave.  The places
//     of one k / 8 are padded, so that the writes (consecutive lanes: consecutive k of a row) spread over the banks.
//   * The loads of a chunk leave between the products of the chunk DEPTH before it, a few per product (three parts): in a row behind
//     the barrier, sixteen cycles of the address unit each, they held up all waves and the products behind them (512 x 3072 x 768
//     22.4 -> 19.9 us, 256 x 3072 x 768 16.6 -> 14.6, 512 x 768 x 3072 25.0 -> 23.0, 256 x 50304 x 512 100 -> 93).
//   * WN waves side by side times KS = 4 / WN slices of K; two steps of 16 k per wave and chunk, one barrier per chunk, LDS
//     double buffered, DEPTH chunks of both operands in flight in registers: a launch of a small transformer has a few
//     chunks per workgroup and is a chain of trips to memory otherwise.
//   * The K slices of a workgroup meet in LDS and every wave finishes an equal share of the tile (a quarter of it where
//     four waves share one 32x32 tile); splits of K over workgroups meet in the stream's workspace, share by share.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>

#include "fl_common.h"
#include "matmul_args.h"

namespace fl {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// four floats next to each other, at any float's address, one access
struct __attribute__((packed, aligned(4))) FourFloats {
  float v[4];
};

constexpr int kPackThreads = 256;
constexpr int kSteps = 2;  // steps of 16 k per wave and chunk

template <int PARTS, int TM, int WN, int KS, int DEPTH, int EXTRA>
__global__ __launch_bounds__(64 * WN *KS, 2) void MatmulPartsKernel(float *C_, const float *A, MatmulArgs p) {
  // (no __restrict__ on what is loaded ahead of its use: see conv_parts.hip)
  constexpr int kWaves = WN * KS, kThreads = 64 * kWaves;
  constexpr int BM = 32 * TM, BN = 32 * WN;
  constexpr int kChunkSteps = kSteps * KS;          // steps of 16 k per chunk of the workgroup
  constexpr int BK = 16 * kChunkSteps;
  constexpr int kK8 = BK / 8;
  // 16-byte places per k / 8: sixteen lanes write kK8 values of k / 8 in 16 / kK8 rows, to sixteen different places
  constexpr int kPitch = BM + (kK8 >= 16 ? 1 : 16 / kK8);
  constexpr int kItems = BM * kK8;                  // eight k of a row
  constexpr int kPer = (kItems + kThreads - 1) / kThreads;
  constexpr bool kWhole = kItems % kThreads == 0;   // else the last item of some threads lies past the tile's rows
  constexpr int kStage = PARTS * kK8 * kPitch;      // 16-byte places per LDS buffer
  constexpr int kShare = TM * 16 / KS;              // values per lane a wave finishes
  constexpr int kRed = KS > 1 ? TM * kWaves * 256 : 0;   // 16-byte places of the K slices' partial tiles
  constexpr int kLds = 2 * kStage > kRed ? 2 * kStage : kRed;
  constexpr bool NORM = EXTRA == 1;
  __shared__ u32x4 lds[kLds + (NORM ? BM / 2 : 0)];
  float *const ln_rows = reinterpret_cast<float *>(lds + kLds);  // mean, then 1 / sqrt(var + eps), per row

  float *C = C_;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int ks = wave / WN, wn = wave % WN;
  const int lrow = lane % 32, half = lane / 32;

  asm volatile("" ::"s"(p.M), "s"(p.N), "s"(p.K), "s"(p.sAm), "s"(p.sCm), "s"(p.sCn), "s"(p.tiles_m),
               "s"(p.tiles_n), "s"(p.n_splits), "s"(p.chunks_per_split), "s"(p.n_groups), "s"(p.n_inner), "s"(p.sCn_outer),
               "s"(p.bias), "s"(p.sDm), "s"(p.sDn), "s"(p.ca), "s"(p.cb), "s"(p.partials), "s"(p.counters), "s"(p.chain_n),
               "s"(p.packed));

  // ---- which tile: a contiguous run of ids per XCD, row tiles of one column tile next to each other ------------
  const uint32_t n_tiles = p.tiles_m * p.tiles_n;
  const uint32_t q = n_tiles / 8, r8 = n_tiles % 8, xcd = blockIdx.x % 8;
  const uint32_t bid = xcd * q + min(xcd, r8) + blockIdx.x / 8;
  const int m0 = static_cast<int>(bid % p.tiles_m) * BM, n0 = static_cast<int>(bid / p.tiles_m) * BN;

  const float *bias = p.bias;
  const u32x4 *packed = static_cast<const u32x4 *>(p.packed);
  int32_t sCm = p.sCm, sCn = p.sCn, sCn_outer = p.sCn_outer;
  if (p.n_groups > 1 && blockIdx.y > 0) {
    const uint32_t g = blockIdx.y - 1;
    C = p.gC[g];
    packed = static_cast<const u32x4 *>(p.g_packed[g]);
    bias = p.gbias[g];
    sCm = p.g_sCm[g];
    sCn = p.g_sCn[g];
    sCn_outer = p.g_sCn_outer[g];
  }
  const int all_steps = (p.K + 15) / 16, n_chunks = (all_steps + kChunkSteps - 1) / kChunkSteps;
  const int c_begin = static_cast<int>(blockIdx.z) * p.chunks_per_split;
  const int c_end = min(n_chunks, c_begin + p.chunks_per_split);

  // ---- loads -----------------------------------------------------------------------------------------------------
  // A: item i of a thread is eight k of one row; rows past M repeat the last one, k past K read as zero
  const char *a_base = reinterpret_cast<const char *>(A + static_cast<int64_t>(m0) * p.sAm);
  uint32_t a_at[kPer];
  int a_k[kPer], a_to[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int i = tid + t * kThreads, row = i / kK8, k8 = i % kK8;
    a_at[t] = 4u * (static_cast<uint32_t>(min(row, p.M - 1 - m0)) * static_cast<uint32_t>(p.sAm) + 8 * k8);
    a_k[t] = 8 * k8;
    a_to[t] = k8 * kPitch + row;
  }
  const int col_tile = min(n0 / 32 + wn, (p.N + 31) / 32 - 1);
  const char *b_base = reinterpret_cast<const char *>(packed) + static_cast<int64_t>(col_tile) * all_steps * (PARTS * 1024);
  constexpr int kSets = DEPTH + 1;
  floatx4 ar[kSets][kPer][2];
  u32x4 br[kSets][kSteps][PARTS];
  const int last = c_end - 1;
  constexpr int kLoads = 2 * kPer + kSteps * PARTS;  // of a wave per chunk, 16 bytes per lane each
  // load i of chunk c: the items of A, then the weights
  auto load = [&](int c, auto set_c, auto load_c) __attribute__((always_inline)) {
    constexpr int S = decltype(set_c)::value, i = decltype(load_c)::value;
    const int cc = min(c, last);  // (past the end: the last chunk again, so that the number of loads in flight is known)
    if constexpr (i < 2 * kPer) {
      // (k past K: the first eight of the row, replaced by zero when they are stored)
      constexpr int t = i / 2;
      const uint32_t off = a_at[t] + (cc * BK + a_k[t] < p.K ? 4u * static_cast<uint32_t>(cc) * BK : 0u - 4u * a_k[t]);
      ar[S][t][i % 2] = *reinterpret_cast<const floatx4 *>(a_base + off + 16 * (i % 2));
    } else {
      constexpr int u = (i - 2 * kPer) / PARTS, s = (i - 2 * kPer) % PARTS;
      const char *from = b_base + static_cast<int64_t>(min(cc * kChunkSteps + ks * kSteps + u, all_steps - 1)) * (PARTS * 1024);  // (uniform)
      br[S][u][s] = *reinterpret_cast<const u32x4 *>(from + s * 1024 + lane * 16u);
    }
  };
  // item t of chunk c: its parts, into LDS
  auto store_item = [&](int c, int buf, auto set_c, int t) {
    constexpr int S = decltype(set_c)::value;
    const bool live = min(c, last) * BK + a_k[t] < p.K;
    const floatx4 lo = ar[S][t][0], hi = ar[S][t][1];
    const float x[8] = {live ? lo.x : 0.0f, live ? lo.y : 0.0f, live ? lo.z : 0.0f, live ? lo.w : 0.0f,
                        live ? hi.x : 0.0f, live ? hi.y : 0.0f, live ? hi.z : 0.0f, live ? hi.w : 0.0f};
    u32x4 parts[PARTS];
    SplitParts<PARTS>(x, parts);
#pragma unroll
    for (int s = 0; s < PARTS; ++s) {
      if (kWhole || t + 1 < kPer || tid + t * kThreads < kItems) lds[buf * kStage + s * (kK8 * kPitch) + a_to[t]] = parts[s];
    }
  };

  floatx16 acc[TM], low[PARTS == 3 ? TM : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = low[PARTS == 3 ? i : 0][e] = 0.0f;

  StaticFor<DEPTH>([&](auto d) {
    StaticFor<kLoads>([&](auto i) { load(c_begin + decltype(d)::value, d, i); });
  });

  // ---- what the epilogue needs, requested behind the first tiles ------------------------------------------------
  const int n = n0 + wn * 32 + lrow;
  const bool bias_by_col = bias != nullptr && p.sDm == 0;
  const float bias_col = bias_by_col && n < p.N ? bias[n * p.sDn] : 0.0f;
  // value v of a lane's share: tile ks * kShare / 16, ... of the wave's column, element e of it
  auto share_row = [&](int v) {
    const int g = ks * kShare + v, e = g % 16;
    return g / 16 * 32 + (e / 4) * 8 + half * 4 + (e % 4);
  };
  int64_t col = static_cast<int64_t>(n) * sCn;
  if (p.n_inner != 0) {
    uint32_t hi, lo;
    p.div_inner.DivMod(static_cast<uint32_t>(n < p.N ? n : 0), hi, lo);
    col = static_cast<int64_t>(hi) * sCn_outer + static_cast<int64_t>(lo) * sCn;
  }
  // The addends: with a few values per lane here, else behind the K loop, where the registers of the tiles are free; all of a lane's
  // together, and with K slices or splits before their exchange (us, asked for sixteen by sixteen where they are used and so: 512 x 768 x
  // 3072 with row statistics 29.3, 28.1; without an exchange 300 x 33000 x 512 86.3, 80.2, one part 1024 x 3072 x 1024 21.7, 19.7).  The
  // second one is rare: with more than sixteen values per lane it is asked for where it is used.  Held beside the first it costs
  // 64x128 tiles of one part a wave per SIMD (128 x 50304 x 512 27.3, now 25.5) and those of 96 rows scalar registers (53.0, 48.0).
  constexpr bool EARLY_ADD = EXTRA != 0 && kShare <= 8, BOTH_ADD = EXTRA != 0 && kShare <= 16;
  float pre_add[EXTRA != 0 ? kShare : 1], pre_add2[BOTH_ADD ? kShare : 1];
  auto load_addend = [&](const float *from, float *to, int v) {
    const int m = m0 + share_row(v);
    *to = m < p.M && n < p.N ? from[static_cast<int64_t>(m) * sCm + col] : 0.0f;
  };
  auto load_addends = [&] {
    if (p.addend == nullptr) return;
#pragma unroll
    for (int v = 0; v < kShare; ++v) load_addend(p.addend, pre_add + v, v);
    if constexpr (BOTH_ADD) {
      if (p.addend2 == nullptr) return;
#pragma unroll
      for (int v = 0; v < kShare; ++v) load_addend(p.addend2, pre_add2 + v, v);
    }
  };
  if constexpr (EARLY_ADD) load_addends();
  constexpr int kNormLanes = NORM ? (kThreads / BM > 16 ? 16 : kThreads / BM) : 1;  // lanes that merge a row's statistics
  constexpr int kNormPer = 32 / kNormLanes;                                         // partials each: rows of up to 1024 elements
  float ln_col = 0.0f, ln_col2 = 0.0f;
  float part_mean[NORM ? kNormPer : 1], part_m2[NORM ? kNormPer : 1];
  const int ln_row = tid / kNormLanes, ln_sub = tid % kNormLanes;
  if constexpr (NORM) {
    if (p.ln_mode != 0 && ln_row < BM) {
      const int m = min(m0 + ln_row, p.M - 1);
#pragma unroll
      for (int u = 0; u < kNormPer; ++u) {
        const float2 e = *reinterpret_cast<const float2 *>(
            p.ln_stats + (static_cast<int64_t>(m) * p.ln_parts + min(ln_sub + u * kNormLanes, p.ln_parts - 1)) * 2);
        part_mean[u] = e.x;
        part_m2[u] = e.y;
      }
    }
    if (p.ln_mode == 1 && n < p.N) {
      const float *c1 = blockIdx.y > 0 && p.n_groups > 1 ? p.g_ln_c1[blockIdx.y - 1] : p.ln_c1;
      ln_col = c1[n * p.ln_s_c1];
    } else if (p.ln_mode == 2 && n < p.N) {
      ln_col = p.ln_scale[n * p.ln_s_scale];
      ln_col2 = p.ln_shift[n * p.ln_s_shift];
    }
  }

#pragma unroll
  for (int t = 0; t < kPer; ++t) store_item(c_begin, 0, std::integral_constant<int, 0>{}, t);
  if constexpr (NORM) {
    // the mean of the row is the weighted mean of the partial means, its squared deviations the partials' own plus
    // count * (partial mean - mean)^2 each (as in matmul.hip)
    if (p.ln_mode != 0 && ln_row < BM) {
      float cnt[kNormPer], sum = 0.0f;
#pragma unroll
      for (int u = 0; u < kNormPer; ++u) {
        const int w = ln_sub + u * kNormLanes;
        cnt[u] = w < p.ln_parts ? static_cast<float>(min(32, p.ln_width - 32 * w)) : 0.0f;
        sum += cnt[u] * part_mean[u];
      }
      const float mean = GroupSum<kNormLanes>(sum) * p.ln_inv_width;
      float m2 = 0.0f;
#pragma unroll
      for (int u = 0; u < kNormPer; ++u) {
        const float d = part_mean[u] - mean;
        m2 += cnt[u] > 0.0f ? part_m2[u] + cnt[u] * d * d : 0.0f;
      }
      m2 = GroupSum<kNormLanes>(m2);
      if (ln_sub == 0) {
        ln_rows[ln_row] = mean;
        ln_rows[BM + ln_row] = 1.0f / sqrtf(m2 * p.ln_inv_width + p.ln_eps);
      }
    }
  }
  __syncthreads();

  // ---- K loop ------------------------------------------------------------------------------------------------------
  // Chunk c lies in LDS buffer (c - c_begin) % 2, its weights in register set (c - c_begin) % kSets.  With one workgroup on
  // a compute unit nobody else fills the matrix pipe while a wave converts, so the conversion of the next chunk runs
  // between the products of this one: a product keeps the pipe busy for 32 cycles, in which eight other instructions issue.
  constexpr int kGroups = kSteps * TM;
  // With one chunk ahead its rows are asked for and converted between the products of the same chunk: the loads leave with the first
  // groups of products, the rows' before the weights', and the last groups convert.  (In the order of the deeper tiles the first
  // conversion waited for loads that it was one product behind, in every chunk: us, 96 x 50304 x 512 47, now 44, 70 x 33000 x 2048 131
  // and 119, 90 x 40000 x 1024 with an addend 73 and 67.)
  constexpr int kLoadGroups = DEPTH == 1 ? kGroups - kPer : kGroups;
  constexpr auto load_group = [](int i) { return i * kLoadGroups / kLoads; };
  constexpr auto store_group = [](int t) { return DEPTH == 1 ? kLoadGroups + t : t * kGroups / kPer; };
  static_assert(DEPTH > 1 || store_group(0) >= load_group(2 * kPer - 1) + 2, "products between a chunk's rows and their conversion");
  auto chunk = [&](int c, auto idx_c) __attribute__((always_inline)) {
    constexpr int I = decltype(idx_c)::value;
    if constexpr (PARTS == 1) {
      StaticFor<kLoads>([&](auto i) { load(c + DEPTH, std::integral_constant<int, (I + DEPTH) % kSets>{}, i); });
      __builtin_amdgcn_sched_barrier(0);  // (the loads keep their place: they are DEPTH chunks early)
    }
    const u32x4 *as = lds + (I % 2) * kStage + (ks * kSteps * 2 + half) * kPitch + lrow;
    u32x4 a[2][PARTS];
    auto load_a = [&](int g) {
#pragma unroll
      for (int s = 0; s < PARTS; ++s) a[g % 2][s] = as[s * (kK8 * kPitch) + 2 * (g / TM) * kPitch + 32 * (g % TM)];
    };
    load_a(0);
    StaticFor<kGroups>([&](auto group_c) {
      constexpr int g = decltype(group_c)::value;
      if constexpr (g + 1 < kGroups) load_a(g + 1);
      if constexpr (PARTS == 3) {
        StaticFor<kLoads>([&](auto i) {
          if constexpr (load_group(i) == g) load(c + DEPTH, std::integral_constant<int, (I + DEPTH) % kSets>{}, i);
        });
        __builtin_amdgcn_sched_barrier(0);
      }
      MfmaParts<PARTS>(a[g % 2], br[I % kSets][g / TM], acc[g % TM], low[PARTS == 3 ? g % TM : 0]);
      // (also behind the last chunk, which is then converted again: a condition would end the block that is scheduled)
#pragma unroll
      for (int t = 0; t < kPer; ++t) {
        if (store_group(t) == g) store_item(c + 1, (I + 1) % 2, std::integral_constant<int, (I + 1) % kSets>{}, t);
      }
#pragma unroll
      for (int k = 0; k < (PARTS == 3 ? 6 : 1); ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);  // vector instructions
      }
    });
    // one barrier per chunk: the buffer written here was last read in the previous chunk
    __syncthreads();
  };
  constexpr int kPeriod = kSets % 2 == 0 ? kSets : 2 * kSets;
  int c = c_begin;
  for (; c + kPeriod <= c_end; c += kPeriod) {
    StaticFor<kPeriod>([&](auto k) { chunk(c + decltype(k)::value, k); });
  }
  StaticFor<kPeriod - 1>([&](auto k) {
    if (c + decltype(k)::value < c_end) chunk(c + decltype(k)::value, k);
  });

  if constexpr (PARTS == 3) {
    bool bad = false, zero = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][e] += low[i][e];
        bad |= BadSum(acc[i][e], false);
        zero |= acc[i][e] == 0.0f;
      }
    if (!__any(bad) && __any(zero && n < p.N)) {
      // Exact zeros: look for activations of this wave's steps whose products may have vanished.  Here and not while they are
      // staged, since only rows (or columns) of zeros come this way: noting it there cost 0.6 of 26 us at 512 rows.
      uint32_t tiny_key = 0xffffffffu;
      for (int cc = c_begin; cc < c_end; ++cc) {
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
          const int k = (cc * kChunkSteps + ks * kSteps + u) * 16 + 8 * half;
          if (k >= p.K) continue;
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            const float *at = A + static_cast<int64_t>(min(m0 + 32 * i + lrow, p.M - 1)) * p.sAm + k;
            const floatx4 lo = *reinterpret_cast<const floatx4 *>(at), hi = *reinterpret_cast<const floatx4 *>(at + 4);
            const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            tiny_key = TinyKey(tiny_key, x);
          }
        }
      }
      bad = tiny_key < kTinyKey;
    }
    if (__any(bad)) {
      // this wave's steps once more with the fp32 instruction, operands straight from memory
      const uint16_t *b_src = reinterpret_cast<const uint16_t *>(b_base) + lrow * 8;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
      for (int cc = c_begin; cc < c_end; ++cc) {
        const int k0 = (cc * kChunkSteps + ks * kSteps) * 16;
        for (int k = k0; k < min(p.K, k0 + 16 * kSteps); k += 2) {
          const bool live = k + half < p.K;
          const float b = live && n < p.N ? JoinParts(b_src + (k + half) / 16 * (PARTS * 512) + (k + half) % 16 / 8 * 256 + (k + half) % 8, 512) : 0.0f;
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            const int m = m0 + 32 * i + lrow;
            const float a = live && m < p.M ? A[static_cast<int64_t>(m) * p.sAm + k + half] : 0.0f;
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
          }
        }
      }
    }
  }

  if constexpr (EXTRA != 0 && !EARLY_ADD) load_addends();

  // ---- the K slices of the workgroup meet in LDS; every wave takes its share on --------------------------------
  float vals[kShare];
  if constexpr (KS > 1) {
    float *red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int g = 0; g < TM * 16; ++g) red[(wave * TM * 16 + g) * 64 + lane] = acc[g / 16][g % 16];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kShare; ++v) {
      const float *at = red + (wn * TM * 16 + ks * kShare + v) * 64 + lane;
      float sum = at[0];
#pragma unroll
      for (int z = 1; z < KS; ++z) sum += at[z * WN * TM * 16 * 64];  // in slice order
      vals[v] = sum;
    }
  } else {
#pragma unroll
    for (int v = 0; v < kShare; ++v) vals[v] = acc[v / 16][v % 16];
  }

  // ---- K split over workgroups: the hand-off of matmul.hip, one arrival per wave --------------------------------
  if (p.n_splits > 1) {
    const uint32_t n_splits = p.n_splits, slot = (blockIdx.y * n_tiles + blockIdx.x) * kWaves + wave;
    float *all = p.partials + static_cast<size_t>(slot) * n_splits * (kShare * 64);
    float *mine = all + blockIdx.z * (kShare * 64);
#pragma unroll
    for (int v = 0; v < kShare; ++v) __hip_atomic_store(mine + v * 64 + lane, vals[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t arrived = 0;
    if (lane == 0) arrived = __hip_atomic_fetch_add(&p.counters[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    arrived = __shfl(arrived, 0);
    if (arrived != n_splits - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // compiler ordering only: no instruction on gfx9
    if (lane == 0) __hip_atomic_store(&p.counters[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int v = 0; v < kShare; ++v) vals[v] = 0.0f;
    constexpr uint32_t kTogether = kShare <= 16 ? 4 : 1;  // splits whose loads are in flight together
    for (uint32_t z0 = 0; z0 < n_splits; z0 += kTogether) {
      float part[kTogether][kShare];
#pragma unroll
      for (uint32_t u = 0; u < kTogether; ++u) {
        const uint32_t z = z0 + u < n_splits ? z0 + u : z0;  // repeats a valid slot, ignored below
#pragma unroll
        for (int v = 0; v < kShare; ++v) {
          part[u][v] = __hip_atomic_load(all + static_cast<size_t>(z) * (kShare * 64) + v * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < kTogether; ++u) {
        if (z0 + u < n_splits) {
#pragma unroll
          for (int v = 0; v < kShare; ++v) vals[v] += part[u][v];
        }
      }
    }
  }

  // ---- epilogue, sixteen values (one tile) or less at a time -----------------------------------------------------
  constexpr int EV = kShare < 16 ? kShare : 16;
  StaticFor<kShare / EV>([&](auto tile_c) {
    constexpr int v0 = decltype(tile_c)::value * EV;
    float out[EV];
#pragma unroll
    for (int e = 0; e < EV; ++e) {
      const int r = share_row(v0 + e), m = m0 + r;
      float v = vals[v0 + e];
      if constexpr (NORM) {
        if (p.ln_mode == 1) v = ln_rows[BM + r] * (v - ln_rows[r] * ln_col);
      }
      if (bias_by_col) {
        v = p.ca * v + p.cb * bias_col;
      } else if (bias != nullptr && m < p.M && n < p.N) {
        v = p.ca * v + p.cb * bias[m * p.sDm + n * p.sDn];
      }
      out[e] = v;
    }
    if (p.chain_n != 0) RunChainBlock<EV>(p.chain, out);
    if constexpr (EXTRA != 0) {
      if (p.addend != nullptr) {
        float add[EV];
#pragma unroll
        for (int e = 0; e < EV; ++e) add[e] = pre_add[v0 + e];
        if (p.ln_mode == 2) {
          // the addend is the un-normalised tensor of a LayerNormalization: normalise it on the way in
#pragma unroll
          for (int e = 0; e < EV; ++e) {
            const int r = share_row(v0 + e);
            add[e] = (add[e] - ln_rows[r]) * ln_rows[BM + r] * ln_col + ln_col2;
          }
        }
#pragma unroll
        for (int e = 0; e < EV; ++e) out[e] = p.addend_is_factor != 0 ? out[e] * add[e] : out[e] + add[e];
        if (p.addend2 != nullptr) {
          float add2[EV];
#pragma unroll
          for (int e = 0; e < EV; ++e) {
            if constexpr (BOTH_ADD) add2[e] = pre_add2[v0 + e];
            else load_addend(p.addend2, add2 + e, v0 + e);
          }
#pragma unroll
          for (int e = 0; e < EV; ++e) out[e] += add2[e];
        }
      }
    }
    if (sCm == 1) {
      // a result whose rows lie next to each other (K of an attention block, a third of its launch): a lane's four rows in one
      // store.  One by one each takes a line per lane, four times over (512 rows, 3 x 768 columns, K = 768: 22.9 us, now 20.4; the
      // few-rows kernel and the tiled one at 37 and 128 rows gained nothing by the same)
#pragma unroll
      for (int e = 0; e < EV; e += 4) {
        const int m = m0 + share_row(v0 + e);
        if (m + 3 < p.M && n < p.N) {
          *reinterpret_cast<FourFloats *>(C + (m + col)) = {{out[e], out[e + 1], out[e + 2], out[e + 3]}};
        } else {
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            if (m + u < p.M && n < p.N) C[m + u + col] = out[e + u];
          }
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const int m = m0 + share_row(v0 + e);
        if (m < p.M && n < p.N) C[static_cast<int64_t>(m) * sCm + col] = out[e];
      }
    }
    if constexpr (NORM) {
      if (p.ln_stats_out != nullptr) {
        // mean and squared deviations of this 32-column run of every row the half wave holds
        const int first = n0 + wn * 32;
        const float inv_cols = 1.0f / static_cast<float>(min(32, p.N - first));
        const int parts = (p.N + 31) / 32;
#pragma unroll
        for (int e = 0; e < EV; ++e) {
          const float mean = GroupSum<32>(n < p.N ? out[e] : 0.0f) * inv_cols;
          const float d = n < p.N ? out[e] - mean : 0.0f;
          const float sq = GroupSum<32>(d * d);
          const int m = m0 + share_row(v0 + e);
          if (lrow == 0 && m < p.M && first < p.N) {
            *reinterpret_cast<float2 *>(p.ln_stats_out + (static_cast<int64_t>(m) * parts + first / 32) * 2) = make_float2(mean, sq);
          }
        }
      }
    }
  });
}

// One thread per (column tile, step, lane): eight k of a column, their parts, 16 bytes per part.
template <int PARTS>
__global__ __launch_bounds__(kPackThreads) void MatmulPackKernel(u32x4 *__restrict__ packed, const float *__restrict__ b, int N, int K,
                                                             int steps, int64_t items, int64_t sBk, int64_t sBn) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kPackThreads + threadIdx.x;
  if (i >= items) return;
  const int lane = static_cast<int>(i % 64);
  const int64_t block = i / 64;
  const int n = static_cast<int>(block / steps) * 32 + lane % 32, k0 = static_cast<int>(block % steps) * 16 + 8 * (lane / 32);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = n < N && k0 + e < K ? b[(k0 + e) * sBk + n * sBn] : 0.0f;
  u32x4 parts[PARTS];
  SplitParts<PARTS>(x, parts);
#pragma unroll
  for (int s = 0; s < PARTS; ++s) packed[(block * PARTS + s) * 64 + lane] = parts[s];
}

// range[0]: the smallest magnitude but zero, as TinyKey has it; range[1]: the bits of the largest finite one.
struct RangeArgs {
  uint32_t n;
  int32_t rank;
  FastDiv shape[4];
  int32_t strides[4];
};
__global__ __launch_bounds__(kPackThreads) void WeightRangeKernel(uint32_t *range, const float *__restrict__ w, RangeArgs a) {
  uint32_t low = 0xffffffffu, high = 0;
  for (uint32_t i = blockIdx.x * kPackThreads + threadIdx.x; i < a.n; i += gridDim.x * kPackThreads) {
    uint32_t rem = i;
    int32_t at = 0;
    for (int d = a.rank - 1; d >= 0; --d) {
      uint32_t q, r;
      a.shape[d].DivMod(rem, q, r);
      at += static_cast<int32_t>(r) * a.strides[d];
      rem = q;
    }
    const uint32_t bits = __builtin_bit_cast(uint32_t, w[at]) & 0x7fffffffu;
    low = min(low, 2 * bits - 1);
    if (bits < 0x7f800000u) high = max(high, bits);
  }
  low = WaveReduce(low, [](uint32_t x, uint32_t y) { return min(x, y); });
  high = WaveReduce(high, [](uint32_t x, uint32_t y) { return max(x, y); });
  // (all waves of a large matrix at one address took 99 us; a stale value here only costs the atomic it was to spare)
  if (threadIdx.x % kWave == 0 && low < __hip_atomic_load(range, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(range, low);
  if (threadIdx.x % kWave == 0 && high > __hip_atomic_load(range + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(range + 1, high);
}

// ---- which weights have a packed form -----------------------------------------------------------------------------
struct PackedWeights {
  void *packed;
  int64_t K, N, sBk, sBn;
  int parts;
};
std::mutex g_packed_mutex;
std::map<const void *, PackedWeights> g_packed;  // by the address of the weights

const void *FindPacked(const float *b, const MatmulArgs &p, int parts) {
  std::lock_guard<std::mutex> lock(g_packed_mutex);
  const auto it = g_packed.find(b);
  if (it == g_packed.end()) return nullptr;
  const PackedWeights &w = it->second;
  return w.K == p.K && w.N == p.N && w.sBk == p.sBk && w.sBn == p.sBn && w.parts == parts ? w.packed : nullptr;
}

// B (or a member's) is the packed form itself
bool StandsPacked(const float *b) {
  std::lock_guard<std::mutex> lock(g_packed_mutex);
  const auto it = g_packed.find(b);
  return it != g_packed.end() && it->second.packed == b;
}

// Whether the packed form is worth having: `cols` are those of all members of a launch together.
// Three parts cost six bytes per weight instead of four (beside them, where somebody reads the weights as they stand too), so it
// is taken where a launch gets about a tenth faster against the best of the other tiles, as a tuner would pick it: from 65 rows, 280000 results and
// 580 million products on.  Measured with weights that come from HBM, gain of the best packed tile:
//   K =  512: 512x1536 5 %, 512x2048 4 %, 77x50304 15 %, 128x50304 18 %, 256x50304 23 %; but 20x50304 -14 %, 64x50304 10 %
//   K =  768: 128x2304 2 %, 512x768 6 %, 128x3072 5 %, 192x3072 6 %, 320x2304 4 %, 224x3072 7 % (528 million products);
//             256x3072 13 %, 512x1536 12 % (604 million), 288x3072 12 %, 384x2304 13 %, 512x2304 19 %, 512x3072 23 %
//   K = 1024: 128x3072 4 %, 128x4096 7 %, 384x1024 10 %, 512x1024 9 %; 192x4096 9 %, 256x4096 13 %, 300x3072 13 %; 64x32000 -8 %
//   K = 2048: 128x2048 -8 %, 512x512 -8 %; 256x2048 14 %, 384x2048 15 %, 128x8192 17 %; 64x8192 1 %
//   K = 3072: 256x768 1 %, 320x768 0 % (245760 results); 384x768 10 % (294912), 448x768 12 %, 512x768 10 %
//   K = 4096: 64x4096 -3 %, 64x11008 4 %, 256x1024 6 % (262144 results); 96x4096 19 %, 128x4096 14 %, 384x1024 22 %, 256x4096 31 %
// One part: two bytes per weight and half the traffic, faster throughout (128x3072 6.1 / 10.7 us, 256x512 4.6 / 5.2); at most
// eight rows stream the fp32 weights instead, whatever the precision asked for.
bool WorthPacking(int64_t rows, int64_t cols, int64_t K, int parts) {
  if (parts == 1) return rows > 8;
  return rows > 64 && rows * cols >= 280000 && static_cast<double>(rows) * static_cast<double>(cols) * static_cast<double>(K) >= 5.8e8;
}

template <int PARTS, int TM, int WN, int KS, int DEPTH, int EXTRA>
int LaunchTile(MatmulArgs q, uint32_t n_batch, float *C, const float *A, hipStream_t s, int splits) {
  constexpr int BK = 16 * kSteps * KS, kWaves = WN * KS;
  q.chain_n = q.chain.n;
  q.tiles_m = static_cast<uint32_t>((q.M + 32 * TM - 1) / (32 * TM));
  q.tiles_n = static_cast<uint32_t>((q.N + 32 * WN - 1) / (32 * WN));
  const int64_t tiles = static_cast<int64_t>(q.tiles_m) * q.tiles_n * n_batch, chunks = (q.K + BK - 1) / BK;
  if (splits > chunks || (chunks + splits - 1) / splits * (splits - 1) >= chunks) return FL_ERR_UNSUPPORTED;
  q.n_splits = static_cast<uint32_t>(splits);
  q.chunks_per_split = static_cast<int32_t>((chunks + splits - 1) / splits);
  if (splits > 1) {
    // (a wave's counter and its share of the tile per split)
    if (tiles * kWaves > static_cast<int64_t>(kWorkspaceTiles) || tiles * WN * TM * splits > static_cast<int64_t>(kWorkspaceTiles)) return FL_ERR_UNSUPPORTED;
    StreamWorkspace *ws = GetStreamWorkspace(s);
    if (ws == nullptr) return FL_ERR_UNSUPPORTED;
    q.partials = ws->partials;
    q.counters = ws->counters;
  }
  FL_LAUNCH((MatmulPartsKernel<PARTS, TM, WN, KS, DEPTH, EXTRA>), dim3(q.tiles_m * q.tiles_n, n_batch, splits), dim3(64 * kWaves), 0, s, C, A, q);
  return FL_OK;
}

// 96 rows by 128 columns, the rule's alone: 65 to 96 rows against so many columns that tiles of 96 rows still fill the chip.  Two
// tiles of 64 rows multiply up to twice as many rows and take the weights in twice (us, 64x128 and this: 77 x 50304 x 512 58, 46; 65 rows
// 58, 46; 96 rows 57, 47; 80 x 33024 x 256 28.0, 24.8; 90 x 40000 x 1024 69, 64; 70 x 33000 x 2048 132, 121).  Before the conversions went
// behind the loads nothing was gained with more rows (280 x 33000 x 768 109, 111) or with one part (90 x 40000 x 1024 32.4, 34.7).
constexpr int kPacked96x128 = 1 << 8;

template <int PARTS, int EXTRA>
int LaunchTiles(const MatmulArgs &p, uint32_t n_batch, float *C, const float *A, hipStream_t s, int tile, int splits) {
  switch (tile) {
    case FL_TILE_PACKED_32x64: return LaunchTile<PARTS, 1, 2, 4, 2, EXTRA>(p, n_batch, C, A, s, splits);
    case FL_TILE_PACKED_64x64: return LaunchTile<PARTS, 2, 2, 2, 2, EXTRA>(p, n_batch, C, A, s, splits);
    case FL_TILE_PACKED_64x128: return LaunchTile<PARTS, 2, 4, 1, 3, EXTRA>(p, n_batch, C, A, s, splits);
    case FL_TILE_PACKED_64x128_K2: return LaunchTile<PARTS, 2, 4, 2, 2, EXTRA>(p, n_batch, C, A, s, splits);
    default: break;
  }
  if constexpr (PARTS == 3) {
    if (tile == kPacked96x128) return LaunchTile<PARTS, 3, 4, 1, 1, EXTRA>(p, n_batch, C, A, s, splits);
  }
  return FL_ERR_UNSUPPORTED;
}

}  // namespace

bool OnlyPacked(const MatmulArgs &p, const float *B) {
  bool only = StandsPacked(B);
  for (int g = 1; g < p.n_groups; ++g) only |= StandsPacked(p.gB[g - 1]);
  return only;
}

int PartsCanCarry(const fl_tensor *weights, int64_t terms, hipStream_t s) {
  if (weights->rank < 1 || weights->rank > 4) return FL_ERR_RANK;
  RangeArgs a;
  std::memset(&a, 0, sizeof(a));
  a.n = static_cast<uint32_t>(Numel(weights));
  a.rank = weights->rank;
  for (int d = 0; d < a.rank; ++d) {
    a.shape[d] = FastDiv(static_cast<uint32_t>(weights->shape[d]));
    a.strides[d] = static_cast<int32_t>(weights->strides[d]);
  }
  uint32_t range[2] = {0xffffffffu, 0}, *device = nullptr;
  FL_HIP_CHECK(hipMalloc(&device, sizeof(range)));
  hipError_t err = hipMemcpyAsync(device, range, sizeof(range), hipMemcpyHostToDevice, s);
  if (err == hipSuccess) {
    const uint32_t blocks = std::min<uint32_t>((a.n + kPackThreads - 1) / kPackThreads, 1024);
    FL_LAUNCH(WeightRangeKernel, dim3(blocks), dim3(kPackThreads), 0, s, device, static_cast<const float *>(weights->base), a);
    err = hipGetLastError();
  }
  if (err == hipSuccess) err = hipMemcpyAsync(range, device, sizeof(range), hipMemcpyDeviceToHost, s);
  if (err == hipSuccess) err = hipStreamSynchronize(s);
  (void)hipFree(device);
  FL_HIP_CHECK(err);
  const float largest = __builtin_bit_cast(float, range[1]);
  const bool ok = range[0] >= 2 * 0x21800000u - 1 && static_cast<double>(terms) * largest <= 0x1p20;  // (2^-60)
  return ok ? FL_OK : FL_ERR_UNSUPPORTED;
}

int LaunchPacked(const MatmulArgs &args, uint32_t n_batch, bool extra, int parts, float *C, const float *A, const float *B,
                 hipStream_t s, TileChoice choice) {
  if (choice.tile != FL_TILE_RULE && choice.tile < FL_TILE_PACKED_32x64) return FL_ERR_UNSUPPORTED;
  MatmulArgs p = args;
  if (p.batch.rank != 0 || (p.n_groups <= 1 && n_batch != 1) || p.k_scale != nullptr) return FL_ERR_UNSUPPORTED;
  if (p.sAk != 1 || p.K % 8 != 0 || p.sAm % 4 != 0 || p.sAm < 0 || !IsAligned(A, 16)) return FL_ERR_UNSUPPORTED;
  if (static_cast<int64_t>(p.sAm) * 128 + p.K > 0x3fffffff) return FL_ERR_UNSUPPORTED;  // (32-bit byte offsets inside a tile)
  p.packed = FindPacked(B, p, parts);
  if (p.packed == nullptr) return FL_ERR_UNSUPPORTED;
  for (int g = 1; g < p.n_groups; ++g) {
    p.g_packed[g - 1] = FindPacked(p.gB[g - 1], p, parts);
    if (p.g_packed[g - 1] == nullptr) return FL_ERR_UNSUPPORTED;
  }
  int tile = choice.tile, splits = choice.splits > 0 ? choice.splits : 1;
  if (tile == FL_TILE_RULE) {
    if (choice.splits != 0 || !WorthPacking(p.M, static_cast<int64_t>(p.N) * std::max(1, p.n_groups), p.K, parts)) return FL_ERR_UNSUPPORTED;
    // One workgroup per compute unit is the aim.  More 64x128 tiles than compute units: four waves each, two of them fit one
    // (96x128 where one row of such tiles takes all rows, see above).
    // Half as many and more: eight waves each (a second K slice).  Fewer: K split over workgroups until they fill the chip,
    // from a length on at which the exchange of the partial tiles pays; below it smaller tiles.  Measured (us):
    //   three parts  512x3072, K = 768: 64x128_K2 21.8, 64x128 23.6, 64x64 24.9; 256x50304, K = 512: 64x128 94, 64x64 106, K2 124;
    //                512x4096, K = 4096 (256 tiles): K2 98, 64x128 112
    //                256x3072, K = 768: 64x64 16.1, K2 in two 17.3; 256x4096, K = 1024: 64x64 20.8, K2 in two 22.4, in one 26.6;
    //                640x1280, K = 1280: 22.5 both; 512x2048, K = 2048: K2 in two 32.7, 64x64 35.4, K2 in one 44.5
    //                256x4096: K = 4096 K2 in two 55, in one 81, K = 11008 137, 223; 512x1024, K = 4096: K2 in four 33.1, in three 36.5
    //                512x768, K = 3072: K2 in four 24.9, 64x64 in four 26.7; 256x2048, K = 2048: K2 in three 23.3, in four 24.1
    //   one part     512x768, K = 3072 (192 tiles of 32x64): 32x64 14.9, K2 in four 14.6; 256x4096, K = 4096 (512): K2 in two 26.6, in
    //                one 36.3; 640x1280, K = 5120 (400): K2 in two 29, 32x64 38; 256x4096, K = 1024: 32x64 10.1, K2 10.7
    auto tiles = [&](int bm, int bn) { return static_cast<int64_t>((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn) * n_batch; };
    const int64_t t128 = tiles(64, 128), t64 = tiles(64, 64), t32 = tiles(32, 64);
    if (t128 > 256) {
      tile = parts == 3 && p.M > 64 && p.M <= 96 && tiles(96, 128) > 256 ? kPacked96x128 : FL_TILE_PACKED_64x128;
    } else if (t128 > 128) {
      tile = FL_TILE_PACKED_64x128_K2;
    } else if (parts == 3 ? p.K >= 1280 && t128 >= 32 : p.K >= 2048 && t32 > 256) {
      tile = FL_TILE_PACKED_64x128_K2;
      splits = static_cast<int>(std::min<int64_t>({256 / t128, 4, p.K / 640}));
    } else if (parts == 3 && t64 >= 144) {
      tile = FL_TILE_PACKED_64x64;
    } else {
      tile = FL_TILE_PACKED_32x64;
      if (p.K >= 2048) splits = static_cast<int>(std::clamp<int64_t>(256 / t32, 1, 4));
    }
    const int64_t chunk = tile == FL_TILE_PACKED_32x64 ? 128 : 64, chunks = (p.K + chunk - 1) / chunk;
    while (splits > 1 && (chunks + splits - 1) / splits * (splits - 1) >= chunks) --splits;
  }
  const int rc = parts == 3 ? (extra ? LaunchTiles<3, 1>(p, n_batch, C, A, s, tile, splits) : LaunchTiles<3, 0>(p, n_batch, C, A, s, tile, splits))
                            : (extra ? LaunchTiles<1, 1>(p, n_batch, C, A, s, tile, splits) : LaunchTiles<1, 0>(p, n_batch, C, A, s, tile, splits));
  if (rc == FL_OK) NotePackedParts(parts);
  return rc;
}

}  // namespace fl

extern "C" {

int fluidml_hip_contract_pack(const fl_tensor *rhs, int32_t trans_b, int64_t rows, int32_t parts, void *stream, void **packed, size_t *bytes) {
  using namespace fl;
  if (packed == nullptr || bytes == nullptr) return FL_ERR_NULL;
  *packed = nullptr;
  *bytes = 0;
  FL_CHECK(CheckView(rhs));
  if (parts != 1 && parts != 3) return FL_ERR_ATTR;
  if (rhs->dtype != FL_FLOAT32) return FL_ERR_DTYPE;
  if (rhs->rank != 2) return FL_ERR_RANK;
  PackedWeights w;
  w.K = rhs->shape[trans_b ? 1 : 0], w.sBk = rhs->strides[trans_b ? 1 : 0];
  w.N = rhs->shape[trans_b ? 0 : 1], w.sBn = rhs->strides[trans_b ? 0 : 1];
  w.parts = parts;
  if (!WorthPacking(rows, w.N, w.K, parts)) return FL_ERR_UNSUPPORTED;
  if (w.K <= 0 || w.N <= 0 || w.K > 0x3fffffff || w.N > 0x3fffffff || w.sBk < 0 || w.sBn < 0) return FL_ERR_UNSUPPORTED;
  const int64_t steps = (w.K + 15) / 16, items = (w.N + 31) / 32 * steps * 64;
  if ((items + kPackThreads - 1) / kPackThreads > 0x7fffffff) return FL_ERR_TOO_LARGE;
  {
    std::lock_guard<std::mutex> lock(g_packed_mutex);
    if (g_packed.count(rhs->base)) return FL_ERR_UNSUPPORTED;  // (packed already)
  }
  if (parts == 3) FL_CHECK(PartsCanCarry(rhs, w.K, AsStream(stream)));
  *bytes = static_cast<size_t>(items) * 16 * parts;
  FL_HIP_CHECK(hipMalloc(&w.packed, *bytes));
  const dim3 grid(static_cast<uint32_t>((items + kPackThreads - 1) / kPackThreads));
  const float *b = static_cast<const float *>(rhs->base);
  u32x4 *to = static_cast<u32x4 *>(w.packed);
  if (parts == 3) {
    FL_LAUNCH(MatmulPackKernel<3>, grid, dim3(kPackThreads), 0, AsStream(stream), to, b, static_cast<int>(w.N), static_cast<int>(w.K),
              static_cast<int>(steps), items, w.sBk, w.sBn);
  } else {
    FL_LAUNCH(MatmulPackKernel<1>, grid, dim3(kPackThreads), 0, AsStream(stream), to, b, static_cast<int>(w.N), static_cast<int>(w.K),
              static_cast<int>(steps), items, w.sBk, w.sBn);
  }
  const int rc = LaunchStatus();
  if (rc != FL_OK) {
    (void)hipFree(w.packed);
    *bytes = 0;
    return rc;
  }
  std::lock_guard<std::mutex> lock(g_packed_mutex);
  g_packed[rhs->base] = w;
  *packed = w.packed;
  return FL_OK;
}

int fluidml_hip_contract_adopt(void *packed) {
  using namespace fl;
  if (packed == nullptr) return FL_ERR_NULL;
  std::lock_guard<std::mutex> lock(g_packed_mutex);
  auto it = g_packed.begin();
  while (it != g_packed.end() && it->second.packed != packed) ++it;
  if (it == g_packed.end()) return FL_ERR_ATTR;
  const PackedWeights w = it->second;
  g_packed.erase(it);
  g_packed[packed] = w;
  return FL_OK;
}

int fluidml_hip_contract_unpack(void *packed) {
  using namespace fl;
  if (packed == nullptr) return FL_OK;
  {
    std::lock_guard<std::mutex> lock(g_packed_mutex);
    auto it = g_packed.begin();
    while (it != g_packed.end() && it->second.packed != packed) ++it;
    if (it == g_packed.end()) return FL_ERR_ATTR;
    g_packed.erase(it);
  }
  FL_HIP_CHECK(hipFree(packed));
  return FL_OK;
}

}  // extern "C"
