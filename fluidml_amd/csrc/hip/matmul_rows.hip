// Contractions of few rows and short sums: MatMul, Gemm and pointwise Conv with every epilogue of the tiled kernel in
// matmul.hip, operands as they stand.  Reference: src/structure/kernel/kernel/matmul.cpp:28-59, gemm.cpp:39-182, conv.cpp.
//
// Such a launch is no matter of throughput: what it takes are the trips to memory one after the other, the bytes a compute
// unit has to be fed and the tail behind the last product.  So here
//   * every wave has its own slice of K and requests two stages of 32 k of both operands before it waits for anything; the
//     K loop has no barrier, and no exchange between workgroups follows;
//   * B (n-contiguous) goes from memory straight into the registers the matrix instruction reads: a lane takes W columns
//     next to each other of the rows 4g .. 4g + 3 of every 16 (g = lane / 16), W values per load, and product w of the W takes
//     the columns W c + w (c = lane % 16).  The order of columns inside a tile is free, so no lane waits for another's value.
//   * A (k-contiguous) would need sixteen rows per load that way, which a compute unit takes in at a quarter of its rate (16
//     rows of 64 bytes: 64 cycles per load, contiguous: 16).  It goes straight into LDS, 128 bytes of eight rows per load, in
//     the part of LDS that only this wave reads; the 16-byte groups of row r stand permuted (q ^ r / 2 % 8) so that sixteen
//     rows read from sixteen different places.
//   * the slices meet in LDS once; from there on every thread has one to four values of the tile: bias, chain, addends and
//     row statistics, all requested while the tiles travel, are spread over the whole workgroup.
#include <algorithm>
#include <cstring>

#include "fl_common.h"
#include "matmul_args.h"

namespace fl {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// W floats at any float's address, one load
template <int W>
struct __attribute__((packed, aligned(4))) Run {
  float v[W];
};

// Waits until at most N vector loads are outstanding.  The builtin, not assembly: the compiler, which does not rely on loads to
// LDS and loads to registers returning in order, would otherwise wait for all of them in front of the registers' first use.
template <int N>
__device__ __forceinline__ void WaitLoads() {
  static_assert(N >= 0 && N < 64, "six bits");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | 7 << 4 | 15 << 8 | (N >> 4) << 14);  // (the other counters: no wait)
  asm volatile("" ::: "memory");
}

template <int S>
using Slot = std::integral_constant<int, S>;

// TM x W matrix tiles of 16 x 16 per wave, WN waves side by side times KS slices of K, R stages of a wave in flight
// EXTRA: 0 = none, 1 = addends and deferred LayerNormalization, 2 = addends and a scale per row of B
template <int TM, int W, int WN, int KS, int R, int EXTRA>
__global__ __launch_bounds__(64 * WN *KS) void MatmulRowsKernel(float *C_, const float *A, const float *B_, MatmulArgs p) {
  // (no __restrict__: the loads ahead of their use would be moved to it)
  constexpr int kThreads = 64 * WN * KS;
  constexpr int BM = 16 * TM, BN = 16 * W;  // of a wave
  constexpr int kStageK = 32;
  constexpr int kPlace = TM * 512;          // floats of A per stage
  constexpr int kLoads = 2 * TM + 8 + (EXTRA == 2 ? 2 : 0);  // load instructions per stage
  constexpr int kValues = TM * W * 256;     // of a wave's tile
  constexpr int EV = KS == 1 ? TM * W * 4 : (kValues + 64 * KS - 1) / (64 * KS);  // values per thread behind the K loop
  constexpr int kRing = WN * KS * R * kPlace, kRed = KS > 1 ? WN * KS * kValues : 0;
  constexpr bool NORM = EXTRA == 1;
  // (one LDS object: with a second one the compiler waits for all loads in front of every read)
  __shared__ __attribute__((aligned(16))) float lds[(kRing > kRed ? kRing : kRed) + (NORM ? 2 * BM : 0)];
  float *const ln_rows = lds + (kRing > kRed ? kRing : kRed);  // mean, then 1 / sqrt(var + eps), per row

  asm volatile("" ::"s"(p.M), "s"(p.N), "s"(p.K), "s"(p.sAm), "s"(p.sBk), "s"(p.sCm), "s"(p.sCn), "s"(p.tiles_m),
               "s"(p.tiles_n), "s"(p.n_groups), "s"(p.n_inner), "s"(p.sCn_outer), "s"(p.bias), "s"(p.sDm), "s"(p.sDn), "s"(p.ca),
               "s"(p.cb), "s"(p.chain_n));
  if constexpr (EXTRA != 0) asm volatile("" ::"s"(p.addend), "s"(p.addend2), "s"(p.k_scale), "s"(p.addend_is_factor));
  if constexpr (NORM) {
    asm volatile("" ::"s"(p.ln_mode), "s"(p.ln_parts), "s"(p.ln_width), "s"(p.ln_eps), "s"(p.ln_inv_width), "s"(p.ln_stats), "s"(p.ln_c1),
                 "s"(p.ln_scale), "s"(p.ln_shift), "s"(p.ln_s_scale), "s"(p.ln_s_shift), "s"(p.ln_s_c1), "s"(p.ln_stats_out));
  }

  float *C = C_;
  const float *B = B_;
  const int tid = threadIdx.x, lane = tid % 64, c = lane % 16, g = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int ks = wave % KS, wn = wave / KS;

  // ---- which tile: a contiguous run of ids per XCD, row tiles of one column tile next to each other ------------
  const uint32_t n_tiles = p.tiles_m * p.tiles_n;
  const uint32_t q8 = n_tiles / 8, r8 = n_tiles % 8, xcd = blockIdx.x % 8;
  const uint32_t bid = xcd * q8 + min(xcd, r8) + blockIdx.x / 8;
  const int m0 = static_cast<int>(bid % p.tiles_m) * BM, n0 = static_cast<int>(bid / p.tiles_m) * (BN * WN) + wn * BN;

  const float *bias = p.bias;
  int32_t sCm = p.sCm, sCn = p.sCn, sCn_outer = p.sCn_outer;
  if (p.n_groups > 1 && blockIdx.y > 0) {
    const uint32_t m = blockIdx.y - 1;
    B = p.gB[m];
    C = p.gC[m];
    bias = p.gbias[m];
    sCm = p.g_sCm[m];
    sCn = p.g_sCn[m];
    sCn_outer = p.g_sCn_outer[m];
  }

  // ---- deferred LayerNormalization: the partial statistics of the rows leave first, they are merged while the tiles travel
  constexpr int kNormLanes = NORM ? (kThreads / BM > 32 ? 32 : kThreads / BM) : 1;  // lanes per row
  constexpr int kNormPer = 32 / kNormLanes;                                         // partials each: rows of up to 1024 elements
  static_assert(!NORM || kNormLanes >= 1, "a lane per row at least");
  const int ln_row = tid / kNormLanes, ln_sub = tid % kNormLanes;
  float part_mean[NORM ? kNormPer : 1], part_m2[NORM ? kNormPer : 1];
  // (all loads ahead of the tiles go without a branch, to A where there is nothing to ask for: what a branch may have asked
  // for makes the compiler wait for everything in flight behind it)
  if constexpr (NORM) {
    const bool any = p.ln_mode != 0;
    const float *stats = any ? p.ln_stats : A;
    const int64_t row_at = any ? static_cast<int64_t>(min(m0 + ln_row, p.M - 1)) * p.ln_parts * 2 : 0;
    const int most = any ? p.ln_parts - 1 : 0;
#pragma unroll
    for (int u = 0; u < kNormPer; ++u) {
      const float *e = stats + row_at + 2 * min(ln_sub + u * kNormLanes, most);
      part_mean[u] = e[0];
      part_m2[u] = e[1];
    }
  }

  // ---- what the epilogue needs, requested ahead of the tiles: one round trip less behind them ---------------
  // value v of this thread: KS > 1: element tid + 64 KS v of its wave column's tile, row by row; KS == 1: its own accumulators
  // B: a lane's W columns from n_first on; the last ones of N where the tile reaches past it
  const int n_first = min(n0 + W * c, p.N - W);
  const int gt = ks * 64 + lane;
  auto row_of = [&](int v) { return KS > 1 ? (gt + v * 64 * KS) / BN : v / (4 * W) * 16 + 4 * g + v % (4 * W) / W; };
  auto col_of = [&](int v) { return KS > 1 ? n0 + (gt + v * 64 * KS) % BN : n_first + v % W; };
  // (KS == 1: a lane moved left to lie inside N repeats columns of its neighbours and stores only those that are its own: one
  // thread per element, which may then be the addend's too)
  auto lives = [&](int v) {
    if constexpr (KS == 1) return m0 + row_of(v) < p.M && col_of(v) >= n0 + W * c;
    return m0 + row_of(v) < p.M && col_of(v) < p.N && (kValues % (64 * KS) == 0 || gt + v * 64 * KS < kValues);
  };
  auto place = [&](int r, int n) {
    int64_t col = static_cast<int64_t>(n) * sCn;
    if (p.n_inner != 0) {
      uint32_t hi, lo;
      p.div_inner.DivMod(static_cast<uint32_t>(n < p.N ? n : 0), hi, lo);
      col = static_cast<int64_t>(hi) * sCn_outer + static_cast<int64_t>(lo) * sCn;
    }
    return static_cast<int64_t>(m0 + r) * sCm + col;
  };
  static_assert(EV <= 8, "more values would take the registers of the tiles in flight");
  float pre_bias[EV], pre_add[EXTRA != 0 ? EV : 1], pre_add2[EXTRA != 0 ? EV : 1], ln_col[NORM ? EV : 1], ln_col2[NORM ? EV : 1];
  {
    auto ask = [&](const float *from, int64_t at) { return (from != nullptr ? from : A)[from != nullptr ? at : 0]; };
    const float *c1 = NORM && p.ln_mode == 1 ? (blockIdx.y > 0 && p.n_groups > 1 ? p.g_ln_c1[blockIdx.y - 1] : p.ln_c1) : nullptr;
#pragma unroll
    for (int v = 0; v < EV; ++v) {
      const int r = min(row_of(v), p.M - 1 - m0), m = m0 + r, n = min(col_of(v), p.N - 1);
      pre_bias[v] = ask(bias, m * p.sDm + n * p.sDn);
      if constexpr (EXTRA != 0) {
        const int64_t at = place(r, n);
        pre_add[v] = ask(p.addend, at);
        pre_add2[v] = ask(p.addend2, at);
      }
      if constexpr (NORM) {
        ln_col[v] = ask(c1 != nullptr ? c1 : p.ln_scale, n * (c1 != nullptr ? p.ln_s_c1 : p.ln_s_scale));
        ln_col2[v] = ask(p.ln_shift, n * p.ln_s_shift);
      }
    }
  }

  // ---- loads -----------------------------------------------------------------------------------------------------
  const int stages = (p.K + kStageK - 1) / kStageK, per = (stages + KS - 1) / KS;
  const int s0 = ks * per, n_st = min(per, stages - s0);  // (not positive: nothing left for this slice)
  // A: load i takes rows 8i .. 8i + 7; place lane % 8 of a row holds group (lane % 8) ^ (row / 2 % 8).  Rows past M repeat the
  // last one; groups past K (K is a multiple of four) the first of the row, and are replaced by zero when they are read.
  const float *a_row[2 * TM];
  int a_k[2 * TM];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    const int r = 8 * i + lane / 8;
    a_row[i] = A + static_cast<int64_t>(min(m0 + r, p.M - 1)) * p.sAm;
    a_k[i] = s0 * kStageK + 4 * ((lane % 8) ^ (r / 2 % 8));
  }
  const float *b_col = B + n_first;
  float *const ring = lds + wave * R * kPlace;
  Run<W> b[R][8];
  floatx4 bs[EXTRA == 2 ? R : 1][2];
  auto load = [&](int t, auto slot_c) {
    constexpr int S = decltype(slot_c)::value;
    const int k0 = (s0 + t) * kStageK;
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
      const int k = a_k[i] + t * kStageK;
      const float *from = a_row[i] + (k < p.K ? k : 0);
      float *to = ring + S * kPlace + i * 256;
      __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = min(k0 + 16 * (j / 4) + 4 * g + j % 4, p.K - 1);
      b[S][j] = *reinterpret_cast<const Run<W> *>(b_col + static_cast<int64_t>(k) * p.sBk);
    }
    if constexpr (EXTRA == 2) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = min(k0 + 16 * h + 4 * g, p.K - 4);
        const Run<4> s = *reinterpret_cast<const Run<4> *>(p.k_scale + k);
        bs[S][h] = floatx4{s.v[0], s.v[1], s.v[2], s.v[3]};
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto merge_rows = [&](auto behind_c) {  // behind_c: stages requested since
    if constexpr (NORM) {
      WaitLoads<decltype(behind_c)::value * kLoads>();
      // the mean of the row is the weighted mean of the partial means, its squared deviations the partials' own plus
      // count * (partial mean - mean)^2 each (as in matmul.hip)
      if (p.ln_mode != 0 && (kThreads == BM * kNormLanes || ln_row < BM)) {
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
  };

  // ---- K loop ------------------------------------------------------------------------------------------------------
  floatx4 acc[TM][W];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int w = 0; w < W; ++w) acc[i][w] = floatx4{0, 0, 0, 0};
  auto multiply = [&](int t, auto slot_c, auto ragged_c) {
    constexpr int S = decltype(slot_c)::value;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool live = !decltype(ragged_c)::value || (s0 + t) * kStageK + 16 * h + 4 * g < p.K;
      floatx4 a[TM];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = 16 * i + c;
        a[i] = *reinterpret_cast<const floatx4 *>(ring + S * kPlace + r * 32 + 4 * ((4 * h + g) ^ (r / 2 % 8)));
        if (!live) a[i] = floatx4{0, 0, 0, 0};
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
          float x = b[S][4 * h + j].v[w];
          if constexpr (EXTRA == 2) x *= bs[S][h][j];
          if (!live) x = 0.0f;
#pragma unroll
          for (int i = 0; i < TM; ++i) acc[i][w] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][j], x, acc[i][w], 0, 0, 0);
        }
      }
    }
  };
  // Loads complete in order: with the loads of the stage behind it outstanding at most, this wave's loads of a stage have landed
  // (the others left before them).  The stages are walked without a condition around a load:
  // the compiler, which waits for B's registers by itself, otherwise loses count and waits for everything in flight.
  auto refill = [&](int t, auto slot_c) {
    __builtin_amdgcn_sched_barrier(0);  // (the place's values have gone into products)
    load(t, slot_c);
  };
  if (n_st >= R) {
    StaticFor<R>([&](auto d) { load(decltype(d)::value, d); });
    merge_rows(Slot<R>{});
    int t = 0;
    for (; t + 2 * R <= n_st; t += R) {
      StaticFor<R>([&](auto d) {
        WaitLoads<(R - 1) * kLoads>();
        multiply(t + decltype(d)::value, d, std::false_type{});
        refill(t + R + decltype(d)::value, d);
      });
    }
    // R .. 2 R - 1 stages are left
    StaticFor<R>([&](auto more_c) {
      constexpr int kLeft = R + decltype(more_c)::value;
      if (n_st - t == kLeft) {
        StaticFor<kLeft>([&](auto d_c) {
          constexpr int d = decltype(d_c)::value;
          WaitLoads<((d + R < kLeft ? d + R : kLeft) - 1 - d) * kLoads>();
          multiply(t + d, Slot<d % R>{}, std::integral_constant<bool, d + 1 == kLeft>{});
          if constexpr (d + R < kLeft) refill(t + d + R, Slot<d % R>{});
        });
      }
    });
  } else {
    // (a slice without a stage asks for some bytes of A and B, which go nowhere)
    StaticFor<R - 1>([&](auto most_c) {
      constexpr int kLeft = 1 + decltype(most_c)::value;
      if (n_st == kLeft || (kLeft == 1 && n_st < 1)) {
        StaticFor<kLeft>([&](auto d) { load(decltype(d)::value, d); });
        merge_rows(Slot<kLeft>{});
        StaticFor<kLeft>([&](auto d_c) {
          constexpr int d = decltype(d_c)::value;
          WaitLoads<(kLeft - 1 - d) * kLoads>();
          if (kLeft > 1 || n_st == 1) multiply(d, Slot<d>{}, std::integral_constant<bool, d + 1 == kLeft>{});
        });
      }
    });
  }

  // ---- the slices meet in LDS ---------------------------------------------------------------------------------------
  float vals[EV];
  if constexpr (KS > 1) {
    __syncthreads();  // (every wave is done with its stages)
    // element (row 16 i + 4 g + e, column W c + w) of a wave's tile: the lanes of a store lie next to each other, and so that a
    // row's columns, read by consecutive lanes, come from different places, the groups g of product w are turned by w
    float *red = lds + wave * kValues;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[((i * 4 + e) * W + w) * 64 + 16 * ((g + 2 * w) % 4) + c] = acc[i][w][e];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < EV; ++v) {
      const int r = min(row_of(v), BM - 1), n = col_of(v);
      // (a lane whose columns reach past N holds the last ones instead)
      const int cc = (n - n0) / W, w = n < p.N ? n - min(n0 + W * cc, p.N - W) : 0;
      const float *at = lds + wn * KS * kValues + (((r / 16) * 4 + r % 4) * W + w) * 64 + 16 * ((r % 16 / 4 + 2 * w) % 4) + cc;
      float sum = at[0];
#pragma unroll
      for (int z = 1; z < KS; ++z) sum += at[z * kValues];  // in slice order
      vals[v] = sum;
    }
  } else {
    if constexpr (NORM) __syncthreads();
#pragma unroll
    for (int v = 0; v < EV; ++v) vals[v] = acc[v / (4 * W)][v % W][v % (4 * W) / W];
  }

  // ---- epilogue -------------------------------------------------------------------------------------------------------
#pragma unroll
  for (int v = 0; v < EV; ++v) {
    if constexpr (NORM) {
      const int r = row_of(v);
      if (p.ln_mode == 1) vals[v] = ln_rows[BM + min(r, BM - 1)] * (vals[v] - ln_rows[min(r, BM - 1)] * ln_col[v]);
    }
    if (bias != nullptr) vals[v] = p.ca * vals[v] + p.cb * pre_bias[v];
  }
  if (p.chain_n != 0) RunChainBlock<EV>(p.chain, vals);
  if constexpr (EXTRA != 0) {
    if (p.addend != nullptr) {
#pragma unroll
      for (int v = 0; v < EV; ++v) {
        float add = pre_add[v];
        if constexpr (NORM) {
          // the addend is the un-normalised tensor of a LayerNormalization: normalise it on the way in
          const int r = min(row_of(v), BM - 1);
          if (p.ln_mode == 2) add = (add - ln_rows[r]) * ln_rows[BM + r] * ln_col[v] + ln_col2[v];
        }
        vals[v] = p.addend_is_factor != 0 ? vals[v] * add : vals[v] + add;
        if (p.addend2 != nullptr) vals[v] += pre_add2[v];
      }
    }
  }
#pragma unroll
  for (int v = 0; v < EV; ++v) {
    if (lives(v)) C[place(row_of(v), col_of(v))] = vals[v];
  }
  if constexpr (NORM && KS > 1 && BN % 32 == 0) {
    if (p.ln_stats_out != nullptr) {
      // mean and squared deviations of the 32-column run this half wave holds a row of
      const int parts = (p.N + 31) / 32;
#pragma unroll
      for (int v = 0; v < EV; ++v) {
        const int n = col_of(v), first = n - lane % 32;
        const float inv_cols = 1.0f / static_cast<float>(min(32, p.N - first));
        const float mean = GroupSum<32>(n < p.N ? vals[v] : 0.0f) * inv_cols;
        const float d = n < p.N ? vals[v] - mean : 0.0f;
        const float sq = GroupSum<32>(d * d);
        const int m = m0 + row_of(v);
        if (lane % 32 == 0 && m < p.M && first < p.N) {
          *reinterpret_cast<float2 *>(p.ln_stats_out + (static_cast<int64_t>(m) * parts + first / 32) * 2) = make_float2(mean, sq);
        }
      }
    }
  }
}

template <int TM, int W, int WN, int KS, int EXTRA>
int Launch(MatmulArgs q, uint32_t n_batch, float *C, const float *A, const float *B, hipStream_t s) {
  if constexpr (EXTRA == 1) {
    if (q.ln_stats_out != nullptr && (KS == 1 || 16 * W % 32 != 0)) return FL_ERR_UNSUPPORTED;
  }
  q.chain_n = q.chain.n;
  q.tiles_m = static_cast<uint32_t>((q.M + 16 * TM - 1) / (16 * TM));
  q.tiles_n = static_cast<uint32_t>((q.N + 16 * W * WN - 1) / (16 * W * WN));
  FL_LAUNCH((MatmulRowsKernel<TM, W, WN, KS, 2, EXTRA>), dim3(q.tiles_m * q.tiles_n, n_batch), dim3(64 * WN * KS), 0, s, C, A, B, q);
  return FL_OK;
}

// Workgroup tiles: rows x columns, slices of K
enum Shape { kNone, k16x16, k16x32, k16x48, k32x32, k32x48, k16x128_K2, k16x256_K1 };

template <int EXTRA>
int LaunchShape(const MatmulArgs &p, uint32_t n_batch, float *C, const float *A, const float *B, hipStream_t s, Shape shape) {
  switch (shape) {
    case k16x16: return Launch<1, 1, 1, 8, EXTRA>(p, n_batch, C, A, B, s);
    case k16x32: return Launch<1, 2, 1, 8, EXTRA>(p, n_batch, C, A, B, s);
    case k16x48: return Launch<1, 3, 1, 8, EXTRA>(p, n_batch, C, A, B, s);
    case k32x32: return Launch<2, 2, 1, 8, EXTRA>(p, n_batch, C, A, B, s);
    case k32x48: return Launch<2, 3, 1, 8, EXTRA>(p, n_batch, C, A, B, s);
    default: break;
  }
  if constexpr (EXTRA != 1) {
    if (shape == k16x128_K2) return Launch<1, 2, 4, 2, EXTRA>(p, n_batch, C, A, B, s);
    if (shape == k16x256_K1) return Launch<1, 2, 8, 1, EXTRA>(p, n_batch, C, A, B, s);
  }
  return FL_ERR_UNSUPPORTED;
}

// The smallest tile that leaves a compute unit one workgroup: a second round of workgroups, or a second one beside the first,
// costs more than a larger tile does.  Measured (us, in the replayed networks; "before": the best of the other kernels'
// tiles as the tuner picked it):
//   M x N x K            before   16x16  16x32  16x48  32x32  32x48
//   128 x 54 x 384         6.4     4.0    4.5    5.3    6.0    7.0
//   77 x 512 x 512         5.2     4.1    4.8    5.7    5.8    7.4
//   384 x 128 x 768        8.6     5.4    6.5    8.3    9.0    12
//   320 x 49 x 1152       10.0     6.0    7.5    9.3    10     13
//   77 x 512 x 2048        7.6     7.6    10     14     15     21    (another 37 x 768 x 3072: 10.6, 12.8)
//   37 x 2304 x 768        8.9     8.1    7.6    9.8    9.6    12    (432 tiles of 16x16, 216 of 16x32)
//   77 x 1536 x 512        6.7     6.3    5.5    6.5    6.9    9.1
//   256 x 512 x 512        5.6     5.2    4.7    5.8    6.0    7.6
//   128 x 768 x 768        8.5            7.3           9.7          (with the statistics of a deferred LayerNormalization)
//   77 x 2048 x 512        8.3     8.8    8.6    7.8    8.1    10
//   128 x 1536 x 768       8.3     9.2    9.6    8.4    9.0    11
//   256 x 1536 x 512      10.5    12.6   11.2   12.6   11.4    9.4
//   128 x 3072 x 768      14.7    17.9   16.5   19.0   16.4   13.9   (256 tiles of 32x48)
//   256 x 2048 x 512      12.3    18     15.5   21     13     19     (344 of 32x48: left to the others)
//   256 x 512 x 2048      10.4    13     11.3   14     16     21     (long sums of more than one 16x16 tile likewise)
// Sums of at most 64 terms are pointwise convolutions of many pixels, whose slices of K would stand idle; past 1536 tiles of
// 16x16 their waves stand side by side:
//   144 x 3136 x 24        6.5     8.2    7.7    12     6.1    10     16x128 5.5, 16x256 5.9
//   96 x 12544 x 16       10.8     19     17     26     14     20     16x128 10.5, 16x256 8.7
// Where the tiled kernel's rule is the faster one (us, this rule without the exceptions behind it; sixteen sets of operands in turn, the
// pointwise convolutions one):
//   * tiles larger than 16x32: eight slices share 4, 12 or 20 stages unevenly, and the chunks of 128 terms of the tiled kernel divide
//     those sums: 192 x 1024 x 384 5.5, 6.4, x 512 6.1, 6.4, x 640 6.8, 8.2, x 704 9.6, 8.1, x 1152 12.2, 11.1; 192 x 768 x 384
//     5.5, 6.2, x 640 6.8, 7.6; 512 x 768 x 128 4.9, 5.5 (with 16x48 and 32x32 as fast), x 192 6.4, 6.4, x 384 7.9, 8.4
//   * waves side by side, more than three workgroups to a compute unit: tiles of 64 rows read B a quarter as often, and are
//     faster where they pad less than a third: 240 x 6400 x 64 (750) 9.1, 8.6, 128 x 12544 x 64 (784) 9.4, 10.2,
//     1024 x 50176 x 48 119, 167; 72 x 50176 x 64 19.9, 17.1, 144 x 50176 x 64 28.3, 27.8
//   * the same with a scale per row of B, which every row tile multiplies by again, in the tile of 16x256 past one workgroup to a
//     compute unit: 256 x 3136 x 32 (208) 6.7, 5.2, 192 x 12544 x 32 (588) 9.0, 10.6, 1024 x 50176 x 32 107, 127;
//     112 x 50176 x 32, which 64 rows pad by a seventh, 19.4, 18.7
// The limits of K, this kernel over the tiled one's time on the other side too: 16x16, x 1536 0.83 to 0.88, x 2048 0.90 to 0.97 (32 x
// 2048 1.11), x 2432 0.98 to 1.05, x 3072 1.00 to 1.08; the larger tiles, x 1088 and 1152 0.80 to 0.98 (192 x 768 and 96 x 1536 1.02 to
// 1.09), x 1408 0.83 to 1.12, x 1664 0.88 to 1.14, x 2048 0.79 to 1.05.
Shape Choose(const MatmulArgs &p, uint32_t n_batch, bool extra) {
  auto tiles = [&](int bm, int bn) { return static_cast<int64_t>((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn) * n_batch; };
  auto fits = [&](int bm, int bn) { return tiles(bm, bn) <= 256; };
  const bool stats = extra && p.ln_stats_out != nullptr;  // runs of 32 columns
  if (p.K <= 2048 && !stats && fits(16, 16)) return k16x16;
  if (p.K <= 1152) {
    const Shape shape = fits(16, 32) ? k16x32 : !stats && fits(16, 48) ? k16x48 : fits(32, 32) ? k32x32 : !stats && fits(32, 48) ? k32x48 : kNone;
    const bool uneven = p.K % 256 == 128 && p.K <= 640 && (p.K > 128 || shape == k32x48);
    if (shape != kNone) return shape != k16x32 && uneven ? kNone : shape;
  }
  if (p.K > 64 || extra) return kNone;
  const int64_t padded = (p.M + 63) / 64 * 64;  // the rows that the tiled kernel multiplies
  if (p.K <= 32 && !fits(16, 128)) return p.k_scale == nullptr || fits(16, 256) || 7 * padded >= int64_t{8} * p.M ? k16x256_K1 : kNone;
  return tiles(16, 128) <= 3 * 256 || 3 * padded >= int64_t{4} * p.M ? k16x128_K2 : kNone;
}

}  // namespace

int LaunchRows(const MatmulArgs &p, uint32_t n_batch, bool extra, float *C, const float *A, const float *B, hipStream_t s) {
  if (p.batch.rank != 0 || (p.n_groups <= 1 && n_batch != 1)) return FL_ERR_UNSUPPORTED;
  // A: 16-byte pieces of its rows; B: columns next to each other, at any float's address
  if (p.sAk != 1 || p.K % 4 != 0 || p.sAm % 4 != 0 || !IsAligned(A, 16)) return FL_ERR_UNSUPPORTED;
  if (p.sBn != 1 || p.N < 4) return FL_ERR_UNSUPPORTED;
  if (p.k_scale != nullptr && p.sKs != 1) return FL_ERR_UNSUPPORTED;
  const Shape shape = Choose(p, n_batch, extra && p.k_scale == nullptr);
  if (shape == kNone) return FL_ERR_UNSUPPORTED;
  if (p.k_scale != nullptr) return LaunchShape<2>(p, n_batch, C, A, B, s, shape);
  return extra ? LaunchShape<1>(p, n_batch, C, A, B, s, shape) : LaunchShape<0>(p, n_batch, C, A, B, s, shape);
}

}  // namespace fl
