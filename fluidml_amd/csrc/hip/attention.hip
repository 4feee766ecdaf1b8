// One launch for the core of an attention block:
//   scores = Q . K^T ; scores = scores / c (or * c) [+ mask] [where(cond, scores, fill)] ;
//   P = softmax(scores, last axis) ; out = P . V
// i.e. the chain MatMulKernel -> DivConstantRhs/MulConstant -> AddCommon / WhereConstantCond -> SoftmaxKernel
// -> MatMulKernel (reference matmul.cpp:28-59, div.cpp:24-56, mul.cpp, add.cpp:75-137, where.cpp:17-150,
// softmax.cpp:22-139) without writing the [.., Sq, Skv] score and probability tensors.
//
// One workgroup owns 16 (or 32, below) query rows of one batch element (head), so that even a single sequence spreads over many
// compute units, and its waves share out the keys.  The kernel is a chain of latencies more than anything else, so
// nothing stands in it that could be left out: no operand is staged in LDS, and no value changes its lane.
//   1. scores, transposed: v_mfma_f32_16x16x4_f32 with the keys as rows and the queries as columns.  A lane feeds it
//      K^T[d][key lane % 16] and Q[query lane % 16][d] and receives the scores of ITS query (lane % 16) with the keys
//      16 t + 4 (lane / 16) + i of every key tile t.
//   2. scale, mask, condition, and the maximum over the wave's own keys: registers and two swaps of rows.
//   3. context, transposed: the product with V^T (head columns as rows, queries as columns) wants of a lane
//      P[key 4 (lane / 16) + i][query lane % 16] in step i -- register i of the scores as they lie.
//   4. every wave leaves its context, its maximum and its sum of exponentials in LDS; after the only barrier the
//      contexts are added, each scaled by exp(its maximum - the row's), and divided by the row's sum.
// The loads run ahead of the products, and none needs more than the alignment of a float, so odd lengths cost nothing.  What
// that takes: one fetch of all arguments, no branch around a single load (each makes the compiler wait for what is under way),
// and offsets of 32 bits from a base that all lanes share.  More than 256 keys and more such workgroups than compute units:
// a workgroup's registers fill a compute unit, so the rest would come in a second round; it takes two tiles of queries with
// the same keys and values instead.  Measured (us in a replayed graph, heads x queries x keys, 64 columns; first: scores through
// an LDS strip, K and V staged in LDS; then: one load, one branch, 64-bit addresses, 16 queries throughout; now):
//   12 x 128 x 128 6.8, 5.5, 4.5; 12 x 37 x 37 9.6, 4.4, 4.2; 8 x 256 x 256 11.4, 9.7, 8.0; 12 x 512 x 512 31 (score MatMul,
//   Softmax, MatMul), 23.4, 16.0 (21.6 with two tiles of queries alone)
// What bounds the last one: the matrix pipes 6.8 us, exponentials 2, and each phase waits for the one before.
// Every operand is addressed through element strides, so the head split of the producers and the head merge
// of the consumer need no copies.
#include <cmath>

#include "fl_common.h"

namespace fl {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kQ = 16;       // query rows per tile
constexpr int kMaxD = 64;    // head dim limit
constexpr int kMaxKeys = 512;

// What every launch reads comes first, in two lines and a half: each missing line is one round trip more in front of the first load.
struct alignas(16) AttentionArgs {
  FastDiv q_blocks;         // workgroups per batch element
  FastDiv inner;            // extent of the inner batch dim
  uint32_t per_xcd;         // workgroups / 8, or 0 where they do not divide
  int32_t batch_rank;       // batch dims; more than two: `batch` instead of the next two
  int32_t sb_in[8], sb_out[8];  // strides of the inner and the outer batch dim: out, q, kt, v, mask, cond, nothing twice
  int32_t Sq, Skv, D, sQm, sKd, sKn, sVn, vec_q;  // vec_q: four consecutive d of a query are 16 aligned bytes
  int32_t sMm, sMn, sCm, sCn;  // additive mask / keep condition strides along (query, key)
  int32_t sQd, sVd, sOm, sOd;
  float scale;
  int32_t scale_is_divisor;
  float fill;
  NestArgs<6> batch;
};
static_assert(offsetof(AttentionArgs, sb_in) == 32 && offsetof(AttentionArgs, sQd) == 144, "five times eight words, and the strides of V, Q and the result");

template <typename T, typename O>
__device__ __forceinline__ T At(const void *base, O bytes) {
  return *reinterpret_cast<const T *>(static_cast<const char *>(base) + bytes);
}

// Two workgroups of eight waves fit a compute unit if they make do with 128 registers, and with V's columns one by one up to
// 8 tiles of keys times tiles of columns do (128 heads x 257 x 257, 32 columns, V transposed: with 130 registers 75 us, with 128 60).
constexpr int MinWaves(int waves, int tiles, bool vec) { return !vec && waves == 8 && tiles <= 8 ? 4 : 1; }

// Consecutive floats, at any address.
template <int N>
struct __attribute__((packed, aligned(4))) Run {
  float v[N];
};

// NW waves with KT tiles of 16 keys each, DT tiles of 16 head columns; FULL: D = 16 DT.
// VEC: head columns lie at unit stride in V (FULL).  Which of them is row r of which tile is free: the tiles are then
// interleaved, row r of tile j is column DT r + j, so that one load brings a lane its row of every tile (12 heads x 128 x 128
// 6.0 -> 5.5 us).  The same for the keys, one load for a lane's row of every key tile, was slower (6.1, with 256 keys 9.0
// instead of 8.1).
// MASK, COND: an additive mask, a condition may be there.
// QT: tiles of 16 queries a workgroup takes with the keys and values it has loaded.
template <int NW, int KT, int DT, int QT, bool FULL, bool VEC, bool MASK, bool COND>
__global__ __launch_bounds__(64 * NW, MinWaves(NW, KT * DT, VEC)) void AttentionKernel(
    AttentionArgs a, float *__restrict__ out, const float *__restrict__ q, const float *__restrict__ kt, const float *__restrict__ v,
    const float *__restrict__ mask, const uint8_t *__restrict__ cond) {
  constexpr int kLd = 16 * DT + 4;  // floats per query in LDS: lanes of consecutive queries in different banks
  __shared__ __attribute__((aligned(16))) float ctx[QT * NW * kQ * kLd];
  __shared__ float stat[2][QT][NW][kQ];  // the waves' maxima and sums

  // Workgroup ids go round the 8 XCDs; renumbered so that each XCD takes a contiguous run of (head, query block)
  // pairs, a head's K and V are fetched by one or two of the L2s instead of all eight.
  // (all arguments at once, and no branch before them: the compiler fetches each where it is used, a round trip every time)
  typedef int32_t Line __attribute__((ext_vector_type(8), aligned(4)));
  const Line *lines = reinterpret_cast<const Line *>(&a);
  asm volatile("" ::"s"(lines[0]), "s"(lines[1]), "s"(lines[2]), "s"(lines[3]), "s"(lines[4]), "s"(q), "s"(kt), "s"(v), "s"(mask), "s"(cond));
  const uint32_t bid = a.per_xcd != 0 ? (blockIdx.x % 8) * a.per_xcd + blockIdx.x / 8 : blockIdx.x;
  uint32_t element, qb;
  a.q_blocks.DivMod(bid, element, qb);
  int32_t off[6] = {0, 0, 0, 0, 0, 0};
  if (a.batch_rank <= 2) {
    uint32_t outer, inner;
    a.inner.DivMod(element, outer, inner);
#pragma unroll
    for (int o = 0; o < 6; ++o) off[o] = static_cast<int32_t>(outer) * a.sb_out[o] + static_cast<int32_t>(inner) * a.sb_in[o];
  } else {
    a.batch.AddOffsets(element, off);
  }
  const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, grp = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int m0 = static_cast<int>(qb) * (QT * kQ), n0 = wave * KT * 16;
  const int last_key = a.Skv - 1;
  auto key = [&](int t, int r) { return n0 + 16 * t + r; };
  auto column = [&](int j, int r) { return VEC ? DT * r + j : 16 * j + r; };

  // ---- requests: K, Q, mask and condition, then V --------------------------------------------------------------
  // d runs in the order 16 j + 4 (lane / 16) + e, the same for both operands, so that a lane's Q is four consecutive d
  float kreg[KT][DT][4], qreg[QT][DT][4];
  const float *kb = kt + off[2];
  if (a.vec_q) {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const float *qp = q + off[1] + min(m0 + kQ * u + l16, a.Sq - 1) * a.sQm;
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        const int d0 = 16 * j + 4 * grp;
        const floatx4 x = *reinterpret_cast<const floatx4 *>(qp + (FULL || d0 < a.D ? d0 : 0));
        qreg[u][j][0] = x.x, qreg[u][j][1] = x.y, qreg[u][j][2] = x.z, qreg[u][j][3] = x.w;
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const float *qp = q + off[1] + min(m0 + kQ * u + l16, a.Sq - 1) * a.sQm;
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = 16 * j + 4 * grp + e;
          qreg[u][j][e] = qp[(FULL ? d : min(d, a.D - 1)) * a.sQd];
        }
    }
  }
  using Offset = std::conditional_t<VEC, uint32_t, uint64_t>;  // bytes from a base that all lanes share
  auto bytes = [](int32_t elements) { return static_cast<Offset>(elements) * 4; };
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    if constexpr (FULL) {
      const Offset at = bytes(min(key(t, l16), last_key) * a.sKn + 4 * grp * a.sKd);
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) kreg[t][j][e] = At<float>(kb + (16 * j + e) * a.sKd, at);
    } else {
      const float *at = kb + min(key(t, l16), last_key) * a.sKn;
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) kreg[t][j][e] = at[min(16 * j + 4 * grp + e, a.D - 1) * a.sKd];
    }
  }
  // (without a condition around each load: where there is no mask they read the queries' first value)
  const bool masked = MASK && mask != nullptr, conditional = COND && cond != nullptr;
  float mreg[QT][KT][4];
  uint8_t creg[QT][KT][4];
  const float *mb = masked ? mask + off[4] : q;
  const uint8_t *cb = conditional ? cond + off[5] : reinterpret_cast<const uint8_t *>(q);
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const int m = min(m0 + kQ * u + l16, a.Sq - 1);
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = min(key(t, 4 * grp + i), last_key);
        if constexpr (MASK) mreg[u][t][i] = At<float>(mb, bytes(m * a.sMm + n * a.sMn));
        if constexpr (COND) creg[u][t][i] = At<uint8_t>(cb, static_cast<Offset>(m * a.sCm + n * a.sCn));
      }
  }
  float vreg[KT][4][DT];
  const float *vb = v + off[3];
  auto load_v = [&] {
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = min(key(t, 4 * grp + i), last_key);
        if constexpr (VEC) {
          const Run<DT> x = At<Run<DT>>(vb, bytes(n * a.sVn + column(0, l16)));
#pragma unroll
          for (int j = 0; j < DT; ++j) vreg[t][i][j] = x.v[j];
        } else {
          const float *at = vb + n * a.sVn;
#pragma unroll
          for (int j = 0; j < DT; ++j) vreg[t][i][j] = at[(FULL ? column(j, l16) : min(column(j, l16), a.D - 1)) * a.sVd];
        }
      }
  };
  // V's columns one by one: these loads keep the other waves' loads of K waiting, so they leave once this wave's K is there, and
  // with many of them (or with some and a mask) behind the scores, where K's registers are free again.  Measured (us; before the loads were put ahead
  // of the scores, with all of them there, now): 128 heads x 200 x 200, 40 columns, a condition
  // 39.0, 47.5, 33.8; V transposed: 128 x 256 x 256, 48, a condition 72.0, 90.3, 67.5; 128 x 300 x 300, 48 134, 155, 136;
  // 128 x 300 x 300, 64 157, 174, 167.
  constexpr bool kBehindScores = !VEC && KT == 4 && (DT == 4 || (DT == 2 && (MASK || COND)));
  if constexpr (!VEC && !kBehindScores) {
#pragma unroll
    for (int t = 0; t < KT; ++t) asm volatile("" ::"v"(kreg[t][DT - 1][3]));
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (!kBehindScores) load_v();

  // ---- scores ------------------------------------------------------------------------------------------------------
  if constexpr (!FULL) {
    // head columns past D: both operands are zero there
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = 16 * j + 4 * grp + e < a.D;
#pragma unroll
        for (int u = 0; u < QT; ++u) qreg[u][j][e] = ok ? qreg[u][j][e] : 0.0f;
#pragma unroll
        for (int t = 0; t < KT; ++t) kreg[t][j][e] = ok ? kreg[t][j][e] : 0.0f;
      }
  }
  float s[QT][KT][4];
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kreg[t][j][e], qreg[u][j][e], acc, 0, 0, 0);
      s[u][t][0] = acc.x, s[u][t][1] = acc.y, s[u][t][2] = acc.z, s[u][t][3] = acc.w;
    }

  if constexpr (kBehindScores) {
    __builtin_amdgcn_sched_barrier(0);
    load_v();
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- scale, mask, condition; exponentials about the maximum of the wave's keys ---------------------------------
  const bool ragged = n0 + 16 * KT > a.Skv;  // some of the wave's keys do not exist
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    auto each = [&](auto &&f) {
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[u][t][i] = f(s[u][t][i], t, i);
    };
    if (a.scale_is_divisor) each([&](float y, int, int) { return y / a.scale; });
    else each([&](float y, int, int) { return y * a.scale; });
    if constexpr (MASK) {
      if (masked) each([&](float y, int t, int i) { return y + mreg[u][t][i]; });
    }
    if constexpr (COND) {
      if (conditional) each([&](float y, int t, int i) { return creg[u][t][i] != 0 ? y : a.fill; });
    }
    if (ragged) each([&](float y, int t, int i) { return key(t, 4 * grp + i) <= last_key ? y : -__FLT_MAX__; });
    float mx = -__FLT_MAX__;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[u][t][i]);
    mx = AcrossHalves(AcrossRows(mx, MaxOp{}), MaxOp{});
    each([&](float y, int, int) { return expf(y - mx); });
    if (ragged) each([&](float y, int t, int i) { return key(t, 4 * grp + i) <= last_key ? y : 0.0f; });
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += s[u][t][i];
    sum = AcrossHalves(AcrossRows(sum, SumOp{}), SumOp{});
    if (grp == 0) {
      stat[0][u][wave][l16] = mx;
      stat[1][u][wave][l16] = sum;
    }
  }

  // ---- the wave's context --------------------------------------------------------------------------------------------
  floatx4 o[QT][DT];
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int j = 0; j < DT; ++j) o[u][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  if (ragged) {
    // (keys past the last one repeat its row of V under a probability of zero; zero themselves, should it hold an infinity)
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DT; ++j) vreg[t][i][j] = key(t, 4 * grp + i) <= last_key ? vreg[t][i][j] : 0.0f;
  }
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int u = 0; u < QT; ++u) o[u][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vreg[t][i][j], s[u][t][i], o[u][j], 0, 0, 0);

  // ---- the waves' contexts meet in LDS --------------------------------------------------------------------------------
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) ctx[((u * NW + wave) * kQ + l16) * kLd + column(j, 4 * grp + i)] = o[u][j][i];
  __syncthreads();
  for (int it = tid; it < QT * kQ * DT * 4; it += 64 * NW) {
    const int row = it / (4 * DT), u = row / kQ, m = row % kQ, k = it % (4 * DT) * 4;
    float row_max = stat[0][u][0][m];
#pragma unroll
    for (int w = 1; w < NW; ++w) row_max = fmaxf(row_max, stat[0][u][w][m]);
    float row_sum = 0.0f;
    floatx4 r = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = expf(stat[0][u][w][m] - row_max);
      row_sum += f * stat[1][u][w][m];
      const floatx4 x = *reinterpret_cast<const floatx4 *>(ctx + ((u * NW + w) * kQ + m) * kLd + k);
      r.x += f * x.x, r.y += f * x.y, r.z += f * x.z, r.w += f * x.w;
    }
    if (m0 + row >= a.Sq) continue;
    float *at = out + off[0] + (m0 + row) * a.sOm;
    const float res[4] = {r.x / row_sum, r.y / row_sum, r.z / row_sum, r.w / row_sum};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (FULL || k + e < a.D) at[(k + e) * a.sOd] = res[e];
    }
  }
}

}  // namespace
}  // namespace fl

using namespace fl;

extern "C" {

int fluidml_hip_attention(const fl_tensor *q, const fl_tensor *kt, const fl_tensor *v, const fl_tensor *out, double scale,
                          int32_t scale_is_divisor, const fl_tensor *add_mask, const fl_tensor *keep_cond, double fill,
                          void *stream) {
  FL_CHECK(CheckView(q));
  FL_CHECK(CheckView(kt));
  FL_CHECK(CheckView(v));
  FL_CHECK(CheckView(out));
  if (q->dtype != FL_FLOAT32 || kt->dtype != FL_FLOAT32 || v->dtype != FL_FLOAT32 || out->dtype != FL_FLOAT32) return FL_ERR_DTYPE;
  const int rank = out->rank;
  if (rank < 2 || q->rank != rank || kt->rank != rank || v->rank != rank) return FL_ERR_RANK;
  AttentionArgs a;
  std::memset(&a, 0, sizeof(a));
  a.Sq = static_cast<int32_t>(q->shape[rank - 2]);
  a.D = static_cast<int32_t>(q->shape[rank - 1]);
  a.Skv = static_cast<int32_t>(kt->shape[rank - 1]);
  if (kt->shape[rank - 2] != a.D || v->shape[rank - 2] != a.Skv || v->shape[rank - 1] != a.D ||
      out->shape[rank - 2] != a.Sq || out->shape[rank - 1] != a.D) return FL_ERR_SHAPE;
  if (a.D > kMaxD || a.Skv > kMaxKeys) return FL_ERR_UNSUPPORTED;
  a.sQm = static_cast<int32_t>(q->strides[rank - 2]);
  a.sQd = static_cast<int32_t>(q->strides[rank - 1]);
  a.sKd = static_cast<int32_t>(kt->strides[rank - 2]);
  a.sKn = static_cast<int32_t>(kt->strides[rank - 1]);
  a.sVn = static_cast<int32_t>(v->strides[rank - 2]);
  a.sVd = static_cast<int32_t>(v->strides[rank - 1]);
  a.sOm = static_cast<int32_t>(out->strides[rank - 2]);
  a.sOd = static_cast<int32_t>(out->strides[rank - 1]);
  a.scale = static_cast<float>(scale);
  a.scale_is_divisor = scale_is_divisor;
  // (a division by a power of two is the product with its inverse, to the bit, and a tenth of the instructions)
  int exponent = 0;
  if (scale_is_divisor && std::frexp(std::fabs(a.scale), &exponent) == 0.5f && exponent > -100 && exponent < 100) {
    a.scale = 1.0f / a.scale;
    a.scale_is_divisor = 0;
  }
  a.fill = static_cast<float>(fill);
  // score-shaped index space [batch..., Sq, Skv] for the broadcast operands
  int64_t score_shape[kMaxRank], ms[kMaxRank] = {}, cs[kMaxRank] = {};
  for (int i = 0; i < rank - 2; ++i) score_shape[i] = out->shape[i];
  score_shape[rank - 2] = a.Sq;
  score_shape[rank - 1] = a.Skv;
  if (add_mask != nullptr) {
    FL_CHECK(CheckView(add_mask));
    if (add_mask->dtype != FL_FLOAT32) return FL_ERR_DTYPE;
    FL_CHECK(BroadcastStrides(add_mask, rank, score_shape, ms));
    a.sMm = static_cast<int32_t>(ms[rank - 2]);
    a.sMn = static_cast<int32_t>(ms[rank - 1]);
  }
  if (keep_cond != nullptr) {
    FL_CHECK(CheckView(keep_cond));
    if (keep_cond->dtype != FL_BOOL) return FL_ERR_DTYPE;
    FL_CHECK(BroadcastStrides(keep_cond, rank, score_shape, cs));
    a.sCm = static_cast<int32_t>(cs[rank - 2]);
    a.sCn = static_cast<int32_t>(cs[rank - 1]);
  }
  LoopNest nest;
  nest.n_operands = 6;
  nest.rank = rank - 2;
  int64_t n_batch = 1;
  for (int i = 0; i < rank - 2; ++i) {
    if (q->shape[i] != out->shape[i] || kt->shape[i] != out->shape[i] || v->shape[i] != out->shape[i]) return FL_ERR_SHAPE;
    nest.shape[i] = out->shape[i];
    nest.strides[0][i] = out->strides[i];
    nest.strides[1][i] = q->strides[i];
    nest.strides[2][i] = kt->strides[i];
    nest.strides[3][i] = v->strides[i];
    nest.strides[4][i] = ms[i];
    nest.strides[5][i] = cs[i];
    n_batch *= out->shape[i];
  }
  nest.Canonicalise();
  a.batch_rank = nest.rank;
  a.batch = MakeNestArgs<6>(nest);
  const int inner = nest.rank - 1;
  a.inner = FastDiv(static_cast<uint32_t>(inner >= 0 ? nest.shape[inner] : 1));
  for (int o = 0; o < 6; ++o) {
    a.sb_in[o] = inner >= 0 ? static_cast<int32_t>(nest.strides[o][inner]) : 0;
    a.sb_out[o] = inner >= 1 ? static_cast<int32_t>(nest.strides[o][inner - 1]) : 0;
  }
  // (offsets inside a matrix of V, of K, of the mask and the condition are 32-bit counts of bytes there)
  auto small = [](int64_t rows, int64_t row, int64_t columns, int64_t column) { return (rows - 1) * row + (columns - 1) * column < (1 << 30); };
  const bool runs = a.sVd == 1 && small(a.Skv, a.sVn, a.D, 1) && small(a.Skv, a.sKn, a.D, a.sKd) &&
                    small(a.Sq, a.sMm, a.Skv, a.sMn) && small(a.Sq, a.sCm, a.Skv, a.sCn);
  int64_t blocks = n_batch * ((a.Sq + kQ - 1) / kQ);
  // (16 queries per workgroup where one round takes them all: more compute units for a short sequence; the paths of unaligned
  // head dims keep more operands in registers)
  const bool pairs = a.Skv > 256 && blocks > 256 && runs && a.D % 16 == 0 && a.D != 48;
  const int64_t queries = pairs ? 2 * kQ : kQ;
  a.q_blocks = FastDiv(static_cast<uint32_t>((a.Sq + queries - 1) / queries));
  blocks = n_batch * ((a.Sq + queries - 1) / queries);
  if (blocks > INT32_MAX) return FL_ERR_TOO_LARGE;
  if (blocks == 0 || a.D == 0) return FL_OK;
  if (a.Skv == 0) return FL_ERR_UNSUPPORTED;
  a.per_xcd = blocks % 8 == 0 ? static_cast<uint32_t>(blocks / 8) : 0;
  const dim3 grid(static_cast<uint32_t>(blocks));
  float *o = static_cast<float *>(out->base);
  const float *qp = static_cast<const float *>(q->base), *kp = static_cast<const float *>(kt->base),
              *vp = static_cast<const float *>(v->base);
  const float *mp = add_mask ? static_cast<const float *>(add_mask->base) : nullptr;
  const uint8_t *cp = keep_cond ? static_cast<const uint8_t *>(keep_cond->base) : nullptr;
  auto mult4 = [](int64_t x) { return x % 4 == 0; };
  bool vec = a.sQd == 1 && a.D % 4 == 0 && mult4(a.sQm) && reinterpret_cast<uintptr_t>(qp) % 16 == 0;
  for (int i = 0; i < rank - 2; ++i) vec = vec && mult4(q->strides[i]);
  a.vec_q = vec ? 1 : 0;
#define FL_ATTENTION_AS(...) \
  FL_LAUNCH((AttentionKernel<__VA_ARGS__>), grid, block, 0, AsStream(stream), a, o, qp, kp, vp, mp, cp)
#define FL_ATTENTION_SCATTERED(NW_, KT_, DT_, FULL_)                                                                 \
  do {                                                                                                               \
    if (mp == nullptr && cp == nullptr) FL_ATTENTION_AS(NW_, KT_, DT_, 1, FULL_, false, false, false);               \
    else if (cp == nullptr) FL_ATTENTION_AS(NW_, KT_, DT_, 1, FULL_, false, true, false);                            \
    else if (mp == nullptr) FL_ATTENTION_AS(NW_, KT_, DT_, 1, FULL_, false, false, true);                            \
    else FL_ATTENTION_AS(NW_, KT_, DT_, 1, FULL_, false, true, true);                                                \
  } while (0)
#define FL_ATTENTION_D(NW_, KT_, DT_, QT_)                                                                           \
  do {                                                                                                               \
    const dim3 block(64 * NW_);                                                                                      \
    if (a.D == 16 * DT_ && runs && cp == nullptr) FL_ATTENTION_AS(NW_, KT_, DT_, QT_, true, true, true, false);      \
    else if (a.D == 16 * DT_ && runs && mp == nullptr) FL_ATTENTION_AS(NW_, KT_, DT_, QT_, true, true, false, true); \
    else if (a.D == 16 * DT_ && runs) FL_ATTENTION_AS(NW_, KT_, DT_, QT_, true, true, true, true);                   \
    else if (a.D == 16 * DT_) FL_ATTENTION_SCATTERED(NW_, KT_, DT_, true);                                           \
    else FL_ATTENTION_SCATTERED(NW_, KT_, DT_, false);                                                               \
  } while (0)
#define FL_ATTENTION(NW_, KT_, QT_)                       \
  do {                                                    \
    if (a.D <= 16) FL_ATTENTION_D(NW_, KT_, 1, QT_);      \
    else if (a.D <= 32) FL_ATTENTION_D(NW_, KT_, 2, QT_); \
    else FL_ATTENTION_D(NW_, KT_, 4, QT_);                \
  } while (0)
  // enough waves that each has few keys (and its loads are in flight together), no more than have any (512 keys: 16 waves
  // with two tiles each 23.8 us, 4 with eight 25.3, 8 with four 23.1)
  if (a.Skv <= 64) FL_ATTENTION(4, 1, 1);
  else if (a.Skv <= 128) FL_ATTENTION(4, 2, 1);
  else if (a.Skv <= 256) FL_ATTENTION(8, 2, 1);
  else if (pairs) FL_ATTENTION(8, 4, 2);
  else FL_ATTENTION(8, 4, 1);
#undef FL_ATTENTION
#undef FL_ATTENTION_D
#undef FL_ATTENTION_SCATTERED
#undef FL_ATTENTION_AS
  return LaunchStatus();
}

}  // extern "C"
