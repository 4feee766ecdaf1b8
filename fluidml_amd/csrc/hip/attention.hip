// One launch for the core of an attention block:
//   scores = Q . K^T ; scores = scores / c (or * c) [+ mask] [where(cond, scores, fill)] ;
//   P = softmax(scores, last axis) ; out = P . V
// i.e. the chain MatMulKernel -> DivConstantRhs/MulConstant -> AddCommon / WhereConstantCond -> SoftmaxKernel
// -> MatMulKernel (reference matmul.cpp:28-59, div.cpp:24-56, mul.cpp, add.cpp:75-137, where.cpp:17-150,
// softmax.cpp:22-139) without writing the [.., Sq, Skv] score and probability tensors.
//
// One workgroup owns 16 query rows of one batch element (head), so that even a single sequence spreads over many
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
// All loads leave at once, and none needs more than the alignment of a float, so odd lengths cost nothing.  Measured
// (us in a replayed graph, heads x queries x keys, 64 columns; before: scores through an LDS strip, K and V staged in LDS):
//   12 x 128 x 128 6.8 -> 5.5, 12 x 37 x 37 9.6 -> 4.3, 8 x 77 x 77 9.5 -> 5.3, 8 x 256 x 256 11.4 -> 7.8,
//   12 x 512 x 512 31 (score MatMul, Softmax, MatMul) -> 23
// Every operand is addressed through element strides, so the head split of the producers and the head merge
// of the consumer need no copies.
#include "fl_common.h"

namespace fl {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kQ = 16;       // query rows per workgroup
constexpr int kMaxD = 64;    // head dim limit
constexpr int kMaxKeys = 512;

struct AttentionArgs {
  NestArgs<6> batch;  // operands: 0 out, 1 q, 2 kt, 3 v, 4 mask, 5 cond
  int32_t Sq, Skv, D;
  int32_t sQm, sQd, sKd, sKn, sVn, sVd, sOm, sOd;
  int32_t sMm, sMn, sCm, sCn;  // additive mask / keep condition strides along (query, key)
  float scale;
  int32_t scale_is_divisor;
  float fill;
  uint32_t q_blocks;
  int32_t vec_q;  // four consecutive d of a query are 16 aligned bytes
};

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
template <int NW, int KT, int DT, bool FULL, bool VEC>
__global__ __launch_bounds__(64 * NW) void AttentionKernel(AttentionArgs a, float *__restrict__ out, const float *__restrict__ q,
                                                           const float *__restrict__ kt, const float *__restrict__ v,
                                                           const float *__restrict__ mask, const uint8_t *__restrict__ cond) {
  constexpr int kLd = 16 * DT + 4;  // floats per query in LDS: lanes of consecutive queries in different banks
  __shared__ __attribute__((aligned(16))) float ctx[NW * kQ * kLd];
  __shared__ float stat[2][NW][kQ];  // the waves' maxima and sums

  // Workgroup ids go round the 8 XCDs; renumbered so that each XCD takes a contiguous run of (head, query block)
  // pairs, a head's K and V are fetched by one or two of the L2s instead of all eight.
  uint32_t bid = blockIdx.x;
  if (gridDim.x % 8 == 0) bid = (bid % 8) * (gridDim.x / 8) + bid / 8;
  const uint32_t qb = bid % a.q_blocks;
  int32_t off[6] = {0, 0, 0, 0, 0, 0};
  a.batch.AddOffsets(bid / a.q_blocks, off);
  const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, grp = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int m0 = static_cast<int>(qb) * kQ, n0 = wave * KT * 16;
  const int last_key = a.Skv - 1;
  auto key = [&](int t, int r) { return n0 + 16 * t + r; };
  auto column = [&](int j, int r) { return VEC ? DT * r + j : 16 * j + r; };

  // ---- requests: K, Q, mask and condition, then V --------------------------------------------------------------
  // d runs in the order 16 j + 4 (lane / 16) + e, the same for both operands, so that a lane's Q is four consecutive d
  float kreg[KT][DT][4], qreg[DT][4];
  const float *kb = kt + off[2], *qp = q + off[1] + min(m0 + l16, a.Sq - 1) * a.sQm;
#pragma unroll
  for (int j = 0; j < DT; ++j) {
    const int d0 = 16 * j + 4 * grp;
    if (a.vec_q) {
      const floatx4 x = *reinterpret_cast<const floatx4 *>(qp + (FULL || d0 < a.D ? d0 : 0));
      qreg[j][0] = x.x, qreg[j][1] = x.y, qreg[j][2] = x.z, qreg[j][3] = x.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) qreg[j][e] = qp[(FULL ? d0 + e : min(d0 + e, a.D - 1)) * a.sQd];
    }
  }
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const float *at = kb + min(key(t, l16), last_key) * a.sKn;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 16 * j + 4 * grp + e;
        kreg[t][j][e] = at[(FULL ? d : min(d, a.D - 1)) * a.sKd];
      }
  }
  float mreg[KT][4];
  uint32_t keep = ~0u;  // bit 4 t + i
  {
    const int m = min(m0 + l16, a.Sq - 1);
    uint8_t creg[KT][4];
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = min(key(t, 4 * grp + i), last_key);
        mreg[t][i] = mask != nullptr ? mask[off[4] + m * a.sMm + n * a.sMn] : 0.0f;
        creg[t][i] = cond != nullptr ? cond[off[5] + m * a.sCm + n * a.sCn] : uint8_t{1};
      }
    if (cond != nullptr) {
      keep = 0;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) keep |= static_cast<uint32_t>(creg[t][i] != 0) << (4 * t + i);
    }
  }
  float vreg[KT][4][DT];
  const float *vb = v + off[3];
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float *at = vb + min(key(t, 4 * grp + i), last_key) * a.sVn;
      if constexpr (VEC) {
        const Run<DT> x = *reinterpret_cast<const Run<DT> *>(at + column(0, l16));
#pragma unroll
        for (int j = 0; j < DT; ++j) vreg[t][i][j] = x.v[j];
      } else {
#pragma unroll
        for (int j = 0; j < DT; ++j) vreg[t][i][j] = at[(FULL ? column(j, l16) : min(column(j, l16), a.D - 1)) * a.sVd];
      }
    }

  // ---- scores ------------------------------------------------------------------------------------------------------
  if constexpr (!FULL) {
    // head columns past D: both operands are zero there
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = 16 * j + 4 * grp + e < a.D;
        qreg[j][e] = ok ? qreg[j][e] : 0.0f;
#pragma unroll
        for (int t = 0; t < KT; ++t) kreg[t][j][e] = ok ? kreg[t][j][e] : 0.0f;
      }
  }
  float s[KT][4];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kreg[t][j][e], qreg[j][e], acc, 0, 0, 0);
    s[t][0] = acc.x, s[t][1] = acc.y, s[t][2] = acc.z, s[t][3] = acc.w;
  }

  // ---- scale, mask, condition; exponentials about the maximum of the wave's keys ---------------------------------
  float mx = -__FLT_MAX__;
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y = a.scale_is_divisor ? s[t][i] / a.scale : s[t][i] * a.scale;
      if (mask != nullptr) y = y + mreg[t][i];
      if ((keep >> (4 * t + i) & 1u) == 0) y = a.fill;
      if (key(t, 4 * grp + i) > last_key) y = -__FLT_MAX__;
      s[t][i] = y;
      mx = fmaxf(mx, y);
    }
  mx = AcrossHalves(AcrossRows(mx, MaxOp{}), MaxOp{});
  float sum = 0.0f;
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[t][i] = key(t, 4 * grp + i) <= last_key ? expf(s[t][i] - mx) : 0.0f;
      sum += s[t][i];
    }
  sum = AcrossHalves(AcrossRows(sum, SumOp{}), SumOp{});

  // ---- the wave's context --------------------------------------------------------------------------------------------
  floatx4 o[DT];
#pragma unroll
  for (int j = 0; j < DT; ++j) o[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // (keys past the last one repeat its row of V under a probability of zero; zero themselves, should it hold an infinity)
      const bool ok = key(t, 4 * grp + i) <= last_key;
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ok ? vreg[t][i][j] : 0.0f, s[t][i], o[j], 0, 0, 0);
      }
    }

  // ---- the waves' contexts meet in LDS --------------------------------------------------------------------------------
#pragma unroll
  for (int j = 0; j < DT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) ctx[(wave * kQ + l16) * kLd + column(j, 4 * grp + i)] = o[j][i];
  if (grp == 0) {
    stat[0][wave][l16] = mx;
    stat[1][wave][l16] = sum;
  }
  __syncthreads();
  for (int it = tid; it < kQ * DT * 4; it += 64 * NW) {
    const int m = it / (4 * DT), k = it % (4 * DT) * 4;
    float row_max = stat[0][0][m];
#pragma unroll
    for (int w = 1; w < NW; ++w) row_max = fmaxf(row_max, stat[0][w][m]);
    float row_sum = 0.0f;
    floatx4 r = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = expf(stat[0][w][m] - row_max);
      row_sum += f * stat[1][w][m];
      const floatx4 x = *reinterpret_cast<const floatx4 *>(ctx + (w * kQ + m) * kLd + k);
      r.x += f * x.x, r.y += f * x.y, r.z += f * x.z, r.w += f * x.w;
    }
    if (m0 + m >= a.Sq) continue;
    float *at = out + off[0] + (m0 + m) * a.sOm;
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
  a.batch = MakeNestArgs<6>(nest);
  a.q_blocks = static_cast<uint32_t>((a.Sq + kQ - 1) / kQ);
  const int64_t blocks = n_batch * a.q_blocks;
  if (blocks > INT32_MAX) return FL_ERR_TOO_LARGE;
  if (blocks == 0 || a.D == 0) return FL_OK;
  if (a.Skv == 0) return FL_ERR_UNSUPPORTED;
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
  const bool runs = a.sVd == 1;
#define FL_ATTENTION_D(NW_, KT_, DT_)                                                                                           \
  do {                                                                                                                          \
    if (a.D == 16 * DT_ && runs) FL_LAUNCH((AttentionKernel<NW_, KT_, DT_, true, true>), grid, dim3(64 * NW_), 0, AsStream(stream), a, o, qp, kp, vp, mp, cp); \
    else if (a.D == 16 * DT_) FL_LAUNCH((AttentionKernel<NW_, KT_, DT_, true, false>), grid, dim3(64 * NW_), 0, AsStream(stream), a, o, qp, kp, vp, mp, cp); \
    else FL_LAUNCH((AttentionKernel<NW_, KT_, DT_, false, false>), grid, dim3(64 * NW_), 0, AsStream(stream), a, o, qp, kp, vp, mp, cp); \
  } while (0)
#define FL_ATTENTION(NW_, KT_)                      \
  do {                                              \
    if (a.D <= 16) FL_ATTENTION_D(NW_, KT_, 1);     \
    else if (a.D <= 32) FL_ATTENTION_D(NW_, KT_, 2); \
    else FL_ATTENTION_D(NW_, KT_, 4);               \
  } while (0)
  // enough waves that each has few keys (and its loads are in flight together), no more than have any (512 keys: 16 waves
  // with two tiles each 23.8 us, 4 with eight 25.3, 8 with four 23.1)
  if (a.Skv <= 64) FL_ATTENTION(4, 1);
  else if (a.Skv <= 128) FL_ATTENTION(4, 2);
  else if (a.Skv <= 256) FL_ATTENTION(8, 2);
  else FL_ATTENTION(8, 4);
#undef FL_ATTENTION
#undef FL_ATTENTION_D
  return LaunchStatus();
}

}  // extern "C"
