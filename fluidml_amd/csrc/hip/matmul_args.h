// Arguments of the contraction kernels (matmul.hip, matmul_parts.hip).
#ifndef FLUIDML_AMD_HIP_MATMUL_ARGS_H_
#define FLUIDML_AMD_HIP_MATMUL_ARGS_H_

#include <cstddef>

#include "fl_common.h"

namespace fl {

// Geometry of a convolution run as an implicit GEMM: M = output channels, N = images x output pixels,
// K = input channels x kernel taps.  B[k][n] is gathered from the input on the fly (padding reads as 0),
// C[m][n] is scattered to out[image, m, oh, ow].  1-d convolutions use H = OH = KH = 1.
struct ConvGeom {
  int32_t H, W;                  // input extents
  int32_t sh, sw, dh, dw, ph, pw;
  int32_t sXn, sXc, sXh, sXw;    // input element strides
  int32_t sOn, sOh, sOw;         // output element strides (the channel stride is sCm)
  FastDiv div_ohw, div_ow;       // n -> (image, oh, ow)
  FastDiv div_khw, div_kw;       // k -> (channel, kh, kw)
};

// Batch dims of a contraction after merging (operand 0 = C, 1 = A, 2 = B), innermost last.  Kept small and
// statically indexed: the kernel's scalar loads of its arguments are a serial chain of cache misses otherwise.
constexpr int kMaxBatchDims = 4;
struct BatchArgs {
  int32_t rank;  // 0: a single batch element
  FastDiv div[kMaxBatchDims];
  int32_t strides[3][kMaxBatchDims];
};

// Kernel arguments.  Every workgroup needs the first block before it can issue its first load, and a cold
// 64-byte line of kernel arguments costs a few hundred nanoseconds: what every launch reads comes first and
// is packed (two lines), what the EXTRA instantiations read follows (the next line and a half), and what only some
// launches read (batch dims, chain, siblings, convolution geometry) comes last.
struct MatmulArgs {
  int32_t M, N, K;
  int32_t sAm, sAk, sBk, sBn, sCm, sCn;
  uint32_t tiles_m, tiles_n;
  // split K over `n_splits` workgroups per tile (blockIdx.z): each takes `chunks_per_split` chunks, writes its
  // partial tile to `partials`, and the workgroup that arrives last at `counters[tile]` adds them up in split order
  uint32_t n_splits;
  int32_t chunks_per_split;
  // sibling contractions that share A and every extent, one per blockIdx.y (n_groups <= 1: none; batch
  // dims are then absent).  Member 0 uses the fields here, member g > 0 the entries g - 1 of the g* arrays.
  int32_t n_groups;
  // optional two-level column addressing of C: column n lives at (n / n_inner) * sCn_outer + (n % n_inner) * sCn
  // (the last output dim reshaped into two dims that a transpose moved apart); n_inner == 0: n * sCn
  int32_t n_inner, sCn_outer;
  // epilogue: C = ca * acc + cb * bias[m * sDm + n * sDn]   (bias may be null)
  const float *bias;
  int32_t sDm, sDn;
  float ca, cb;
  float *partials;
  uint32_t *counters;
  // copies of batch.rank and chain.n (set at launch), so that a launch without batch dims or chain never touches
  // the lines those live in
  int32_t batch_rank, chain_n;
  // EXTRA == 1 instantiations only, one batch element: a LayerNormalization kept out of memory (fl_norm_fusion).
  // ln_mode 1: A holds the un-normalised tensor, the epilogue turns acc into rstd * (acc - mean * c1[n]) + bias[n];
  // ln_mode 2: the addend does, and enters as (t - mean) * rstd * scale[n] + shift[n].  Row statistics come as
  // ln_parts (mean, M2) pairs per row, each over 32 consecutive columns of the ln_width wide tensor.
  int32_t ln_mode, ln_parts, ln_width;
  float ln_eps;
  // ---- byte 128 ----
  // EXTRA instantiations only (plain contraction, B kept [k][n]), all optional:
  // a tensor with the strides of C, added to the value after the chain (read at the element offset the value is
  // stored at);
  const float *addend;
  // a second one, added after the first;
  const float *addend2;
  // one batch element: row k of B is multiplied by k_scale[k * sKs] while it is staged, each product rounded like
  // a separate Mul kernel's
  const float *k_scale;
  int32_t sKs;
  float ln_inv_width;  // (1 / ln_width, rounded once on the host)
  const float *ln_stats;
  const float *ln_c1;                 // mode 1, member 0 (members g > 0: g_ln_c1[g - 1])
  const float *ln_scale, *ln_shift;   // mode 2
  // ---- byte 192 ----
  float *ln_stats_out;                // non-null: (mean, M2) of every 32-column run of C's rows, ceil(N / 32) per row
  int32_t ln_s_scale, ln_s_shift, ln_s_c1;  // element strides of the three vectors
  int32_t addend_is_factor;                 // EXTRA: the value is multiplied by `addend` instead
  FastDiv div_inner;
  const float *g_ln_c1[3];
  const float *gB[3];
  float *gC[3];
  const float *gbias[3];
  int32_t g_sCm[3], g_sCn[3], g_sCn_outer[3];
  // matmul_parts.hip: the packed form of B, one per member
  const void *packed;
  const void *g_packed[3];
  BatchArgs batch;
  // optional elementwise chain applied after the bias (chain.n == 0: none)
  fl_ew_program chain;
  ConvGeom conv;  // read by the CONV instantiations only
};
static_assert(offsetof(MatmulArgs, addend) == 128 && offsetof(MatmulArgs, ln_stats_out) == 192,
              "the packing of the kernel arguments into lines is deliberate");

// What the caller fixed of a launch's configuration (fl_contract_tile, K splits; 0 = the library's rule decides).
struct TileChoice {
  int tile = FL_TILE_RULE;
  int splits = 0;
};

// matmul_parts.hip: the contraction against weights that fluidml_hip_contract_pack has laid out.  FL_ERR_UNSUPPORTED, with
// nothing launched, where they are not among them, the operands do not fit or the choice is not one of its tiles (with
// FL_TILE_RULE also where its own rule leaves the problem to the other kernels).
int LaunchPacked(const MatmulArgs &p, uint32_t n_batch, bool extra, int parts, float *C, const float *A, const float *B,
                 hipStream_t s, TileChoice choice);

// matmul_rows.hip: the contraction of few rows and short sums.  FL_ERR_UNSUPPORTED, with nothing launched, where the operands
// do not fit or its rule leaves the problem to the other kernels.
int LaunchRows(const MatmulArgs &p, uint32_t n_batch, bool extra, float *C, const float *A, const float *B, hipStream_t s);

// Whether B, or that of a member, exists in its packed form only: no other kernel can read it.
bool OnlyPacked(const MatmulArgs &p, const float *B);

}  // namespace fl

#endif
