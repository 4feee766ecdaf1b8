// Dense 2-d convolutions whose sums have at most 32 terms: the first layer over an image of a few channels.
// Reference: src/structure/kernel/kernel/conv.cpp:27-280.
//
// Such a layer writes far more than it reads or multiplies (64 filters over 3 channels: 27 products per value written), so
// it is bound by the stores, provided the products take no longer than they have to.  The whole K = channels x taps of a
// wave's filters fits its registers; the activations, of which an image holds a few hundred kilobytes, come from the caches
// straight into the matrix operand: a wave takes 64 output pixels of 32 filters through
// v_mfma_f32_16x16x4_f32, K padded to a multiple of four (conv_halo.hip stages eight channels of which three exist, 2.7 times the
// products; the implicit GEMM gathers element by element through LDS in chunks of 32 to 128 terms).
//   * the weights go through LDS once per workgroup: a lane wants its filter's terms one by one, and loads whose lanes lie in
//     different rows take a compute unit four times as long (64 cycles each; 28 of them per wave were half the launch);
//   * filters are the rows of the products, pixels the columns: lane % 16 is a filter of the one operand and four pixels of the
//     other, lane / 16 the term inside a group of four.  Which of the four goes into which product is free, so a lane takes four
//     neighbours of a row, one 16-byte load per term and one 16-byte store per filter, 256 bytes side by side over the lanes.
//     A row's last four are filled up and not stored.
// Measured, bias and ReLU included (us; before: conv_halo.hip): 8 x 3 x 224^2 -> 64 filters 75 -> 38 (103 MB written), one
// image 16.4 -> 10.5.  With the weights read from memory by every wave and the loads left where the compiler puts them: 52 and 14.
#include "fl_common.h"

namespace fl {
namespace {

constexpr int kThreads = 256;
constexpr int FT = 2;  // tiles of 16 filters per wave (four: two waves per SIMD instead of four, one image 14.1 against 10.3 us, eight 37 both)

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Four consecutive floats at any float's address
struct __attribute__((packed, aligned(4))) Quad {
  float v[4];
};

struct ShortArgs {
  int32_t F, K, fours, runs;  // runs of four pixels, of all images together; sixteen of them are a wave's
  int32_t H, W, OW, sh, dh, dw, ph, pw;
  int32_t sXn, sXc, sXh;
  int32_t sOn, sOf, sOh;
  int32_t sWf, sWc, sWh, sWw;
  FastDiv div_image, div_row, div_khw, div_kw;  // fours of an image, of a row; terms of a channel, of a tap's row
  const float *bias;
  int32_t sB;
  int32_t chain_n;
  fl_ew_program chain;
};

template <int STEPS>
__global__ __launch_bounds__(kThreads, 4) void ConvShortKernel(float *out, const float *in, const float *w, ShortArgs p) {
  // (no __restrict__, and barriers for the scheduler: the loads would be moved to their use, one round trip after the other)
  constexpr int kTerms = 4 * STEPS, kPitch = kTerms + 1;  // (odd: lanes of consecutive filters in different banks)
  __shared__ float filters[16 * FT * kPitch], bias[16 * FT];
  const int lane = threadIdx.x % 64, c = lane % 16, g = lane / 16;
  const int f0 = static_cast<int>(blockIdx.y) * (16 * FT);
  // (runs past the last, all of whose pixels are, take part up to the barrier)
  const int run = static_cast<int>(blockIdx.x) * (kThreads / 64) + static_cast<int>(threadIdx.x / 64);

  // ---- the pixels: four neighbours of a row (past the last: the first four again, not stored) ------------------------
  const int n = run * 16 + c, count = n < p.fours ? n : 0;
  uint32_t img, rest, oh, four;
  p.div_image.DivMod(static_cast<uint32_t>(count), img, rest);
  p.div_row.DivMod(rest, oh, four);
  const int ow = 4 * static_cast<int>(four), stored = n < p.fours ? min(4, p.OW - ow) : 0;
  const int ih0 = static_cast<int>(oh) * p.sh - p.ph, iw0 = ow - p.pw;
  const int base = static_cast<int>(img) * p.sXn;
  const int dst = static_cast<int>(img) * p.sOn + static_cast<int>(oh) * p.sOh + ow;
  // the terms of this lane: 4 s + g
  float b[STEPS][4];
  int32_t shift[STEPS];  // columns the four were moved left by to lie in the image (-1: right); 4: nothing of them is wanted
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int k = 4 * s + g;
    uint32_t ch, tap, y, x;
    p.div_khw.DivMod(static_cast<uint32_t>(min(k, p.K - 1)), ch, tap);
    p.div_kw.DivMod(tap, y, x);
    const int ih = ih0 + static_cast<int>(y) * p.dh, iw = iw0 + static_cast<int>(x) * p.dw;
    const int row = min(max(ih, 0), p.H - 1), first = min(max(iw, 0), p.W - 4);
    const Quad q = *reinterpret_cast<const Quad *>(in + (base + static_cast<int>(ch) * p.sXc + row * p.sXh + first));
#pragma unroll
    for (int j = 0; j < 4; ++j) b[s][j] = q.v[j];
    shift[s] = row == ih && k < p.K ? min(iw - first, 4) : 4;
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the weights, through LDS ---------------------------------------------------------------------------------------
  constexpr int kAll = 16 * FT * kTerms, kPer = (kAll + kThreads - 1) / kThreads;
  float weight[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int i = static_cast<int>(threadIdx.x) + t * kThreads, f = i / kTerms, k = i % kTerms;
    uint32_t ch, tap, y, x;
    p.div_khw.DivMod(static_cast<uint32_t>(min(k, p.K - 1)), ch, tap);
    p.div_kw.DivMod(tap, y, x);
    weight[t] = w[min(f0 + f, p.F - 1) * p.sWf + static_cast<int32_t>(ch) * p.sWc + static_cast<int32_t>(y) * p.sWh + static_cast<int32_t>(x) * p.sWw];
  }
  const float *bias_at = p.bias != nullptr ? p.bias + min(f0 + static_cast<int>(threadIdx.x) % (16 * FT), p.F - 1) * p.sB : w;
  const float added = *bias_at;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int i = static_cast<int>(threadIdx.x) + t * kThreads, f = i / kTerms, k = i % kTerms;
    if (f < 16 * FT) filters[f * kPitch + k] = k < p.K ? weight[t] : 0.0f;
  }
  if (threadIdx.x < 16 * FT) bias[threadIdx.x] = p.bias != nullptr ? added : 0.0f;
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const bool right = shift[s] < 0, none = shift[s] == 4, one = !right && (shift[s] & 1) != 0, two = !right && (shift[s] & 2) != 0;
    const float v0 = b[s][0], v1 = b[s][1], v2 = b[s][2], v3 = b[s][3];
    // (one to the left, then two)
    const float u0 = one ? v1 : v0, u1 = one ? v2 : v1, u2 = one ? v3 : v2, u3 = one ? 0.0f : v3;
    b[s][0] = none || right ? 0.0f : two ? u2 : u0;
    b[s][1] = none ? 0.0f : right ? v0 : two ? u3 : u1;
    b[s][2] = none || two ? 0.0f : right ? v1 : u2;
    b[s][3] = none || two ? 0.0f : right ? v2 : u3;
  }
  __syncthreads();
  if (run >= p.runs) return;

  floatx4 acc[FT][4];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < STEPS; ++s)
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      const float a = filters[(16 * i + c) * kPitch + 4 * s + g];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[s][j], acc[i][j], 0, 0, 0);
    }

  StaticFor<FT>([&](auto i_c) {
    constexpr int i = decltype(i_c)::value;
    float vals[16];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) vals[4 * e + j] = acc[i][j][e] + bias[16 * i + 4 * g + e];
    if (p.chain_n != 0) RunChainBlock<16>(p.chain, vals);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int f = f0 + 16 * i + 4 * g + e;
      if (f >= p.F) continue;
      float *to = out + f * p.sOf + dst;
      if (stored == 4) {
        *reinterpret_cast<Quad *>(to) = Quad{{vals[4 * e], vals[4 * e + 1], vals[4 * e + 2], vals[4 * e + 3]}};
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          if (j < stored) to[j] = vals[4 * e + j];
        }
      }
    }
  });
}

}  // namespace

// FL_ERR_UNSUPPORTED (nothing launched) when the convolution does not fit this kernel.  Operands were validated by the caller.
int ConvShort(const fl_tensor *in, const fl_tensor *weights, const fl_tensor *bias, const fl_tensor *out, const int64_t *pads,
              const int64_t *strides, const int64_t *dilations, const fl_ew_program *chain, void *stream) {
  if (out->rank != 4) return FL_ERR_UNSUPPORTED;
  const int64_t C = in->shape[1], H = in->shape[2], W = in->shape[3], KH = weights->shape[2], KW = weights->shape[3];
  const int64_t F = out->shape[1], OH = out->shape[2], OW = out->shape[3];
  // (a single tap is a plain contraction, and goes there)
  if (C * KH * KW > 32 || KH * KW == 1 || F > 32 * 65535) return FL_ERR_UNSUPPORTED;
  // four neighbours of an output row read four neighbours of an input row
  if ((strides && strides[1] != 1) || in->strides[3] != 1 || out->strides[3] != 1 || W < 4 || (pads && pads[1] > 1)) return FL_ERR_UNSUPPORTED;
  // A launch of few waves takes the one trip to memory that every wave starts with, 6 to 7 us, and the implicit GEMM less.  Measured
  // (us, implicit GEMM and here, one image, kernels of 2 x 2 over eight channels): 16 filters of 56^2 5.7, 5.9, 96^2 6.4, 5.9; 32 of
  // 56^2 5.8, 6.6, 88^2 6.0, 6.6, 96^2 6.6, 6.7, 112^2 7.9, 6.8; 64 of 64^2 6.0, 6.7, 80^2 6.7, 6.8, 96^2 10.9, 6.9; 128 of 28^2 5.9,
  // 6.6, 56^2 6.7, 6.8: the line lies where there are 144 waves, whatever the kernel, the channels and the images.  The 3 x 3 kernels
  // of unit stride that conv_halo.hip takes otherwise cost more there: few waves 5.9, 5.9 to 6.1, 9216 pixels 6.9, 6.1; with
  // weights that it does not take, channels last, they do not: 64 filters of 14^2 4.9, 6.3.
  const bool halo = KH == 3 && KW == 3 && (!strides || strides[0] == 1) && (!dilations || (dilations[0] == 1 && dilations[1] == 1)) &&
                    weights->strides[3] == 1 && weights->strides[2] == 3 && weights->strides[1] == 9;
  if (!halo && out->shape[0] * OH * OW * ((F + 16 * FT - 1) / (16 * FT)) < 144 * 64) return FL_ERR_UNSUPPORTED;
  const int64_t fours = out->shape[0] * OH * ((OW + 3) / 4);
  if (fours > INT32_MAX - 64) return FL_ERR_UNSUPPORTED;
  ShortArgs p;
  std::memset(&p, 0, sizeof(p));
  p.F = static_cast<int32_t>(F), p.K = static_cast<int32_t>(C * KH * KW), p.fours = static_cast<int32_t>(fours);
  p.runs = static_cast<int32_t>((fours + 15) / 16);
  p.H = static_cast<int32_t>(H), p.W = static_cast<int32_t>(W), p.OW = static_cast<int32_t>(OW);
  p.sh = strides ? static_cast<int32_t>(strides[0]) : 1;
  p.dh = dilations ? static_cast<int32_t>(dilations[0]) : 1, p.dw = dilations ? static_cast<int32_t>(dilations[1]) : 1;
  p.ph = pads ? static_cast<int32_t>(pads[0]) : 0, p.pw = pads ? static_cast<int32_t>(pads[1]) : 0;
  p.sXn = static_cast<int32_t>(in->strides[0]), p.sXc = static_cast<int32_t>(in->strides[1]), p.sXh = static_cast<int32_t>(in->strides[2]);
  p.sOn = static_cast<int32_t>(out->strides[0]), p.sOf = static_cast<int32_t>(out->strides[1]), p.sOh = static_cast<int32_t>(out->strides[2]);
  p.sWf = static_cast<int32_t>(weights->strides[0]), p.sWc = static_cast<int32_t>(weights->strides[1]);
  p.sWh = static_cast<int32_t>(weights->strides[2]), p.sWw = static_cast<int32_t>(weights->strides[3]);
  p.div_image = FastDiv(static_cast<uint32_t>(OH * ((OW + 3) / 4))), p.div_row = FastDiv(static_cast<uint32_t>((OW + 3) / 4));
  p.div_khw = FastDiv(static_cast<uint32_t>(KH * KW)), p.div_kw = FastDiv(static_cast<uint32_t>(KW));
  if (bias != nullptr) p.bias = static_cast<const float *>(bias->base), p.sB = static_cast<int32_t>(bias->strides[0]);
  if (chain != nullptr) p.chain = *chain;
  p.chain_n = p.chain.n;
  float *o = static_cast<float *>(out->base);
  const float *x = static_cast<const float *>(in->base), *w = static_cast<const float *>(weights->base);
  const dim3 grid((p.runs + kThreads / 64 - 1) / (kThreads / 64), (p.F + 16 * FT - 1) / (16 * FT)), block(kThreads);
  if (p.K <= 28) FL_LAUNCH(ConvShortKernel<7>, grid, block, 0, AsStream(stream), o, x, w, p);
  else FL_LAUNCH(ConvShortKernel<8>, grid, block, 0, AsStream(stream), o, x, w, p);
  return LaunchStatus();
}

}  // namespace fl
