// Shared by the decode step's GEMMs (wgemm.hip, wgemm_wide.hip).
#pragma once

#include "pdk_common.h"

namespace wg {

using pdk::v8;

typedef __bf16 bf16x8_t __attribute__((__vector_size__(16)));
typedef float f32x4 __attribute__((__vector_size__(16)));

__device__ __forceinline__ f32x4 mfma(const v8& a, const v8& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

constexpr int kStepK = 128;        // k per wave step: 4 MFMA of 32
constexpr int kBlock = 16 * kStepK;  // tiled W: one tile's k step, 4 KiB

// kResidualSsq: kResidual that also writes, per 16-column tile and row, the
// sum of squares of the bf16 outputs (ssq[row][tile]): the raw material of the
// next RMSNorm. kSwiGLURms: kSwiGLU on weights with that norm's gain folded
// into their columns, whose input x is the un-normalised residual: each row's
// two sums are scaled by r = rsqrt(sum(ssq[row][.]) / K + eps) before SwiGLU,
// so rmsnorm(x) . W^T = r * (x . (W diag g)^T) takes no launch of its own.
//
// kPartialFinal: kPartial whose last-arriving split of each column group adds
// the splits' partials in split order to the residual (y = bf16(r + sum), r
// may alias y: the update pdk_rmsnorm_partials makes) and writes that
// group's sums of squares as kResidualSsq does, so the next RMSNorm needs no
// launch. kArgmaxRms: kArgmax on weights with the final norm's gain folded in,
// each row's logits scaled by its r (from ssq) before rounding. kPartialRms:
// kPartial on weights with a norm's gain folded in, each row's partial scaled
// by its r (the q|k|v projection: its consumer adds the scaled halves).
enum Epilogue { kPlain = 0, kResidual = 1, kSwiGLU = 2, kArgmax = 3, kPartial = 4,
                kResidualSsq = 5, kSwiGLURms = 6, kPartialFinal = 7, kArgmaxRms = 8,
                kPartialRms = 9 };

// Greedy-token key of one bf16 logit: the value in an order-preserving code
// above the complement of the column, so the unsigned maximum is the largest
// value at its lowest column (torch.argmax: NaN above every number, the first
// of equal values; -0 counts as +0). 0 is below every key.
__device__ __forceinline__ uint64_t argmax_key(uint32_t h, int n) {
  h &= 0xffffu;
  if (h == 0x8000u) h = 0;                                   // -0 -> +0
  uint32_t ord;
  if ((h & 0x7fffu) > 0x7f80u) ord = 0xffffu;               // NaN
  else ord = (h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u);
  return ((uint64_t)ord << 32) | (uint64_t)(0xffffffffu - (uint32_t)n);
}

// The canonical order of a sum over K. The k steps of 128 fall into 8 classes
// (step % 8), each class is one chain of MFMA in increasing step order, and
// the 8 class sums p0 .. p7 are added in a fixed order that every kernel of
// the same epilogue follows, so a row's result does not depend on which of
// them ran (a stream's tokens are then the same at any batch size):
//   kSwiGLURms, kArgmaxRms   (p0 + p1 + p2 + p3) + (p4 + p5 + p6 + p7), each
//                            half from 0 in order (two wavefronts with four
//                            classes each);
//   kResidualSsq, kResidual  c0 + c1 + c2 + c3 in order, cs = ps + p(s+4) (four
//                            workgroups, each with two classes);
//   the others               p0 + .. + p7 in order.
template <int kEpi>
__device__ __forceinline__ float sum_classes(const float p[8]) {
  if (kEpi == kResidualSsq || kEpi == kResidual)
    return (((p[0] + p[4]) + (p[1] + p[5])) + (p[2] + p[6])) + (p[3] + p[7]);
  if (kEpi == kSwiGLURms || kEpi == kArgmaxRms) {
    const float a = (((0.f + p[0]) + p[1]) + p[2]) + p[3];
    const float b = (((0.f + p[4]) + p[5]) + p[6]) + p[7];
    return a + b;
  }
  float sum = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) sum += p[q];
  return sum;
}

// The kernels of wgemm_wide.hip for more than 16 rows (tiled weights and
// activations), and the shapes they are used for.
bool wide_swiglu(int B, int K, int M);
bool wide_argmax(int B, int K, int N);
bool wide_ssq(int B, int K, int N);
int launch_wide_swiglu(const uint16_t* x, const uint16_t* w, int B, int K, int M, const float* ssq,
                       float eps, uint16_t* y, hipStream_t st);
int launch_wide_argmax(const uint16_t* x, const uint16_t* w, int B, int K, int N, const float* ssq,
                       float eps, uint16_t* logits, uint64_t* keys, hipStream_t st);
// part: kWideSplits * B * N floats; counters: ceil(N / 64) of kWideCounters
// zeros, left zero.
constexpr int kWideSplits = 4, kWideCounters = 4096;
int launch_wide_ssq(const uint16_t* x, const uint16_t* w, int B, int K, int N, const uint16_t* r,
                    uint16_t* y, float* ssq, float* part, int* counters, hipStream_t st);

}  // namespace wg
