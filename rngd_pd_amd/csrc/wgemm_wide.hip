// The decode step's GEMMs for 17 to 64 rows on tiled weights and activations
// (gate|up with SwiGLU, the lm_head with its argmax, the down projection), for
// gfx950.
//
// wgemm_kernel gives every wavefront all rows and its own k steps, so each
// workgroup reads the whole X for its 16 or 32 columns: at B = 50 that is 4 or
// 2 times the weight bytes out of L2, which bounds it (27-30 bytes per clock
// and CU in all), not HBM. Here four wavefronts take 16 columns each at the
// same k step and read that step of X from LDS, where the workgroup put it
// once: X costs as many bytes as W. Two such groups share the workgroup, each
// with half of the k step classes, so that 8 wavefronts stream weights.
//
// Per step a wavefront reads its W tile (pair) straight into registers, two
// steps ahead; X goes global -> registers two steps ahead -> LDS one step
// ahead, in the MFMA operand order of pdk::act_at (linear 16-byte units, no
// bank conflicts). One barrier per step. Four steps of W ahead instead of two
// were no faster (gate|up 40.9 and 41.2 us at B = 20).
//
// Sums follow wg::sum_classes, so the results are bit for bit those of
// wgemm_kernel. K / 128 must be a multiple of 16: 8 classes of an even number
// of steps (two steps per loop turn, whose LDS buffers alternate). Widths such as
// 3072, 5120, 11008 and 13824 are not, and their products keep wgemm_kernel.
//
// Measured (us, launches of a HIP graph over weights that do not fit the last-
// level cache, before -> after): gate|up M = 14336, K = 4096 B=50 66.9 -> 44.5,
// B=20 41.7 -> 40.8; lm_head N = 128256 B=50 443 -> 214, B=20 213 -> 180; down
// N = 4096, K = 14336 B=50 35.7 -> 27.0, B=20 27.6 -> 23.6. HBM alone would take
// 39, 175 and 20 at 6 TB/s. The O projection (K = 4096) does not gain (B=50 13.7
// and 13.7, B=20 10.2 and 10.9): its 4 steps per wavefront do not pay for the
// second pass over the partial sums.

#include <math.h>

#include <type_traits>

#include "wgemm_common.h"

namespace {

using namespace wg;

constexpr int kWn = 4, kWk = 2;                  // wavefronts over columns, over classes
constexpr int kThreads = 64 * kWn * kWk, kGroup = 64 * kWn;

// R row tiles (B <= 16 R). kEpi: kSwiGLURms, kArgmaxRms (one workgroup per 64
// columns, each group of wavefronts four classes in turn) or kResidualSsq
// (gridDim.y = kWideSplits workgroups per 64 columns, group g of workgroup s
// class 4 g + s; the last of them to finish adds the partial sums).
template <int R, int kEpi>
__global__ __launch_bounds__(kThreads) void wgemm_wide_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int B, int K, int N, float* ssq,
    const uint16_t* r, uint16_t* y, uint64_t* keys, float* part, float eps, int* counters) {
  constexpr bool kGLU = kEpi == kSwiGLURms, kArg = kEpi == kArgmaxRms;
  constexpr bool kSplit = kEpi == kResidualSsq;
  constexpr int kW = kGLU ? 2 : 1;               // W tiles per wavefront and step
  constexpr int kCpg = kSplit ? 1 : 4;           // classes per wavefront
  constexpr int kU = R;                          // 16-byte units of X per thread and step
  constexpr int kBuf = kWk * R * kBlock;         // one step of X for both groups
  __shared__ __align__(16) uint16_t xs[2 * kBuf];
  __shared__ float rms[kSplit ? 1 : 16 * R];
  __shared__ uint64_t kbest[kArg ? 16 * R : 1][kArg ? kWn : 1];
  __shared__ int is_last;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wn = wave % kWn, wk = wave / kWn;
  const int col = lane & 15, kg = lane >> 4;
  const int n_tiles = (N + 15) >> 4;
  const int tile = blockIdx.x * kWn + wn;        // the wavefront's column tile
  const int64_t step_stride = (int64_t)kW * n_tiles * kBlock;
  const uint16_t* wp[kW];
#pragma unroll
  for (int p = 0; p < kW; ++p)
    wp[p] = w + ((int64_t)p * n_tiles + min(tile, n_tiles - 1)) * kBlock + lane * 8;
  // Unit u of a step of X: row tile u / 256, its 16-byte unit v = u % 256 (rows
  // past B read row B - 1, as everywhere).
  const int tg = threadIdx.x % kGroup;
  const uint16_t* xp[kU];
#pragma unroll
  for (int i = 0; i < kU; ++i) {
    const int row = min(i * 16 + (tg & 15), B - 1);
    xp[i] = x + (int64_t)(row >> 4) * 16 * K + ((tg >> 4) * 16 + (row & 15)) * 8;
  }
  static_assert(kGroup == 256, "one row tile's units are one per thread of a group");
  const int n = K / kStepK >> 3;                 // steps of a class, even
  const int total = kCpg * n;
  struct Step { int q, j; };                     // class, step of it: k step q + 8 j
  auto next = [&](Step& s) { if (++s.j == n) { s.j = 0; ++s.q; } };
  Step cx{kSplit ? 4 * wk + (int)blockIdx.y : 4 * wk, 0}, cw = cx;

  v8 wv[2][kW][4], xv[2][kU];
  auto load_x = [&](int set) __attribute__((always_inline)) {
    const int64_t at = (int64_t)(cx.q + 8 * cx.j) * kBlock;
#pragma unroll
    for (int i = 0; i < kU; ++i) xv[set][i] = pdk::ld16(xp[i] + at);
    next(cx);
  };
  auto load_w = [&](int set) __attribute__((always_inline)) {
    const int64_t at = (cw.q + 8 * cw.j) * step_stride;
#pragma unroll
    for (int p = 0; p < kW; ++p)
#pragma unroll
      for (int c = 0; c < 4; ++c) wv[set][p][c] = pdk::ld16_stream(wp[p] + at + 512 * c);
    next(cw);
  };
  auto stash = [&](int set) __attribute__((always_inline)) {
    uint16_t* d = xs + set * kBuf + wk * R * kBlock + tg * 8;
#pragma unroll
    for (int i = 0; i < kU; ++i) pdk::st16(d + i * kBlock, xv[set][i]);
  };

  f32x4 acc[kW][R], tot[kW][R];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < kW; ++p)
#pragma unroll
    for (int t = 0; t < R; ++t) acc[p][t] = tot[p][t] = zero;
  load_x(0);
  load_w(0);
  load_x(1);
  load_w(1);
  if constexpr (!kSplit) {                       // row scales of the folded norm
    const int n_ssq = K >> 4;
    for (int m = threadIdx.x >> 5; m < 16 * R; m += kThreads / 32) {
      const int mc = min(m, B - 1);
      const pdk::RowRms rr = pdk::row_rms_load(ssq, mc, n_ssq, lane);
      const float s = pdk::row_rms_finish(rr, ssq, mc, n_ssq, K, eps, lane);
      if ((lane & 31) == 0) rms[m] = s;
    }
  }
  stash(0);
  __syncthreads();

  // One step from buffer `set`. Its X registers were stashed a step ago and
  // take the step after next; the W registers are refilled once used. No load
  // is conditional at run time (a path around a load would make the waits
  // before the products drain the loads behind it): the last two steps, which
  // load nothing, are code of their own.
  int left = n;
  auto step = [&](auto set_c, auto load_c, auto stash_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    if (decltype(load_c)::value) load_x(set);
    const uint16_t* xb = xs + set * kBuf + wk * R * kBlock + lane * 8;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const v8 xf = pdk::ld16(xb + t * kBlock + 512 * c);
#pragma unroll
        for (int p = 0; p < kW; ++p) acc[p][t] = mfma(xf, wv[set][p][c], acc[p][t]);
      }
    if (decltype(load_c)::value) load_w(set);
    if constexpr (!kSplit && set == 1) {
      if ((left -= 2) == 0) {                    // a class is complete
#pragma unroll
        for (int p = 0; p < kW; ++p)
#pragma unroll
          for (int t = 0; t < R; ++t) {
            tot[p][t] += acc[p][t];
            acc[p][t] = zero;
          }
        left = n;
      }
    }
    if (decltype(stash_c)::value) stash(set ^ 1);
    __syncthreads();
  };
  constexpr std::integral_constant<int, 0> even;
  constexpr std::integral_constant<int, 1> odd;
  for (int i = 2; i < total; i += 2) {
    step(even, std::true_type{}, std::true_type{});
    step(odd, std::true_type{}, std::true_type{});
  }
  step(even, std::false_type{}, std::true_type{});
  step(odd, std::false_type{}, std::false_type{});

  // The two groups exchange their sums of the row tiles the other one
  // finishes (group g finishes tiles t with t % 2 == g), through the X buffers
  // (free since the last barrier; kW <= 2 tiles of 4 KiB per wavefront fit).
  static_assert(kWn * R * kW * 64 * 16 <= 2 * kBuf * 2, "the exchange fits the X buffers");
  f32x4* red = reinterpret_cast<f32x4*>(xs);
  auto mine = [&](int p, int t) { return kSplit ? acc[p][t] : tot[p][t]; };
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int p = 0; p < kW; ++p)
      if ((t & 1) != wk) red[((wn * R + t) * kW + p) * 64 + lane] = mine(p, t);
  __syncthreads();
  f32x4 sum[kW][R];
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int p = 0; p < kW; ++p)
      if ((t & 1) == wk) sum[p][t] = mine(p, t) + red[((wn * R + t) * kW + p) * 64 + lane];

  // sum[p][t][i] is row 16 t + 4 kg + i, column n of tile p.
  const int nc = 16 * tile + col;
  auto finish = [&](int t, int i, float v, float u) __attribute__((always_inline)) {
    const int m = 16 * t + 4 * kg + i;
    const bool ok = m < B && nc < N;
    const int64_t at = kArg ? (int64_t)m * N + nc : pdk::act_at(m, nc, N);
    float out = v;
    if (kSplit && ok) out += pdk::bf16_to_f32(r[at]);
    if (kGLU) {
      const float a = v * rms[m], b = u * rms[m];
      out = a / (1.f + expf(-a)) * b;
    }
    if (kArg) out = v * rms[m];
    const uint32_t h = pdk::f32_to_bf16_rne(out);
    if (ok && y) y[at] = (uint16_t)h;
    if (kSplit) {                                // 16 lanes hold a row's 16 columns
      const float hv = pdk::bf16_to_f32(h);
      float sq = ok ? hv * hv : 0.f;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) sq += __shfl_xor(sq, o);
      if (col == 0 && ok) ssq[(int64_t)m * (N >> 4) + tile] = sq;
    }
    if (kArg) {
      uint64_t key = ok ? argmax_key(h, nc) : 0;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const uint64_t other = __shfl_xor(key, o);
        key = other > key ? other : key;
      }
      if (col == 0) kbest[m][wn] = key;
    }
  };
  if constexpr (kSplit) {
    // Partial sums to the workspace and a ticket, as in wgemm_kernel's
    // kPartialFinal (where the ordering is argued): agent-scope accesses, the
    // stores complete before the ticket, the last workgroup finishes and
    // resets the count. No workgroup waits for another.
    float* mp = part + (int64_t)blockIdx.y * B * N;
#pragma unroll
    for (int t = 0; t < R; ++t)
      if ((t & 1) == wk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 16 * t + 4 * kg + i;
          if (m < B && nc < N)
            __hip_atomic_store(mp + (int64_t)m * N + nc, sum[0][t][i], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
      int* cnt = counters + blockIdx.x;
      const int done = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = done == kWideSplits - 1;
      if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      is_last = last;
    }
    __syncthreads();
    if (!is_last) return;
    float pv[(R + 1) / 2][4][kWideSplits];
#pragma unroll
    for (int t = 0; t < R; ++t)
      if ((t & 1) == wk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int s = 0; s < kWideSplits; ++s)
            pv[t >> 1][i][s] = __hip_atomic_load(
                part + ((int64_t)s * B + min(16 * t + 4 * kg + i, B - 1)) * N + min(nc, N - 1),
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int t = 0; t < R; ++t)
      if ((t & 1) == wk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* p = pv[t >> 1][i];
          finish(t, i, ((p[0] + p[1]) + p[2]) + p[3], 0.f);
        }
    return;
  }
#pragma unroll
  for (int t = 0; t < R; ++t)
    if ((t & 1) == wk)
#pragma unroll
      for (int i = 0; i < 4; ++i) finish(t, i, sum[0][t][i], sum[kW - 1][t][i]);
  if constexpr (kArg) {
    __syncthreads();
    const int m = threadIdx.x;                   // 16 R <= 64 rows, one thread each
    if (m < min(16 * R, B)) {
      uint64_t best = kbest[m][0];
#pragma unroll
      for (int c = 1; c < kWn; ++c) best = kbest[m][c] > best ? kbest[m][c] : best;
      uint64_t* slot = keys + m;
      if (best > __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        __hip_atomic_fetch_max(slot, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

template <int kEpi>
int go(const uint16_t* x, const uint16_t* w, int B, int K, int N, float* ssq, const uint16_t* r,
       uint16_t* y, uint64_t* keys, float* part, float eps, int* counters, hipStream_t st) {
  const dim3 grid((N + 16 * kWn - 1) / (16 * kWn), kEpi == kResidualSsq ? kWideSplits : 1);
#define PDK_WIDE(R)                                                                            \
  hipLaunchKernelGGL((wgemm_wide_kernel<R, kEpi>), grid, dim3(kThreads), 0, st, x, w, B, K, N, \
                     ssq, r, y, keys, part, eps, counters)
  switch ((B + 15) / 16) {
    case 2: PDK_WIDE(2); break;
    case 3: PDK_WIDE(3); break;
    default: PDK_WIDE(4); break;
  }
#undef PDK_WIDE
  return pdk::check_launch("wgemm_wide_kernel");
}

// More than one row tile, and whole classes of an even number of steps.
bool fits(int B, int K) { return B > 16 && B <= 64 && K > 0 && K % (16 * kStepK) == 0; }

}  // namespace

namespace wg {

// 64 columns per workgroup: below 192 workgroups wgemm_kernel's narrower ones
// fill the chip better (lm_head N = 8016, 126 workgroups: 23.3 against 20.7 us at
// B = 20, 29.5 against 26.7 at B = 50; N = 16032, 251: 30.5 against 30.9, 36.1
// against 36.6).
bool wide_swiglu(int B, int K, int M) { return fits(B, K) && (M + 63) / 64 >= 192; }
bool wide_argmax(int B, int K, int N) { return fits(B, K) && (N + 63) / 64 >= 192; }
// Each class needs enough steps to pay for the partial sums (8 and more; with
// 4 it is slower, above), and the 4 x N / 64 workgroups have to fill the chip.
bool wide_ssq(int B, int K, int N) {
  return fits(B, K) && K / kStepK >= 64 && N >= 4096 && N % kStepK == 0 &&
         N <= 64 * kWideCounters;
}

int launch_wide_swiglu(const uint16_t* x, const uint16_t* w, int B, int K, int M, const float* ssq,
                       float eps, uint16_t* y, hipStream_t st) {
  return go<kSwiGLURms>(x, w, B, K, M, const_cast<float*>(ssq), nullptr, y, nullptr, nullptr, eps,
                        nullptr, st);
}

int launch_wide_argmax(const uint16_t* x, const uint16_t* w, int B, int K, int N, const float* ssq,
                       float eps, uint16_t* logits, uint64_t* keys, hipStream_t st) {
  return go<kArgmaxRms>(x, w, B, K, N, const_cast<float*>(ssq), nullptr, logits, keys, nullptr,
                        eps, nullptr, st);
}

int launch_wide_ssq(const uint16_t* x, const uint16_t* w, int B, int K, int N, const uint16_t* r,
                    uint16_t* y, float* ssq, float* part, int* counters, hipStream_t st) {
  return go<kResidualSsq>(x, w, B, K, N, ssq, r, y, nullptr, part, 0.f, counters, st);
}

}  // namespace wg
