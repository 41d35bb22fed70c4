// The prefill's GEMMs for prompts of up to 512 tokens, for gfx950:
//   part[s][T][N] = X[T][K_s] . W[N][K_s]^T      fp32 partial sums of K range s
//   Y[T][M]       = silu(X . Wg^T) * (X . Wu^T)   (W = [Wg; Wu]), bf16
// W is [out][in] bf16 as the caller holds it; the sums stay fp32 up to the one
// rounding by whoever reads them (RoPE, the norm's residual add) or, for
// SwiGLU, in the epilogue.
//
// Up to some 150 tokens a projection is bound by reading W once, beyond that by
// the matrix cores on too few tiles: N = 4096 at 470 tokens has 128 tiles of 128
// x 128 for 256 CUs. So K is split until every CU has a workgroup, and W and X
// stream through LDS: each stage is 64 columns of K of both, loaded by
// global_load_lds (16 bytes a lane, no registers), kStages - 1 stages ahead. One
// barrier per stage: it waits for the wavefront's own loads of the oldest stage
// (vmcnt counts the younger ones) and for its LDS reads of the stage whose
// buffer is refilled next.
//
// LDS rows are 64 columns (128 bytes, eight 16-byte chunks); chunk c of row r
// holds columns 8 (c ^ (r / 2 & 7)) .., so that each group of 16 lanes that a
// ds_read_b128 serves in one cycle touches all 64 banks: no conflicts counted,
// where c ^ (r & 7) has as many conflict cycles as useful ones. global_load_lds
// writes LDS in lane order, so the swizzle is applied to the addresses the lanes
// load from.
//
// With one or two K splits (gate|up, the lm_head) the workgroups would read the
// same columns at a time, rows 8 KiB apart, which the memory channels serve
// unevenly: each column tile starts 8 stages after its neighbour and wraps around
// (gate|up at 41 tokens 46.4 -> 42.1 us, 1 token 44.0 -> 42.0, 100 tokens 49.5 ->
// 47.3; the lm_head of 16032 rows 30.9 -> 24.0).
//
// W is the A operand and X the B operand of v_mfma_f32_16x16x32_bf16: a lane
// then holds four consecutive output columns of one token.
//
// Measured in us, library GEMM -> this one (launches in a HIP graph over
// weights that do not fit the last-level cache; HBM alone at 6 TB/s in brackets):
//   tokens                     1            41           128          470
//   q|k|v   4096 -> 6144  [8]  14.5 -> 10.4 17.7 -> 11.9 25.6 -> 16.0
//   O       4096 -> 4096  [6]  15.5 ->  7.4 13.7 ->  8.5 24.4 -> 11.7 28.7 -> 24.1
//   down   14336 -> 4096 [20]  26.5 -> 21.2 39.4 -> 22.8 75.4 -> 29.4 93.0 -> 64.3
//   gate|up 4096 -> 28672 [39] 57.0 -> 42.0 48.5 -> 42.1 55.1 -> 50
// (gate|up with its SwiGLU, which is a launch of its own after the library's).
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "wgemm_common.h"

namespace {

using namespace wg;

constexpr int kBK = 64;                   // columns of K per stage
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// All but the youngest N of this wavefront's loads have arrived and its LDS
// reads are done; then the workgroup's barrier. (__syncthreads would wait for
// every load.) The memory clobber keeps LDS accesses on their side.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// BM tokens x BN weight rows per workgroup, WM x WN wavefronts. kGlu: BN / 2
// gate rows and the matching up rows, a lane holding both of an output.
// Consecutive workgroups go to the 8 XCDs in turn; each XCD gets a contiguous
// run of units with the token tile fastest, so the token tiles that share a
// part of W read it through one L2.
template <int BM, int BN, int WM, int WN, int kStages, bool kGlu, int kMinWaves>
__global__ __launch_bounds__(64 * WM * WN, kMinWaves) void prefill_gemm_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int T, int K, int N,
    int splits, int m_tiles, void* __restrict__ out) {
  constexpr int kWaves = WM * WN;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;  // fragments per wavefront
  constexpr int BC = kGlu ? BN / 2 : BN;               // output columns
  constexpr int kStage = (BM + BN) * kBK;
  constexpr int kLoads = (BM + BN) / 8;                // of 8 rows (1 KiB) per stage
  constexpr int L = (kLoads + kWaves - 1) / kWaves;    // per wavefront
  static_assert(BM % (16 * WM) == 0 && BN % ((kGlu ? 32 : 16) * WN) == 0, "whole fragments");
  static_assert((kStages - 2) * L < 64, "vmcnt is 6 bits");
  __shared__ __align__(1024) uint16_t sm[kStages * kStage];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave % WM, wn = wave / WM;
  int unit;
  {
    const int q = gridDim.x >> 3, r = gridDim.x & 7, xcd = blockIdx.x & 7;
    unit = xcd * q + min(xcd, r) + (blockIdx.x >> 3);
  }
  const int m0 = unit % m_tiles * BM;
  unit /= m_tiles;
  const int split = unit % splits, n0 = unit / splits * BC;
  const int steps_all = K / kBK;
  const int first = (int)((int64_t)split * steps_all / splits);
  const int n = (int)((int64_t)(split + 1) * steps_all / splits) - first;   // >= kStages - 1

  // This lane's source of each load: stage row r (W's BN rows, then X's BM;
  // rows past the end read the last one, their results are dropped). When the
  // loads do not divide evenly the last one is made more than once.
  const uint16_t* src[L];
  int dst[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int at = min(wave + i * kWaves, kLoads - 1);
    const int r = at * 8 + (lane >> 3);
    const uint16_t* p;
    if (at >= BN / 8) p = x + (int64_t)min(m0 + r - BN, T - 1) * K;
    else if (kGlu && r >= BC) p = w + (int64_t)(N + min(n0 + r - BC, N - 1)) * K;
    else p = w + (int64_t)min(n0 + r, N - 1) * K;
    src[i] = p + (int64_t)first * kBK + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
    dst[i] = at * 512;
  }
  f32x4 acc[FN][FM];
#pragma unroll
  for (int a = 0; a < FN; ++a)
#pragma unroll
    for (int b = 0; b < FM; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A fragment's lane reads row lane % 16, columns 32 kc + 8 (lane / 16) .. + 7.
  const int frag = (lane & 15) * kBK + ((lane >> 4) ^ ((lane >> 1) & 7)) * 8;
  int row[FN];                                         // first W row of fragment a
#pragma unroll
  for (int a = 0; a < FN; ++a)
    row[a] = kGlu ? (a < FN / 2 ? 0 : BC) + wn * (BC / WN) + a % (FN / 2) * 16
                  : wn * (BN / WN) + a * 16;

  const int rot = splits <= 2 ? n0 / BC * 8 % n : 0;
  auto issue = [&](uint16_t* __restrict__ to, int i) __attribute__((always_inline)) {
    const int step = i + rot - (i + rot >= n ? n : 0);
#pragma unroll
    for (int l = 0; l < L; ++l)
      __builtin_amdgcn_global_load_lds((global_void*)(src[l] + (int64_t)step * kBK),
                                       (lds_void*)(to + dst[l]), 16, 0, 0);
  };
  auto products = [&](const uint16_t* __restrict__ from) __attribute__((always_inline)) {
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      v8 fw[FN], fx[FM];
#pragma unroll
      for (int a = 0; a < FN; ++a) fw[a] = pdk::ld16(from + row[a] * kBK + (frag ^ (32 * kc)));
#pragma unroll
      for (int b = 0; b < FM; ++b)
        fx[b] = pdk::ld16(from + (BN + wm * (BM / WM) + b * 16) * kBK + (frag ^ (32 * kc)));
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b) acc[a][b] = mfma(fw[a], fx[b], acc[a][b]);
    }
  };
  // The two buffers are different ones; without __restrict__ the compiler
  // would wait for the loads just issued before it reads.
  auto both = [&](const uint16_t* __restrict__ from, uint16_t* __restrict__ to,
                  int step) __attribute__((always_inline)) {
    issue(to, step);
    products(from);
  };
#pragma unroll
  for (int j = 0; j < kStages - 1; ++j) issue(sm + j * kStage, j);
  int rb = 0, wb = kStages - 1;
  for (int i = 0; i < n - (kStages - 1); ++i) {
    stage_barrier<(kStages - 2) * L>();
    both(sm + rb * kStage, sm + wb * kStage, i + kStages - 1);
    rb = rb + 1 == kStages ? 0 : rb + 1;
    wb = wb + 1 == kStages ? 0 : wb + 1;
  }
  auto tail = [&](auto j) __attribute__((always_inline)) {   // the last stages load nothing
    stage_barrier<(kStages - 2 - decltype(j)::value) * L>();
    products(sm + rb * kStage);
    rb = rb + 1 == kStages ? 0 : rb + 1;
  };
  static_assert(kStages == 3 || kStages == 4, "two or three stages in the tail");
  tail(std::integral_constant<int, 0>{});
  tail(std::integral_constant<int, 1>{});
  if constexpr (kStages == 4) tail(std::integral_constant<int, 2>{});

  // acc[a][b][e]: token m0 + .. + lane % 16, column n0 + .. + 4 (lane / 16) + e.
#pragma unroll
  for (int b = 0; b < FM; ++b) {
    const int t = m0 + wm * (BM / WM) + b * 16 + (lane & 15);
    if (t >= T) continue;
#pragma unroll
    for (int a = 0; a < (kGlu ? FN / 2 : FN); ++a) {
      const int c = n0 + row[a] + 4 * (lane >> 4);     // N % 4 == 0: four columns or none
      if (c >= N) continue;
      if constexpr (kGlu) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = acc[a][b][e], u = acc[a + FN / 2][b][e];
          o[e] = g / (1.f + expf(-g)) * u;
        }
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + (int64_t)t * N + c) =
            make_uint2(pdk::pack_bf16x2_rne(o[0], o[1]), pdk::pack_bf16x2_rne(o[2], o[3]));
      } else {
        *reinterpret_cast<f32x4*>(static_cast<float*>(out) + ((int64_t)split * T + t) * N + c) =
            acc[a][b];
      }
    }
  }
}

// The best wg::argmax_key of 1024 columns of one row of partial sums, added in
// order and rounded to bf16 (the logit), per workgroup.
__global__ __launch_bounds__(256) void prefill_argmax_kernel(const float* part, int splits, int N,
                                                             uint64_t* keys) {
  __shared__ uint64_t best[4];
  const int c = (blockIdx.x * 256 + threadIdx.x) * 4;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  const int at = min(c, N - 4);                        // N % 4 == 0
  for (int s = 0; s < splits; ++s)
    sum += *reinterpret_cast<const f32x4*>(part + (int64_t)s * N + at);
  uint64_t key = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c < N) key = max(key, argmax_key(pdk::pack_bf16x2_rne(sum[e], 0.f), c + e));
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) key = max(key, (uint64_t)__shfl_xor((unsigned long long)key, o));
  if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = key;
  __syncthreads();
  if (threadIdx.x == 0) keys[blockIdx.x] = max(max(best[0], best[1]), max(best[2], best[3]));
}

// Tiles by the number of tokens. At most 64 of them leave the kernel bound by
// W, where 128 weight rows x 3 stages (48 KiB; 64 KiB of LDS) per CU are in flight
// and more rows of X would only take LDS; from 129 on two token tiles share each
// part of W. Without a K split (gate|up) the 64-column tiles of 17 to 32 tokens make a
// nearly empty second wave: 51.3 us at 17 tokens in the model, 64 x 128 tiles
// take 42.7.
// Splits fill 256 CUs (two workgroups each for the 36 KiB tiles), at most 8
// and each of at least 4 stages: one split more costs T * N * 8 bytes.
//
// narrow: where 128 columns would need those 8 splits of a short K (the O
// projection: N and K 4096), 64 columns and 4 splits: O at 1 token 8.0 -> 7.4 us,
// 24 8.5 -> 7.9, 41 9.6 -> 8.5, 100 12.2 -> 10.9, and half the partial sums to read.
// The down projection (K 14336) has stages enough and gains nothing from it.
struct Plan {
  int bm, bn, target;
  bool narrow;
};
Plan plan_for(int T, int K, int cols, bool glu) {
  if (T > 128) return {128, 256, 256, false};
  const bool narrow = !glu && K <= 4096 && (cols + 127) / 128 <= 32;
  if (T <= 16) return {16, narrow ? 64 : 128, 256, narrow};
  if (T <= 32 && !glu) return {32, 64, narrow ? 256 : 512, narrow};
  if (T <= 64) return {64, narrow ? 64 : 128, 256, narrow};
  return {128, narrow ? 64 : 128, 256, narrow};
}
int64_t tiles_of(const Plan& p, int T, int cols) {
  return (int64_t)((T + p.bm - 1) / p.bm) * ((cols + p.bn - 1) / p.bn);
}

// Up to 256 tokens always; up to 512 where the library's tiles leave most of
// the chip idle (at most 64 tiles of 128 x 256 here: N = 4096 and less). At 470
// tokens: O 28.7 library, 24.1 here, down 93.0 and 64.3; but q|k|v 33.4 and 36.5,
// gate|up 104 (with SwiGLU 115) and 120 of the best tile, 132 of these.
// Around the second token tile (us with the kernel that reads the result,
// library -> here):
//   tokens   112          128          129          160          192          256
//   q|k|v    27.2 -> 20.7 28.7 -> 21.5 41.4 -> 27.5 31.5 -> 27.8 37.1 -> 28.7 43.6 -> 29.2
//   O        19.8 -> 15.2 27.9 -> 16.1 25.3 -> 23.0 30.3 -> 22.9 36.2 -> 23.7 26.2 -> 25.4
//   down     53.6 -> 32.5 78.7 -> 33.6 57.3 -> 42.9 86.9 -> 43.8  106 -> 44.8 65.1 -> 46.9
//   gate|up  59.4 -> 49.7 56.9 -> 51.3 60.3 -> 72.4 61.4 -> 74.0 66.3 -> 73.3 73.0 -> 76.5
// From 129 tokens on gate|up by itself is slower here, in the model by less: a
// prefill of 4 layers takes 767 us with it and 751 with the library's at 129
// tokens, 783 and 765 at 160, 811 and 831 at 200, 847 and 866 at 256. It stays the
// kernel's over the whole range because its sums are 32-bit up to SwiGLU's result:
// the error of the KV against 64 bits is 0.0072 instead of 0.0078.
bool takes(int T, int K, int rows) {
  if (T < 1 || K < 4 * kBK || K % kBK || rows < 4 || rows % 4) return false;
  return T <= 256 || (T <= 512 && tiles_of(plan_for(T, K, rows, false), T, rows) <= 64);
}

int splits_for(int T, int K, int N) {
  const Plan p = plan_for(T, K, N, false);
  const int64_t s = p.target / tiles_of(p, T, N);
  return (int)std::max<int64_t>(1, std::min<int64_t>({s, 8, K / kBK / 4}));
}

template <bool kGlu>
int launch(const uint16_t* x, const uint16_t* w, int T, int K, int N, int splits, void* out,
           hipStream_t st) {
  const Plan p = plan_for(T, K, N, kGlu);
  const int m_tiles = (T + p.bm - 1) / p.bm;
  const int64_t blocks = tiles_of(p, T, kGlu ? 2 * N : N) * splits;
  PDK_REQUIRE(blocks < (1ll << 31), "launch too large");
#define PDK_PG(BM, BN, WM, WN, S, OCC)                                                        \
  hipLaunchKernelGGL((prefill_gemm_kernel<BM, BN, WM, WN, S, kGlu, OCC>), dim3((unsigned)blocks), \
                     dim3(64 * WM * WN), 0, st, x, w, T, K, N, splits, m_tiles, out)
  if constexpr (!kGlu) {                         // tiles gate|up never takes
    if (p.narrow) {
      if (T <= 16) PDK_PG(16, 64, 1, 4, 4, 2);
      else if (T <= 32) PDK_PG(32, 64, 1, 4, 4, 2);
      else if (T <= 64) PDK_PG(64, 64, 2, 2, 4, 2);
      else PDK_PG(128, 64, 4, 2, 4, 1);
      return pdk::check_launch("prefill_gemm_kernel");
    }
    if (p.bm == 32) {
      PDK_PG(32, 64, 2, 2, 3, 4);
      return pdk::check_launch("prefill_gemm_kernel");
    }
  }
  if (T <= 16) PDK_PG(16, 128, 1, 4, 4, 1);
  else if (T <= 64) PDK_PG(64, 128, 2, 4, 4, 1);
  else if (T <= 128) PDK_PG(128, 128, 2, 4, 4, 2);
  else PDK_PG(128, 256, 2, 4, 3, 2);
#undef PDK_PG
  return pdk::check_launch("prefill_gemm_kernel");
}

int check(const void* x, const void* w, const void* out) {
  PDK_REQUIRE(x && w && out, "null pointer argument");
  PDK_REQUIRE(pdk::aligned16(x) && pdk::aligned16(w) && pdk::aligned16(out),
              "tensors must be 16-byte aligned");
  return PDK_OK;
}

}  // namespace

extern "C" int pdk_prefill_gemm_splits(int T, int K, int N) {
  return takes(T, K, N) ? splits_for(T, K, N) : 0;
}

extern "C" int pdk_prefill_gemm(const uint16_t* x, const uint16_t* w, int T, int K, int N,
                                float* partials, uintptr_t stream) {
  pdk::clear_error();
  if (int rc = check(x, w, partials)) return rc;
  PDK_REQUIRE(takes(T, K, N), "T=%d K=%d N=%d is not a shape this GEMM takes", T, K, N);
  return launch<false>(x, w, T, K, N, splits_for(T, K, N), partials, pdk::as_stream(stream));
}

// Without a K split the SwiGLU's tiles alone fill the chip, or do not.
extern "C" int pdk_prefill_gemm_swiglu_takes(int T, int K, int M) {
  return T <= 256 && M >= 1 && M < (1 << 30) && M % 4 == 0 && takes(T, K, 2 * M);
}

extern "C" int pdk_prefill_gemm_swiglu(const uint16_t* x, const uint16_t* w_gate_up, int T, int K,
                                       int M, uint16_t* y, uintptr_t stream) {
  pdk::clear_error();
  if (int rc = check(x, w_gate_up, y)) return rc;
  PDK_REQUIRE(pdk_prefill_gemm_swiglu_takes(T, K, M), "T=%d K=%d M=%d is not a shape this GEMM takes",
              T, K, M);
  return launch<true>(x, w_gate_up, T, K, M, 1, y, pdk::as_stream(stream));
}

extern "C" int pdk_prefill_argmax(const float* partials, int splits, int N, uint64_t* keys,
                                  uintptr_t stream) {
  pdk::clear_error();
  PDK_REQUIRE(partials && keys, "null pointer argument");
  PDK_REQUIRE(pdk::aligned16(partials) && ((uintptr_t)keys & 7u) == 0,
              "partials must be 16-byte aligned and keys 8-byte aligned");
  PDK_REQUIRE(N >= 4 && N % 4 == 0, "N must be a positive multiple of 4 (got %d)", N);
  PDK_REQUIRE(splits >= 1 && splits <= 64, "splits must be in [1, 64] (got %d)", splits);
  hipLaunchKernelGGL(prefill_argmax_kernel, dim3((N + 1023) / 1024), dim3(256), 0,
                     pdk::as_stream(stream), partials, splits, N, keys);
  return pdk::check_launch("prefill_argmax_kernel");
}
