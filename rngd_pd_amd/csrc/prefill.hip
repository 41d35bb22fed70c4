// The prefill's non-GEMM kernels for gfx950: RoPE fused with the KV outputs,
// and causal GQA attention over one prompt of T tokens (head_dim 128).
//
// rope_kv_kernel reads the q|k|v projection [T][(NH + 2 NKV) 128] once. It
// rotates q in place, writes the rotated k and v to the caller's [T][NKV][128]
// rows (the handoff's source), and lays k and v out a second time as the
// attention's MFMA operands, one 32-token tile (8 KiB each) after another:
//   kt [kvh][tile][s = 0..7][lane][8]: MFMA A operand of k-step s (dims 16s ..
//      16s + 15): lane 32 hh + r holds token pi(r), dims 16 s + 8 hh + e;
//   vt [kvh][tile][n = 0..3][ks = 0..1][lane][8]: lane 32 hh + r holds dim 32 n
//      + r of tokens 16 ks + 8 hh + e (V transposed);
// pi swaps bits 2 and 3 of the index. Tokens past T are zero in both.
//
// attn kernel: S^T = K Q^T with v_mfma_f32_32x32x16_bf16, so a lane holds one
// query (column j = lane & 31) and 16 of the tile's 32 scores; with pi its
// accumulators 8 ks .. 8 ks + 7 are tokens 16 ks + 8 (lane >> 5) + 0..7, which
// is the B operand that O^T += V^T P^T needs, with no exchange between lanes.
// Maximum, sum and rescale are per lane (one lane swap each).
//
// The weights P stay 32-bit: each is split exactly into three bf16 parts (8
// mantissa bits each; truncation, so hi + mid + lo is the float itself) and
// multiplied part by part into one fp32 accumulator: 3 MFMA per V operand read
// instead of a 16-bit P.
//
// Measured per layer at Llama-3.1-8B shape (32 query, 8 KV heads): the attention
// takes 273 us at T = 4000 and 25 us at T = 470, RoPE with the KV outputs 22 and
// 6 us; as fp32 torch operations over a [32, T, T] score matrix in HBM the two
// took 5.4 ms and 0.17 ms.
#include <math.h>

#include <algorithm>

#include "pdk_common.h"

namespace {

using pdk::v8;

typedef __bf16 bf16x8_t __attribute__((__vector_size__(16)));
typedef float f32x16 __attribute__((__vector_size__(64)));

constexpr int kD = 128;
constexpr int kTile = 32;                 // tokens per K/V tile and queries per wavefront
constexpr int kTileElems = kTile * kD;    // 4096 bf16 = 8 KiB
constexpr int kAttnWaves = 4;

__device__ __forceinline__ f32x16 mfma32(const v8& a, const v8& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ float vmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// The row of the S^T tile that holds token x of the tile, and the reverse.
__device__ __forceinline__ int pi(int x) { return (x & 0x13) | ((x & 4) << 1) | ((x & 8) >> 1); }

// table[t][i] = (cos, sin)(t * inv_freq[i]), fp32.
__global__ __launch_bounds__(256) void rope_table_kernel(const float* inv_freq, int T, int half,
                                                         float2* table) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= T * half) return;
  const int t = idx / half, i = idx - t * half;
  float s, c;
  sincosf((float)t * inv_freq[i], &s, &c);
  table[idx] = make_float2(c, s);
}

// Eight elements of `splits` partial rows, added in order and rounded to bf16.
__device__ __forceinline__ v8 partial_sum(const float* p, int splits, int64_t stride) {
  float s[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) s[k] = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 4) {          // four splits' loads in flight
    float4 u[4], v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* q = p + min(s0 + i, splits - 1) * stride;
      u[i] = *reinterpret_cast<const float4*>(q);
      v[i] = *reinterpret_cast<const float4*>(q + 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (s0 + i >= splits) break;
      s[0] += u[i].x; s[1] += u[i].y; s[2] += u[i].z; s[3] += u[i].w;
      s[4] += v[i].x; s[5] += v[i].y; s[6] += v[i].z; s[7] += v[i].w;
    }
  }
  v8 r;
#pragma unroll
  for (int w = 0; w < 4; ++w) r.w[w] = pdk::pack_bf16x2_rne(s[2 * w], s[2 * w + 1]);
  return r;
}

// One workgroup: a 32-token tile of kRopeHeads consecutive heads (of NH q, NKV
// k, NKV v). Thread (r, o) = (tid / 8, tid % 8) holds token r, dims 8o..8o+7
// and 64+8o..+7 (a rotation pair per element), and its 8 (cos, sin) pairs stay
// in registers for all the heads: reading them per head would move as many
// bytes as the heads themselves. Bound by the bytes of q|k|v in and out.
//
// kPart: q|k|v comes as `splits` fp32 partial sums [s][T][(NH + 2 NKV) 128]
// (pdk_prefill_gemm's), added in order and rounded to bf16 once, and q goes to
// rows of its own. Those are prompts of at most a few tiles: one head per
// workgroup, so that more than 12 workgroups per tile share the reads.
constexpr int kRopeHeads = 4;
constexpr int kVRow = kD + 2;             // LDS row of the V transpose

template <bool kPart>
__global__ __launch_bounds__(256) void rope_kv_kernel(uint16_t* qkv, const float* part, int splits,
                                                      const float2* table, int T, int NH, int NKV,
                                                      uint16_t* k_out, int64_t k_ld,
                                                      uint16_t* v_out, int64_t v_ld, uint16_t* kt,
                                                      uint16_t* vt) {
  constexpr int kHeads = kPart ? 1 : kRopeHeads;
  __shared__ uint16_t vs[kTile][kVRow];
  const int tile = blockIdx.x, n_tiles = gridDim.x;
  const int r = threadIdx.x >> 3, o = threadIdx.x & 7;
  const int t = tile * kTile + r;
  const bool live = t < T;
  const int tc = min(t, T - 1);
  float2 cs[8];
  {
    const float4* p = reinterpret_cast<const float4*>(table + (int64_t)tc * (kD / 2) + 8 * o);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 x = p[i];
      cs[2 * i] = make_float2(x.x, x.y);
      cs[2 * i + 1] = make_float2(x.z, x.w);
    }
  }
  const int n_heads = NH + 2 * NKV;
  uint16_t* row = qkv + (int64_t)tc * (kPart ? NH : n_heads) * kD + 8 * o;
  const int h0 = blockIdx.y * kHeads;
  v8 a[kHeads], b[kHeads];
#pragma unroll
  for (int i = 0; i < kHeads; ++i) {
    const int hd = min(h0 + i, n_heads - 1);
    if constexpr (kPart) {
      const float* p = part + ((int64_t)tc * n_heads + hd) * kD + 8 * o;
      a[i] = partial_sum(p, splits, (int64_t)T * n_heads * kD);
      b[i] = partial_sum(p + kD / 2, splits, (int64_t)T * n_heads * kD);
    } else {
      a[i] = pdk::ld16(row + (int64_t)hd * kD);
      b[i] = pdk::ld16(row + (int64_t)hd * kD + kD / 2);
    }
  }
#pragma unroll
  for (int i = 0; i < kHeads; ++i) {
    const int hd = h0 + i;
    if (hd >= n_heads) break;                      // uniform
    if (hd < NH + NKV) {
      v8 x, y;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float u0, u1, v0, v1;
        pdk::rope_pair(pdk::bf16_to_f32(a[i].w[w] & 0xffffu), pdk::bf16_to_f32(b[i].w[w] & 0xffffu),
                       cs[2 * w].x, cs[2 * w].y, u0, v0);
        pdk::rope_pair(pdk::bf16_to_f32(a[i].w[w] >> 16), pdk::bf16_to_f32(b[i].w[w] >> 16),
                       cs[2 * w + 1].x, cs[2 * w + 1].y, u1, v1);
        x.w[w] = pdk::pack_bf16x2_rne(u0, u1);
        y.w[w] = pdk::pack_bf16x2_rne(v0, v1);
      }
      if (hd < NH) {
        if (live) {
          pdk::st16(row + (int64_t)hd * kD, x);
          pdk::st16(row + (int64_t)hd * kD + kD / 2, y);
        }
      } else {
        const int h = hd - NH;
        if (live) {
          uint16_t* p = k_out + (int64_t)t * k_ld + h * kD + 8 * o;
          pdk::st16(p, x);
          pdk::st16(p + kD / 2, y);
        } else {
          x = y = pdk::zero8();
        }
        // dims 8o.. are k-step o / 2, half o % 2; dims 64 + 8o.. k-step o / 2 + 4.
        uint16_t* p = kt + ((int64_t)h * n_tiles + tile) * kTileElems +
                      ((o >> 1) * 64 + (o & 1) * 32 + pi(r)) * 8;
        pdk::st16(p, x);
        pdk::st16(p + 4 * 64 * 8, y);
      }
    } else {
      const int h = hd - NH - NKV;
      v8 x = a[i], y = b[i];
      if (live) {
        uint16_t* p = v_out + (int64_t)t * v_ld + h * kD + 8 * o;
        pdk::st16(p, x);
        pdk::st16(p + kD / 2, y);
      } else {
        x = y = pdk::zero8();
      }
      __syncthreads();                             // the previous V head has left vs
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        *reinterpret_cast<uint32_t*>(&vs[r][8 * o + 2 * w]) = x.w[w];
        *reinterpret_cast<uint32_t*>(&vs[r][kD / 2 + 8 * o + 2 * w]) = y.w[w];
      }
      __syncthreads();
      uint16_t* p = vt + ((int64_t)h * n_tiles + tile) * kTileElems;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int u = threadIdx.x + 256 * j;       // unit (n, ks, lane)
        const int lane = u & 63, ks = (u >> 6) & 1, n = u >> 7;
        const int d = 32 * n + (lane & 31), t0 = 16 * ks + 8 * (lane >> 5);
        v8 g;
#pragma unroll
        for (int w = 0; w < 4; ++w)
          g.w[w] = (uint32_t)vs[t0 + 2 * w][d] | ((uint32_t)vs[t0 + 2 * w + 1][d] << 16);
        pdk::st16(p + u * 8, g);
      }
    }
  }
}

// One wavefront: 32 queries (tile qt) of one query head. Units (qt, head of the
// KV group) are laid end to end, G heads of a tile next to each other, and a
// workgroup takes kAttnWaves consecutive units of one KV head, so that its
// wavefronts read the same K/V tiles from LDS (for G = 4 exactly the group's
// heads at one tile). Workgroups go longest first (the last query tile has the
// most K/V tiles), with the KV head the fastest index: 8 KV heads spread over
// the 8 XCDs and each XCD's L2 holds one head's K/V (2 MiB at T = 4096).
// K/V tiles are double buffered in LDS (32 KiB); the next tile's global loads
// are in flight during a tile's products.
//
// Per tile a wavefront issues 8 MFMA for QK and 24 for PV (three parts of P),
// 1024 cycles of matrix work against 16 KiB of LDS reads and the softmax of 16
// scores per lane; two workgroups per CU overlap one's softmax with the
// other's products.
__global__ __launch_bounds__(64 * kAttnWaves, 2) void prefill_attn_kernel(
    const uint16_t* q, int64_t q_ld, const uint16_t* kt, const uint16_t* vt, int T, int NH,
    int NKV, float c, uint16_t* out) {
  __shared__ __align__(16) uint16_t smem[2][2 * kTileElems];   // [buffer][K tile, V tile]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int j = lane & 31, hh = lane >> 5;
  const int n_tiles = (T + kTile - 1) / kTile;
  const int G = NH / NKV, units = n_tiles * G;
  const int kvh = blockIdx.x % NKV;
  const int wg = (units + kAttnWaves - 1) / kAttnWaves - 1 - (int)(blockIdx.x / NKV);
  const int unit = min(wg * kAttnWaves + wave, units - 1);     // a spare wavefront repeats the last
  const int qt = unit / G, head = kvh * G + (unit - qt * G);
  // K/V tiles the workgroup walks: up to its last unit's query tile.
  const int n_kv = min(wg * kAttnWaves + kAttnWaves - 1, units - 1) / G + 1;

  v8 qv[8];
  {
    const uint16_t* p = q + (int64_t)min(qt * kTile + j, T - 1) * q_ld + head * kD + 8 * hh;
#pragma unroll
    for (int s = 0; s < 8; ++s) qv[s] = pdk::ld16(p + 16 * s);
  }
  const uint16_t* kp = kt + (int64_t)kvh * n_tiles * kTileElems + threadIdx.x * 8;
  const uint16_t* vp = vt + (int64_t)kvh * n_tiles * kTileElems + threadIdx.x * 8;
  v8 pre[4];
  auto fetch = [&](int tile) __attribute__((always_inline)) {
    const int64_t at = (int64_t)tile * kTileElems;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      pre[i] = pdk::ld16(kp + at + 2048 * i);
      pre[2 + i] = pdk::ld16(vp + at + 2048 * i);
    }
  };
  auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      pdk::st16(&smem[buf][threadIdx.x * 8 + 2048 * i], pre[i]);
      pdk::st16(&smem[buf][kTileElems + threadIdx.x * 8 + 2048 * i], pre[2 + i]);
    }
  };

  f32x16 o[4];
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.f;
  float m = -INFINITY, l = 0.f;           // m: raw-score maximum in use; l: this lane's tokens

  fetch(0);
  stash(0);
  __syncthreads();
  for (int tile = 0; tile < n_kv; ++tile) {
    const int buf = tile & 1;
    if (tile + 1 < n_kv) fetch(tile + 1);
    if (tile <= qt) {                     // uniform across the wavefront
      const uint16_t* ks_ = &smem[buf][lane * 8];
      const uint16_t* vs_ = &smem[buf][kTileElems + lane * 8];
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) s = mfma32(pdk::ld16(ks_ + 512 * k), qv[k], s);
      if (tile == qt) {                   // tokens after the query (and so those past T)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (16 * (i >> 3) + 8 * hh + (i & 7) > j) s[i] = -INFINITY;
      }
      float mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = vmax(mx, s[i]);
      {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx),
                                                        false, false);
        mx = vmax(__uint_as_float(x[0]), __uint_as_float(x[1]));
      }
      // The maximum in use follows the running one only when it falls more than
      // 2^8 behind: P then stays within 2^8 in fp32 (no precision is lost by a
      // common factor) and O is rescaled a few times per query instead of at
      // almost every tile.
      if (__any((mx - m) * c > 8.f)) {
        const float m_new = vmax(m, mx);
        const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - m_new) * c);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[n][i] *= alpha;
      }
      const float mc = m == -INFINITY ? 0.f : m * c;
      v8 p0[2], p1[2], p2[2];
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c, -mc));
        const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i + 1], c, -mc));
        l += x;
        l += y;
        const uint32_t xu = __float_as_uint(x), yu = __float_as_uint(y);
        const float x1 = x - __uint_as_float(xu & 0xffff0000u);
        const float y1 = y - __uint_as_float(yu & 0xffff0000u);
        const uint32_t x1u = __float_as_uint(x1), y1u = __float_as_uint(y1);
        const uint32_t x2u = __float_as_uint(x1 - __uint_as_float(x1u & 0xffff0000u));
        const uint32_t y2u = __float_as_uint(y1 - __uint_as_float(y1u & 0xffff0000u));
        const int k = i >> 3, w = (i & 7) >> 1;
        p0[k].w[w] = __builtin_amdgcn_perm(yu, xu, 0x07060302u);
        p1[k].w[w] = __builtin_amdgcn_perm(y1u, x1u, 0x07060302u);
        p2[k].w[w] = __builtin_amdgcn_perm(y2u, x2u, 0x07060302u);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const v8 va = pdk::ld16(vs_ + 512 * (2 * n + k));
          o[n] = mfma32(va, p2[k], o[n]);
          o[n] = mfma32(va, p1[k], o[n]);
          o[n] = mfma32(va, p0[k], o[n]);
        }
    }
    if (tile + 1 < n_kv) stash(buf ^ 1);  // last read before the previous barrier
    __syncthreads();
  }
  {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false,
                                                    false);
    l = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  const float inv = 1.f / l;              // the query's own token is always there: l > 0
  const int t = qt * kTile + j;
  // Lane (hh, j) holds dims 32n + 8g + 4hh + 0..3 of query j (g = 0..3); a lane
  // swap of groups g, g + 1 gives each half 8 consecutive dims: 16-byte stores.
  uint16_t* op = out + ((int64_t)min(t, T - 1) * NH + head) * kD + 8 * hh;
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      uint32_t w[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          w[i][e] = pdk::pack_bf16x2_rne(o[n][4 * (g + i) + 2 * e] * inv,
                                         o[n][4 * (g + i) + 2 * e + 1] * inv);
      const auto a = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
      const auto b = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
      const v8 res{{a[0], b[0], a[1], b[1]}};
      if (t < T && wg * kAttnWaves + wave < units) pdk::st16(op + 32 * n + 8 * g, res);
    }
}

int check_prefill(int T, int NH, int NKV) {
  PDK_REQUIRE(T >= 1 && T <= (1 << 20), "T must be in [1, 2^20] (got %d)", T);
  PDK_REQUIRE(NKV >= 1 && NH >= NKV && NH % NKV == 0 && NH + 2 * NKV <= 65535,
              "n_q_heads=%d must be a multiple of n_kv_heads=%d", NH, NKV);
  return PDK_OK;
}

}  // namespace

extern "C" int pdk_rope_table(const float* inv_freq, int T, int half, float* table,
                              uintptr_t stream) {
  pdk::clear_error();
  PDK_REQUIRE(inv_freq && table && pdk::aligned16(table), "null pointer or table not 16-byte aligned");
  PDK_REQUIRE(T >= 1 && half >= 1 && (int64_t)T * half < (1ll << 31) - 256, "T or half out of range");
  hipLaunchKernelGGL(rope_table_kernel, dim3((T * half + 255) / 256), dim3(256), 0,
                     pdk::as_stream(stream), inv_freq, T, half, reinterpret_cast<float2*>(table));
  return pdk::check_launch("rope_table_kernel");
}

extern "C" int64_t pdk_prefill_kv_tile_elems(int T, int n_kv_heads) {
  if (T < 1 || n_kv_heads < 1) return 0;
  return (int64_t)n_kv_heads * ((T + kTile - 1) / kTile) * kTileElems;
}

namespace {

template <bool kPart>
int rope_kv(uint16_t* qkv, const float* part, int splits, const float* table, int T,
            int n_q_heads, int n_kv_heads, int head_dim, uint16_t* k_out, int64_t k_tok_stride,
            uint16_t* v_out, int64_t v_tok_stride, uint16_t* kt, uint16_t* vt, uintptr_t stream) {
  pdk::clear_error();
  if (head_dim != kD) {
    pdk::set_error("the prefill kernels implement head_dim %d only (got %d)", kD, head_dim);
    return PDK_ENOTSUP;
  }
  if (int rc = check_prefill(T, n_q_heads, n_kv_heads)) return rc;
  PDK_REQUIRE(qkv && table && k_out && v_out && kt && vt, "null pointer argument");
  PDK_REQUIRE(pdk::aligned16(qkv) && pdk::aligned16(table) && pdk::aligned16(k_out) &&
                  pdk::aligned16(v_out) && pdk::aligned16(kt) && pdk::aligned16(vt),
              "tensors must be 16-byte aligned");
  PDK_REQUIRE(k_tok_stride >= (int64_t)n_kv_heads * kD && k_tok_stride % 8 == 0 &&
                  v_tok_stride >= (int64_t)n_kv_heads * kD && v_tok_stride % 8 == 0,
              "token strides must be multiples of 8 and hold Hkv * D elements");
  PDK_REQUIRE(!kPart || (part && pdk::aligned16(part)), "partials must be 16-byte aligned");
  PDK_REQUIRE(!kPart || (splits >= 1 && splits <= 64), "splits must be in [1, 64] (got %d)",
              splits);
  const int heads = kPart ? 1 : kRopeHeads;
  const dim3 grid((T + kTile - 1) / kTile, (n_q_heads + 2 * n_kv_heads + heads - 1) / heads);
  hipLaunchKernelGGL(rope_kv_kernel<kPart>, grid, dim3(256), 0, pdk::as_stream(stream), qkv, part,
                     splits, reinterpret_cast<const float2*>(table), T, n_q_heads, n_kv_heads,
                     k_out, k_tok_stride, v_out, v_tok_stride, kt, vt);
  return pdk::check_launch("rope_kv_kernel");
}

}  // namespace

extern "C" int pdk_prefill_rope_kv(uint16_t* qkv, const float* table, int T, int n_q_heads,
                                   int n_kv_heads, int head_dim, uint16_t* k_out,
                                   int64_t k_tok_stride, uint16_t* v_out, int64_t v_tok_stride,
                                   uint16_t* kt, uint16_t* vt, uintptr_t stream) {
  return rope_kv<false>(qkv, nullptr, 0, table, T, n_q_heads, n_kv_heads, head_dim, k_out,
                        k_tok_stride, v_out, v_tok_stride, kt, vt, stream);
}

extern "C" int pdk_prefill_rope_kv_partials(const float* partials, int splits, const float* table,
                                            int T, int n_q_heads, int n_kv_heads, int head_dim,
                                            uint16_t* q_out, uint16_t* k_out, int64_t k_tok_stride,
                                            uint16_t* v_out, int64_t v_tok_stride, uint16_t* kt,
                                            uint16_t* vt, uintptr_t stream) {
  return rope_kv<true>(q_out, partials, splits, table, T, n_q_heads, n_kv_heads, head_dim, k_out,
                       k_tok_stride, v_out, v_tok_stride, kt, vt, stream);
}

extern "C" int pdk_prefill_attn(const uint16_t* q, int64_t q_tok_stride, const uint16_t* kt,
                                const uint16_t* vt, int T, int n_q_heads, int n_kv_heads,
                                int head_dim, float scale, uint16_t* out, uintptr_t stream) {
  pdk::clear_error();
  if (head_dim != kD) {
    pdk::set_error("the prefill kernels implement head_dim %d only (got %d)", kD, head_dim);
    return PDK_ENOTSUP;
  }
  if (int rc = check_prefill(T, n_q_heads, n_kv_heads)) return rc;
  PDK_REQUIRE(q && kt && vt && out, "null pointer argument");
  PDK_REQUIRE(pdk::aligned16(q) && pdk::aligned16(kt) && pdk::aligned16(vt) && pdk::aligned16(out),
              "tensors must be 16-byte aligned");
  PDK_REQUIRE(q_tok_stride >= (int64_t)n_q_heads * kD && q_tok_stride % 8 == 0,
              "the token stride must be a multiple of 8 and hold Hq * D elements");
  PDK_REQUIRE(scale > 0.f && scale < INFINITY, "scale must be positive and finite (got %g)",
              (double)scale);
  const int64_t units = (int64_t)((T + kTile - 1) / kTile) * (n_q_heads / n_kv_heads);
  const int64_t blocks = (units + kAttnWaves - 1) / kAttnWaves * n_kv_heads;
  PDK_REQUIRE(units < (1ll << 30) && blocks < (1ll << 31), "launch too large");
  hipLaunchKernelGGL(prefill_attn_kernel, dim3((unsigned)blocks), dim3(64 * kAttnWaves), 0,
                     pdk::as_stream(stream), q, q_tok_stride, kt, vt, T, n_q_heads, n_kv_heads,
                     scale * 1.4426950408889634f, out);
  return pdk::check_launch("prefill_attn_kernel");
}
