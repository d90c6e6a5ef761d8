// Projections of up to 16 rows, out[M, N] = f(x[M, K]) W[N, K]^T in bf16 with fp32
// sums: the products of a decode step of few sequences (gfx950).
//
// Bound by the weights' bytes, each needed once, and below about 30 MB by the fixed
// costs of a launch; so one launch does what surrounds the product too, and even a
// matrix of a few MB is in flight on the whole chip at once.
//
//   - Operands go straight from memory into the layout of
//     v_mfma_f32_16x16x32_bf16 (A = weights: row = lane%16, k = 8*(lane/16)..+7;
//     B = tokens: column = lane%16; C: column = lane%16, rows 4*(lane/16)+r).
//   - With M tokens only 16/KH >= M of the 16 columns are needed, so K is cut in KH
//     slices that take the rest: A's rows are 16/KH weight rows times KH slices, B's
//     columns 16/KH tokens times KH slices, and the result is the sum of the
//     blocks on C's diagonal. That sets a workgroup's share to 16, 8 or 4 weight
//     rows (KH = 1, 2, 4) without a masked lane.
//   - The workgroup's waves share out the slices in chunks and add up through LDS. A
//     wave with several chunks asks for the next one's weights ahead of a chunk's
//     products, under a condition, so that the wait before those covers them too.
//   - NORM: the tokens are RMS-normalised on the way in: x times the norm's weights
//     (rounded, as a normalised row is) goes to LDS once per workgroup, while the
//     first weights travel, its squares are summed beside, and the row's factor
//     meets the fp32 sums at the end. (Weighting each operand where it is used cost
//     16384 x 2048 pairs with one token 25.3 instead of 17.3 us: more vector work than the
//     weights' bytes leave time for.)
//   - RES: the sums are added to the residual in place. ACT: half of the weight
//     rows are gates, half the values that they act on (x = [gate | up]).
//   - ROPE (the q/k/v projection): a workgroup takes channel pairs of one head, rotates
//     q and k and writes k and v into the paged cache too; positions and
//     angles are read while the weights travel. A launch of its own for that took 4.5 us
//     a layer (a step of llama-3.2-1b, one sequence: 902 us, 873 without it).

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short sg_s16x8;
typedef __attribute__((ext_vector_type(4))) unsigned sg_u32x4;
typedef __attribute__((ext_vector_type(4))) float sg_f32x4;
typedef __attribute__((ext_vector_type(2))) float sg_f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 sg_bf16x2;

enum : int { kSgPlain = 0, kSgResidual = 1, kSgSilu = 2, kSgGelu = 3, kSgRope = 4 };

// What kSgRope needs: the paged caches [blocks, kv_heads, bs, D] (bf16 or e4m3),
// cos_sin [positions, D] as cosines | sines, a cache slot per row (negative: none).
struct SgRope {
  void *k_cache, *v_cache;
  const long *positions, *slots;
  const float* cos_sin;
  int heads, kv_heads, D, bs;
  bool fp8;
};

// Places of weighted tokens in LDS (shorts): the 16 columns of an operand read lie in
// 16 different 16-byte bank groups where slices are multiples of 128.
template <int KH>
struct SgTokens {
  static constexpr int kPlaces = 16 / KH;
  __host__ __device__ static int slice(int K) { return K / KH + 8 * kPlaces; }
  __host__ __device__ static int row(int K) { return (KH * slice(K) + 127) / 128 * 128 + 8; }
};

// KH: slices of K (16 / KH >= M); NW: waves; KU: 32-wide K steps of a chunk.
template <int KH, int NW, int KU, bool NORM, int EPI>
__global__ __launch_bounds__(64 * NW) void stream_gemm_kernel(
    __hip_bfloat16* __restrict__ out, long out_stride,
    const __hip_bfloat16* __restrict__ x, long x_stride,
    const __hip_bfloat16* __restrict__ wt, const __hip_bfloat16* __restrict__ bias,
    const __hip_bfloat16* __restrict__ norm_w, float eps, float offset,
    int M, int N, int K, SgRope rope) {
  constexpr int R = 16 / KH, MP = 16 / KH, KC = 32 * KU;   // weight rows, token places
  constexpr bool PAIR = EPI >= kSgSilu;
  constexpr int RO = PAIR ? R / 2 : R;                     // output columns (kSgRope: pairs)
  constexpr int RP = 17;
  __shared__ float red[NW][16 * RP];
  __shared__ float sums[NW][16];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int ks = K / KH;
  // a pair's second row lies `apart` rows behind its first; halves of a head are pairs
  const int half = EPI == kSgRope ? rope.D / 2 : 0;
  const int head = EPI == kSgRope ? blockIdx.x * RO / half : 0;
  const int n0 = blockIdx.x * RO + head * half;
  const int apart = EPI == kSgRope ? half : N / 2;
  const int i = col % R;
  const int wrow = PAIR && i >= RO ? apart + n0 + i - RO : n0 + i;
  const long kslice = (long)(col / R) * ks + grp * 8;
  const __hip_bfloat16* wp = wt + (long)wrow * K + kslice;
  const __hip_bfloat16* xp = x + (long)min(col % MP, M - 1) * x_stride + kslice;
  extern __shared__ __align__(16) short tokens[];
  const short* tp = tokens + min(col % MP, M - 1) * SgTokens<KH>::row(K) +
                    (col / R) * SgTokens<KH>::slice(K) + grp * 8;
  sg_f32x4 acc = {0.f, 0.f, 0.f, 0.f};

  sg_s16x8 wf[KU], wn[KU];
  auto fetch = [&](sg_s16x8 (&f)[KU], int k0) {
#pragma unroll
    for (int u = 0; u < KU; ++u)
      f[u] = __builtin_nontemporal_load(reinterpret_cast<const sg_s16x8*>(wp + k0 + u * 32));
  };
  int k0 = w * KC;
  long slot = -1, position = 0;
  float cosine = 1.f, sine = 0.f;
  if constexpr (EPI == kSgRope) {      // one sum per thread: 4 RO MP <= 64 NW
    const int m = min(((int)threadIdx.x >> 2) / RO, M - 1);
    position = rope.positions[m];
    slot = rope.slots[m];
  }
  if (k0 < ks) fetch(wf, k0);
  if constexpr (EPI == kSgRope) {
    if (head < rope.heads + rope.kv_heads) {
      const float* cs = rope.cos_sin + position * rope.D + (n0 - head * rope.D) +
                        (threadIdx.x >> 2) % RO;
      cosine = cs[0];
      sine = cs[half];
    }
  }
  if constexpr (NORM) {
    for (int m = 0; m < M; ++m) {
      float ss = 0.f;
      for (int k = threadIdx.x * 8; k < K; k += 64 * NW * 8) {
        const Vec8<__hip_bfloat16> xv = load16(x + (long)m * x_stride + k);
        const Vec8<__hip_bfloat16> nv = load16(norm_w + k);
        sg_u32x4 y;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float a = to_f32(xv.data[e]), b = to_f32(xv.data[e + 1]);
          ss += a * a + b * b;
          y[e / 2] = __builtin_bit_cast(unsigned, __builtin_convertvector(
              (sg_f32x2{a * (to_f32(nv.data[e]) + offset), b * (to_f32(nv.data[e + 1]) + offset)}),
              sg_bf16x2));
        }
        *reinterpret_cast<sg_u32x4*>(tokens + m * SgTokens<KH>::row(K) +
                                     (k / ks) * SgTokens<KH>::slice(K) + k % ks) = y;
      }
      ss = wave_reduce_sum(ss);
      if (lane == 0) sums[w][m] = ss;
    }
    __syncthreads();
  }
  for (; k0 < ks; k0 += NW * KC) {
    sg_s16x8 xf[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u)
      xf[u] = NORM ? *reinterpret_cast<const sg_s16x8*>(tp + k0 + u * 32)
                   : *reinterpret_cast<const sg_s16x8*>(xp + k0 + u * 32);
    const int next = k0 + NW * KC;
    if (next < ks) fetch(wn, next);
#pragma unroll
    for (int u = 0; u < KU; ++u)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf[u], acc, 0, 0, 0);
#pragma unroll
    for (int u = 0; u < KU; ++u) wf[u] = wn[u];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[w][(grp * 4 + r) * RP + col] = acc[r];
  __syncthreads();
  // four threads per sum: each takes every fourth wave
  auto total = [&](int m, int row, int part) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NW / 4; ++v)
#pragma unroll
      for (int h = 0; h < KH; ++h)
        s += red[part + v * 4][(h * R + row) * RP + h * MP + m];
    s += __shfl_xor(s, 1, WAVE);
    s += __shfl_xor(s, 2, WAVE);
    return s;
  };
  static_assert(EPI != kSgRope || 4 * RO * MP <= 64 * NW, "angles of one sum per thread");
  for (int t = threadIdx.x; t < 4 * RO * MP; t += 64 * NW) {
    const int part = t & 3, row = (t >> 2) % RO, m = (t >> 2) / RO;
    float y = total(m, row, part);
    float up = 0.f, inv = 1.f;
    if constexpr (PAIR) up = total(m, row + RO, part);
    if constexpr (NORM) {
      float q = 0.f;
#pragma unroll
      for (int v = 0; v < NW / 4; ++v) q += sums[part + v * 4][min(m, M - 1)];
      q += __shfl_xor(q, 1, WAVE);
      q += __shfl_xor(q, 2, WAVE);
      inv = rsqrtf(q / K + eps);
    }
    if (part != 0 || m >= M) continue;
    const int n = n0 + row;
    y *= inv;
    if (bias) y += to_f32(bias[n]);
    if constexpr (EPI == kSgRope) {
      up *= inv;
      if (bias) up += to_f32(bias[n + half]);
      const __hip_bfloat16 a = __float2bfloat16(y * cosine - up * sine);
      const __hip_bfloat16 b = __float2bfloat16(up * cosine + y * sine);
      __hip_bfloat16* o = out + (long)m * out_stride + n;
      o[0] = a;
      o[half] = b;
      if (head < rope.heads || slot < 0) continue;
      const bool is_v = head >= rope.heads + rope.kv_heads;
      const int kh = head - rope.heads - (is_v ? rope.kv_heads : 0);
      const long at = ((slot / rope.bs * rope.kv_heads + kh) * rope.bs + slot % rope.bs) * rope.D +
                      n - head * rope.D;
      void* cache = is_v ? rope.v_cache : rope.k_cache;
      if (rope.fp8) {                      // from the rounded rows, as elsewhere
        __hip_fp8_e4m3* c = static_cast<__hip_fp8_e4m3*>(cache) + at;
        c[0] = from_f32<__hip_fp8_e4m3>(to_f32(a));
        c[half] = from_f32<__hip_fp8_e4m3>(to_f32(b));
      } else {
        __hip_bfloat16* c = static_cast<__hip_bfloat16*>(cache) + at;
        c[0] = a;
        c[half] = b;
      }
      continue;
    }
    if constexpr (EPI == kSgSilu || EPI == kSgGelu) {
      up *= inv;
      if constexpr (EPI == kSgSilu) {
        y = y / (1.0f + __expf(-y)) * up;
      } else {               // tanh form of GELU
        y = 0.5f * y * (1.0f + tanhf(0.7978845608028654f * (y + 0.044715f * y * y * y))) * up;
      }
    }
    __hip_bfloat16* o = out + (long)m * out_stride + n;
    if constexpr (EPI == kSgResidual) y += to_f32(*o);
    *o = __float2bfloat16(y);
  }
}
