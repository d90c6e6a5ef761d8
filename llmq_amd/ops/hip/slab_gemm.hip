// Projections of up to 128 rows, x[M, K] W[N, K]^T with fp32 sums, by 64-bit addresses:
// for operands that ring_gemm.hip cannot reach with 32-bit offsets (rows spread over
// 4 GiB). And the kernels that add up the slabs of either.
//
// A workgroup owns 64 weight rows, all M tokens and, as it is launched, all of K (a grid
// of several parts in y would leave a slab each). Weights go straight from memory into the
// matrix layout; the tokens, which every workgroup reads again, are staged once per
// workgroup in LDS by global_load_lds (16-byte granules placed by row, so operand reads
// meet no bank conflict). v_mfma_f32_16x16x32_bf16, A = weights (row = lane%16, k =
// 8*(lane/16)..+7), B = tokens likewise, C: column = token, rows = 4 weight rows.
// A step of 128 channels asks for the next step's tokens at its start and for the
// weights of the one after at its end, but its products wait for both: the loads sit
// under conditions, and the compiler's count of what may still travel is the least over
// all paths: 2.6 to 2.7 TB/s, where the ring kernel reads 3.7 to 6 (64 rows, 2048 x 8192:
// 12.4 us against 9.0). Gate and value rows (PAIR) are activated here.

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short sl_s16x8;
typedef __attribute__((ext_vector_type(4))) float sl_f32x4;

enum : int { kSlabSums = 0, kSlabSilu = 1, kSlabGelu = 2 };

constexpr int kSlabBK = 128;

// TM: token tiles of 16; WK: groups of four waves that take the K steps in turn (gate
// and value rows).
template <int TM, int WK, int EPI>
__global__ __launch_bounds__(256 * WK) void slab_gemm_kernel(
    float* __restrict__ slabs, __hip_bfloat16* __restrict__ out, long out_stride,
    const __hip_bfloat16* __restrict__ x, long x_stride,
    const __hip_bfloat16* __restrict__ wt, int M, int N, int K, int steps_per_split) {
  constexpr bool PAIR = EPI != kSlabSums;
  static_assert(PAIR || WK == 1, "groups' sums meet in LDS for gate and value rows only");
  constexpr int ROWS = TM * 16, TILE = ROWS * kSlabBK;       // one staged token tile
  __shared__ __align__(16) short lds[2 * WK * TILE];         // and fewer fp32 sums later
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = w & 3, kg = w >> 2;
  const int col = lane & 15, grp = lane >> 4;
  const int step0 = blockIdx.y * steps_per_split;
  const int total = min(steps_per_split, K / kSlabBK - step0);
  const int loops = (total + WK - 1) / WK;
  const int n0 = blockIdx.x * (PAIR ? 32 : 64);
  const int wrow = PAIR ? (nt < 2 ? n0 + nt * 16 : N / 2 + n0 + (nt - 2) * 16) : n0 + nt * 16;
  // Through an opaque asm: as a plain kernel argument that nothing aliases, the compiler
  // might move its loads across the barriers' memory clobbers, and step() counts them.
  auto wp = (const __attribute__((address_space(1))) __hip_bfloat16*)(
      wt + (long)(wrow + col) * K + (long)step0 * kSlabBK + grp * 8);
  asm volatile("" : "+v"(wp) :: "memory");
  // staging: load j of this wave fills rows 4 (nt + 4 j) + lane/16 of its group's tile
  const int srow = nt * 4 + (lane >> 4);
  const int sgran = ((lane & 15) ^ (srow & 15)) << 3;
  const __hip_bfloat16* xp[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j)
    xp[j] = x + (long)min(srow + j * 16, M - 1) * x_stride + (long)step0 * kSlabBK + sgran;
  short* const mine = lds + kg * TILE;                        // + stage * WK * TILE
  auto stage = [&](int i) {
    const int s = i * WK + kg;
    if (s >= total) return;
#pragma unroll
    for (int j = 0; j < TM; ++j)
      glds16(xp[j] + s * kSlabBK, mine + (i & 1) * (WK * TILE) + (nt + j * 4) * 512);
    __builtin_amdgcn_sched_barrier(0);                        // before any weights
  };
  auto fetch = [&](sl_s16x8 (&f)[4], int i) {
    const int s = min(i * WK + kg, total - 1);                // past the end: unused
#pragma unroll
    for (int u = 0; u < 4; ++u)
      f[u] = __builtin_nontemporal_load(
          reinterpret_cast<const __attribute__((address_space(1))) sl_s16x8*>(
              wp + s * kSlabBK + u * 32));
  };
  sl_f32x4 acc[TM];
#pragma unroll
  for (int m = 0; m < TM; ++m) acc[m] = sl_f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int i, sl_s16x8 (&f)[4]) {
    // this step's tokens and weights have landed, the next weights may travel: the last
    // four loads are fetch(i + 1)'s, issued after stage(i)'s and nothing after them
    if (i + 1 < loops) pipe_barrier_vm<4>();
    else pipe_barrier_vm<0>();
    if (i + 1 < loops) stage(i + 1);
    if (i * WK + kg < total) {
      const short* xt = mine + (i & 1) * (WK * TILE) + col * kSlabBK;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int m = 0; m < TM; ++m) {
          const sl_s16x8 xf = *reinterpret_cast<const sl_s16x8*>(
              xt + m * 16 * kSlabBK + (((u * 4 + grp) ^ col) << 3));
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[u], xf, acc[m], 0, 0, 0);
        }
    }
    if (i + 2 < loops) fetch(f, i + 2);
    __builtin_amdgcn_sched_barrier(0);                        // not past the next barrier
  };
  sl_s16x8 wa[4], wb[4];
  stage(0);
  fetch(wa, 0);
  if (loops > 1) fetch(wb, 1);
  for (int i = 0; i < loops; i += 2) {
    step(i, wa);
    if (i + 1 < loops) step(i + 1, wb);
  }

  if constexpr (!PAIR) {
    float* slab = slabs + (long)blockIdx.y * M * N + wrow + grp * 4;
#pragma unroll
    for (int m = 0; m < TM; ++m)
      if (m * 16 + col < M)
        *reinterpret_cast<sl_f32x4*>(slab + (long)(m * 16 + col) * N) = acc[m];
    return;
  }
  // sums of the groups, and of gate and value rows, meet in LDS
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int m = 0; m < TM; ++m)
    *reinterpret_cast<sl_f32x4*>(red + ((w * TM + m) * 64 + lane) * 4) = acc[m];
  __syncthreads();
  for (int unit = w; unit < 2 * TM; unit += 4 * WK) {         // (n tile, m tile) of 64 lanes
    const int t = unit / TM, m = unit % TM;
    auto sum = [&](int tile) {
      sl_f32x4 s = *reinterpret_cast<const sl_f32x4*>(red + ((tile * TM + m) * 64 + lane) * 4);
#pragma unroll
      for (int g = 1; g < WK; ++g)
        s += *reinterpret_cast<const sl_f32x4*>(
            red + (((g * 4 + tile) * TM + m) * 64 + lane) * 4);
      return s;
    };
    const int row = m * 16 + col;
    const sl_f32x4 y = sum(t), up = sum(t + 2);
    Vec4<__hip_bfloat16> v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float g = y[r];
      const float a = EPI == kSlabSilu
          ? g / (1.0f + __expf(-g))
          : 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
      v.data[r] = __float2bfloat16(a * up[r]);
    }
    if (row < M)
      *reinterpret_cast<int2*>(out + (long)row * out_stride + n0 + t * 16 + grp * 4) =
          *reinterpret_cast<const int2*>(v.data);
  }
}

// ------------------------------------------------------- readers of the slabs --

// The first S of NE slabs (one at the least) added to y, all loads in flight together:
// their L2 is another XCD's.
template <int NE>
DEVINL void slab_add(sl_f32x4& y, const float* __restrict__ from, long stride, int S) {
  sl_f32x4 v[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e)
    v[e] = *reinterpret_cast<const sl_f32x4*>(from + min(e, S - 1) * stride);
#pragma unroll
  for (int e = 0; e < NE; ++e)
    if (e < S) y += v[e];
}

// Sum of S slabs at one place.
DEVINL sl_f32x4 slab_sum(const float* __restrict__ slabs, long at, long stride, int S) {
  sl_f32x4 y = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += 16) {
    const float* from = slabs + s0 * stride + at;
    const int n = S - s0;
    if (n <= 4) slab_add<4>(y, from, stride, n);
    else if (n <= 8) slab_add<8>(y, from, stride, n);
    else if (n <= 12) slab_add<12>(y, from, stride, n);
    else slab_add<16>(y, from, stride, min(n, 16));
  }
  return y;
}

DEVINL sl_f32x4 slab_bf4(const __hip_bfloat16* p) {
  const Vec4<__hip_bfloat16> v = load8(p);
  return sl_f32x4{to_f32(v.data[0]), to_f32(v.data[1]), to_f32(v.data[2]), to_f32(v.data[3])};
}

DEVINL Vec4<__hip_bfloat16> slab_store(__hip_bfloat16* p, sl_f32x4 y) {
  Vec4<__hip_bfloat16> v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v.data[r] = __float2bfloat16(y[r]);
  *reinterpret_cast<int2*>(p) = *reinterpret_cast<const int2*>(v.data);
  return v;
}

// residual += y, or with POST += rmsnorm(y) (w_post + offset), y the summed slabs;
// h = rmsnorm(residual) (w + offset). One workgroup per row, the row in registers:
// up to 8192 channels. Bound by latency: few rows, each behind S slabs; so everything is
// asked for at once, norm weights too, and a sum over the row takes one barrier.
// Measured (us, with weights read behind the sums, three barriers a sum and rounds of eight
// slabs -> now; a sequence of such launches): 96 rows of 3584, 9 slabs, two norms 6.8 -> 5.7;
// 48 rows 6.4 -> 5.5; 189 rows of 3072, 10 slabs 7.5 -> 6.9; 64 rows of 2048, 8 slabs 3.8,
// as before (with 512 channels a wave instead of 256 4.5). Slabs that the same L2 still holds
// from the launch before hide that: 64 rows of 3072, 8 slabs 4.4 -> 4.8; behind the products that
// write them whole layers take 0 to 2 % less.
constexpr int kSlabNT = 1024;

// x plus the x of the lane that DPP control `CTRL` names, in the rows of 16 that ROWS has.
template <int CTRL, int ROWS>
DEVINL float slab_dpp_add(float x) {
  return x + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), CTRL, ROWS, 0xf,
                                                         false));
}

// The workgroup's sum, in all threads; `red` is not used again. Sums go up within rows of 16
// lanes, from row to row and through LDS once, without the LDS crossbar.
DEVINL float slab_block_sum(float x, float (&red)[kSlabNT / WAVE]) {
  x = slab_dpp_add<0x111, 0xf>(x);                         // row_shr 1, 2, 4, 8
  x = slab_dpp_add<0x112, 0xf>(x);
  x = slab_dpp_add<0x114, 0xf>(x);
  x = slab_dpp_add<0x118, 0xf>(x);
  x = slab_dpp_add<0x142, 0xa>(x);                         // row_bcast 15, 31
  x = slab_dpp_add<0x143, 0xc>(x);
  if ((threadIdx.x & (WAVE - 1)) == WAVE - 1) red[threadIdx.x / WAVE] = x;
  __syncthreads();
  const int waves = blockDim.x / WAVE;
  x = 0.f;
#pragma unroll
  for (int i = 0; i < kSlabNT / WAVE; ++i) {
    const float v = red[i];
    x += i < waves ? v : 0.f;
  }
  return x;
}

template <bool POST>
__global__ __launch_bounds__(kSlabNT) void slab_add_norm_kernel(
    __hip_bfloat16* __restrict__ h, __hip_bfloat16* __restrict__ residual,
    const float* __restrict__ slabs, int S, const __hip_bfloat16* __restrict__ w_post,
    const __hip_bfloat16* __restrict__ w, int M, int N, float eps, float offset) {
  __shared__ float red[2][kSlabNT / WAVE];
  const long row = (long)blockIdx.x * N;
  const long stride = (long)M * N;
  sl_f32x4 y[2], r[2];
  int2 was[2], wn[2], wp[2];               // bf16 as read
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = (k * blockDim.x + threadIdx.x) * 4;
    y[k] = r[k] = sl_f32x4{0.f, 0.f, 0.f, 0.f};
    if (i >= N) continue;
    was[k] = *reinterpret_cast<const int2*>(residual + row + i);
    wn[k] = *reinterpret_cast<const int2*>(w + i);
    if (POST) wp[k] = *reinterpret_cast<const int2*>(w_post + i);
    y[k] = slab_sum(slabs, row + i, stride, S);
    if (POST) ss += y[k][0] * y[k][0] + y[k][1] * y[k][1] + y[k][2] * y[k][2] + y[k][3] * y[k][3];
  }
  float inv = 1.f;
  if (POST) inv = rsqrtf(slab_block_sum(ss, red[0]) / N + eps);
  ss = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = (k * blockDim.x + threadIdx.x) * 4;
    if (i >= N) continue;
    r[k] = slab_bf4(reinterpret_cast<const __hip_bfloat16*>(&was[k]));
    if (POST)
      r[k] += y[k] * inv * (slab_bf4(reinterpret_cast<const __hip_bfloat16*>(&wp[k])) + offset);
    else r[k] += y[k];
    const Vec4<__hip_bfloat16> v = slab_store(residual + row + i, r[k]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[k][e] = to_f32(v.data[e]);           // the rounded stream is what is normalised
      ss += r[k][e] * r[k][e];
    }
  }
  inv = rsqrtf(slab_block_sum(ss, red[1]) / N + eps);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = (k * blockDim.x + threadIdx.x) * 4;
    if (i < N)
      slab_store(h + row + i,
                 r[k] * inv * (slab_bf4(reinterpret_cast<const __hip_bfloat16*>(&wn[k])) + offset));
  }
}

// The summed slabs of a q/k/v projection (+ bias): q and k rotated (halves of a head,
// as in rope_and_cache_kernel), all written as packed bf16 rows and k, v into the
// paged cache. Workgroups of (token, quarter of the heads), four channel pairs per
// thread.
template <typename TC>
__global__ __launch_bounds__(256) void slab_rope_cache_kernel(
    __hip_bfloat16* __restrict__ qkv, const float* __restrict__ slabs, int S,
    const __hip_bfloat16* __restrict__ bias, TC* __restrict__ k_cache, TC* __restrict__ v_cache,
    const long* __restrict__ positions, const float* __restrict__ cos_sin,
    const long* __restrict__ slots, int M, int heads, int kv_heads, int D, int block_size) {
  const int token = blockIdx.x, half = D / 2, quads = half / 4;
  const int N = (heads + 2 * kv_heads) * D;
  const long row = (long)token * N, stride = (long)M * N;
  const float* cs = cos_sin + positions[token] * D;
  const long slot = slots[token];
  for (int t = blockIdx.y * 256 + threadIdx.x; t < (heads + 2 * kv_heads) * quads;
       t += gridDim.y * 256) {
    const int hd = t / quads, d = (t % quads) * 4;
    const int i = hd * D + d;
    sl_f32x4 a = slab_sum(slabs, row + i, stride, S);
    sl_f32x4 b = slab_sum(slabs, row + i + half, stride, S);
    if (bias) {
      a += slab_bf4(bias + i);
      b += slab_bf4(bias + i + half);
    }
    if (hd < heads + kv_heads) {
      const sl_f32x4 c = *reinterpret_cast<const sl_f32x4*>(cs + d);
      const sl_f32x4 s = *reinterpret_cast<const sl_f32x4*>(cs + half + d);
      const sl_f32x4 ra = a * c - b * s;
      b = b * c + a * s;
      a = ra;
    }
    const Vec4<__hip_bfloat16> va = slab_store(qkv + row + i, a);
    const Vec4<__hip_bfloat16> vb = slab_store(qkv + row + i + half, b);
    if (hd < heads || slot < 0) continue;
    const bool is_v = hd >= heads + kv_heads;
    const int kh = hd - heads - (is_v ? kv_heads : 0);
    const long block = slot / block_size;
    const int off = (int)(slot - block * block_size);
    TC* dst = (is_v ? v_cache : k_cache) +
              ((block * kv_heads + kh) * (long)block_size + off) * D + d;
    if constexpr (std::is_same_v<TC, __hip_bfloat16>) {
      *reinterpret_cast<int2*>(dst) = *reinterpret_cast<const int2*>(va.data);
      *reinterpret_cast<int2*>(dst + half) = *reinterpret_cast<const int2*>(vb.data);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {          // from the rounded rows, as the other path
        dst[e] = from_f32<TC>(to_f32(va.data[e]));
        dst[half + e] = from_f32<TC>(to_f32(vb.data[e]));
      }
    }
  }
}
