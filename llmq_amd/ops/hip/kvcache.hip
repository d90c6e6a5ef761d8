// Paged-KV scatter: write this step's k/v vectors into the paged cache.
// Cache layout: [num_blocks, kv_heads, block_size, head_dim] (a (block,head)
// pair is a contiguous [block_size, head_dim] tile for the decode kernel).

#include "common.h"

template <typename T, typename TC = T>
__global__ void reshape_and_cache_kernel(
    const T* __restrict__ key,     // [T, kv_heads, D] (row stride key_stride)
    const T* __restrict__ value,
    TC* __restrict__ k_cache,      // [blocks, kv_heads, bs, D]
    TC* __restrict__ v_cache,
    const long* __restrict__ slots,  // [T] global slot id
    int kv_heads, int head_dim, int block_size,
    long key_stride, long val_stride) {
  constexpr int VE = Vec8<T>::kElems;
  const int token = blockIdx.x;
  const long slot = slots[token];
  if (slot < 0) return;  // padding
  const long block = slot / block_size;
  const int off = (int)(slot % block_size);
  const int chunks = (kv_heads * head_dim) / VE;
  for (int i = threadIdx.x; i < chunks; i += blockDim.x) {
    const int h = (i * VE) / head_dim;
    const int d = (i * VE) % head_dim;
    const long dst =
        ((block * kv_heads + h) * (long)block_size + off) * head_dim + d;
    Vec8<T> kv = load16(key + (long)token * key_stride + (long)h * head_dim + d);
    Vec8<T> vv = load16(value + (long)token * val_stride + (long)h * head_dim + d);
    if constexpr (std::is_same_v<T, TC>) {
      store16(k_cache + dst, kv);
      store16(v_cache + dst, vv);
    } else {  // quantizing cache write (e.g. bf16 → fp8)
#pragma unroll
      for (int j = 0; j < VE; ++j) {
        k_cache[dst + j] = from_f32<TC>(to_f32(kv.data[j]));
        v_cache[dst + j] = from_f32<TC>(to_f32(vv.data[j]));
      }
    }
  }
}

// Fused RoPE + cache write: rotates q and k in place AND scatters the rotated k
// plus v into the paged cache in one launch. A thread takes NP channel pairs (d,
// half + d) of a head: NP = 8 bytes' worth where rows and head size allow it, else 1.
// Workgroups: (token, part of the heads). Bound by bytes on prompts (8192 tokens, 16
// + 8 + 8 heads of 256: 89 us with 2-byte accesses, 57 with 8-byte ones), by latency
// on decode steps (189 tokens, 24 + 8 + 8 heads of 128: 7.5 -> 4.9 us).
template <typename T, typename TC, int NP>
__global__ __launch_bounds__(256) void rope_and_cache_kernel(
    T* __restrict__ q,             // [T, Hq, D] (row stride q_stride)
    T* __restrict__ k,             // [T, Hk, D]
    const T* __restrict__ value,   // [T, Hk, D]
    TC* __restrict__ k_cache,      // [blocks, Hk, bs, D]
    TC* __restrict__ v_cache,
    const long* __restrict__ positions,
    const float* __restrict__ cos_sin,  // [max_pos, D] f32
    const long* __restrict__ slots,
    int num_q_heads, int num_k_heads, int head_dim, int block_size,
    long q_stride, long k_stride, long v_stride) {
  struct alignas(NP * sizeof(T)) Part { T e[NP]; };
  struct alignas(NP * sizeof(float)) Angles { float e[NP]; };
  const int token = blockIdx.x;
  const int half = head_dim / 2, parts = half / NP;
  const float* cs = cos_sin + positions[token] * head_dim;
  const long slot = slots[token];
  const long block = slot / block_size;
  const int off = (int)(slot % block_size);
  const int total = (num_q_heads + 2 * num_k_heads) * parts;
  for (int t = blockIdx.y * 256 + threadIdx.x; t < total; t += gridDim.y * 256) {
    const int h = t / parts, d = (t % parts) * NP;
    const bool is_q = h < num_q_heads, is_v = h >= num_q_heads + num_k_heads;
    if (is_v && slot < 0) continue;
    const int kh = h - num_q_heads - (is_v ? num_k_heads : 0);
    const T* src = is_q ? q + (long)token * q_stride + (long)h * head_dim
                 : is_v ? value + (long)token * v_stride + (long)kh * head_dim
                        : k + (long)token * k_stride + (long)kh * head_dim;
    Part a = *reinterpret_cast<const Part*>(src + d);
    Part b = *reinterpret_cast<const Part*>(src + half + d);
    if (!is_v) {
      const Angles c = *reinterpret_cast<const Angles*>(cs + d);
      const Angles s = *reinterpret_cast<const Angles*>(cs + half + d);
#pragma unroll
      for (int e = 0; e < NP; ++e) {
        const float x1 = to_f32(a.e[e]), x2 = to_f32(b.e[e]);
        a.e[e] = from_f32<T>(x1 * c.e[e] - x2 * s.e[e]);
        b.e[e] = from_f32<T>(x2 * c.e[e] + x1 * s.e[e]);
      }
      T* dst = const_cast<T*>(src);
      *reinterpret_cast<Part*>(dst + d) = a;
      *reinterpret_cast<Part*>(dst + half + d) = b;
    }
    if (is_q || slot < 0) continue;
    TC* dst = (is_v ? v_cache : k_cache) +
        ((block * num_k_heads + kh) * (long)block_size + off) * head_dim + d;
    if constexpr (std::is_same_v<T, TC>) {
      *reinterpret_cast<Part*>(dst) = a;
      *reinterpret_cast<Part*>(dst + half) = b;
    } else {
#pragma unroll
      for (int e = 0; e < NP; ++e) {
        dst[e] = from_f32<TC>(to_f32(a.e[e]));
        dst[half + e] = from_f32<TC>(to_f32(b.e[e]));
      }
    }
  }
}
