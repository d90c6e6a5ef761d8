// Paged attention for gfx950.
//
// DECODE (paged_decode_attention_kernel): fp32 and fp16 caches; bf16 and fp8
// ones run on the matrix cores (paged_decode.hip). One workgroup per
// (sequence, kv_head); all GQA query heads of that kv head are processed
// together so the KV stream is read ONCE: 16-byte coalesced K loads,
// two-phase chunk processing with scores staged in LDS, fp32 online softmax.
//
//   phase A: 16-lane groups compute q·k for CHUNK tokens -> s[CHUNK][G] LDS
//   phase B: thread (h, d-slice) runs online softmax over the chunk and
//            accumulates p·V into per-thread fp32 registers; V rows are
//            read coalesced by each 32-thread head-group (L1 serves the
//            G-way reuse across head-groups).
//
// PREFILL (varlen_prefill_attention_kernel): fp32 and fp16 (bf16 prompts run on
// the matrix cores, flash_prefill.hip): packed varlen causal attention, one wave
// per query row, keys across lanes, online softmax.

#include "common.h"

#define DECODE_CHUNK 128  // tokens per two-phase iteration (8 KV blocks @ bs 16)

template <typename T, int HEAD_DIM>
__global__ __launch_bounds__(256) void paged_decode_attention_kernel(
    T* __restrict__ out,                  // [B, H, D] (row stride out_stride)
    const T* __restrict__ q,              // [B, H, D] (row stride q_stride)
    const T* __restrict__ k_cache,        // [nb, KVH, bs, D]
    const T* __restrict__ v_cache,
    const int* __restrict__ block_tables, // [B, max_blocks]
    const int* __restrict__ context_lens, // [B]
    int num_heads, int num_kv_heads, int block_size, int max_blocks,
    float scale, float softcap, int window,
    long q_stride, long out_stride) {
  const int b = blockIdx.x;
  const int kh = blockIdx.y;
  const int G = num_heads / num_kv_heads;  // <= 8
  const int L = context_lens[b];
  if (L <= 0) return;

  constexpr int VE = Vec8<T>::kElems;        // 8 for bf16, 4 for f32
  constexpr int D = HEAD_DIM;
  constexpr int CHUNK = DECODE_CHUNK;
  const int lane16 = threadIdx.x & 15;       // lane within 16-lane score group
  const int g16 = threadIdx.x >> 4;          // score group id (0..15)

  // Phase-B decomposition: SUBS token-parallel sub-groups per head, each of
  // 32 threads covering all D dims. All 256 threads work for G*32*SUBS==256.
  const int tph = 32 * G;                    // threads per head-set
  const int SUBS = 256 / tph;                // 8,4,2,2,1,1,1,1 for G=1..8
  const int sub = threadIdx.x / tph;         // token sub-group (>=SUBS: idle)
  const int h_b = (threadIdx.x % tph) >> 5;  // head
  constexpr int DPT = D / 32;                // dims per thread (2/4/8)
  const int d0 = (threadIdx.x & 31) * DPT;

  // LDS: q (G x D f32, pre-scaled) | scores (CHUNK x G) | chunk block ids |
  //      merge buffers (SUBS x G x (D + 2))
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* q_s = reinterpret_cast<float*>(smem);              // [G][D]
  float* s_s = q_s + G * D;                                 // [CHUNK][G]
  int* bt_s = reinterpret_cast<int*>(s_s + CHUNK * G);      // [CHUNK/bs up to 16]
  float* merge_s = reinterpret_cast<float*>(bt_s + 16);     // [SUBS][G][D+2]

  for (int i = threadIdx.x; i < G * D; i += blockDim.x) {
    const int h = i / D, d = i % D;
    q_s[i] = to_f32(q[(long)b * q_stride + (long)(kh * G + h) * D + d]) * scale;
  }

  const int start = (window > 0 && L > window) ? (L - window) : 0;
  const int* bt = block_tables + (long)b * max_blocks;
  const int base0 = (start / CHUNK) * CHUNK;

  float acc[DPT];
#pragma unroll
  for (int i = 0; i < DPT; ++i) acc[i] = 0.f;
  float m_run = -1e30f, l_run = 0.f;

  for (int base = base0; base < L; base += CHUNK) {
    const int chunk_end = min(base + CHUNK, L);
    const int n = chunk_end - base;
    // stage this chunk's block ids (removes a dependent global load from the
    // phase-B address chain)
    if (threadIdx.x < (unsigned)((n + block_size - 1) / block_size))
      bt_s[threadIdx.x] = bt[(base + threadIdx.x * block_size) / block_size];
    __syncthreads();
    // ---- phase A: scores for tokens [base, chunk_end)
    for (int t0 = g16; t0 < n; t0 += 16) {
      const int t = base + t0;
      const long blk = bt_s[t0 / block_size];
      const int off = t % block_size;
      const T* krow =
          k_cache + (((blk * num_kv_heads + kh) * (long)block_size + off)) * D;
      constexpr int DL = D / 16;  // elems per lane16
      float kf[DL];
      if constexpr (DL % VE == 0) {
#pragma unroll
        for (int c = 0; c < DL; c += VE) {
          Vec8<T> kv = load16(krow + lane16 * DL + c);
#pragma unroll
          for (int j = 0; j < VE; ++j) kf[c + j] = to_f32(kv.data[j]);
        }
      } else {  // e.g. D=64 bf16: 4 elems per lane — scalar loads
#pragma unroll
        for (int c = 0; c < DL; ++c) kf[c] = to_f32(krow[lane16 * DL + c]);
      }
      for (int h = 0; h < G; ++h) {
        float dot = 0.f;
        const float* qrow = q_s + h * D + lane16 * DL;
#pragma unroll
        for (int j = 0; j < DL; ++j) dot += qrow[j] * kf[j];
        dot = group_reduce_sum<16>(dot);
        if (lane16 == 0) {
          if (softcap > 0.f) dot = tanhf(dot / softcap) * softcap;
          if (t < start) dot = -1e30f;
          s_s[t0 * G + h] = dot;
        }
      }
    }
    __syncthreads();
    // ---- phase B: online softmax + V accumulation (sub-group token split)
    if (sub < SUBS) {
      float m_chunk = -1e30f;
      for (int t = sub; t < n; t += SUBS)
        m_chunk = fmaxf(m_chunk, s_s[t * G + h_b]);
      const float m_new = fmaxf(m_run, m_chunk);
      if (m_new > -1e30f) {
        const float alpha = __expf(m_run - m_new);
#pragma unroll
        for (int i = 0; i < DPT; ++i) acc[i] *= alpha;
        l_run *= alpha;
        m_run = m_new;
        // Iterations are independent (chunk-max softmax, no rescale inside)
        // so V loads pipeline across tokens.
        for (int t = sub; t < n; t += SUBS) {
          const float p = __expf(s_s[t * G + h_b] - m_new);
          l_run += p;
          const int tok = base + t;
          const long blk = bt_s[t / block_size];
          const int off = tok % block_size;
          const T* vrow =
              v_cache + (((blk * num_kv_heads + kh) * (long)block_size + off)) * D + d0;
          // Vectorized V row slice: DPT contiguous elems per thread
          // (16B for bf16 D=256, 8B for D=128) — scalar 2B loads here
          // were the v2 bandwidth ceiling.
          if constexpr (DPT % Vec8<T>::kElems == 0) {
            constexpr int VE8 = Vec8<T>::kElems;
#pragma unroll
            for (int c = 0; c < DPT; c += VE8) {
              Vec8<T> vv = load16(vrow + c);
#pragma unroll
              for (int j = 0; j < VE8; ++j) acc[c + j] += p * to_f32(vv.data[j]);
            }
          } else if constexpr (DPT % Vec4<T>::kElems == 0) {
            constexpr int VE4 = Vec4<T>::kElems;
#pragma unroll
            for (int c = 0; c < DPT; c += VE4) {
              Vec4<T> vv = load8(vrow + c);
#pragma unroll
              for (int j = 0; j < VE4; ++j) acc[c + j] += p * to_f32(vv.data[j]);
            }
          } else {
#pragma unroll
            for (int i = 0; i < DPT; ++i) acc[i] += p * to_f32(vrow[i]);
          }
        }
      }
    }
    __syncthreads();  // protect s_s / bt_s for the next chunk
  }

  // ---- merge sub-group partials (flash-decoding style, within the block)
  const int d2 = D + 2;
  if (sub < SUBS && SUBS > 1) {
    float* slot = merge_s + (sub * G + h_b) * d2;
#pragma unroll
    for (int i = 0; i < DPT; ++i) slot[d0 + i] = acc[i];
    if (d0 == 0) {
      slot[D] = m_run;
      slot[D + 1] = l_run;
    }
  }
  __syncthreads();
  if (sub == 0) {
    float m_tot = m_run, l_tot = 0.f;
    if (SUBS > 1) {
      for (int s2 = 0; s2 < SUBS; ++s2)
        m_tot = fmaxf(m_tot, merge_s[(s2 * G + h_b) * d2 + D]);
      float accm[DPT];
#pragma unroll
      for (int i = 0; i < DPT; ++i) accm[i] = 0.f;
      for (int s2 = 0; s2 < SUBS; ++s2) {
        const float* slot = merge_s + (s2 * G + h_b) * d2;
        const float w = __expf(slot[D] - m_tot);
        l_tot += w * slot[D + 1];
#pragma unroll
        for (int i = 0; i < DPT; ++i) accm[i] += w * slot[d0 + i];
      }
#pragma unroll
      for (int i = 0; i < DPT; ++i) acc[i] = accm[i];
    } else {
      l_tot = l_run;
    }
    const float inv = (l_tot > 0.f) ? 1.0f / l_tot : 0.f;
    T* orow = out + (long)b * out_stride + (long)(kh * G + h_b) * D + d0;
#pragma unroll
    for (int i = 0; i < DPT; ++i) orow[i] = from_f32<T>(acc[i] * inv);
  }
}

// --------------------------------------------------------------- prefill --
// Packed varlen causal attention. Grid: (seq, head). 4 waves per block;
// each wave owns query rows i = wave_id + 4*n. Keys go across lanes (one
// key per lane per 64-key chunk), V accumulation is lane-dim-parallel via
// shfl broadcast of the probabilities.

template <typename T, int HEAD_DIM>
__global__ __launch_bounds__(256) void varlen_prefill_attention_kernel(
    T* __restrict__ out,            // [Tq, H, D]
    const T* __restrict__ q,        // [Tq, H, D] (row strides below)
    const T* __restrict__ k,        // [Tk, KVH, D]
    const T* __restrict__ v,
    const int* __restrict__ cu_seqlens,    // [B+1] query offsets
    const int* __restrict__ cu_seqlens_k,  // [B+1] key offsets (chunked)
    int num_heads, int num_kv_heads, float scale, float softcap, int window,
    long q_stride, long k_stride, long v_stride, long o_stride) {
  constexpr int D = HEAD_DIM;
  constexpr int VE = Vec8<T>::kElems;
  constexpr int DPT = D / WAVE;  // dims per lane (1/2/4)
  const int seq = blockIdx.x;
  const int h = blockIdx.y;
  const int kvh = h / (num_heads / num_kv_heads);
  const int s0 = cu_seqlens[seq], s1 = cu_seqlens[seq + 1];
  const int L = s1 - s0;
  const int s0k = cu_seqlens_k[seq];
  const int Lk = cu_seqlens_k[seq + 1] - s0k;
  const int off = Lk - L;  // abs position of q row 0
  const int wid = threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);

  __shared__ __attribute__((aligned(16))) float q_lds[4][D];

  for (int i = wid; i < L; i += 4) {  // query row
    // stage q row (pre-scaled) into this wave's LDS slot
    for (int d = lane; d < D; d += WAVE)
      q_lds[wid][d] = to_f32(q[(long)(s0 + i) * q_stride + (long)h * D + d]) * scale;
    __builtin_amdgcn_wave_barrier();

    float m_run = -1e30f, l_run = 0.f;
    float acc[DPT];
#pragma unroll
    for (int t = 0; t < DPT; ++t) acc[t] = 0.f;

    const int iabs = off + i;  // absolute position of this query row
    const int kstart = (window > 0 && iabs + 1 > window) ? (iabs + 1 - window) : 0;
    for (int base = (kstart / WAVE) * WAVE; base <= iabs; base += WAVE) {
      const int j = base + lane;  // this lane's key (absolute)
      float score = -1e30f;
      if (j <= iabs && j >= kstart && j < Lk) {
        const T* krow = k + (long)(s0k + j) * k_stride + (long)kvh * D;
        float dot = 0.f;
#pragma unroll 4
        for (int d = 0; d < D; d += VE) {
          Vec8<T> kv = load16(krow + d);
#pragma unroll
          for (int e = 0; e < VE; ++e) dot += q_lds[wid][d + e] * to_f32(kv.data[e]);
        }
        score = (softcap > 0.f) ? tanhf(dot / softcap) * softcap : dot;
      }
      const float m_chunk = wave_reduce_max(score);
      const float m_new = fmaxf(m_run, m_chunk);
      const float alpha = __expf(m_run - m_new);
      const float p = (score > -1e29f) ? __expf(score - m_new) : 0.f;
      const float psum = wave_reduce_sum(p);
      l_run = l_run * alpha + psum;
      m_run = m_new;
#pragma unroll
      for (int t = 0; t < DPT; ++t) acc[t] *= alpha;
      const int jn = min(iabs - base + 1, WAVE);
      for (int jj = 0; jj < jn; ++jj) {
        const float pj = __shfl(p, jj, WAVE);
        if (pj != 0.f) {
          const T* vrow = v + (long)(s0k + base + jj) * v_stride + (long)kvh * D;
#pragma unroll
          for (int t = 0; t < DPT; ++t)
            acc[t] += pj * to_f32(vrow[lane * DPT + t]);
        }
      }
    }
    const float inv = (l_run > 0.f) ? 1.0f / l_run : 0.f;
    T* orow = out + (long)(s0 + i) * o_stride + (long)h * D;
#pragma unroll
    for (int t = 0; t < DPT; ++t) orow[lane * DPT + t] = from_f32<T>(acc[t] * inv);
    __builtin_amdgcn_wave_barrier();
  }
}
