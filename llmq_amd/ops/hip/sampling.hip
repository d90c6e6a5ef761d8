// Fused token sampling for gfx950.
//
// One pass over the fp32 logits [B, V]: each workgroup scans a vocab chunk
// of one row and computes a local argmax of
//   temp <= 0:  logit                      (greedy)
//   temp  > 0:  logit / temp + Gumbel(g)   (Gumbel-max == softmax sampling)
// then leaves it as a packed (orderable-f32 | index) key; the row's largest is its token.
// Replaces the torch sampler's 4+ full passes (softmax, multinomial, ...)
// with a single logits read — at B=256, V=256k fp32 that is 262 MB ≈ 35 µs
// at stream rate. Top-k/top-p rows fall back to the torch path (wrapper).
//
// RNG: counter-based (seed, step, element) hash — deterministic per engine
// step, independent of launch geometry, so eager and hipGraph runs sample
// identical tokens.

#include "common.h"

DEVINL unsigned int hash_u32(unsigned int x) {
  // finalizer-strength integer hash (xxhash/murmur-style avalanche)
  x ^= x >> 16; x *= 0x7feb352dU;
  x ^= x >> 15; x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

DEVINL float uniform01(unsigned int seed, unsigned int step, unsigned int b,
                       unsigned int v) {
  // Weyl-style multiplicative mixing of the coordinates BEFORE the
  // finalizers: xor-combining (b<<20)^v leaves nearby (b, v) pairs
  // jointly dependent enough to bias argmax sampling by ~3% (verified
  // against the softmax distribution; see TestFusedSampler).
  unsigned int key = b * 0x9E3779B9u ^ v * 0x85EBCA6Bu ^ step * 0xC2B2AE35u ^ seed;
  unsigned int h = hash_u32(hash_u32(key));
  // (0, 1]: avoid 0 so log() is finite
  return (h + 1u) * (1.0f / 4294967296.0f);
}

DEVINL unsigned long long pack_key(float val, int idx) {
  unsigned int u = __float_as_uint(val);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // order-preserving map
  // index bits inverted so equal values tie-break toward the LOWER index
  // (matches torch argmax) under atomicMax
  return ((unsigned long long)u << 32) | (unsigned int)(~idx);
}

// Per-row RNG keying: rows with a user seed (req_seeds[b] != 0) draw from
// (request_seed, output_position) — REPRODUCIBLE for a given request
// regardless of batch placement or engine step. Unseeded rows draw from
// (engine seed, step, row).
__global__ __launch_bounds__(256) void sample_argmax_kernel(
    unsigned long long* __restrict__ parts,     // [B, gridDim.y], each chunk's best
    const float* __restrict__ logits,           // [B, V]
    const float* __restrict__ temps,            // [B]
    const unsigned int* __restrict__ req_seeds, // [B] (0 = unseeded)
    const unsigned int* __restrict__ req_pos,   // [B] output position
    const float* __restrict__ bounds,           // [B] top-k/p keep-bound or null
    int V, unsigned int seed, unsigned int step, int chunk, bool vec) {
  const int b = blockIdx.x;
  const int v0 = blockIdx.y * chunk;
  const int v1 = min(v0 + chunk, V);
  const float temp = temps[b];
  const bool greedy = temp <= 0.f;
  const float inv_t = greedy ? 1.0f : 1.0f / temp;
  const float* row = logits + (long)b * V;
  const unsigned int rs = req_seeds[b];
  const unsigned int kseed = rs ? rs : seed;
  const unsigned int kstep = rs ? req_pos[b] : step;
  const unsigned int kb = rs ? 0u : (unsigned int)b;
  // top-k/top-p truncation: only logits >= bound are candidates (the
  // bound kernel guarantees the row max passes; greedy rows get -inf)
  const float bound = bounds ? bounds[b] : -3e38f;

  float best = -3e38f;
  int best_i = v0;
  auto take = [&](float l, int v) {
    if (l < bound) return;
    float x = l * inv_t;
    if (!greedy) {
      const float u = uniform01(kseed, kstep, kb, v);
      x += -__logf(-__logf(u));  // Gumbel(0,1)
    }
    if (x > best) { best = x; best_i = v; }
  };
  if (vec) {
#pragma unroll 4
    for (int v = v0 + threadIdx.x * 4; v < v1; v += 1024) {
      const float4 l = *reinterpret_cast<const float4*>(row + v);
      take(l.x, v);
      take(l.y, v + 1);
      take(l.z, v + 2);
      take(l.w, v + 3);
    }
  } else {
    for (int v = v0 + threadIdx.x; v < v1; v += 256) take(row[v], v);
  }
  // wave reduce (value, index)
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, WAVE);
    const int oi = __shfl_xor(best_i, off, WAVE);
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
  }
  __shared__ float vals[4];
  __shared__ int idxs[4];
  const int wid = threadIdx.x / WAVE;
  if ((threadIdx.x & (WAVE - 1)) == 0) { vals[wid] = best; idxs[wid] = best_i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      if (vals[w] > best || (vals[w] == best && idxs[w] < best_i)) {
        best = vals[w]; best_i = idxs[w];
      }
    }
    parts[(long)b * gridDim.y + blockIdx.y] = pack_key(best, best_i);
  }
}

// ------------------------------------------------- top-k / top-p select --
// Per-row LOGIT-space bound L_min such that keeping {v : logit_v >= L_min}
// realises nucleus (top-p) and top-k truncation without a full-vocab sort: the
// row's maximum m; a 512-bin histogram of x = (l - m) / T over [-32, 0] with
// exp-mass and counts, scanned from the top bin until the mass reaches top_p Z or
// the count k; and the same again, 512 times finer, within the crossing bin. The
// crossing sub-bin is kept whole (overshoot at most its mass, about Z p / 512^2).
// Sampling from the truncated set then uses the same one-pass gumbel-max.
//
// Bound by three readings of the logits (262 MB each at 256 x 256000) and, in the
// first histogram, by LDS atomics that meet in the populated bins. A row is cut in
// chunks so that few rows fill the chip too, loads are 16 bytes, every fourth lane
// has a histogram of its own. With a top-k the first reading also leaves a value that at least
// k elements reach; the first histogram counts no bin below it. Measured (us; one workgroup a row, 4-byte loads and a serial scan
// before): 256 x 256000 normal logits, top-k 50 and top-p 0.95 1026 -> 143, top-p
// alone 1035 -> 422 (LDS atomics: half of the row is in the nucleus); 1 x 256000
// 678 -> 29.

constexpr int kThBins = 512;
constexpr int kThCopies = 4;
constexpr float kThMin = -32.0f;

// Scratch of one row, zeroed before every call.
struct ThRow {
  unsigned max_key;             // row maximum, order-preserving map
  unsigned many_key;            // value that 64 elements of one chunk reach
  unsigned not_all_key;         // complement of one that 64 of every chunk reach
  float tail;                   // mass below the first window
  // set by the first scan: window of the second, mass and count above it
  float lo, hi, keep_above, z, p_above;
  int n_above;
  unsigned done;                // no crossing in the first window
  float sum[2][kThBins];
  int cnt[2][kThBins];
};

DEVINL unsigned th_key(float x) {
  const unsigned u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
DEVINL float th_value(unsigned key) {
  return __uint_as_float((key & 0x80000000u) ? key & 0x7fffffffu : ~key);
}
// f(value) for the chunk's elements of a row; 16-byte loads where rows allow them,
// four in flight
template <typename F>
DEVINL void th_scan(const float* row, int v0, int v1, bool vec, F&& f) {
  if (!vec) {
    for (int v = v0 + threadIdx.x; v < v1; v += 256) f(row[v]);
    return;
  }
  int v = v0 + threadIdx.x * 4;
  for (; v + 3072 < v1; v += 4096) {
    float4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const float4*>(row + v + u * 1024);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f(x[u].x); f(x[u].y); f(x[u].z); f(x[u].w);
    }
  }
  for (; v < v1; v += 1024) {
    const float4 x = *reinterpret_cast<const float4*>(row + v);
    f(x.x); f(x.y); f(x.z); f(x.w);
  }
}

DEVINL bool th_limits(float temp, float p_lim, long k_lim, int V, bool& need_p, bool& need_k) {
  need_p = p_lim < 1.0f;
  need_k = k_lim > 0 && k_lim < V;
  // greedy rows take argmax regardless; unconstrained rows keep all
  return temp > 0.f && (need_p || need_k);
}

__global__ __launch_bounds__(256) void topk_topp_max_kernel(
    float* __restrict__ out_bound, ThRow* __restrict__ rows, const float* __restrict__ logits,
    const float* __restrict__ temps, const float* __restrict__ top_ps,
    const long* __restrict__ top_ks, int V, long stride, int chunk, bool vec) {
  const int b = blockIdx.x;
  bool need_p, need_k;
  if (!th_limits(temps[b], top_ps[b], top_ks[b], V, need_p, need_k)) {
    if (blockIdx.y == 0 && threadIdx.x == 0) out_bound[b] = -3e38f;
    return;
  }
  const int v0 = blockIdx.y * chunk, v1 = min(v0 + chunk, V);
  float m = -3e38f;
  th_scan(logits + (long)b * stride, v0, v1, vec, [&](float x) { m = fmaxf(m, x); });
  // the least of 64 maxima of four threads each: at least 64 elements reach it
  float many = fmaxf(m, __shfl_xor(m, 1, WAVE));
  many = fmaxf(many, __shfl_xor(many, 2, WAVE));
#pragma unroll
  for (int off = 4; off < WAVE; off <<= 1) many = fminf(many, __shfl_xor(many, off, WAVE));
  m = wave_reduce_max(m);
  __shared__ float red[4], red2[4];
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = m;
    red2[threadIdx.x >> 6] = many;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const unsigned key = th_key(fminf(fminf(red2[0], red2[1]), fminf(red2[2], red2[3])));
  atomicMax(&rows[b].max_key, th_key(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))));
  atomicMax(&rows[b].many_key, key);
  atomicMax(&rows[b].not_all_key, ~key);
}

// ITER 0: the whole range; 1: the crossing bin. The window is [lo, hi): elements
// >= keep_above are kept already (counted in p_above, n_above), elements < lo are
// dropped. An element EXACTLY at the crossing bin's lower edge belongs to the
// refinement window.
template <int ITER>
__global__ __launch_bounds__(256) void topk_topp_hist_kernel(
    ThRow* __restrict__ rows, const float* __restrict__ logits,
    const float* __restrict__ temps, const float* __restrict__ top_ps,
    const long* __restrict__ top_ks, int V, long stride, int chunk, bool vec) {
  const int b = blockIdx.x;
  const float temp = temps[b];
  const long k_lim = top_ks[b];
  bool need_p, need_k;
  if (!th_limits(temp, top_ps[b], k_lim, V, need_p, need_k)) return;
  ThRow& R = rows[b];
  if (ITER == 1 && R.done) return;           // bound written by the first scan
  const int tid = threadIdx.x, lane = tid & 63;
  const float m = th_value(R.max_key);
  const float inv_t = 1.0f / temp;
  const float lo = ITER == 0 ? kThMin : R.lo, hi = ITER == 0 ? 0.0f : R.hi;
  const float keep_above = ITER == 0 ? 3e38f : R.keep_above;
  const float width = (hi - lo) / kThBins;
  const float inv_w = 1.0f / width;

  // Bins below `from` cannot hold the crossing: k elements lie above them.
  int from = 0;
  if (ITER == 0 && need_k && k_lim <= 64 * (long)gridDim.y) {
    const float reach = th_value(k_lim <= 64 ? R.many_key : ~R.not_all_key);
    const float at = ((reach - m) * inv_t - lo) * inv_w;
    from = at > 1.f ? min((int)at - 1, kThBins - 1) : 0;   // a bin's room for rounding
  }
  const float count_from = lo + from * width;
  __shared__ float h_sum[kThCopies][kThBins];
  __shared__ int h_cnt[kThCopies][kThBins];
  for (int i = tid; i < kThCopies * kThBins; i += 256) {
    (&h_sum[0][0])[i] = 0.f;
    (&h_cnt[0][0])[i] = 0;
  }
  __syncthreads();
  const int copy = lane & (kThCopies - 1);
  const int v0 = blockIdx.y * chunk, v1 = min(v0 + chunk, V);
  float tail = 0.f;                          // mass below lo (first window: used for Z)
  th_scan(logits + (long)b * stride, v0, v1, vec, [&](float l) {
    const float x = (l - m) * inv_t;
    if (x >= keep_above) return;
    if (x < (ITER == 0 ? count_from : lo)) {
      if (ITER == 0) tail += __expf(fmaxf(x, -80.f));
      return;
    }
    int bin = (int)((x - lo) * inv_w);
    bin = bin < 0 ? 0 : (bin >= kThBins ? kThBins - 1 : bin);
    atomicAdd(&h_sum[copy][bin], __expf(x));
    if (need_k) atomicAdd(&h_cnt[copy][bin], 1);
  });
  __syncthreads();
  for (int i = tid; i < kThBins; i += 256) {
    float s = 0.f;
    int c = 0;
#pragma unroll
    for (int k = 0; k < kThCopies; ++k) {
      s += h_sum[k][i];
      c += h_cnt[k][i];
    }
    if (s != 0.f) atomicAdd(&R.sum[ITER][i], s);         // e^-32 at the least
    if (c) atomicAdd(&R.cnt[ITER][i], c);
  }
  if (ITER == 0) {
    tail = wave_reduce_sum(tail);
    if (lane == 0 && tail != 0.f) atomicAdd(&R.tail, tail);
  }
}

// One workgroup per row: the crossing bin of the histogram, and what it says.
template <int ITER>
__global__ __launch_bounds__(256) void topk_topp_scan_kernel(
    float* __restrict__ out_bound, ThRow* __restrict__ rows, const float* __restrict__ temps,
    const float* __restrict__ top_ps, const long* __restrict__ top_ks, int V) {
  const int b = blockIdx.x;
  const float temp = temps[b], p_lim = top_ps[b];
  const long k_lim = top_ks[b];
  bool need_p, need_k;
  if (!th_limits(temp, p_lim, k_lim, V, need_p, need_k)) return;
  ThRow& R = rows[b];
  if (ITER == 1 && R.done) return;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const float m = th_value(R.max_key);
  const float lo = ITER == 0 ? kThMin : R.lo, hi = ITER == 0 ? 0.0f : R.hi;
  const float keep_above = ITER == 0 ? 3e38f : R.keep_above;
  const float width = (hi - lo) / kThBins;

  // thread t holds bins 511 - 2t and 510 - 2t; sums run from the top bin down
  const int b0 = kThBins - 1 - 2 * tid, b1 = b0 - 1;
  const float s0 = R.sum[ITER][b0], s1 = R.sum[ITER][b1];
  const int c0 = R.cnt[ITER][b0], c1 = R.cnt[ITER][b1];
  float cs = s0 + s1;
  int cc = c0 + c1;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const float ys = __shfl_up(cs, off, WAVE);
    const int yc = __shfl_up(cc, off, WAVE);
    if (lane >= off) {
      cs += ys;
      cc += yc;
    }
  }
  __shared__ float ws[4];
  __shared__ int wc[4];
  __shared__ int cross;
  if (lane == 63) {
    ws[wid] = cs;
    wc[wid] = cc;
  }
  if (tid == 0) cross = kThBins;
  __syncthreads();
  const float p_above = ITER == 0 ? 0.f : R.p_above;
  const int n_above = ITER == 0 ? 0 : R.n_above;
  float before_s = p_above;
  int before_c = n_above;
  for (int k = 0; k < wid; ++k) {
    before_s += ws[k];
    before_c += wc[k];
  }
  const float z = ITER == 0 ? R.tail + (ws[0] + ws[1] + ws[2] + ws[3]) : R.z;
  before_s += cs - (s0 + s1);                // above this thread's bins
  before_c += cc - (c0 + c1);
  const float p_target = need_p ? p_lim * z : 3e38f;
  const long k_target = need_k ? k_lim : 0x7fffffffffffffffL;
  const bool hit0 = before_s + s0 >= p_target || before_c + c0 >= k_target;
  const bool hit1 = before_s + s0 + s1 >= p_target || before_c + c0 + c1 >= k_target;
  if (hit0 || hit1) atomicMin(&cross, hit0 ? 2 * tid : 2 * tid + 1);
  __syncthreads();
  if (cross == kThBins) {
    // No crossing in the window. First: the target needs mass below it too, keep
    // everything. Second: rounding; keep the WHOLE window.
    if (tid == 0) {
      out_bound[b] = ITER == 0 ? -3e38f : m + lo * temp;
      if (ITER == 0) R.done = 1;
    }
    return;
  }
  if (tid != cross / 2) return;
  const int bin = cross & 1 ? b1 : b0;
  if (ITER == 1) {
    out_bound[b] = m + (lo + bin * width) * temp;
    return;
  }
  R.lo = lo + bin * width;
  R.hi = lo + (bin + 1) * width;
  // The window's top lies INSIDE the top bin: where that bin is the crossing one,
  // the row's maximum must stay in the refinement.
  R.keep_above = bin == kThBins - 1 ? keep_above : lo + (bin + 1) * width;
  R.z = z;
  R.p_above = before_s + (cross & 1 ? s0 : 0.f);
  R.n_above = before_c + (cross & 1 ? c0 : 0);
}

// fp32 logits of bf16 ones, through cap * tanh(x / cap): one pass instead of a
// conversion, a division, tanh and a product.
__global__ __launch_bounds__(256) void softcap_logits_kernel(
    float* __restrict__ out, const __hip_bfloat16* __restrict__ in, long n, float cap) {
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8; i < n; i += (long)gridDim.x * 2048) {
    float y[8];
    if (i + 8 <= n) {
      const Vec8<__hip_bfloat16> x = load16(in + i);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = tanhf(to_f32(x.data[e]) / cap) * cap;
      *reinterpret_cast<float4*>(out + i) = make_float4(y[0], y[1], y[2], y[3]);
      *reinterpret_cast<float4*>(out + i + 4) = make_float4(y[4], y[5], y[6], y[7]);
    } else {
      for (long e = i; e < n; ++e) out[e] = tanhf(to_f32(in[e]) / cap) * cap;
    }
  }
}

// A row's best chunk, by a wave: the packed key and the token that it names. (Chunks that met
// in one word by atomics needed it cleared, a launch a step: head and sampler of one row
// 77.4 us, 76.3 without; of 142 rows, 131072 tokens 202.5 and 201.1.)
__global__ __launch_bounds__(256) void unpack_keys_kernel(
    long* __restrict__ out, unsigned long long* __restrict__ keys,
    const unsigned long long* __restrict__ parts, int splits, int B) {
  const int b = blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  if (b >= B) return;
  unsigned long long best = 0;
  for (int i = lane; i < splits; i += WAVE) best = max(best, parts[(long)b * splits + i]);
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1)
    best = max(best, (unsigned long long)__shfl_xor((long long)best, off, WAVE));
  if (lane == 0) {
    keys[b] = best;
    out[b] = (long)(unsigned int)(~(best & 0xffffffffu));
  }
}
