// Single-token GQA attention over the paged cache on the matrix cores (gfx950):
// bf16 queries; head size 128 or 256 with a bf16 or fp8 (OCP e4m3) cache and up to 16
// query heads per kv head, head size 64 with a bf16 cache and up to 8; optional score
// cap and sliding window.
//
// Bound by the cache's bytes: at 16 query columns the products take a few percent
// of the matrix cores, so everything here serves to keep loads in flight on all
// CUs until the last byte has come. Measured (us, with the merge; before = one
// workgroup per pair, VALU at head size 64, K and V through one shared LDS
// pipeline else): 64 x 1040 keys, 8 kv heads of 64: 391 -> 34 (136 MB);
// 189 ragged up to 1100, 8 of 128: 152 -> 108 (473 MB); 3 ragged up to 16000,
// 8 of 128: 83 -> 40 (147 MB); 96 x 1064, 8 of 256, capped: 197 -> 161 (837 MB);
// 512 x 1064: 889 -> 772 (4.46 GB, 5.8 TB/s); 48 ragged up to 2000, 8 of 256,
// fp8: 132 -> 55 (219 MB). Below about 100 MB the two launches, the walk from
// lengths to block table to keys and the merge (together 8 us) count most.
//
//   - The work is cut in tiles of 16 NK keys of one (sequence, kv head) pair, and
//     the tiles of the whole batch, in order, are dealt to a fixed number of waves
//     in equal contiguous ranges. Every wave finds its range by itself from
//     context_lens, so lengths may differ and change under a captured graph, and
//     neither a long sequence nor a last round of workgroups leaves CUs idle. Where a
//     sequence is cut, and with it the order of its sums, depends on the lengths of the
//     whole batch and on the table's width: its result may differ in the last bf16
//     digit between batches, and between a captured graph and an eager call.
//   - Waves are independent: no barrier anywhere. K operands come straight from
//     memory in matrix layout; V rows pass through a wave-private LDS tile
//     (row-major, 32-byte column groups swizzled by key) and are read transposed
//     with ds_read_b64_tr_b16. The next tile's rows are in flight during the
//     current tile's products.
//   - Both products run transposed, S^T = K Q^T and O^T = V^T P^T (A: row =
//     lane%16, k = 8*(lane/16)..+7; B: column = lane%16; C: column = lane%16, rows
//     4*(lane/16)+r), so a lane's scores belong to one query and its weights are
//     already the second product's operand: slot 8h+4b+i = key 16b+4h+i.
//   - Weights enter as bf16 planes, a product each, which is not the bound. Head sizes
//     128 and 256: two, 16 mantissa bits. Head size 64: three, all 24 bits, as the fp32
//     kernel that still serves fp32 caches has them: 64 x 1040 keys, queries of size 3,
//     outputs other than the 64-bit result's nearest bf16: that kernel 4.3e-4, three
//     planes 3.8e-4, two 1.5e-3; 1b decode step of 64 sequences 1726 and 1708 us with
//     two and three.
//   - A pair that lies in one wave's range is written at once; the pieces of the
//     others go to `part` (output, maximum in the log2 domain, sum) and are merged
//     by paged_decode_merge_kernel.

#include "common.h"

typedef __attribute__((ext_vector_type(4))) short pd_s16x4;
typedef __attribute__((ext_vector_type(8))) short pd_s16x8;
typedef __attribute__((ext_vector_type(4))) unsigned pd_u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned pd_u32x2;
typedef __attribute__((ext_vector_type(4))) float pd_f32x4;
typedef __attribute__((ext_vector_type(2))) float pd_f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 pd_bf16x2;
typedef __attribute__((ext_vector_type(4))) __bf16 pd_bf16x4;
typedef __attribute__((address_space(3))) pd_bf16x4 pd_lds_bf16x4;

// Tiles of 2^TS keys that a sequence's visible keys touch.
template <int TS>
DEVINL int pd_tiles(int len, int window) {
  if (len <= 0) return 0;
  const int lo = window > 0 && len > window ? len - window : 0;
  return ((len - 1) >> TS) - (lo >> TS) + 1;
}

// The visible tiles of all sequences, one kv head. `first` is lane's entry of
// context_lens, loaded by the caller.
template <int TS>
DEVINL int pd_total(const int* __restrict__ lens, int B, int window, int lane, int first) {
  int n = lane < B ? pd_tiles<TS>(first, window) : 0;
  for (int b = lane + WAVE; b < B; b += WAVE) n += pd_tiles<TS>(lens[b], window);
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, WAVE);
  return __builtin_amdgcn_readfirstlane(n);
}

// Tiles per wave: an equal share. One tile while that leaves CUs without work
// (latency); two from there on, so that short pairs are not cut needlessly. Head size 64's
// tiles are half as many keys and bytes: two where pairs of one or two tiles would be cut for
// nothing and where one would make over 64 pieces of a pair; four beyond 2048 tiles, unless
// pairs are short and two make one round. Measured (us, with the merge, least share of 1 / 2):
// 1 x 20 keys, 8 kv heads 6.5 / 7.6, 8 x 60 8.3 / 7.4, 32 ragged up to 50 8.3 / 7.7, 1 x 200
// 8.6 / 9.4, 1 x 4000, 2 kv heads 12.0 / 10.1; of 2 / 4: 200 ragged up to 100 14.7 / 16.3,
// 512 x 60 (three, by count) 29.4 / 24.7.
template <int D>
DEVINL int pd_share(int total, int waves, int pairs) {
  int least = total > 1024 ? 2 : 1;
  if constexpr (D == 64) {
    // without branches: 1 x 200 keys 8.1 us with them, 7.9 so
    const bool two = total > 512 || (unsigned)(total - pairs - 1) < (unsigned)pairs ||
                     total > 64 * pairs;
    const bool four = total > 2048 && (total > 3 * pairs || total > 2 * waves);
    least = 1 + two + 2 * four;
  }
  return max((total + waves - 1) / waves, least);
}

// The first sequence whose tiles reach past `t` (all pairs counted, kv heads
// innermost), its length and the tiles of one kv head before it.
template <int TS>
DEVINL void pd_locate(const int* __restrict__ lens, int B, int KVH, int window, int lane, int t,
                      int first, int& b, int& len, int& before) {
  int base = 0;
  b = len = before = 0;
  for (int c = 0; c < B; c += WAVE) {
    const int mine = c == 0 ? first : c + lane < B ? lens[c + lane] : 0;
    const int n = c + lane < B ? pd_tiles<TS>(mine, window) : 0;
    int x = n;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const int y = __shfl_up(x, off, WAVE);
      if (lane >= off) x += y;
    }
    const unsigned long long hit = __ballot((base + x) * KVH > t);
    if (hit) {
      const int at = __ffsll((long long)hit) - 1;
      b = c + at;
      len = __builtin_amdgcn_readlane(mine, at);
      before = base + __builtin_amdgcn_readlane(x - n, at);
      return;
    }
    base += __builtin_amdgcn_readlane(x, WAVE - 1);
  }
}

// 8 fp8 -> 8 bf16, exact: e4m3 has fewer bits than bf16 in both fields.
DEVINL pd_s16x8 pd_widen(unsigned lo, unsigned hi) {
  pd_u32x4 r;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int v = (int)(w ? hi : lo);
    const pd_f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
    const pd_f32x2 c = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
    r[w * 2] = __builtin_amdgcn_perm(__float_as_uint(a[1]), __float_as_uint(a[0]), 0x07060302u);
    r[w * 2 + 1] = __builtin_amdgcn_perm(__float_as_uint(c[1]), __float_as_uint(c[0]), 0x07060302u);
  }
  return __builtin_bit_cast(pd_s16x8, r);
}

// Two weights -> their bf16 planes: hi cut off, lo the rounded rest (16 mantissa bits),
// or with three planes the rest cut off and rounded again, exact: 24 bits.
template <int PL>
DEVINL void pd_planes(float p0, float p1, unsigned (&w)[PL]) {
#pragma unroll
  for (int i = 0; i + 1 < PL; ++i) {
    const unsigned b0 = __float_as_uint(p0), b1 = __float_as_uint(p1);
    w[i] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
    p0 -= __uint_as_float(b0 & 0xffff0000u);
    p1 -= __uint_as_float(b1 & 0xffff0000u);
  }
  w[PL - 1] = __builtin_bit_cast(
      unsigned, __builtin_convertvector((pd_f32x2{p0, p1}), pd_bf16x2));
}

// Swizzle of the V tile's 16-byte granules: the 8 keys that one transposing read
// takes together lie in 8 different 32-byte bank groups.
template <int D>
DEVINL int pd_swz(int key) {
  return D >= 128 ? (key & 7) << 1 : ((key >> 1) & 3) << 1;
}

template <int D, typename TC, int NK>
struct PdShape {
  static constexpr int kTileShift = NK == 2 ? 5 : 4;
  static constexpr int kKeys = 16 * NK;
  static constexpr size_t kLds = 4 * sizeof(short) * (size_t)kKeys * D;
};

template <int D, typename TC, int NK, int OCC, bool CAP>
__global__ __launch_bounds__(256, OCC) void paged_decode_kernel(
    __hip_bfloat16* __restrict__ out, long out_stride,
    const __hip_bfloat16* __restrict__ q, long q_stride,
    const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ lens,
    int B, int KVH, int G, int bs_shift, int window, float scale_log2, float cap_log2,
    float cap_in, float* __restrict__ part_o, float* __restrict__ part_ml) {
  constexpr bool F8 = sizeof(TC) == 1;
  constexpr int TS = PdShape<D, TC, NK>::kTileShift, KT = 16 * NK;
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int PL = D == 64 ? 3 : 2;                // bf16 planes of a weight
  constexpr int KL = F8 ? KS / 2 : KS;               // 16-byte loads of a K operand row
  constexpr int GPR = D * (int)sizeof(TC) / 16;      // 16-byte granules of a V row
  constexpr int RPI = WAVE / GPR;                    // V rows per load
  constexpr int NV = KT / RPI;
  extern __shared__ __align__(16) unsigned char pd_smem[];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  short* const Vt = reinterpret_cast<short*>(pd_smem) + w * (KT * D);

  // consecutive ranges on different CUs
  const int waves = gridDim.x * 4;
  const int wave = w * gridDim.x + blockIdx.x;
  const int first = lens[min(lane, B - 1)];
  const int total = pd_total<TS>(lens, B, window, lane, first) * KVH;
  const int share = pd_share<D>(total, waves, B * KVH);
  int t = wave * share;
  const int t_end = min(total, t + share);
  if (t >= t_end) return;
  int b, len, before, kh, i0;
  pd_locate<TS>(lens, B, KVH, window, lane, t, first, b, len, before);
  int nt = pd_tiles<TS>(len, window);
  {
    const int r = t - before * KVH;
    kh = r / nt;
    i0 = r % nt;
  }
  const int t_begin = t;
  const int bs_mask = (1 << bs_shift) - 1;

  // this lane's part of the K operands and of the V tile
  const unsigned klane = col * D + grp * (16 / (int)sizeof(TC));
  const int vrow = lane / GPR, vgran = lane % GPR;
  const unsigned vlane = vrow * D + vgran * (16 / (int)sizeof(TC));
  // transposing reads: 16 lanes take 4 keys x 16 channels
  const int tkey = grp * 4 + (col >> 2);
  const int tsw = pd_swz<D>(tkey);
  const int tbase = tkey * D + (col & 1) * 4;
  const int tg = (col & 3) >> 1;

  while (t < t_end) {
    const int pos = len - 1;
    const int lo = window > 0 && len > window ? len - window : 0;
    const int n = min(nt - i0, t_end - t);
    const int* bt = block_tables + (long)b * bt_stride;
    int key0 = ((lo >> TS) + i0) << TS;

    // cache rows of the tile's 16-key groups (a group past the end takes the last
    // live block: its scores are masked and its values zeroed)
    long rb[NK];
    auto rows = [&](int k0) {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const int key = k0 + i * 16;
        const int at = __builtin_amdgcn_readfirstlane(min(key, pos) >> bs_shift);
        rb[i] = (((long)bt[at] * KVH + kh) << bs_shift) + (key & bs_mask);
      }
    };
    pd_s16x8 kf[NK][KL], vf[NV];
    auto fetch_k = [&]() {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const TC* kr = k_cache + rb[i] * D;    // uniform; the lane adds 32 bits
#pragma unroll
        for (int ks = 0; ks < KL; ++ks)
          kf[i][ks] = *reinterpret_cast<const pd_s16x8*>(kr + (klane + ks * (F8 ? 64 : 32)));
      }
    };
    auto fetch_v = [&]() {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const TC* vr = v_cache + rb[(i * RPI) >> 4] * D;
        vf[i] = *reinterpret_cast<const pd_s16x8*>(vr + (vlane + ((i * RPI) & 15) * D));
      }
    };
    rows(key0);
    fetch_k();
    fetch_v();
    if (n > 1) rows(key0 + KT);

    pd_s16x8 qf[KS];
    {
      const __hip_bfloat16* qr = q + (long)b * q_stride + (long)(kh * G + col) * D;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d8 = F8 ? (ks >> 1) * 64 + grp * 16 + (ks & 1) * 8 : ks * 32 + grp * 8;
        qf[ks] = col < G ? *reinterpret_cast<const pd_s16x8*>(qr + d8)
                         : pd_s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
    float m = -INFINITY, l = 0.f;              // log2 domain
    pd_f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = pd_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int i = 0; i < n; ++i, key0 += KT) {
      const bool more = i + 1 < n;
      pd_f32x4 s[NK];
#pragma unroll
      for (int g = 0; g < NK; ++g) s[g] = pd_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KL; ++ks)
#pragma unroll
        for (int g = 0; g < NK; ++g) {
          if constexpr (F8) {
            const pd_u32x4 raw = __builtin_bit_cast(pd_u32x4, kf[g][ks]);
            s[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pd_widen(raw[0], raw[1]),
                                                           qf[2 * ks], s[g], 0, 0, 0);
            s[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pd_widen(raw[2], raw[3]),
                                                           qf[2 * ks + 1], s[g], 0, 0, 0);
          } else {
            s[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[g][ks], qf[ks], s[g], 0, 0, 0);
          }
        }
      if (more) fetch_k();

      if constexpr (CAP) cap_tile<NK, 4>(s, scale_log2, cap_log2, cap_in);
      const bool ragged = key0 < lo || key0 + KT - 1 > pos;
      float tmax = -INFINITY;
#pragma unroll
      for (int g = 0; g < NK; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x = CAP ? s[g][r] : s[g][r] * scale_log2;
          if (ragged) {
            const int key = key0 + g * 16 + grp * 4 + r;
            x = key >= lo && key <= pos ? x : -INFINITY;
          }
          s[g][r] = x;
          tmax = fmaxf(tmax, x);
        }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, WAVE));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, WAVE));
      const float m_new = fmaxf(m, tmax);
      const float mb = m_new > -INFINITY ? m_new : 0.f;
      if (__any(m_new > m)) {
        const float alpha = __builtin_amdgcn_exp2f(m - mb);    // m = -inf -> 0
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
        m = m_new;
      }

      // V rows to the wave's tile; rows past the end as zeros (a weight of zero
      // does not cancel what an unwritten row may hold)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int key = v * RPI + vrow;
        if (ragged && key0 + key > pos) vf[v] = pd_s16x8{0, 0, 0, 0, 0, 0, 0, 0};
        short* row = Vt + key * D;
        if constexpr (F8) {
          const pd_u32x4 raw = __builtin_bit_cast(pd_u32x4, vf[v]);
          short* dst = row + (((2 * vgran) ^ pd_swz<D>(key)) << 3);
          *reinterpret_cast<pd_s16x8*>(dst) = pd_widen(raw[0], raw[1]);
          *reinterpret_cast<pd_s16x8*>(dst + 8) = pd_widen(raw[2], raw[3]);
        } else {
          *reinterpret_cast<pd_s16x8*>(row + ((vgran ^ pd_swz<D>(key)) << 3)) = vf[v];
        }
      }
      if (more) {
        fetch_v();
        if (i + 2 < n) rows(key0 + 2 * KT);
      }
      // one wave, LDS in order: the tile's writes come before its reads
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();

      if constexpr (NK == 1) {
        pd_u32x2 pw[PL];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float p0 = __builtin_amdgcn_exp2f(s[0][2 * e] - mb);
          const float p1 = __builtin_amdgcn_exp2f(s[0][2 * e + 1] - mb);
          l += p0 + p1;
          unsigned w2[PL];
          pd_planes(p0, p1, w2);
#pragma unroll
          for (int pl = 0; pl < PL; ++pl) pw[pl][e] = w2[pl];
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const pd_s16x4 va = __builtin_bit_cast(pd_s16x4, __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (pd_lds_bf16x4*)(Vt + tbase + (((dt * 2 + tg) ^ tsw) << 3))));
#pragma unroll
          for (int pl = 0; pl < PL; ++pl)
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                va, __builtin_bit_cast(pd_s16x4, pw[pl]), o[dt], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < NK / 2; ++j) {
          pd_u32x4 pw[PL];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p0 = __builtin_amdgcn_exp2f(s[2 * j + e / 2][(e & 1) * 2] - mb);
            const float p1 = __builtin_amdgcn_exp2f(s[2 * j + e / 2][(e & 1) * 2 + 1] - mb);
            l += p0 + p1;
            unsigned w2[PL];
            pd_planes(p0, p1, w2);
#pragma unroll
            for (int pl = 0; pl < PL; ++pl) pw[pl][e] = w2[pl];
          }
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            short* at = Vt + j * 32 * D + tbase + (((dt * 2 + tg) ^ tsw) << 3);
            const pd_s16x4 v0 = __builtin_bit_cast(pd_s16x4,
                __builtin_amdgcn_ds_read_tr16_b64_v4bf16((pd_lds_bf16x4*)at));
            const pd_s16x4 v1 = __builtin_bit_cast(pd_s16x4,
                __builtin_amdgcn_ds_read_tr16_b64_v4bf16((pd_lds_bf16x4*)(at + 16 * D)));
            const pd_s16x8 va = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int pl = 0; pl < PL; ++pl)
              o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  va, __builtin_bit_cast(pd_s16x8, pw[pl]), o[dt], 0, 0, 0);
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    l += __shfl_xor(l, 16, WAVE);
    l += __shfl_xor(l, 32, WAVE);
    if (col < G) {
      if (n == nt) {
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        __hip_bfloat16* orow = out + (long)b * out_stride + (long)(kh * G + col) * D + grp * 4;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          Vec4<__hip_bfloat16> v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v.data[r] = __float2bfloat16(o[dt][r] * inv);
          *reinterpret_cast<int2*>(orow + dt * 16) = *reinterpret_cast<const int2*>(v.data);
        }
      } else {
        // a range holds at most two pieces: one from its start, one to its end
        const long slot = ((long)wave * 2 + (t == t_begin ? 0 : 1)) * G + col;
        float* po = part_o + slot * D + grp * 4;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<pd_f32x4*>(po + dt * 16) = o[dt];
        if (grp == 0) *reinterpret_cast<pd_f32x2*>(part_ml + slot * 2) = pd_f32x2{m, l};
      }
    }
    t += n;
    i0 = 0;
    if (t < t_end && ++kh == KVH) {
      kh = 0;
      do {
        len = __builtin_amdgcn_readfirstlane(lens[++b]);
        nt = pd_tiles<TS>(len, window);
      } while (nt == 0);
    }
  }
}

// The pieces of a (sequence, query head) that several waves shared, merged by WPP
// waves: each takes every WPP-th piece, eight at a time. WPP = 1: four heads per
// workgroup (64 sequences, 32 heads of 64: 4.6 us, four waves each 7.1).
template <int D, int TS, int WPP>
__global__ __launch_bounds__(256) void paged_decode_merge_kernel(
    __hip_bfloat16* __restrict__ out, long out_stride, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const int* __restrict__ lens, int B, int KVH, int G,
    int window, int waves) {
  constexpr int DL = D / WAVE;               // channels per lane
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = WPP == 1 ? 0 : wave;
  const int b = blockIdx.x, h = WPP == 1 ? blockIdx.y * 4 + wave : blockIdx.y;
  const int nt = pd_tiles<TS>(lens[b], window);
  if (nt == 0) return;
  int all = 0, before = 0;
  for (int c = lane; c < B; c += WAVE) {
    const int n = pd_tiles<TS>(lens[c], window);
    all += n;
    before += c < b ? n : 0;
  }
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    all += __shfl_xor(all, off, WAVE);
    before += __shfl_xor(before, off, WAVE);
  }
  const int share = pd_share<D>(all * KVH, waves, B * KVH);
  const int first_tile = before * KVH + (h / G) * nt;
  const int first = first_tile / share, last = (first_tile + nt - 1) / share;
  if (first == last) return;                 // written by its wave
  // the first piece starts inside its wave's range unless it opens it
  const int head = first_tile % share ? 1 : 0;
  const int g = h % G;
  float m = -INFINITY, l = 0.f, o[DL];
#pragma unroll
  for (int c = 0; c < DL; ++c) o[c] = 0.f;
  for (int s0 = first + w; s0 <= last; s0 += 8 * WPP) {
    float pm[8], pl[8], po[8][DL];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int s = min(s0 + e * WPP, last); // past the end: weight zero below
      const long slot = ((long)s * 2 + (s == first ? head : 0)) * G + g;
      const pd_f32x2 ml = *reinterpret_cast<const pd_f32x2*>(part_ml + slot * 2);
      pm[e] = s0 + e * WPP <= last ? ml[0] : -INFINITY;
      pl[e] = ml[1];
#pragma unroll
      for (int c = 0; c < DL; ++c) po[e][c] = part_o[slot * D + c * WAVE + lane];
    }
    float top = m;
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, pm[e]);
    const float tb = top > -INFINITY ? top : 0.f;
    const float f0 = __builtin_amdgcn_exp2f(m - tb);
    l *= f0;
#pragma unroll
    for (int c = 0; c < DL; ++c) o[c] *= f0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = __builtin_amdgcn_exp2f(pm[e] - tb);
      if (pm[e] > -INFINITY) {
        l += pl[e] * f;
#pragma unroll
        for (int c = 0; c < DL; ++c) o[c] += po[e][c] * f;
      }
    }
    m = top;
  }
  if constexpr (WPP == 1) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
    for (int c = 0; c < DL; ++c)
      out[(long)b * out_stride + (long)h * D + c * WAVE + lane] = __float2bfloat16(o[c] * inv);
    return;
  }
  __shared__ float so[4][D], sm[4], sl[4];
#pragma unroll
  for (int c = 0; c < DL; ++c) so[w][c * WAVE + lane] = o[c];
  if (lane == 0) {
    sm[w] = m;
    sl[w] = l;
  }
  __syncthreads();
  if (threadIdx.x >= D) return;
  const float top = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
  const float tb = top > -INFINITY ? top : 0.f;
  float a = 0.f, ll = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float f = __builtin_amdgcn_exp2f(sm[e] - tb);
    a += so[e][threadIdx.x] * f;
    ll += sl[e] * f;
  }
  out[(long)b * out_stride + (long)h * D + threadIdx.x] =
      __float2bfloat16(ll > 0.f ? a / ll : 0.f);
}
