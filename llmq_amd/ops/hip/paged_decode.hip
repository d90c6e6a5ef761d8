// Single-token GQA attention over the paged cache on the matrix cores (gfx950):
// bf16 queries; head size 128 or 256 with a bf16 or fp8 (OCP e4m3) cache and up to 16
// query heads per kv head, head size 64 with a bf16 cache and up to 8; optional score
// cap and sliding window.
//
// Bound by the cache's bytes: at 16 query columns the products take a few percent
// of the matrix cores, so everything here serves to keep loads in flight on all
// CUs until the last byte has come. Measured (us; before = a wave a range, waves' pieces
// merged by a second launch): 1 x 200 keys, 8 kv heads of 64: 7.6 -> 4.6; 16 ragged up to 300,
// the same: 10.7 -> 7.0; 1 x 1000: 8.7 -> 8.1; 64 x 1040: 33.4 -> 26.2 (136 MB); 7 ragged up to
// 1900, 2 of 128, 6 heads each: 12.0 -> 10.6; 189 ragged up to 1100, 8 of 128: 97 -> 87 (5.4 TB/s);
// 3 ragged up to 16000, the same: 33.8 -> 28.9; 96 x 1064, 8 of 256, capped: 156 -> 142 (837 MB,
// 5.9 TB/s); 64 ragged up to 300, the same: 26.3 -> 24.9; 48 ragged up to 2000, fp8: 52.1 -> 48.5;
// 64 x 1040, 2 of 256, 16 heads each: 41.5 -> 39.2. Below about 100 MB the launch, the walk from
// lengths to block table to keys and every instruction around it (4 clocks each) count most.
//
//   - The work is cut in tiles of 16 NK keys of one (sequence, kv head) pair, in order, and
//     dealt to a fixed number of workgroups: a piece of a pair or a whole one each, or equal
//     ranges (pd_deal). Every workgroup finds its part by itself from
//     context_lens, so lengths may differ and change under a captured graph, and
//     neither a long sequence nor a last round of workgroups leaves CUs idle. Where a
//     sequence is cut, and with it the order of its sums, depends on the lengths of the
//     whole batch and on the table's width: its result may differ in the last bf16
//     digit between batches, and between a captured graph and an eager call.
//   - The four waves of a workgroup share the tiles of a pair, each with its own sums; they
//     meet in LDS, while the range's next pair is on its way. Until then they are independent:
//     K operands come straight from memory in matrix layout; V rows pass through a wave-private
//     LDS tile (row-major, 32-byte column groups swizzled by key) and are read transposed
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
//   - A pair that lies in one workgroup's range is written at once; the pieces of the
//     others go to `part` (output, maximum in the log2 domain, sum), and the last workgroup to
//     arrive at a pair, counted in `arrivals`, merges its pieces in their order. (The launch
//     that did so took 3.7 to 7.6 us, this 1 to 2.)

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
__host__ __device__ __forceinline__ int pd_tiles(int len, int window) {
  if (len <= 0) return 0;
  const int lo = window > 0 && len > window ? len - window : 0;
  return ((len - 1) >> TS) - (lo >> TS) + 1;
}

// x of this lane and all before it, without the LDS crossbar (whose six exchanges take 0.3 us).
DEVINL int pd_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr 1, 2, 4, 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast 15, 31
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}
DEVINL int pd_max(int x) {                       // of values >= 0
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(x, WAVE - 1);
}
DEVINL int pd_sum(int x) { return __builtin_amdgcn_readlane(pd_scan(x), WAVE - 1); }

// Here and on the host, where the deal is tested. Quotients below 2^20 are exact: the reciprocal's
// error moves them by less than the half that keeps them off whole numbers.
__host__ __device__ __forceinline__ float pd_rcp(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.f / x;
#endif
}
__host__ __device__ __forceinline__ float pd_sqrt(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_sqrtf(x);
#else
  return sqrtf(x);
#endif
}
__host__ __device__ __forceinline__ int pd_quotient(int x, float inv) {
  return (int)(((float)x + 0.5f) * inv);
}

// Pieces of a pair of nt tiles, of up to c each; up to twice the least piece stays whole. One
// workgroup reads the partial sums of all, each as many bytes as `thick` tiles, so that a piece has
// at least sqrt(nt `thick`) tiles, with a factor for the merge's longer way, in whole rounds of four
// waves. us, without that floor / with it: 1 x 16000 keys, 1 kv head of 256, 8 heads 62.6 / 30.8; 3 x
// 16000, 2 of 128, 6 heads each 29.5 / 21.0; 1 x 16000, 8 of 64, 4 heads each 17.2 / 15.3. Factors of 1
// to 3 are within 1 % over 86 batches; at 2 one of 4000 keys, 2 of 128, fp8 loses 13 %.
__host__ __device__ __forceinline__ int pd_piece(int nt, int c, float thick) {
  const int floor = ((int)pd_sqrt(1.5f * nt * thick) + 3) & ~3;    // four waves share them
  return c > floor ? c : floor;
}
__host__ __device__ __forceinline__ int pd_pieces(int nt, int c, int least, float thick) {
  if (nt <= 2 * least) return nt > 0;
  const int size = pd_piece(nt, c, thick);
  return pd_quotient(nt + size - 1, pd_rcp((float)size));
}

// How the tiles of all pairs (in order, kv heads innermost) are dealt to `wgs` workgroups, of
// which `resident` run at a time: piece > 0: a piece of a pair each, of up to that many tiles;
// else `share` tiles each to `resident` of them. In turn:
//   - pieces of the least size (64 KiB, what a CU takes in in 1 us; of 32 KiB and more of them 1 x
//     12000 keys, 8 kv heads of 64 26.4 us, of 64 15.2) where all find a workgroup;
//   - whole pairs unless the longest is over twice the mean share; short ones (three least pieces
//     in the mean) up to three times, and also more of them than run at a time. us, whole / equal
//     ranges: 64 x 1040, 8 of 64 26.6 / 33; 120 ragged up to 700, the same 25.1 / 29.0; 200 up to
//     700, 8 of 128, fp8 40.0 / 45.3; 100 up to 300, 8 of 256 35.7 / 38.9; 120 up to 400, the same,
//     fp8 33.3 / 37.9; 200 up to 400, 8 of 256 (3.5 least pieces) 77.3 / 80.1, 150 up to 500 (4.4)
//     73.2 / 70.9; 48 up to 2000, 8 of 256, fp8 (2.45 times) 57.8 / 46.9;
//   - pieces that surely find a workgroup, where they are at most 1.5 mean shares (24 ragged up
//     to 1500, 8 of 256, 1.6: 43.3, equal ranges 38.8);
//   - equal ranges, whose ends cut pairs and whose segments follow each other; at head size 256
//     with a bf16 cache one workgroup a CU where that is 2 MiB each (96 x 1064: 143.7 / 142.3).
struct PdDeal { int piece, share, total; };

// tiles: of all pairs; most: of one; their least pieces are too many.
__host__ __device__ __forceinline__ PdDeal pd_choose(int tiles, int most, int pairs, int wgs,
                                                     int resident, int least, bool lone) {
  const int share = (tiles + resident - 1) / resident;
  const bool brief = tiles <= 3 * least * pairs;
  if (pairs <= (brief ? wgs : resident) && most <= (brief ? 3 : 2) * share) return {most, 1, pairs};
  const int room = resident - pairs;
  if (room > 0) {
    const int c = (tiles + room - 1) / room;   // sum of ceil(n / c) <= tiles / c + pairs
    if (c * 2 <= share * 3) return {c, 1, wgs};
  }
  return {0, lone && share >= 64 ? 2 * share : share, tiles};
}

// Workgroups of a launch: as many as are resident, so that every range is in work at once, and
// one for every pair. tiles: of a pair, at most.
inline long pd_workgroups(long pairs, long tiles, int least, long resident) {
  const long most = pairs * ((tiles + least - 1) / least), all = resident > pairs ? resident : pairs;
  return all < most ? all : most;
}

// The lengths of sequences c + lane, c + 64 + lane, ..: four loads in flight.
struct PdLens { int of[4]; };
DEVINL PdLens pd_lens(const int* __restrict__ lens, int B, int lane, int c) {
  PdLens r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r.of[i] = c + i * WAVE < B ? lens[min(c + i * WAVE + lane, B - 1)] : 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (c + i * WAVE + lane >= B) r.of[i] = 0;
  return r;
}

template <int TS>
DEVINL PdDeal pd_deal(const int* __restrict__ lens, int B, int KVH, int window, int lane,
                      const PdLens& first, int wgs, int resident, int least, float thick,
                      bool lone) {
  int tiles = 0, n0 = 0, most = 0;
  auto each = [&](auto f) {
    for (int c = 0; c < B; c += 4 * WAVE) {
      const PdLens l = c == 0 ? first : pd_lens(lens, B, lane, c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (c + i * WAVE >= B) break;
        f(pd_tiles<TS>(l.of[i], window));
      }
    }
  };
  each([&](int n) {
    tiles += n;
    n0 += n <= 2 * least ? min(n, 1) : (n + least - 1) / least;
    most = max(most, n);
  });
  most = pd_max(most);
  // Only where the longest pair's floor is over the least piece is it the count: else none of its
  // branches (189 ragged up to 300 keys, 8 kv heads of 128: 36.0 us with them, 35.2 so).
  if (pd_piece(most, least, thick) > least) {
    n0 = 0;
    each([&](int n) { n0 += pd_pieces(n, least, least, thick); });
  }
  tiles = pd_sum(tiles) * KVH;
  n0 = pd_sum(n0) * KVH;
  if (n0 <= wgs) return {least, 1, n0};
  return pd_choose(tiles, most, B * KVH, wgs, resident, least, lone);
}

// The first sequence whose pieces or tiles reach past `t` (all pairs counted), its length and
// those of one kv head before it.
template <int TS>
DEVINL void pd_locate(const int* __restrict__ lens, int B, int KVH, int window, int lane, int t,
                      const PdLens& first, int piece, int least, float thick, int& b, int& len,
                      int& before) {
  int base = 0;
  for (int c = 0; c < B; c += 4 * WAVE) {
    const PdLens l = c == 0 ? first : pd_lens(lens, B, lane, c);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (c + i * WAVE >= B) break;
      int n = pd_tiles<TS>(l.of[i], window);
      if (piece > 0) n = pd_pieces(n, piece, least, thick);
      const int x = pd_scan(n);
      const unsigned long long hit = __ballot((base + x) * KVH > t);
      if (hit) {
        const int at = __ffsll((long long)hit) - 1;
        b = c + i * WAVE + at;
        len = __builtin_amdgcn_readlane(l.of[i], at);
        before = base + __builtin_amdgcn_readlane(x - n, at);
        return;
      }
      base += __builtin_amdgcn_readlane(x, WAVE - 1);
    }
  }
  b = B;                                       // no piece for this workgroup
  len = before = 0;
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

// A pair in pieces: the workgroups that have them, and the first one's slot among its two.
struct PdPair { int b, kh, w_first, w_last, head; };

// 16 bytes of the cache, which a step reads once: past the last-level cache (us, kept there /
// not: 189 ragged up to 1100 keys, 8 kv heads of 128 95.2 / 87.6; 96 x 1064, 8 of 256 151.5 /
// 141.6; 48 ragged up to 2000, fp8 50.2 / 46.9; 64 x 1040, 8 of 64 27.8 / 26.9).
DEVINL pd_s16x8 pd_stream(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const pd_s16x8*>(p));
}

// The workgroup's LDS accesses are done; loads from memory may travel.
DEVINL void pd_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Words that workgroups on other XCDs, whose L2 is another, read in the same launch: they go
// to and come from memory itself. Whoever has seen the writer's later arrival sees them.
DEVINL void pd_publish(float* to, pd_f32x2 x) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(to),
                     __builtin_bit_cast(unsigned long long, x), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL pd_f32x2 pd_published(const float* from) {
  return __builtin_bit_cast(pd_f32x2, __hip_atomic_load(
      reinterpret_cast<const unsigned long long*>(from), __ATOMIC_RELAXED,
      __HIP_MEMORY_SCOPE_AGENT));
}

// Two or four channels (V) of a head, their sum not yet divided by its weight.
template <typename V>
struct PdSum {
  float top, weight;
  V x;
};
template <typename V>
DEVINL void pd_finish(__hip_bfloat16* to, const PdSum<V>& s) {
  typedef __bf16 Row __attribute__((ext_vector_type(sizeof(V) / 4)));
  const V y = s.x * (s.weight > 0.f ? 1.0f / s.weight : 0.f);
  *reinterpret_cast<Row*>(to) = __builtin_convertvector(y, Row);
}

// The sums of a pair's pieces, of E quads of channels that are 256 quads apart and of which `live`
// are there: pieces `group`, `group` + `groups`, .. At 32-bit offsets of rows of heads from the
// first piece's workgroup: 64-bit places and divisions took 0.5 us (7 ragged up to 1900 keys, 2 kv
// heads of 128, 6 heads each: 11.6 -> 11.1).
template <int D, int E>
DEVINL void pd_sum_pieces(PdSum<pd_f32x4> (&s)[E], const float* part_o, const float* part_ml,
                          const PdPair& pair, int G, unsigned quad, int live, int group,
                          int groups) {
  const int first = __builtin_amdgcn_readfirstlane(pair.w_first);
  const int last = __builtin_amdgcn_readfirstlane(pair.w_last) - first;
  const unsigned head = pair.head * G, step = 2 * G;
  const float* const from_o = part_o + (long)first * 2 * G * D;
  const float* const from_ml = part_ml + (long)first * 2 * G * 2;
#pragma unroll
  for (int k = 0; k < E; ++k) s[k] = PdSum<pd_f32x4>{-INFINITY, 0.f, {0.f, 0.f, 0.f, 0.f}};
  // N pieces from r0 on, asked for together
  auto take = [&]<int N>(int r0) {
    pd_f32x2 ml[E][N], x[E][N], y[E][N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = min(r0 + i * groups, last);  // past the end: weight zero below
      unsigned at = r * step;
      if (i == 0) at += r == 0 ? head : 0;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        const unsigned e = k < live ? quad + k * 256 : quad;
        ml[k][i] = pd_published(from_ml + (at + e / (D / 4)) * 2);
        const float* const o = from_o + (at * D + e * 4);
        x[k][i] = pd_published(o);
        y[k][i] = pd_published(o + 2);
      }
    }
#pragma unroll
    for (int k = 0; k < E; ++k) {
      float top = s[k].top;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if (r0 + i * groups > last) ml[k][i][0] = -INFINITY;
        top = fmaxf(top, ml[k][i][0]);
      }
      const float tb = top > -INFINITY ? top : 0.f;
      const float f0 = __builtin_amdgcn_exp2f(s[k].top - tb);
      s[k].weight *= f0;
      s[k].x *= f0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float f = __builtin_amdgcn_exp2f(ml[k][i][0] - tb);
        if (ml[k][i][0] > -INFINITY) {
          s[k].weight += ml[k][i][1] * f;
          s[k].x += __builtin_shufflevector(x[k][i], y[k][i], 0, 1, 2, 3) * f;
        }
      }
      s[k].top = top;
    }
  };
  constexpr int kMost = E == 4 ? 4 : 8;
  for (int r0 = group; r0 <= last; r0 += kMost * groups) {
    if (r0 + 2 * groups > last) take.template operator()<2>(r0);
    else take.template operator()<kMost>(r0);
  }
}

template <int D, typename TC, int NK>
struct PdShape {
  static constexpr int kTileShift = NK == 2 ? 5 : 4;
  static constexpr int kKeys = 16 * NK;
  // LDS of a wave: its V tile, and after its last tile its sums of G heads in the same place
  __host__ __device__ static constexpr int wave_lds(int G) {
    return D * (kKeys * (int)sizeof(short) > G * (int)sizeof(float) ? kKeys * (int)sizeof(short)
                                                                    : G * (int)sizeof(float));
  }
  // the least piece of a pair: 64 KiB of keys and values
  static constexpr int kLeastPiece = 64 * 1024 / (2 * kKeys * D * (int)sizeof(TC));
};

// 16-key groups of a tile and workgroups a CU, by registers; their LDS fits at every G. us, so / else:
// head size 64, four groups and two workgroups: 16 ragged up to 300 keys 6.9 / 7.8, 64 x 1040 26.3 /
// 28.6, 200 ragged up to 100 12.6 / 17.4, 6 ragged up to 15000 31.1 / 30.5; 128, four and one: 189
// ragged up to 1100 86.3 / 104, 60 up to 800 29.4 / 35.0, 3 up to 16000 28.5 / 28.2, two and one: 86.3
// / 91.8, 29.4 / 32.6, 28.5 / 27.8; 256, one and one: 64 up to 300 24.6 / 29.1, 40 up to 500 26.2 /
// 28.8; fp8 of 128, two and two: 189 up to 1100 53.8 / 54.0, 3 up to 16000 22.4 / 20.5, four and two: 53.8
// / 59.1, 22.4 / 20.7; of 256, one and one: 48 up to 2000 48.8 / 66.3, 100 up to 500 35.4 / 37.3.
struct PdVariant { int groups, resident; };
constexpr PdVariant pd_variant(int D, bool fp8) {
  return D == 64 ? PdVariant{2, 3} : D == 128 ? PdVariant{2, fp8 ? 3 : 2} : PdVariant{1, 2};
}

template <int D, typename TC, int NK, int OCC, bool CAP>
__global__ __launch_bounds__(256, OCC) void paged_decode_kernel(
    __hip_bfloat16* __restrict__ out, long out_stride,
    const __hip_bfloat16* __restrict__ q, long q_stride,
    const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ lens,
    int B, int KVH, int G, int bs_shift, int window, float scale_log2, float cap_log2,
    float cap_in, float* __restrict__ part_o, float* __restrict__ part_ml,
    unsigned* __restrict__ arrivals, int resident) {
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
  const int wave_lds = PdShape<D, TC, NK>::wave_lds(NK == 2 ? 16 : G);   // 16: no more than a tile
  short* const Vt = reinterpret_cast<short*>(pd_smem + w * wave_lds);

  const int wgs = gridDim.x, wg = blockIdx.x;
  const PdLens first = pd_lens(lens, B, lane, 0);
  constexpr int kLeast = PdShape<D, TC, NK>::kLeastPiece;
  int share = 1, t, t_end, b, len, nt, kh, i0;
  int w_first = 0, w_last = 0;                 // the workgroups of a pair in pieces
  bool pieces = true;
  // Few sequences whose least pieces all find a workgroup, without pd_deal's other sums and a
  // second scan: 150 of the 450 instructions ahead of the first load, 4 clocks each. Of many nothing
  // is counted here (200 ragged up to 100 keys, 8 kv heads of 64: 12.3 us with it, 11.8 so).
  const float thick = G * (2.f / (KT * (int)sizeof(TC)));
  int n_l = 0, upto = 0, n0 = wgs + 1;
  if (B <= WAVE) {
    n_l = pd_pieces(pd_tiles<TS>(first.of[0], window), kLeast, kLeast, thick);
    upto = pd_scan(n_l);                       // pieces of a head of this lane's sequence and before
    n0 = __builtin_amdgcn_readlane(upto, WAVE - 1) * KVH;
  }
  if (n0 <= wgs) {
    if (wg >= n0) return;
    b = __ffsll((long long)__ballot(upto * KVH > wg)) - 1;
    len = __builtin_amdgcn_readlane(first.of[0], b);
    nt = pd_tiles<TS>(len, window);
    const int of = __builtin_amdgcn_readlane(n_l, b);
    const int r = wg - (__builtin_amdgcn_readlane(upto, b) - of) * KVH;
    const float inv = pd_rcp((float)of);
    kh = __builtin_amdgcn_readfirstlane(pd_quotient(r, inv));
    i0 = r - kh * of;
    w_first = wg - i0;
    w_last = w_first + of - 1;
    const int size = __builtin_amdgcn_readfirstlane(pd_quotient(nt + of - 1, inv));
    t = i0 *= size;
    t_end = min(nt, i0 + size);
  } else {
    const PdDeal deal = pd_deal<TS>(lens, B, KVH, window, lane, first, wgs, resident, kLeast,
                                    thick, D == 256 && !F8);
    share = deal.share;
    pieces = deal.piece > 0;
    t = wg * share;
    t_end = min(deal.total, t + share);
    if (t >= t_end) return;
    int before;
    pd_locate<TS>(lens, B, KVH, window, lane, t, first, deal.piece, kLeast, thick, b, len,
                  before);
    if (b >= B) return;
    nt = pd_tiles<TS>(len, window);
    const int of = pieces ? pd_pieces(nt, deal.piece, kLeast, thick) : nt;
    const int r = t - before * KVH;
    kh = r / of;
    i0 = r % of;
    if (pieces) {                              // from here on the range is in tiles of the pair
      const int size = (nt + of - 1) / of;     // no piece is empty
      w_first = wg - i0;
      w_last = w_first + of - 1;
      i0 *= size;
      t = i0;
      t_end = min(nt, i0 + size);
    }
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

  // A segment: the range's tiles of one pair; this wave's are `count` from key0 on.
  int n, count, key0, pos, lo;
  const int* bt;
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
  pd_s16x8 kf[NK][KL], vf[NV], qf[KS];
  auto fetch_k = [&]() {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const TC* kr = k_cache + rb[i] * D;      // uniform; the lane adds 32 bits
#pragma unroll
      for (int ks = 0; ks < KL; ++ks)
        kf[i][ks] = pd_stream(kr + (klane + ks * (F8 ? 64 : 32)));
    }
  };
  auto fetch_v = [&]() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const TC* vr = v_cache + rb[(i * RPI) >> 4] * D;
      vf[i] = pd_stream(vr + (vlane + ((i * RPI) & 15) * D));
    }
  };
  auto open = [&]() {
    pos = len - 1;
    lo = window > 0 && len > window ? len - window : 0;
    n = min(nt - i0, t_end - t);
    const int at = (n * w) >> 2;
    count = ((n * (w + 1)) >> 2) - at;
    bt = block_tables + (long)b * bt_stride;
    key0 = ((lo >> TS) + i0 + at) << TS;
    if (count == 0) return;
    rows(key0);
    fetch_k();
    fetch_v();
    if (count > 1) rows(key0 + KT);
    const __hip_bfloat16* qr = q + (long)b * q_stride + (long)(kh * G + col) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d8 = F8 ? (ks >> 1) * 64 + grp * 16 + (ks & 1) * 8 : ks * 32 + grp * 8;
      qf[ks] = col < G ? *reinterpret_cast<const pd_s16x8*>(qr + d8)
                       : pd_s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  };
  auto mo = [&](int part) { return reinterpret_cast<float*>(pd_smem + part * wave_lds); };
  __shared__ pd_f32x2 ml[4][16];
  __shared__ PdPair pending[2];                // cut at the ends of the range
  __shared__ unsigned arrived[2];
  // The W channels of a thread, number e of a pair's: two at head size 64, where four leave half the
  // threads idle (1 x 1500 keys, 8 kv heads: 8.4 us, 8.0 so).
  constexpr int W = D == 64 ? 2 : 4;
  typedef float Channels __attribute__((ext_vector_type(W)));
  // What `parts` waves or groups left of them in LDS, read together. The other parts may be another
  // pair's: a weight of zero does not cancel an infinity there, so they are put to zero.
  auto meet = [&](int e, int parts) {
    const int g = e / (D / W);
    PdSum<Channels> s{-INFINITY, 0.f, Channels(0.f)};
    pd_f32x2 of[4];
    Channels x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      of[v] = ml[v][g];
      x[v] = *reinterpret_cast<const Channels*>(mo(v) + e * W);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (v >= parts) of[v] = pd_f32x2{-INFINITY, 0.f}, x[v] = Channels(0.f);
      s.top = fmaxf(s.top, of[v][0]);
    }
    const float tb = s.top > -INFINITY ? s.top : 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float f = __builtin_amdgcn_exp2f(of[v][0] - tb);         // -inf -> 0
      s.weight += of[v][1] * f;
      s.x += x[v] * f;
    }
    return s;
  };
  int waiting = 0;
  open();
  while (true) {
    float m = -INFINITY, l = 0.f;              // log2 domain
    pd_f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = pd_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int i = 0; i < count; ++i, key0 += KT) {
      const bool more = i + 1 < count;
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
      tmax = across_32(across_16(tmax, lanes_max), lanes_max);
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
        if (i + 2 < count) rows(key0 + 2 * KT);
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
    l = across_32(across_16(l, lanes_add), lanes_add);
    if (col < G) {
      float* to = mo(w) + col * D + grp * 4;   // the wave has read its last V tile
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<pd_f32x4*>(to + dt * 16) = o[dt];
      if (grp == 0) ml[w][col] = pd_f32x2{m, l};
    }

    // the next segment's first tiles travel while this one's waves meet
    const int s_b = b, s_kh = kh, s_t = t, s_nt = nt, s_first = t - i0;
    const bool whole = n == nt;
    t += n;
    i0 = 0;
    if (t < t_end) {
      if (++kh == KVH) {
        kh = 0;
        do {
          len = __builtin_amdgcn_readfirstlane(lens[++b]);
          nt = pd_tiles<TS>(len, window);
        } while (nt == 0);
      }
      open();
    }

    pd_barrier();
    __hip_bfloat16* const orow = out + (long)s_b * out_stride + (long)s_kh * G * D;
    // a range holds at most two pieces: one from its start, one to its end
    const long slot = ((long)wg * 2 + (pieces || s_t == t_begin ? 0 : 1)) * G;
    for (int e = threadIdx.x; e < G * (D / W); e += 256) {
      const PdSum<Channels> s = meet(e, 4);
      if (whole) {
        pd_finish(orow + e * W, s);
        continue;
      }
#pragma unroll
      for (int c = 0; c < W; c += 2)
        pd_publish(part_o + slot * D + e * W + c, pd_f32x2{s.x[c], s.x[c + 1]});
      if (e % (D / W) == 0)
        pd_publish(part_ml + (slot + e / (D / W)) * 2, pd_f32x2{s.top, s.weight});
    }
    if (!whole) {
      if (threadIdx.x == 0) {
        const int w0 = pieces ? w_first : s_first / share;
        pending[waiting] = PdPair{s_b, s_kh, w0, pieces ? w_last : (s_first + s_nt - 1) / share,
                                  !pieces && s_first % share ? 1 : 0};
      }
      ++waiting;
    }
    if (t >= t_end) break;
    pd_barrier();                              // `mo` and `ml` are read
  }
  if (waiting == 0) return;
  // The last workgroup to arrive with a piece of a pair merges all, in their order. Arrivals
  // wait for the end of the range, so that its loads do not.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // published
  pd_barrier();
  if ((int)threadIdx.x < waiting)
    arrived[threadIdx.x] = __hip_atomic_fetch_add(
        arrivals + pending[threadIdx.x].b * KVH + pending[threadIdx.x].kh, 1u, __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT);
  pd_barrier();
  for (int p = 0; p < waiting; ++p) {
    const PdPair pair = pending[p];
    if ((int)arrived[p] != pair.w_last - pair.w_first) continue;
    __hip_bfloat16* const orow = out + (long)pair.b * out_stride + (long)pair.kh * G * D;
    const int tid = threadIdx.x, quads = G * (D / 4);
    const int groups = 1 + (2 * quads <= 256) + (3 * quads <= 256) + (4 * quads <= 256);
    const int group =
        groups == 1 ? 0 : (tid >= quads) + (tid >= 2 * quads) + (tid >= 3 * quads);
    const int e0 = tid - group * quads;
    const int live = group < groups ? (quads - e0 + 255) / 256 : 0;      // none below zero
    auto merge = [&]<int E>() {
      PdSum<pd_f32x4> s[E];
      pd_sum_pieces<D, E>(s, part_o, part_ml, pair, G, e0, live, group, groups);
#pragma unroll
      for (int k = 0; k < E; ++k) {
        const int e = e0 + k * 256;
        if (k >= live) break;
        if (groups == 1) {
          pd_finish(orow + e * 4, s[k]);
        } else {
          *reinterpret_cast<pd_f32x4*>(mo(group) + e * 4) = s[k].x;
          if (e % (D / 4) == 0) ml[group][e / (D / 4)] = pd_f32x2{s[k].top, s[k].weight};
        }
      }
    };
    // up to D / 64 quads a thread, asked for together (1 x 200 keys, 2 kv heads of 256, 16 heads
    // each: one after the other 15.8 us, so 12.4)
    if (live > 0) {
      if (D == 64 || quads <= 256) merge.template operator()<1>();
      else if (D == 128 || quads <= 512) merge.template operator()<D == 64 ? 1 : 2>();
      else merge.template operator()<D == 256 ? 4 : 1>();
    }
    if (groups > 1) {
      pd_barrier();
      for (int e = tid; e < G * (D / W); e += 256) pd_finish(orow + e * W, meet(e, groups));
    }
    // Zero again for the next launch: nobody else comes to this counter in this one. Behind the
    // merge, whose loads would wait for it too (1 x 1000 keys, 8 kv heads of 64: 8.26 us ahead of
    // them and with an atomic's way to memory, 8.14 so).
    if (tid == 0) arrivals[pair.b * KVH + pair.kh] = 0u;
    if (p + 1 < waiting) pd_barrier();
  }
}
