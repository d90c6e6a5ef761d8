// Gate and value rows of many tokens with their activation, out[M, N / 2] = f(x Wg^T) (x
// Wv^T), W[N, K] = [gates | values], fp32 sums: more than 256 rows of a prompt step or a
// decode batch (gfx950).
//
// Bound by the matrix cores at the clock that they leave, 1.1 to 1.4 PFLOP/s; the
// activation costs no pass over the product and its rounding to bf16 is gone. With few
// tokens the weights come from memory too late for two stages: the rule at the launch says
// where. Measured (us, weights in the caches; before = the library's product and
// act_and_mul_kernel): 512 rows, 17920 x 1536 40.6 -> 32.4;
// 1000, 16384 x 3072 84 -> 74; 1000, 28672 x 3584 179 -> 165; 3953, 17920 x 1536 207 -> 176;
// 8192, 16384 x 2048 454 -> 384, 16384 x 3072 630 -> 577 (1.43 PFLOP/s), 28672 x 3584 1224 ->
// 1208. (Plain products on these tiles lose to the library by 3 to 10 % where they fill
// the chip and by more where they do not: 8192 rows, 8192 x 3584 336 against 309.)
//
//   - A workgroup owns a tile of 256 weight rows by 64 TW tokens, eight waves of 128 x
//     16 TW, and takes tiles in turn until none are left; stages of 64 channels follow each
//     other across tiles, so the next tile's operands travel during a tile's last products.
//   - Weights and tokens go to LDS by global_load_lds, two stages. The products of a
//     stage's first 32 channels run while its second 32 are read from LDS into other
//     registers, those of the second while the next stage's first are read: no product
//     waits for LDS, and a stage has one barrier, which frees the buffer just read for
//     the stage after the next.
//   - v_mfma_f32_16x16x32_bf16, A = weights, B = tokens, C: column = token, rows = 4 weight
//     rows. Weight rows are dealt to A's rows so that a lane ends up with 16 neighbouring
//     outputs of a token and their gates: 32 bytes, 128 over the token's four lanes.
//   - Tiles that run together on an XCD are four weight tiles wide and go through K in step,
//     for its L2. XCDs start at different stages: rows of 7168 bytes lie on few memory
//     channels (8192 rows, 28672 x 3584 1252 -> 1208; a start of its own per workgroup 1440).

#include "common.h"   // and ring_load of stream_gemm.hip, epilogues of slab_gemm.hip

typedef __attribute__((ext_vector_type(8))) short tg_s16x8;
typedef __attribute__((ext_vector_type(4))) float tg_f32x4;

constexpr int kTileRows = 256, kTileBK = 64;

template <int TW>
constexpr size_t tile_lds() { return sizeof(short) * 2 * (kTileRows + 64 * TW) * kTileBK; }

// SiLU or tanh-form GELU of g: both g / (1 + 2^-t).
template <int EPI>
DEVINL float tile_act(float g) {
  constexpr float kLog2e = 1.4426950408889634f;
  const float t = EPI == kSlabSilu
      ? g * kLog2e
      : g * fmaf(g * g, 2.f * 0.7978845608028654f * 0.044715f * kLog2e,
                 2.f * 0.7978845608028654f * kLog2e);
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-t));
}

// EPI: kSlabSilu or kSlabGelu; wtiles x ttiles tiles, no fewer than workgroups.
template <int TW, int EPI>
__global__ __launch_bounds__(512) void tile_gemm_kernel(
    __hip_bfloat16* __restrict__ out, long out_stride, const __hip_bfloat16* __restrict__ x,
    long x_stride, const __hip_bfloat16* __restrict__ wt, int M, int N, int K, int wtiles,
    int ttiles) {
  constexpr int R = kTileRows, T = 64 * TW, BK = kTileBK, STAGE = (R + T) * BK;
  constexpr int NW = 4, NT = TW, NL = NW + NT;             // a wave's loads of a stage
  constexpr int RO = R / 2;                                // output columns of a tile
  extern __shared__ __align__(16) short tile_smem[];       // [2][R weight | T token rows][BK]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = w & 1, wc = w >> 1;
  const int col = lane & 15, grp = lane >> 4;
  const int grid = gridDim.x, id = blockIdx.x;
  const int first = grid % 8 == 0 ? id % 8 * (grid / 8) + id / 8 : id;
  const int mine = (wtiles * ttiles - 1 - first) / grid + 1, steps = K / BK;
  const int total = mine * steps;

  auto place = [&](int row) { return ((lane & 7) ^ ((row >> 1) & 7)) << 3; };
  unsigned woff[NW], xoff[NT];
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    const int lr = (w + j * 8) * 8 + (lane >> 3);          // LDS row: wave column, tile, row
    const int a = lr / 16 % 8, c = lr % 16;
    const int row = lr / 128 * 64 + c / 4 * 16 + a % 4 * 4 + c % 4 + (a < 4 ? 0 : N / 2);
    woff[j] = ((unsigned)row * (unsigned)K + place(lr)) * 2u;
  }
  auto locate = [&](int i, int& n0, int& m0) {
    const int t = first + i * grid;
    const int g = t / (4 * ttiles), in = t - g * (4 * ttiles);
    const int width = min(4, wtiles - g * 4), tt = in / width;
    n0 = (g * 4 + in - tt * width) * RO;
    m0 = tt * T;
  };
  // the loads' place in the sequence of stages; an XCD's tiles start at `rot`
  const int rot = id % 8 * steps / 8;
  int l_tile = 0, l_step = 0, l_at = rot;
  const __hip_bfloat16 *wb, *xb;
  auto aim = [&]() {
    int n0, m0;
    locate(l_tile, n0, m0);
    wb = wt + (long)n0 * K + rot * BK;
    xb = x + (long)m0 * x_stride + rot * BK;
#pragma unroll
    for (int j = 0; j < NT; ++j) {                         // past the last token: repeat it
      const int lr = (w + j * 8) * 8 + (lane >> 3);
      xoff[j] = ((unsigned)min(lr, M - 1 - m0) * (unsigned)x_stride + place(lr)) * 2u;
    }
  };
  aim();
  const unsigned ring_off = (unsigned)(unsigned long)(
      (__attribute__((address_space(3))) char*)tile_smem) + w * 1024;
  auto stage = [&](int buf) {
    const unsigned to = __builtin_amdgcn_readfirstlane(ring_off + (unsigned)buf * (STAGE * 2));
#pragma unroll
    for (int j = 0; j < NW; ++j) ring_load<false>(wb, woff[j], to + j * 8192);
#pragma unroll
    for (int j = 0; j < NT; ++j) ring_load<false>(xb, xoff[j], to + R * BK * 2 + j * 8192);
    wb += BK;
    xb += BK;
    if (++l_at == steps) {
      l_at = 0;
      wb -= K;
      xb -= K;
    }
    if (++l_step == steps) {
      l_step = 0;                                          // and l_at = rot
      if (++l_tile < mine) aim();
    }
  };

  tg_f32x4 acc[8][TW];
  auto clear = [&]() {
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int m = 0; m < TW; ++m) acc[a][m] = tg_f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  // operands of 32 channels, half u of a stage
  struct Half { tg_s16x8 w[8], x[TW]; };
  const int at0 = (grp ^ ((col >> 1) & 7)) << 3;
  const int wat = (wn * 128 + col) * BK + at0, xat = (R + wc * 16 * TW + col) * BK + at0;
  auto read_w = [&](const short* s, int u, int a) {
    return *reinterpret_cast<const tg_s16x8*>(s + ((wat ^ (u * 32)) + a * 16 * BK));
  };
  auto read_x = [&](const short* s, int u, int m) {
    return *reinterpret_cast<const tg_s16x8*>(s + ((xat ^ (u * 32)) + m * 16 * BK));
  };
  // the products of `now` while `then` is read
  auto multiply = [&](const Half& now, Half& then, const short* s, int u) {
#pragma unroll
    for (int m = 0; m < TW; ++m) then.x[m] = read_x(s, u, m);
#pragma unroll
    for (int a = 0; a < 8; ++a) then.w[a] = read_w(s, u, a);
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int m = 0; m < TW; ++m)
        acc[a][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now.w[a], now.x[m], acc[a][m], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 8 + TW; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // two products
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8 * TW, 0);
  };

  stage(0);
  if (total > 1) {
    stage(1);
    pipe_barrier_vm<NL>();
  } else {
    pipe_barrier_vm<0>();
  }
  Half h0, h1;
#pragma unroll
  for (int m = 0; m < TW; ++m) h0.x[m] = read_x(tile_smem, 0, m);
#pragma unroll
  for (int a = 0; a < 8; ++a) h0.w[a] = read_w(tile_smem, 0, a);
  int tile = 0, step = 0;
  for (int it = 0; it < total; ++it) {
    const short* cur = tile_smem + (it & 1) * STAGE;
    const short* nxt = tile_smem + (~it & 1) * STAGE;
    multiply(h0, h1, cur, 1);
    // the next stage is here; this one is in registers, its buffer free
    pipe_barrier_vm<0>();
    if (it + 2 < total) stage(it & 1);
    multiply(h1, h0, nxt, 0);                              // past the last stage: unused
    if (++step < steps) continue;
    step = 0;
    int n0, m0;
    locate(tile++, n0, m0);
#pragma unroll
    for (int m = 0; m < TW; ++m) {
      const int row = m0 + (wc * TW + m) * 16 + col;
      if (row >= M) continue;
      __hip_bfloat16* o = out + (long)row * out_stride + n0 + wn * 64 + grp * 16;
#pragma unroll
      for (int a = 0; a < 4; a += 2) {
        Vec8<__hip_bfloat16> v;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v.data[e] = __float2bfloat16(tile_act<EPI>(acc[a + e / 4][m][e % 4]) *
                                       acc[a + 4 + e / 4][m][e % 4]);
        store16(o + a * 4, v);
      }
    }
    clear();
  }
}
