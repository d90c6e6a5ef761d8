// Torch bindings for the llmq-amd CDNA4 kernels.
// Registered under torch.ops.llmq_amd.* ; loaded via torch.ops.load_library.

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/library.h>

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

// Kernel definitions are included BEFORE this file in the umbrella TU
// (ops.hip) — no forward declarations needed (stale declarations with
// narrower template parameter lists silently generate dead launch stubs).

namespace {

#define CHECK_GPU(x) TORCH_CHECK(x.is_cuda(), #x " must be on GPU")
#define CHECK_LASTDIM(x) \
  TORCH_CHECK(x.stride(-1) == 1, #x " innermost dim must be contiguous")

hipStream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

template <typename F>
void dispatch_dtype(const at::Tensor& t, const char* name, F&& f) {
  switch (t.scalar_type()) {
    case at::kBFloat16:
      f.template operator()<__hip_bfloat16>();
      break;
    case at::kHalf:
      f.template operator()<_Float16>();
      break;
    case at::kFloat:
      f.template operator()<float>();
      break;
    default:
      TORCH_CHECK(false, name, ": unsupported dtype ", t.scalar_type());
  }
}

// ---------------------------------------------------------------- norms --

void rmsnorm(at::Tensor out, at::Tensor in, at::Tensor weight, double eps,
             double offset) {
  CHECK_GPU(in);
  CHECK_LASTDIM(in);
  const int hidden = in.size(-1);
  const long rows = in.numel() / hidden;
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  dispatch_dtype(in, "rmsnorm", [&]<typename T>() {
    hipLaunchKernelGGL(rmsnorm_kernel<T>, dim3(rows), dim3(256), 0, stream(),
                       reinterpret_cast<T*>(out.data_ptr()),
                       reinterpret_cast<const T*>(in.data_ptr()),
                       reinterpret_cast<const T*>(weight.data_ptr()), hidden,
                       (float)eps, (float)offset);
  });
}

void fused_add_rmsnorm(at::Tensor x, at::Tensor residual, at::Tensor weight,
                       double eps, double offset) {
  CHECK_GPU(x);
  CHECK_LASTDIM(x);
  const int hidden = x.size(-1);
  const long rows = x.numel() / hidden;
  dispatch_dtype(x, "fused_add_rmsnorm", [&]<typename T>() {
    hipLaunchKernelGGL(fused_add_rmsnorm_kernel<T>, dim3(rows), dim3(256), 0,
                       stream(), reinterpret_cast<T*>(x.data_ptr()),
                       reinterpret_cast<T*>(residual.data_ptr()),
                       reinterpret_cast<const T*>(weight.data_ptr()), hidden,
                       (float)eps, (float)offset);
  });
}

// ----------------------------------------------------------- activations --

template <bool GELU>
void act_and_mul(at::Tensor out, at::Tensor in) {
  CHECK_GPU(in);
  CHECK_LASTDIM(in);
  const int d = out.size(-1);
  const long rows = out.numel() / d;
  TORCH_CHECK(in.size(-1) == 2 * d, "in must be [..., 2*d]");
  const long chunks = rows * (d / 8);
  const int grid = std::min<long>((chunks + 255) / 256, 2048);
  dispatch_dtype(in, "act_and_mul", [&]<typename T>() {
    hipLaunchKernelGGL((act_and_mul_kernel<T, GELU>), dim3(grid), dim3(256), 0,
                       stream(), reinterpret_cast<T*>(out.data_ptr()),
                       reinterpret_cast<const T*>(in.data_ptr()), rows, d);
  });
}

void silu_and_mul(at::Tensor out, at::Tensor in) { act_and_mul<false>(out, in); }
void gelu_tanh_and_mul(at::Tensor out, at::Tensor in) { act_and_mul<true>(out, in); }

// ----------------------------------------------------------------- rope --

void rope_inplace(at::Tensor q, at::Tensor k, at::Tensor positions,
                  at::Tensor cos_sin) {
  CHECK_GPU(q);
  CHECK_LASTDIM(q);
  CHECK_LASTDIM(k);
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3, "q/k must be [T, H, D]");
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat, "cos_sin must be f32");
  const int T_ = q.size(0);
  if (T_ == 0) return;
  const int hq = q.size(1), hk = k.size(1), d = q.size(2);
  TORCH_CHECK(q.stride(1) == d && k.stride(1) == d, "head dim must be packed");
  dispatch_dtype(q, "rope", [&]<typename T>() {
    hipLaunchKernelGGL(rope_kernel<T>, dim3(T_), dim3(256), 0, stream(),
                       reinterpret_cast<T*>(q.data_ptr()),
                       reinterpret_cast<T*>(k.data_ptr()),
                       positions.data_ptr<long>(), cos_sin.data_ptr<float>(),
                       hq, hk, d, q.stride(0), k.stride(0));
  });
}

void norm_add_norm(at::Tensor x, at::Tensor residual, at::Tensor w_post,
                   at::Tensor w_pre, double eps, double offset) {
  CHECK_GPU(x);
  CHECK_LASTDIM(x);
  const int hidden = x.size(-1);
  const long rows = x.numel() / hidden;
  dispatch_dtype(x, "norm_add_norm", [&]<typename T>() {
    hipLaunchKernelGGL(norm_add_norm_kernel<T>, dim3(rows), dim3(256), 0,
                       stream(), reinterpret_cast<T*>(x.data_ptr()),
                       reinterpret_cast<T*>(residual.data_ptr()),
                       reinterpret_cast<const T*>(w_post.data_ptr()),
                       reinterpret_cast<const T*>(w_pre.data_ptr()), hidden,
                       (float)eps, (float)offset);
  });
}

// ------------------------------------------------------------- KV cache --

void reshape_and_cache(at::Tensor key, at::Tensor value, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor slot_mapping) {
  CHECK_GPU(key);
  CHECK_LASTDIM(key);
  const int T_ = key.size(0);
  if (T_ == 0) return;
  const int kvh = key.size(1), d = key.size(2);
  const int bs = k_cache.size(2);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  const bool fp8_cache = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  dispatch_dtype(key, "reshape_and_cache", [&]<typename T>() {
    if (fp8_cache) {
      if constexpr (std::is_same_v<T, __hip_bfloat16>) {
        hipLaunchKernelGGL((reshape_and_cache_kernel<T, __hip_fp8_e4m3>),
                           dim3(T_), dim3(128), 0, stream(),
                           reinterpret_cast<const T*>(key.data_ptr()),
                           reinterpret_cast<const T*>(value.data_ptr()),
                           reinterpret_cast<__hip_fp8_e4m3*>(k_cache.data_ptr()),
                           reinterpret_cast<__hip_fp8_e4m3*>(v_cache.data_ptr()),
                           slot_mapping.data_ptr<long>(), kvh, d, bs,
                           key.stride(0), value.stride(0));
      } else {
        TORCH_CHECK(false, "fp8 KV cache requires bf16 activations");
      }
      return;
    }
    hipLaunchKernelGGL(reshape_and_cache_kernel<T>, dim3(T_), dim3(128), 0,
                       stream(), reinterpret_cast<const T*>(key.data_ptr()),
                       reinterpret_cast<const T*>(value.data_ptr()),
                       reinterpret_cast<T*>(k_cache.data_ptr()),
                       reinterpret_cast<T*>(v_cache.data_ptr()),
                       slot_mapping.data_ptr<long>(), kvh, d, bs,
                       key.stride(0), value.stride(0));
  });
}

void rope_and_cache(at::Tensor q, at::Tensor k, at::Tensor value,
                    at::Tensor k_cache, at::Tensor v_cache,
                    at::Tensor positions, at::Tensor cos_sin,
                    at::Tensor slot_mapping) {
  CHECK_GPU(q);
  CHECK_LASTDIM(q);
  CHECK_LASTDIM(k);
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3, "q/k must be [T, H, D]");
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  const int T_ = q.size(0);
  if (T_ == 0) return;
  const int hq = q.size(1), hk = k.size(1), d = q.size(2);
  const int bs = k_cache.size(2);
  TORCH_CHECK(q.stride(1) == d && k.stride(1) == d, "head dim must be packed");
  const bool fp8_cache = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  // 8-byte pieces of every row, 16-byte ones of the angles
  auto pieces = [&](const at::Tensor& t, long bytes) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0 &&
           t.stride(0) * (long)t.element_size() % bytes == 0;
  };
  dispatch_dtype(q, "rope_and_cache", [&]<typename T>() {
    constexpr int NP = 8 / sizeof(T);
    const bool wide = d % (2 * NP) == 0 && pieces(q, 8) && pieces(k, 8) && pieces(value, 8) &&
                      pieces(cos_sin, 4 * NP) && (d / 2 * 4) % (4 * NP) == 0 &&
                      reinterpret_cast<uintptr_t>(k_cache.data_ptr()) % 8 == 0 &&
                      reinterpret_cast<uintptr_t>(v_cache.data_ptr()) % 8 == 0;
    auto go = [&]<typename TC, int N>() {
      // few tokens: the heads over four workgroups
      hipLaunchKernelGGL((rope_and_cache_kernel<T, TC, N>), dim3(T_, T_ < 1024 ? 4 : 1), dim3(256),
                         0, stream(), reinterpret_cast<T*>(q.data_ptr()),
                         reinterpret_cast<T*>(k.data_ptr()),
                         reinterpret_cast<const T*>(value.data_ptr()),
                         reinterpret_cast<TC*>(k_cache.data_ptr()),
                         reinterpret_cast<TC*>(v_cache.data_ptr()), positions.data_ptr<long>(),
                         cos_sin.data_ptr<float>(), slot_mapping.data_ptr<long>(), hq, hk, d, bs,
                         q.stride(0), k.stride(0), value.stride(0));
    };
    auto pick = [&]<typename TC>() {
      if (wide) go.template operator()<TC, NP>();
      else go.template operator()<TC, 1>();
    };
    if (fp8_cache) {
      if constexpr (std::is_same_v<T, __hip_bfloat16>) pick.template operator()<__hip_fp8_e4m3>();
      else TORCH_CHECK(false, "fp8 KV cache requires bf16 activations");
      return;
    }
    pick.template operator()<T>();
  });
}

// ------------------------------------------------------------ attention --

// 16-byte loads and 8-byte stores: rows that start elsewhere go through a copy.
bool rows_start_on(const at::Tensor& t, long bytes) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0 &&
         t.stride(0) * (long)t.element_size() % bytes == 0;
}
at::Tensor rows_on_16(const at::Tensor& t) {
  return rows_start_on(t, 16) ? t : t.clone(at::MemoryFormat::Contiguous);
}

int compute_units(const at::Tensor& x) {
  int cus = 0;
  TORCH_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                                    x.get_device()) == hipSuccess);
  return cus;
}

// The matrix-core kernel of paged_decode.hip. arrivals: zeros [B, KVH], zeros again after the
// launch; without it they are made here, a launch of 2 us.
template <int D, typename TC>
void launch_paged_decode(at::Tensor& out, const at::Tensor& q, const at::Tensor& kc,
                         const at::Tensor& vc, const at::Tensor& bt,
                         const at::Tensor& cl, double scale, double softcap,
                         long window, const c10::optional<at::Tensor>& arrivals) {
  constexpr PdVariant kVariant = pd_variant(D, sizeof(TC) == 1);
  constexpr int NK = kVariant.groups, OCC = kVariant.resident;
  using Shape = PdShape<D, TC, NK>;
  static_assert(OCC * (4 * Shape::wave_lds(16) + 1024) <= 160 * 1024, "resident at every G");
  constexpr double kLog2e = 1.4426950408889634;
  const int B = q.size(0), KVH = kc.size(1), G = q.size(1) / KVH;
  const int bs_shift = kc.size(2) == 32 ? 5 : 4;
  const long tiles = (bt.size(1) << bs_shift) / Shape::kKeys + 1;   // of a pair, at most
  const long resident = (long)compute_units(q) * OCC;
  const int wgs = (int)pd_workgroups((long)B * KVH, tiles, Shape::kLeastPiece, resident);
  auto opts = q.options().dtype(at::kFloat);
  at::Tensor part_o = at::empty({2L * wgs, G, D}, opts);
  at::Tensor part_ml = at::empty({2L * wgs, G, 2}, opts);
  const bool given = arrivals.has_value() && arrivals->defined();
  TORCH_CHECK(!given || (arrivals->scalar_type() == at::kInt && arrivals->is_contiguous() &&
                         arrivals->numel() == (long)B * KVH && arrivals->device() == q.device()),
              "arrivals must be int32 zeros [B, kv heads] on q's device");
  const at::Tensor arr = given ? *arrivals : at::zeros({B, KVH}, q.options().dtype(at::kInt));
  auto go = [&]<bool CAP>() {
    hipLaunchKernelGGL((paged_decode_kernel<D, TC, NK, OCC, CAP>), dim3(wgs), dim3(256),
                       4 * Shape::wave_lds(G), stream(),
                       reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), out.stride(0),
                       reinterpret_cast<const __hip_bfloat16*>(q.data_ptr()), q.stride(0),
                       reinterpret_cast<const TC*>(kc.data_ptr()),
                       reinterpret_cast<const TC*>(vc.data_ptr()), bt.data_ptr<int>(),
                       (int)bt.stride(0), cl.data_ptr<int>(), B, KVH, G, bs_shift, (int)window,
                       (float)(scale * kLog2e), (float)(softcap * kLog2e),
                       softcap > 0 ? (float)(2 / softcap) : 0.f,
                       part_o.data_ptr<float>(), part_ml.data_ptr<float>(),
                       reinterpret_cast<unsigned*>(arr.data_ptr<int>()),
                       (int)std::min<long>(resident, wgs));
  };
  if (softcap > 0) go.template operator()<true>();
  else go.template operator()<false>();
}

template <typename T>
void launch_decode(at::Tensor& out, const at::Tensor& q, const at::Tensor& kc,
                   const at::Tensor& vc, const at::Tensor& bt,
                   const at::Tensor& cl, double scale, double softcap,
                   long window, const c10::optional<at::Tensor>& arrivals) {
  const int B = q.size(0), H = q.size(1), D = q.size(2);
  const int KVH = kc.size(1);
  const int bs = kc.size(2);
  const int G = H / KVH;
  TORCH_CHECK(H % KVH == 0, "num_heads must divide num_kv_heads");
  TORCH_CHECK(bs == 16 || bs == 32, "block_size must be 16 or 32");
  if (B == 0) return;
  const bool fp8 = kc.scalar_type() == at::kFloat8_e4m3fn;
  TORCH_CHECK(!fp8 || (std::is_same_v<T, __hip_bfloat16> && (D == 128 || D == 256) && G <= 16),
              "fp8 KV cache requires the MFMA decode path (bf16 q, head_dim "
              "128/256, GQA group <= 16); got head_dim=", D, " group=", G);
  TORCH_CHECK(D == 64 || D == 128 || D == 256, "unsupported head_dim ", D);
  if constexpr (std::is_same_v<T, __hip_bfloat16>) {
    TORCH_CHECK(G <= (D == 64 ? 8 : 16), "GQA group must be <= 8 at head_dim 64, else <= 16");
    const at::Tensor qa = rows_on_16(q);
    const at::Tensor bta = bt.stride(1) == 1 ? bt : bt.contiguous();
    at::Tensor oa = rows_start_on(out, 8) ? out : out.clone(at::MemoryFormat::Contiguous);
    auto go = [&]<int HD, typename TC>() {
      launch_paged_decode<HD, TC>(oa, qa, kc, vc, bta, cl, scale, softcap, window, arrivals);
    };
    using BF = __hip_bfloat16;
    using F8 = __hip_fp8_e4m3;
    if (D == 64) go.template operator()<64, BF>();
    else if (D == 128 && !fp8) go.template operator()<128, BF>();
    else if (D == 256 && !fp8) go.template operator()<256, BF>();
    else if (D == 128) go.template operator()<128, F8>();
    else go.template operator()<256, F8>();
    if (!oa.is_same(out)) out.copy_(oa);
    return;
  } else {
  const int max_blocks = bt.size(1);
  dim3 grid(B, KVH);
  TORCH_CHECK(G <= 8, "GQA group must be <= 8 for the VALU decode kernel");
  const int subs = 256 / (32 * G);
  const int lds = (G * D + DECODE_CHUNK * G + subs * G * (D + 2)) * sizeof(float) +
                  16 * sizeof(int);
  auto l = [&]<int HD>() {
    hipLaunchKernelGGL((paged_decode_attention_kernel<T, HD>), grid, dim3(256),
                       lds, stream(), reinterpret_cast<T*>(out.data_ptr()),
                       reinterpret_cast<const T*>(q.data_ptr()),
                       reinterpret_cast<const T*>(kc.data_ptr()),
                       reinterpret_cast<const T*>(vc.data_ptr()),
                       bt.data_ptr<int>(), cl.data_ptr<int>(), H, KVH, bs,
                       max_blocks, (float)scale, (float)softcap, (int)window,
                       q.stride(0), out.stride(0));
  };
  switch (D) {
    case 64: l.template operator()<64>(); break;
    case 128: l.template operator()<128>(); break;
    case 256: l.template operator()<256>(); break;
  }
  }
}

void paged_decode_attention(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                            at::Tensor v_cache, at::Tensor block_tables,
                            at::Tensor context_lens, double scale,
                            double softcap, long window, c10::optional<at::Tensor> arrivals) {
  CHECK_GPU(q);
  CHECK_LASTDIM(q);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt);
  TORCH_CHECK(context_lens.scalar_type() == at::kInt);
  dispatch_dtype(q, "paged_decode_attention", [&]<typename T>() {
    launch_decode<T>(out, q, k_cache, v_cache, block_tables, context_lens,
                     scale, softcap, window, arrivals);
  });
}

// The matrix-core kernel of flash_prefill.hip on packed rows, or with a block table
// on cache blocks [blocks, kv heads, block, D].
struct PrefillArgs {
  const at::Tensor &q, &k, &v, &cu, &cu_k;
  const at::Tensor* block_tables;            // null: packed rows
  int B, KVH;
  double scale, softcap;
  long window, max_seqlen;
};

template <int D, int HP, int WR, int KT, int MINW>
void launch_flash_prefill(at::Tensor& out, const PrefillArgs& a) {
  constexpr double kLog2e = 1.4426950408889634;
  const int H = a.q.size(1);
  // Tiles on an axis of their own: one axis holds 2^32 threads, which 2048 sequences of
  // up to 40000 tokens, 32 heads, would pass.
  const int n_qt = (int)((std::max<long>(a.max_seqlen, 1) + 32 * WR - 1) / (32 * WR));
  auto go = [&]<bool CAP, bool PAGED>() {
    hipLaunchKernelGGL((flash_prefill_kernel<D, HP, WR, KT, MINW, CAP, PAGED>),
                       dim3(H / HP * a.B, n_qt), dim3(64 * HP * WR), 0, stream(),
                       reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), out.stride(0),
                       reinterpret_cast<const __hip_bfloat16*>(a.q.data_ptr()), a.q.stride(0),
                       reinterpret_cast<const __hip_bfloat16*>(a.k.data_ptr()), a.k.stride(0),
                       reinterpret_cast<const __hip_bfloat16*>(a.v.data_ptr()), a.v.stride(0),
                       a.cu.data_ptr<int>(), a.cu_k.data_ptr<int>(),
                       PAGED ? a.block_tables->data_ptr<int>() : nullptr,
                       PAGED ? (int)a.block_tables->stride(0) : 0,
                       PAGED && a.k.size(2) == 32 ? 5 : 4, H, a.KVH, (int)a.window,
                       (float)(a.scale * kLog2e), (float)(a.softcap * kLog2e),
                       a.softcap > 0 ? (float)(2 / a.softcap) : 0.f);
  };
  if (a.block_tables) {
    if (a.softcap > 0) go.template operator()<true, true>();
    else go.template operator()<false, true>();
  } else {
    if (a.softcap > 0) go.template operator()<true, false>();
    else go.template operator()<false, false>();
  }
}

// flash_prefill.hip counts bytes from a tile's first key, up to 63 rows of k or v on, in 32
// bits: packed copies of rows farther apart (2^25 elements, 64 MiB).
at::Tensor rows_in_reach(const at::Tensor& t) {
  const at::Tensor r = rows_on_16(t);
  return r.size(0) <= 1 || r.stride(0) < (1L << 25) ? r : r.clone(at::MemoryFormat::Contiguous);
}

void launch_flash_prefill_any(at::Tensor& out, const PrefillArgs& args) {
  const int H = args.q.size(1), D = args.q.size(2);
  at::Tensor qa = rows_on_16(args.q);
  const bool paged = args.block_tables != nullptr;       // contiguous caches, 64-bit addresses
  const at::Tensor ka = paged ? args.k : rows_in_reach(args.k);
  const at::Tensor va = paged ? args.v : rows_in_reach(args.v);
  at::Tensor oa = rows_start_on(out, 8) ? out : out.clone(at::MemoryFormat::Contiguous);
  // The kernel masks scores with -inf before it scales them: a negative scale goes into
  // the queries, and zero (every visible key alike) too.
  double scale = args.scale;
  if ((float)scale == 0.f) {
    qa = at::zeros_like(qa, qa.options(), at::MemoryFormat::Contiguous);
    scale = 1;
  } else if (scale < 0) {
    qa = qa.neg().contiguous();
    scale = -scale;
  }
  const PrefillArgs a{qa, ka, va, args.cu, args.cu_k, args.block_tables, args.B, args.KVH,
                      scale, args.softcap, args.window, args.max_seqlen};
  // Two heads of a kv head on one stream of tiles where the group is even
  // (2 x 64 rows at head size 64, 2 x 128 at 256: 138 against 147 us for
  // 8 x 1024 tokens). Tiles of 32 keys where that buys a third wave per SIMD
  // (head size 128: 160 against 187 us for 16 x 1024) or the registers (256).
  const bool even = (H / args.KVH) % 2 == 0;
  // Head size 256: four waves a workgroup instead of eight where the wide ones would not
  // fill the CUs (a wave then has its SIMD to itself) or where a prompt fits in one narrow
  // tile. Measured, us, 16 heads of 8 kv heads, wide / narrow: 1 x 100 21.0 / 15.6, 1 x 500
  // 50.0 / 41.8, 8 x 300 (192 wide workgroups) 37.8 / 33.0, 16 x 200 (256) 35.3 / 41.0,
  // 1 x 5000 (320) 363 / 470, 300 x 33 111 / 99, 64 x 65 (512) 42.7 / 51.1.
  const int wide_rows = even ? 128 : 256;
  const long wide = (args.max_seqlen + wide_rows - 1) / wide_rows * (H / (even ? 2 : 1)) * args.B;
  int cus = 0;
  TORCH_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                                    args.q.get_device()) == hipSuccess);
  const bool narrow = args.max_seqlen <= wide_rows / 2 || wide < cus;
  if (D == 64 && even) launch_flash_prefill<64, 2, 2, 64, 3>(oa, a);
  else if (D == 64) launch_flash_prefill<64, 1, 4, 64, 3>(oa, a);
  else if (D == 128) launch_flash_prefill<128, 1, 4, 32, 3>(oa, a);
  else if (narrow && even) launch_flash_prefill<256, 2, 2, 32, 1>(oa, a);
  else if (narrow) launch_flash_prefill<256, 1, 4, 32, 1>(oa, a);
  else if (even) launch_flash_prefill<256, 2, 4, 32, 1>(oa, a);
  else launch_flash_prefill<256, 1, 8, 32, 1>(oa, a);
  if (!oa.is_same(out)) out.copy_(oa);
}

template <typename T>
void launch_prefill(at::Tensor& out, const at::Tensor& q, const at::Tensor& k,
                    const at::Tensor& v, const at::Tensor& cu,
                    const at::Tensor& cu_k, int B,
                    double scale, double softcap, long window, long max_seqlen) {
  const int H = q.size(1), D = q.size(2);
  const int KVH = k.size(1);
  if (B == 0) return;
  TORCH_CHECK(D == 64 || D == 128 || D == 256, "unsupported head_dim ", D);
  if constexpr (std::is_same_v<T, __hip_bfloat16>) {
    launch_flash_prefill_any(out, PrefillArgs{q, k, v, cu, cu_k, nullptr, B, KVH, scale, softcap,
                                              window, max_seqlen});
    return;
  } else {
  dim3 grid(B, H);
  auto l = [&]<int HD>() {
    hipLaunchKernelGGL((varlen_prefill_attention_kernel<T, HD>), grid,
                       dim3(256), 0, stream(),
                       reinterpret_cast<T*>(out.data_ptr()),
                       reinterpret_cast<const T*>(q.data_ptr()),
                       reinterpret_cast<const T*>(k.data_ptr()),
                       reinterpret_cast<const T*>(v.data_ptr()),
                       cu.data_ptr<int>(), cu_k.data_ptr<int>(), H, KVH,
                       (float)scale, (float)softcap, (int)window,
                       q.stride(0), k.stride(0), v.stride(0), out.stride(0));
  };
  switch (D) {
    case 64: l.template operator()<64>(); break;
    case 128: l.template operator()<128>(); break;
    case 256: l.template operator()<256>(); break;
  }
  }
}

void varlen_prefill_attention(at::Tensor out, at::Tensor q, at::Tensor k,
                              at::Tensor v, at::Tensor cu_seqlens,
                              at::Tensor cu_seqlens_k,
                              long max_seqlen, double scale, double softcap,
                              long window) {
  CHECK_GPU(q);
  CHECK_LASTDIM(q);
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt);
  TORCH_CHECK(cu_seqlens_k.scalar_type() == at::kInt);
  const int B = cu_seqlens.size(0) - 1;
  dispatch_dtype(q, "varlen_prefill_attention", [&]<typename T>() {
    launch_prefill<T>(out, q, k, v, cu_seqlens, cu_seqlens_k, B, scale,
                      softcap, window, max_seqlen);
  });
}

// Prompt portions over the paged bf16 cache: the last rows of contexts of
// cu_k[b+1] - cu_k[b] keys.
void paged_prefill_attention(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                             at::Tensor v_cache, at::Tensor block_tables, at::Tensor cu_seqlens,
                             at::Tensor cu_seqlens_k, long max_seqlen, double scale,
                             double softcap, long window) {
  CHECK_GPU(q);
  CHECK_LASTDIM(q);
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt && cu_seqlens_k.scalar_type() == at::kInt &&
              block_tables.scalar_type() == at::kInt);
  TORCH_CHECK(q.scalar_type() == at::kBFloat16 && k_cache.scalar_type() == at::kBFloat16 &&
                  v_cache.scalar_type() == at::kBFloat16, "bfloat16 queries and cache");
  const int D = q.size(2), B = cu_seqlens.size(0) - 1, KVH = k_cache.size(1);
  const long bs = k_cache.size(2);
  TORCH_CHECK(D == 64 || D == 128 || D == 256, "unsupported head_dim ", D);
  TORCH_CHECK(bs == 16 || bs == 32, "block_size must be 16 or 32");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() && block_tables.stride(1) == 1);
  TORCH_CHECK(q.size(1) % KVH == 0 && block_tables.size(0) == B &&
              cu_seqlens_k.size(0) == B + 1);
  if (B == 0 || q.size(0) == 0) return;
  launch_flash_prefill_any(out, PrefillArgs{q, k_cache, v_cache, cu_seqlens, cu_seqlens_k,
                                            &block_tables, B, KVH, scale, softcap, window,
                                            max_seqlen});
}

// ---------------------------------------------------------- skinny GEMM --

void skinny_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                 c10::optional<at::Tensor> bias, long splitk) {
  CHECK_GPU(x);
  CHECK_LASTDIM(x);
  CHECK_LASTDIM(w);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16);
  TORCH_CHECK(out.scalar_type() == at::kBFloat16 && out.is_contiguous());
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(K % SKG_BK == 0, "K must be a multiple of 64");
  TORCH_CHECK(N % 4 == 0, "N must be a multiple of 4");
  const __hip_bfloat16* bias_ptr = nullptr;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->numel() == N);
    bias_ptr = reinterpret_cast<const __hip_bfloat16*>(bias->data_ptr());
  }
  const int mt = (M + SKG_BM - 1) / SKG_BM;
  const int nt = (N + SKG_BN - 1) / SKG_BN;
  int z = (int)splitk;
  if (z <= 0) {  // auto: fill the chip (>=256 blocks), keep >=8 K-steps/slice
    z = 1;
    while (mt * nt * z < 256 && (K / SKG_BK) / (z * 2) >= 8 && z < 8) z *= 2;
  }
  dim3 grid(mt, nt, z);
  static const int sync_dbg = [] {
    const char* e = getenv("LLMQ_SKG_SYNC");
    return e ? atoi(e) : 0;
  }();
  if (z == 1) {
    if (sync_dbg) {
      hipLaunchKernelGGL((skinny_gemm_kernel<0, 1>), grid, dim3(SKG_NT), 0,
                         stream(), out.data_ptr(),
                         reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                         reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                         bias_ptr, M, N, K, x.stride(0), w.stride(0));
      return;
    }
    hipLaunchKernelGGL((skinny_gemm_kernel<0>), grid, dim3(SKG_NT), 0, stream(),
                       out.data_ptr(),
                       reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                       reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                       bias_ptr, M, N, K, x.stride(0), w.stride(0));
    return;
  }
  at::Tensor slabs = at::empty({z, (long)M * N}, x.options().dtype(at::kFloat));
  hipLaunchKernelGGL((skinny_gemm_kernel<1>), grid, dim3(SKG_NT), 0, stream(),
                     slabs.data_ptr(),
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                     nullptr, M, N, K, x.stride(0), w.stride(0));
  const long MN = (long)M * N;
  const long blocks = (MN / 4 + 255) / 256;
  hipLaunchKernelGGL(skinny_gemm_reduce_kernel, dim3(blocks), dim3(256), 0,
                     stream(),
                     reinterpret_cast<__hip_bfloat16*>(out.data_ptr()),
                     slabs.data_ptr<float>(), bias_ptr, z, MN, N);
}

// Weights that the streaming kernels read: packed rows from a 16-byte boundary. Others
// (a transposed or padded view, one inside a larger buffer) go to the library.
bool streamable(const at::Tensor& w) {
  return w.is_contiguous() && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0;
}

// A norm's weights or a bias as the kernels read them: a copy of any that is a strided
// view or starts elsewhere.
at::Tensor packed(const at::Tensor& t) {
  return streamable(t) ? t : t.clone(at::MemoryFormat::Contiguous);
}

// ------------------------------------------- projections, up to 256 rows --

constexpr long kSlabRows = 128, kRingRows = 256;

bool slab_rows_ok(const at::Tensor& x, const at::Tensor& w, long rows) {
  return x.dim() == 2 && w.dim() == 2 && x.size(0) > 0 && x.size(0) <= rows &&
         x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 &&
         x.stride(1) == 1 && rows_start_on(x, 16) && x.size(1) == w.size(1) &&
         w.size(1) % kSlabBK == 0 && w.size(1) > 0 && w.size(0) % 64 == 0;
}

// Token tiles of 16 that ring_gemm.hip is built for.
int ring_token_tiles(long M) {
  const int tt = (int)(M + 15) / 16;
  for (int t : {1, 2, 3, 4, 6, 8, 12, 16})
    if (tt <= t) return t;
  return 16;
}

// ring_gemm.hip counts bytes from a workgroup's first row in 32 bits.
bool ring_reaches(const at::Tensor& x, const at::Tensor& w) {
  return w.numel() * 2 < (1L << 32) && (x.size(0) - 1) * x.stride(0) * 2 < (1L << 32) - (1 << 20);
}

// Weight rows of a workgroup (64 or 128) and parts of K: what takes least, a CU taking in
// (weight + token rows) x 128 bytes a stage at 46 KB/us and the slabs being written at
// 3.3 and read at 10 MB/us, up to 128 rows what the workgroups that read a row's (`readers`) take
// in at 50 KB/us each, with no more workgroups than CUs while K has parts. Measured
// (us, R x parts): 64 rows, 3584 x 14336: 64 x 4 22.6, 128 x 8 20.6, 128 x 9 19.9; 64 rows,
// 3072 x 2048: 64 x 4 6.2, 64 x 5 5.9, 64 x 8 6.4, 128 x 8 6.5; 96 rows, 8192 x 3584: 64 x 2
// 16.0, 128 x 4 14.7, 128 x 8 18; 189 rows, 3072 x 3072: 64 x 5 11.7, 128 x 10 12.1. With the
// norm that reads the slabs: 12 rows, 2048 x 8192: 128 x 16 12.0, 64 x 8 10.9; 24 rows, 1536 x
// 8960: 128 x 20 12.1, 64 x 10 10.5; 48 rows, 3072 x 8192: 128 x 10 17.6, 64 x 5 16.0; 45 rows,
// 3584 x 4096: 128 x 8 14.6, 64 x 4 13.4; 48 rows, 3584 x 14336: 128 x 9 25.7, 64 x 4 26.1; in a
// step of 150 rows of llama-3.2-1b 128 x 16 and 64 x 8 of 2048 x 8192 1317 and 1358 in all.
struct RingPlan { int rows, parts, steps; };

RingPlan ring_plan(long M, long N, long K, int cus, long readers) {
  RingPlan best{64, 1, (int)(K / kRingBK)};
  double least = 0;
  const int tokens = 16 * ring_token_tiles(M), stages = (int)(K / kRingBK);
  const double read = M <= 128 ? std::min(10e6, 50e3 * M * readers) : 10e6;
  for (int R : {64, 128}) {
    if (N % R) continue;
    const long tiles = N / R;
    for (int p = 1; p <= std::max<long>(1, cus / tiles) && p <= stages; ++p) {
      const int steps = (stages + p - 1) / p, parts = (stages + steps - 1) / steps;
      const long rounds = (tiles * parts + cus - 1) / cus;
      const double us = rounds * (R + tokens) * steps * (128 / 46e3) +
                        parts * M * N * 4 * (1 / 3.3e6 + 1 / read);
      if (least == 0 || us < least) least = us, best = RingPlan{R, parts, steps};
    }
  }
  return best;
}

size_t sums_bytes(long M, const SgScale& scale) {
  return sizeof(float) * (size_t)M * sg_sums_stride(scale);
}

template <int TT, int RT, int WN, int WT, int WK, int ST, int EPI, bool ROT, int TQ = 1>
void launch_ring(float* slabs, __hip_bfloat16* out, long out_stride, const at::Tensor& x,
                 const at::Tensor& w, int parts, int steps, const SgScale& scale = {},
                 float cap = 0) {
  using Shape = RingShape<TT, RT, WN, WT, WK, ST>;
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  hipLaunchKernelGGL((ring_gemm_kernel<TT, RT, WN, WT, WK, ST, EPI, ROT, TQ>),
                     dim3((N + Shape::kRows - 1) / Shape::kRows * parts * TQ),
                     dim3(64 * Shape::kWaves),
                     Shape::kLds + (scale.sq ? sums_bytes(M, scale) : 0),
                     stream(), slabs, out, out_stride,
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()), x.stride(0),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), M, N, K, parts, steps,
                     scale, cap);
}

template <typename F>
void ring_tiles(long M, F&& go) {
  switch (ring_token_tiles(M)) {
    case 1: return go.template operator()<1>();
    case 2: return go.template operator()<2>();
    case 3: return go.template operator()<3>();
    case 4: return go.template operator()<4>();
    case 6: return go.template operator()<6>();
    case 8: return go.template operator()<8>();
    case 12: return go.template operator()<12>();
    default: return go.template operator()<16>();
  }
}

// Two weight tiles and one wave column suit few tokens, four and two (four from 129 rows
// on) the others, whose operand reads from LDS count (128 rows, 3584 x 14336: 25.7 and 26.3).
template <int TT, int EPI, bool ROT = false>
void launch_ring_128(float* slabs, __hip_bfloat16* out, long out_stride, const at::Tensor& x,
                     const at::Tensor& w, int parts, int steps, const SgScale& scale = {}) {
  if constexpr (TT <= 3)
    launch_ring<TT, 2, 4, 1, 1, 4, EPI, ROT>(slabs, out, out_stride, x, w, parts, steps, scale);
  else if constexpr (TT <= 8)
    launch_ring<TT, 4, 2, 2, 1, 3, EPI, ROT>(slabs, out, out_stride, x, w, parts, steps, scale);
  else
    launch_ring<TT, 4, 2, 4, 1, 3, EPI, ROT>(slabs, out, out_stride, x, w, parts, steps, scale);
}

// slab_gemm.hip: operands out of the ring kernels' reach.
template <int EPI>
void launch_slab_gemm(float* slab, __hip_bfloat16* out, long out_stride, const at::Tensor& x,
                      const at::Tensor& w) {
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  auto go = [&]<int TM, int WK>() {
    hipLaunchKernelGGL((slab_gemm_kernel<TM, WK, EPI>), dim3(N / 64), dim3(256 * WK), 0, stream(),
                       slab, out, out_stride,
                       reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()), x.stride(0),
                       reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), M, N, K,
                       K / kSlabBK);
  };
  // Gates need whole sums: two groups of waves instead of parts of K.
  constexpr int WK = EPI == kSlabSums ? 1 : 2;
  const int tm = (M + 15) / 16;
  if (tm == 1) go.template operator()<1, WK>();
  else if (tm == 2) go.template operator()<2, WK>();
  else if (tm == 3) go.template operator()<3, WK>();
  else if (tm == 4) go.template operator()<4, WK>();
  else if constexpr (EPI == kSlabSums) {
    if (tm <= 6) go.template operator()<6, 1>();
    else go.template operator()<8, 1>();
  }
}

constexpr int kRopeReaders = 4;              // workgroups of slab_rope_cache that read a row

// x W^T as fp32 slabs [parts, M, N]; their sum is the product. for_rope: slab_rope_cache will
// read them, else slab_add_norm, a workgroup a row.
at::Tensor ring_linear(const at::Tensor& x, const at::Tensor& w, bool for_rope) {
  CHECK_GPU(x);
  TORCH_CHECK(slab_rows_ok(x, w, kRingRows),
              "ring_linear: 1 to 256 bf16 rows on 16 bytes, K a multiple of 128, N of 64");
  if (!streamable(w)) return at::linear(x, w).to(at::kFloat).unsqueeze(0);
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  const auto opts = x.options().dtype(at::kFloat);
  if (!ring_reaches(x, w)) {
    if (M > kSlabRows) return at::linear(x, w).to(at::kFloat).unsqueeze(0);
    at::Tensor slab = at::empty({1, M, N}, opts);
    launch_slab_gemm<kSlabSums>(slab.data_ptr<float>(), nullptr, 0, x, w);
    return slab;
  }
  const RingPlan plan = ring_plan(M, N, K, compute_units(x), for_rope ? kRopeReaders : 1);
  at::Tensor slabs = at::empty({plan.parts, M, N}, opts);
  float* p = slabs.data_ptr<float>();
  auto go = [&]<int TT, bool ROT>() {
    if (plan.rows == 128)
      launch_ring_128<TT, kSlabSums, ROT>(p, nullptr, 0, x, w, plan.parts, plan.steps);
    else if constexpr (TT <= 8)
      launch_ring<TT, 1, 4, 1, 1, 4, kSlabSums, ROT>(p, nullptr, 0, x, w, plan.parts, plan.steps);
    else
      launch_ring<TT, 2, 2, 4, 1, 4, kSlabSums, ROT>(p, nullptr, 0, x, w, plan.parts, plan.steps);
  };
  const bool rotate = K % 8192 == 0 && N >= 5120 && (M <= 160 || N % 8192 == 0);
  ring_tiles(M, [&]<int TT>() {
    if (rotate) go.template operator()<TT, true>();
    else go.template operator()<TT, false>();
  });
  return slabs;
}

// Gate and value rows: as many weight rows a workgroup as make one round of workgroups.
// Measured (us, 64 / 128 / 256 rows): 64 tokens, 28672 x 3584 42.6 / 35.8 / -; 48 tokens,
// 37888 x 3584 60 / 60 / 51.5; 128, 55296 x 5120 177 / 132 / 107; 128, 16384 x 3072 28.2 / 38 / -.
long ring_act_rows(long N, long cus) {
  if (N / 128 > cus && N % 256 == 0) return 256;
  return N / 64 > cus && N % 128 == 0 ? 128 : 64;
}

template <int EPI>
void launch_ring_act(__hip_bfloat16* out, long out_stride, const at::Tensor& x,
                     const at::Tensor& w, const SgScale& scale = {}) {
  const long rows = ring_act_rows(w.size(0), compute_units(x));
  const int steps = (int)(w.size(1) / kRingBK);
  // over 192 tokens two groups of 128, and as many workgroups (us, one group / two: 16384 x
  // 2048, 200 rows 26.5 / 23.6, 256 rows 27.1 / 24.5; 16384 x 3072, the same 39.0 / 34.2, 40.7 /
  // 35.2; two of 96: 192 rows 23.5 / 23.2, 36.3 / 35.8, 161 rows 23.1 / 23.6)
  if (rows == 64 && x.size(0) > 192 && w.size(0) % 128 == 0)
    return launch_ring<8, 4, 2, 4, 1, 4, EPI, false, 2>(nullptr, out, out_stride, x, w, 1, steps);
  ring_tiles(x.size(0), [&]<int TT>() {
    auto go = [&]<int RT, int WN, int WT, int WK, int ST, bool ROT>() {
      launch_ring<TT, RT, WN, WT, WK, ST, EPI, ROT>(nullptr, out, out_stride, x, w, 1, steps, scale);
    };
    if (rows == 256) {
      if constexpr (TT <= 3) go.template operator()<2, 8, 1, 1, 3, false>();
      else if constexpr (TT <= 8) go.template operator()<4, 4, 2, 1, 3, false>();
      else go.template operator()<4, 4, 2, 1, 2, false>();
    } else if (rows == 128) {
      launch_ring_128<TT, EPI>(nullptr, out, out_stride, x, w, 1, steps, scale);
    } else {
      // eight waves where two groups, or four columns, have work for them (64 rows of 16384 x
      // 2048: one group 14.0, two 14.6; 96 rows 17.1 and 16.5; 45 rows 16.1 and 14.1)
      if constexpr (TT == 1 || TT == 3) go.template operator()<2, 2, 1, 2, 4, true>();
      else if constexpr (TT <= 4) go.template operator()<2, 2, 2, 1, 4, true>();
      else if constexpr (TT == 6) go.template operator()<2, 2, 2, 2, 3, true>();
      else go.template operator()<2, 2, 4, 1, 4, true>();
    }
  });
}

// Whether gate and value rows are worth a product of their own with the activation in
// it: up to 192 rows always, up to 256 while 128 weight rows a workgroup make one round
// (256 rows, the library's product + activation: 28672 x 3584 63.2 + 6 against 62.6,
// 37888 x 3584 79 + 7 / 106; 189 rows, 55296 x 5120 146 + 8 / 138; 96 rows, 28672 x 3584
// 46.8 + 5 / 39.6).
bool ring_act_ok(const at::Tensor& x, const at::Tensor& w) {
  return slab_rows_ok(x, w, kRingRows) && (x.size(0) <= 192 || w.size(0) <= 32768);
}

at::Tensor ring_act_linear(const at::Tensor& x, const at::Tensor& w, bool gelu) {
  CHECK_GPU(x);
  TORCH_CHECK(slab_rows_ok(x, w, kRingRows),
              "ring_act_linear: 1 to 256 bf16 rows on 16 bytes, K a multiple of 128, N of 64");
  at::Tensor out = at::empty({x.size(0), w.size(0) / 2}, x.options());
  auto* p = reinterpret_cast<__hip_bfloat16*>(out.data_ptr());
  if (!streamable(w) || (!ring_reaches(x, w) && x.size(0) > 64)) {
    const at::Tensor y = at::linear(x, w);
    if (gelu) gelu_tanh_and_mul(out, y);
    else silu_and_mul(out, y);
  } else if (!ring_reaches(x, w)) {
    if (gelu) launch_slab_gemm<kSlabGelu>(nullptr, p, out.stride(0), x, w);
    else launch_slab_gemm<kSlabSilu>(nullptr, p, out.stride(0), x, w);
  } else if (gelu) launch_ring_act<kSlabGelu>(p, out.stride(0), x, w);
  else launch_ring_act<kSlabSilu>(p, out.stride(0), x, w);
  return out;
}

// The head: fp32 logits x W^T, capped where cap > 0. Weight rows a workgroup as for gates, but
// any multiple of 64 in all: the last workgroup may have fewer. Token tiles of 160 and 224 too
// where 256 rows a workgroup take most of what a CU takes in. Measured (us, 64 / 128 / 256 rows
// a workgroup, the library's product and conversion): 1 row, 128256 x 2048 81 / 84 / 80, 114 + 5; 7
// rows, 131072 x 1536 61 / 62 / 62, 78 + 5; 96 rows, 256000 x 3584 434 / 385 / 335, 350 + 27; 256
// rows, 32064 x 4096 106 / 75 / -, 86 with its conversion; 49216 x 2048 108 / - / 63, 75; 65600 x
// 3072 189 / - / 157, 149 (257 workgroups, two rounds). Tokens rounded up to 192 or 256 / to 160 or
// 224: 256000 x 4608, 129 rows 526 / 519, library 513; 208 rows 583 / 557, 608; 152064 x 5120, 144
// rows 406 / 405, 372.
bool ring_head_ok(const at::Tensor& x, const at::Tensor& w) {
  return slab_rows_ok(x, w, kRingRows) && streamable(w) && w.size(1) < (1 << 22) &&
         (x.size(0) - 1) * x.stride(0) < (1L << 30);
}

at::Tensor ring_head(const at::Tensor& x, const at::Tensor& w, double cap) {
  CHECK_GPU(x);
  TORCH_CHECK(ring_head_ok(x, w), "ring_head: 1 to 256 bf16 rows on 16 bytes, packed weights, "
                                  "K a multiple of 128, N of 64");
  const long N = w.size(0), cus = compute_units(x);
  at::Tensor out = at::empty({x.size(0), N}, x.options().dtype(at::kFloat));
  auto go = [&]<int TT, int RT, int WN, int WT, int ST>() {
    launch_ring<TT, RT, WN, WT, 1, ST, kRingHead, true>(
        out.data_ptr<float>(), nullptr, 0, x, w, 1, (int)(w.size(1) / kRingBK), {}, (float)cap);
  };
  const int tt = (int)(x.size(0) + 15) / 16;
  const bool wide = N / 128 > cus && (N % 256 == 0 || N % 128 != 0);
  if (wide && (tt == 9 || tt == 10)) go.template operator()<10, 4, 4, 2, 2>();
  else if (wide && (tt == 13 || tt == 14)) go.template operator()<14, 4, 4, 2, 2>();
  else ring_tiles(x.size(0), [&]<int TT>() {
    if (wide) {
      if constexpr (TT <= 3) go.template operator()<TT, 2, 8, 1, 3>();
      else if constexpr (TT <= 8) go.template operator()<TT, 4, 4, 2, 3>();
      else if constexpr (TT == 12) go.template operator()<TT, 4, 4, 2, 2>();
      else go.template operator()<TT, 8, 2, 4, 2>();
    } else if (N / 64 > cus) {
      if constexpr (TT <= 3) go.template operator()<TT, 2, 4, 1, 4>();
      else if constexpr (TT <= 8) go.template operator()<TT, 4, 2, 2, 3>();
      else go.template operator()<TT, 4, 2, 4, 3>();
    } else {
      if constexpr (TT <= 8) go.template operator()<TT, 1, 4, 1, 4>();
      else go.template operator()<TT, 2, 2, 4, 4>();
    }
  });
  return out;
}

// ------------------------------------------- gate and value rows, many tokens --

// Tokens of a tile / 64 for tile_gemm.hip, and whether it is worth it. With weights that
// come from memory, as a model's layers do, a stage of 64 channels takes 1.27, 1.45 or 1.68 us
// with tiles of 128, 192 or 256 tokens (0.93, 1.18 and 1.5 from the caches), a tile 2.5 more;
// all CUs take a tile a round. Against that stand 1.45 PFLOP/s, a pass at 4.5 TB/s and 5 us, what
// the library's product and an activation come to at their best. They are seldom there: over
// 2048 rows they reach 800 to 1500 TFLOP/s, from one row count to the next 30 % apart, so that
// up to 1.4 times that estimate pays up to 6144 channels (27 shapes of 4096 to 73728 rows, 896
// to 5120 channels, 25 row counts each from 2049 to 8192: 13 % less time on average, at worst
// 7 % more). At 8192 channels the tiles take 1.5 % more on average. Below 2048 channels the
// library's tiles fill and drain every few stages: 1.4 at any row count. Else, up to 2048 rows, only where the
// estimate is near: 1.05, up to 3072 channels. Measured (us, weights from memory, library +
// activation / tiles): 512 rows, 17920 x 1536 43 / 36; 1000, the same 83 / 69; 768, 16384 x 2048
// 53 / 51; 1152, the same 86 / 92 (refused); 512, 16384 x 3072 58 / 68 (refused); 1000, the
// same 91 / 85; 2048, 16384 x 4096 and 73728 x 4608 the library by 4 and 5 % (refused); 2305, 16384
// x 3072 297 / 213; 28672 x 3584 404 / 419; 57344 x 8192 1646 / 1720 (refused); 2560, 28672 x
// 3584 418 / 437, 28672 x 4096 459 / 492; 3073, 17920 x 1536 202 / 151, 28672 x 3584 619 / 504;
// 4200, 16384 x 3072 401 / 350, 28672 x 3584 673 / 682, 59136 x 8192 2886 / 3000 (refused); 8192,
// 16384 x 3072 629 / 605, 28672 x 3584 1223 / 1229, 57344 x 8192 5139 / 5379 (refused).
struct TilePlan { int tw; bool worth; };

TilePlan tile_plan(long M, long N, long K, int cus) {
  TilePlan best{0, false};
  double least = 0;
  const double stage_us[] = {1.27, 1.45, 1.68};
  for (int tw = 2; tw <= 4; ++tw) {
    const long tiles = N / kTileRows * ((M + 64 * tw - 1) / (64 * tw));
    const double us = (tiles + cus - 1) / cus * (K / kTileBK * stage_us[tw - 2] + 2.5);
    if (best.tw == 0 || us < least) least = us, best.tw = tw;
  }
  const double library = 2e-9 / 1.45 * M * N * K + M * N * 3 / 4.5e6 + 5;
  best.worth = M > 2048 || K < 2048 ? K <= 6144 && least <= 1.4 * library
                                    : K <= 3072 && least <= 1.05 * library;
  return best;
}

// What tile_gemm.hip takes: it counts bytes from a tile's first row in 32 bits.
bool tile_takes(const at::Tensor& x, const at::Tensor& w) {
  return x.dim() == 2 && w.dim() == 2 && x.size(0) > 0 && x.size(0) < (1L << 30) &&
         x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 &&
         x.size(1) == w.size(1) && w.size(1) > 0 && w.size(1) % kTileBK == 0 &&
         w.size(0) > 0 && w.size(0) % kTileRows == 0 && x.stride(1) == 1 &&
         rows_start_on(x, 16) && streamable(w) && x.is_cuda() && w.get_device() == x.get_device() &&
         w.numel() * 2 < (1L << 32) && x.stride(0) >= 0 && x.stride(0) < (1L << 22);
}

// Whether tile_act_linear beats the library's product and an activation. Up to 256 rows
// are ring_gemm.hip's.
bool tile_act_ok(const at::Tensor& x, const at::Tensor& w) {
  return tile_takes(x, w) && x.size(0) > kRingRows &&
         tile_plan(x.size(0), w.size(0), w.size(1), compute_units(x)).worth;
}

at::Tensor tile_act_linear(const at::Tensor& x, const at::Tensor& w, bool gelu) {
  CHECK_GPU(x);
  TORCH_CHECK(tile_takes(x, w), "tile_act_linear: bf16 rows on 16 bytes, packed weights, K a "
                                "multiple of 64, N of 256");
  const int M = x.size(0), K = x.size(1), N = w.size(0), cus = compute_units(x);
  at::Tensor out = at::empty({M, N / 2}, x.options());
  auto go = [&]<int TW>() {
    const int wtiles = N / kTileRows, ttiles = (M + 64 * TW - 1) / (64 * TW);
    auto kernel = gelu ? &tile_gemm_kernel<TW, kSlabGelu> : &tile_gemm_kernel<TW, kSlabSilu>;
    hipLaunchKernelGGL(kernel, dim3(std::min<long>(cus, (long)wtiles * ttiles)), dim3(512),
                       tile_lds<TW>(), stream(), reinterpret_cast<__hip_bfloat16*>(out.data_ptr()),
                       out.stride(0), reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                       x.stride(0), reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), M, N, K,
                       wtiles, ttiles);
  };
  switch (tile_plan(M, N, K, cus).tw) {
    case 2: go.template operator()<2>(); break;
    case 3: go.template operator()<3>(); break;
    default: go.template operator()<4>();
  }
  return out;
}

// The two for up to 128 and 64 rows.
at::Tensor slab_linear(const at::Tensor& x, const at::Tensor& w) {
  CHECK_GPU(x);
  TORCH_CHECK(slab_rows_ok(x, w, kSlabRows),
              "slab_linear: 1 to 128 bf16 rows on 16 bytes, K a multiple of 128, N of 64");
  return ring_linear(x, w, false);
}

at::Tensor slab_act_linear(const at::Tensor& x, const at::Tensor& w, bool gelu) {
  CHECK_GPU(x);
  TORCH_CHECK(slab_rows_ok(x, w, 64),
              "slab_act_linear: 1 to 64 bf16 rows on 16 bytes, K a multiple of 128, N of 64");
  return ring_act_linear(x, w, gelu);
}

// --------------------------------------------------- projections, few rows --

// Weights that stream_gemm.hip takes: it counts bytes from a workgroup's first row in 32
// bits.
bool few_streams(const at::Tensor& w) { return streamable(w) && w.numel() * 2 < (1L << 32); }

// Slices of K in stream_gemm.hip, 16 / slices weight rows a workgroup: two where that makes
// workgroups for CUs without one and the tokens leave room. Measured (us, one / two slices):
// 3 rows, 2048 x 2048 4.2 / 3.9, 3072 x 2048 4.6 / 4.6, 3072 x 8192 11.1 / 10.5, 5120 x 3072
// 7.6 / 8.2; 7 rows, 1536 x 8960 10.7 / 8.1, 3072 x 3072 5.7 / 7.3. Four were never better.
int stream_slices(long M, long N) {
  return M <= 8 && N / 16 <= (M <= 4 ? 256 : 128) ? 2 : 1;
}

void launch_stream_prep(at::Tensor& g, at::Tensor& sq, const at::Tensor& x, const at::Tensor& w,
                        double offset) {
  hipLaunchKernelGGL(stream_prep_kernel, dim3(x.size(0)), dim3(256), 0, stream(),
                     reinterpret_cast<__hip_bfloat16*>(g.data_ptr()), sq.data_ptr<float>(),
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()), x.stride(0),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), (float)offset,
                     (int)x.size(1));
}

// The library's product of the rows, normalised first where weights are given.
at::Tensor norm_linear(const at::Tensor& x, const at::Tensor& w,
                       const c10::optional<at::Tensor>& bias,
                       const c10::optional<at::Tensor>& norm_w, double eps, double offset) {
  if (!norm_w.has_value() || !norm_w->defined()) return at::linear(x, w, bias);
  at::Tensor h = at::empty({x.size(0), x.size(1)}, x.options());
  rmsnorm(h, x.contiguous(), *norm_w, eps, offset);
  return at::linear(h, w, bias);
}

// out = f(y) of a product y = x W^T.
void finish_product(at::Tensor out, const at::Tensor& y, long epi) {
  if (epi == kSgPlain) out.copy_(y);
  else if (epi == kSgResidual) out.add_(y);
  else if (epi == kSgSilu) silu_and_mul(out, y);
  else gelu_tanh_and_mul(out, y);
}

// Whether gate and value rows of up to 16 tokens go to ring_gemm.hip, whose workgroups own 64
// rows and more and all of K, or to stream_gemm.hip's pairs, 8 or 16 rows each. The ring wants
// many workgroups, a last round that is no small one, and rows whose starts spread over the
// memory channels: multiples of 1 KiB do so badly without the start of its own that a
// workgroup of 64 rows takes, of 4 KiB worse, of 16 KiB in any form. From nine tokens on,
// which the pairs read again for every 16 rows, it wins more. Measured (us, ring / pairs): 1
// token, 2048 x 2048 8.2 / 3.8, 2048 x 8192 25.3 / 8.0, 8192 x 3072 13.8 / 10.2, 9728 x 896
// 6.0 / 6.3, 12288 x 4096 19.7 / 20.5, 16384 x 2048 13.7 / 14.4, 16384 x 8192 62 / 48, 16448 x
// 3072 26.9 / 21.4, 17920 x 1536 14.2 / 12.9, 18432 x 2304 17.9 / 18.2, 24576 x 896 10.1 /
// 11.2, 28672 x 2048 26.6 / 23.3, 28672 x 3584 36.0 / 37.3, 37888 x 3584 53 / 46; 9 tokens,
// 4096 x 896 5.2 / 3.7, 6144 x 896 5.4 / 5.7, 8192 x 3072 14.9 / 12.2, 9728 x 3072 14.4 /
// 15.7, 16448 x 3072 26.9 / 24.5, 24640 x 2048 21.8 / 24.9, 17920 x 1536 14.5 / 16.1, 28672 x
// 3584 35.7 / 42.4, 57344 x 8192 187 / 150.
bool pairs_in_ring(long M, long N, long K, long cus) {
  const bool many = M > 8;
  if (N % 64 != 0 || N <= (many && K < 1536 ? 20 : 32) * cus || K >= 8192) return false;
  const long rows = ring_act_rows(N, cus), tiles = N / rows;
  if (rows == 64) return tiles <= cus || (many && tiles * 4 >= cus * 5);
  if (many || K < 1536 || (rows == 128 && K % 512 != 0)) return true;
  return tiles <= cus && tiles * 5 >= cus * 4 && K % 2048 != 0;
}

// out = f(x) W^T for up to 16 rows: see stream_gemm.hip. norm_w: x is RMS-normalised
// first; epi: 0 plain, 1 added to out in place, 2 / 3 SiLU / tanh-GELU of the first
// half of W's rows times the second half. scale: x's rows await their factors; next:
// what kSgResidual leaves for the next norm.
void launch_stream_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                        c10::optional<at::Tensor> bias, c10::optional<at::Tensor> norm_w,
                        double eps, double offset, long epi, const SgRope& rope = {},
                        const SgScale& scale = {}, const SgNext& next = {}) {
  CHECK_GPU(x);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 2, "x, w and out must be matrices");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  const bool pair = epi == kSgSilu || epi == kSgGelu;
  const int cols = pair ? N / 2 : N;
  auto bf16 = [](const at::Tensor& t) { return t.scalar_type() == at::kBFloat16; };
  auto start16 = [](const at::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  TORCH_CHECK(bf16(x) && bf16(w) && bf16(out), "x, w and out must be bfloat16");
  TORCH_CHECK(M >= 1 && M <= 16, "1 to 16 rows");
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == cols, "shapes differ");
  TORCH_CHECK(K > 0 && K % 128 == 0 && N % 32 == 0, "K must be a multiple of 128, N of 32");
  TORCH_CHECK(w.is_contiguous() && x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
                  out.stride(1) == 1 && start16(x) && start16(w),
              "w must be contiguous, x's rows start on 16 bytes, rows packed");
  const __hip_bfloat16* bp = nullptr;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK(bf16(*bias) && bias->numel() == N && !pair,
                "bias must be bfloat16 [N], without an activation");
    bias = packed(*bias);
    bp = reinterpret_cast<const __hip_bfloat16*>(bias->data_ptr());
  }
  if (!ring_reaches(x, w))                               // rows far apart
    return launch_stream_gemm(out, x.contiguous(), w, bias, norm_w, eps, offset, epi, rope, scale,
                              next);
  if (norm_w.has_value() && norm_w->defined()) {
    TORCH_CHECK(bf16(*norm_w) && norm_w->numel() == K, "norm weights must be bfloat16 [K]");
    norm_w = packed(*norm_w);
    // Either way a launch before the product. Up to six rows of not too much work for the
    // workgroups the rows' factors meet the sums (operands rounded before their scaling),
    // else the rows are normalised: the roundings that each size has had.
    const int R = (long)N * K >= (48L << 20) || M > 8 ? 16 : M > 4 ? 8 : 4;
    at::Tensor h = at::empty({M, K}, x.options());
    if (M <= 6 && (long)(N / R) * M * K <= 12'000'000 && (long)M * (K + 512) * 2 <= (120 << 10)) {
      at::Tensor sq = at::empty({4L * M}, x.options().dtype(at::kFloat));
      launch_stream_prep(h, sq, x, *norm_w, offset);
      launch_stream_gemm(out, h, w, bias, c10::nullopt, 0, 0, epi, rope,
                         SgScale{sq.data_ptr<float>(), 1, (float)eps});
    } else {
      rmsnorm(h, x.is_contiguous() ? x : x.contiguous(), *norm_w, eps, offset);
      launch_stream_gemm(out, h, w, bias, c10::nullopt, 0, 0, epi, rope);
    }
    return;
  }
  if (pair && pairs_in_ring(M, N, K, compute_units(x)) && out.stride(0) % 4 == 0 &&
      reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0) {
    auto* p = reinterpret_cast<__hip_bfloat16*>(out.data_ptr());
    if (epi == kSgSilu) launch_ring_act<kSlabSilu>(p, out.stride(0), x, w, scale);
    else launch_ring_act<kSlabGelu>(p, out.stride(0), x, w, scale);
    return;
  }
  auto go = [&]<int KH, int ST, int NX, bool SCALE, int EPI>() {
    using Shape = StreamShape<KH, ST, NX>;
    hipLaunchKernelGGL((stream_gemm_kernel<KH, ST, NX, SCALE, EPI>), dim3(N / Shape::kRows),
                       dim3(stream_threads(EPI)), Shape::kLds + (SCALE ? sums_bytes(M, scale) : 0), stream(),
                       reinterpret_cast<__hip_bfloat16*>(out.data_ptr()),
                       out.stride(0), reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                       x.stride(0), reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), bp,
                       scale, next, M, N, K, rope);
  };
  // Rings of four stages while each workgroup has a CU to itself; two, and two or three
  // workgroups a CU, where there are more (us, two / four stages: 3 rows, 5120 x 3072
  // 7.6 / 9.1, 3072 x 8192 in slices 10.5 / 11.6, 2048 x 8192 in slices 8.7 / 7.4).
  const bool sliced = stream_slices(M, N) == 2, many = N / (sliced ? 8 : 16) > 256;
  auto shape = [&]<bool SCALE, int EPI>() {
    constexpr int FOUR = SCALE ? 3 : 4;                  // beside the rows' sums in LDS
    if (M > 8) go.template operator()<1, FOUR, 2, SCALE, EPI>();
    else if (!sliced && many) go.template operator()<1, 2, 1, SCALE, EPI>();
    else if (!sliced) go.template operator()<1, 4, 1, SCALE, EPI>();
    else if (M > 4) go.template operator()<2, FOUR, 2, SCALE, EPI>();
    else if (many) go.template operator()<2, 2, 1, SCALE, EPI>();
    else go.template operator()<2, 4, 1, SCALE, EPI>();
  };
  auto epilogue = [&]<bool SCALE>() {
    if (epi == kSgPlain) shape.template operator()<SCALE, kSgPlain>();
    else if (epi == kSgResidual) shape.template operator()<SCALE, kSgResidual>();
    else if (epi == kSgSilu) shape.template operator()<SCALE, kSgSilu>();
    else if (epi == kSgRope) shape.template operator()<SCALE, kSgRope>();
    else shape.template operator()<SCALE, kSgGelu>();
  };
  if (scale.sq) epilogue.template operator()<true>();
  else epilogue.template operator()<false>();
}

void stream_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                 c10::optional<at::Tensor> bias, c10::optional<at::Tensor> norm_w,
                 double eps, double offset, long epi) {
  TORCH_CHECK(epi >= kSgPlain && epi <= kSgGelu, "unknown epilogue");
  if (few_streams(w)) return launch_stream_gemm(out, x, w, bias, norm_w, eps, offset, epi);
  finish_product(out, norm_linear(x, w, bias, norm_w, eps, offset), epi);
}

// out = rmsnorm(x) W^T (+ bias) as q/k/v rows [M, (heads + 2 kv heads) D], q and k
// rotated, k and v also written into the paged cache. scale: in the norm's place.
void launch_stream_qkv(at::Tensor out, at::Tensor x, at::Tensor w, c10::optional<at::Tensor> bias,
                       c10::optional<at::Tensor> norm_w, double eps, double offset,
                       at::Tensor k_cache, at::Tensor v_cache, at::Tensor positions,
                       at::Tensor cos_sin, at::Tensor slots, const SgScale& scale = {}) {
  CHECK_GPU(x);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && k_cache.dim() == 4 && cos_sin.dim() == 2);
  const int M = x.size(0), N = w.size(0), kv_heads = k_cache.size(1), D = k_cache.size(3);
  const bool fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  TORCH_CHECK(D > 0 && D % 16 == 0 && N % D == 0 && N / D > 2 * kv_heads,
              "w must have (heads + 2 kv heads) D rows, D a multiple of 16");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
                  k_cache.sizes() == v_cache.sizes() &&
                  k_cache.scalar_type() == v_cache.scalar_type() &&
                  (fp8 || k_cache.scalar_type() == at::kBFloat16),
              "caches must be contiguous, bfloat16 or e4m3");
  TORCH_CHECK(positions.scalar_type() == at::kLong && positions.numel() == M &&
                  slots.scalar_type() == at::kLong && slots.numel() == M &&
                  positions.is_contiguous() && slots.is_contiguous() &&
                  cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous() &&
                  cos_sin.size(1) == D, "one int64 position and slot per row, fp32 cos_sin [*, D]");
  if (!few_streams(w)) {
    out.copy_(norm_linear(x, w, bias, norm_w, eps, offset));
    const at::Tensor heads = out.view({M, N / D, D});
    const long q = N / D - 2 * kv_heads;
    return rope_and_cache(heads.narrow(1, 0, q), heads.narrow(1, q, kv_heads),
                          heads.narrow(1, q + kv_heads, kv_heads), k_cache, v_cache, positions,
                          cos_sin, slots);
  }
  launch_stream_gemm(out, x, w, bias, norm_w, eps, offset, kSgRope,
                     SgRope{k_cache.data_ptr(), v_cache.data_ptr(), positions.data_ptr<long>(),
                            slots.data_ptr<long>(), cos_sin.data_ptr<float>(),
                            N / D - 2 * kv_heads, kv_heads, D, (int)k_cache.size(2), fp8},
                     scale);
}

void stream_qkv(at::Tensor out, at::Tensor x, at::Tensor w, c10::optional<at::Tensor> bias,
                c10::optional<at::Tensor> norm_w, double eps, double offset, at::Tensor k_cache,
                at::Tensor v_cache, at::Tensor positions, at::Tensor cos_sin, at::Tensor slots) {
  launch_stream_qkv(out, x, w, bias, norm_w, eps, offset, k_cache, v_cache, positions, cos_sin,
                    slots);
}

// The steps of a layer of few rows whose norms ride on its products. Between them go
// g [M, K], the residual rows times the next norm's weights, and sq, n sums of squares a
// row (rounded up to 4): few_prep and few_add leave them and return n, few_qkv and few_act
// take them.

void check_scaled(const at::Tensor& g, const at::Tensor& sq, long n) {
  CHECK_GPU(g);
  TORCH_CHECK(g.dim() == 2 && g.scalar_type() == at::kBFloat16 && g.is_contiguous() &&
                  streamable(g) && g.size(1) % 8 == 0 && g.size(0) >= 1 && g.size(0) <= 16,
              "g must be 1 to 16 packed bf16 rows from a 16-byte boundary");
  TORCH_CHECK(sq.scalar_type() == at::kFloat && sq.is_contiguous() && n >= 1 &&
                  sq.numel() >= g.size(0) * ((n + 3) / 4 * 4) && streamable(sq),
              "sq must hold n fp32 sums a row, rounded up to 4");
}

at::Tensor scaled_rows(const at::Tensor& g, const at::Tensor& sq, long n, double eps) {
  const long M = g.size(0);
  const long ns = (n + 3) / 4 * 4;
  const at::Tensor ms =
      sq.flatten().narrow(0, 0, M * ns).view({M, ns}).narrow(1, 0, n).sum(1, true) / g.size(1);
  return (g.to(at::kFloat) * at::rsqrt(ms + eps)).to(at::kBFloat16);
}

long few_prep(const at::Tensor& x, const at::Tensor& w, double offset, at::Tensor g,
              at::Tensor sq) {
  check_scaled(g, sq, 1);
  TORCH_CHECK(x.sizes() == g.sizes() && x.scalar_type() == at::kBFloat16 && x.stride(1) == 1 &&
                  rows_start_on(x, 16) && w.scalar_type() == at::kBFloat16 &&
                  w.numel() == x.size(1), "x must be bf16 rows on 16 bytes, w bf16 [K]");
  launch_stream_prep(g, sq, x, packed(w), offset);
  return 1;
}

// residual += x W^T, and with next_w what the next norm by next_w + offset needs.
long few_add(const at::Tensor& x, const at::Tensor& w, at::Tensor residual,
             c10::optional<at::Tensor> next_w, double offset, at::Tensor g, at::Tensor sq) {
  const bool more = next_w.has_value() && next_w->defined();
  if (!few_streams(w)) {
    residual.add_(at::linear(x, w));
    return more ? few_prep(residual, *next_w, offset, g, sq) : 0;
  }
  SgNext next{};
  long n = 0;
  at::Tensor wn;
  if (more) {
    TORCH_CHECK(residual.is_contiguous() && g.sizes() == residual.sizes() &&
                    next_w->scalar_type() == at::kBFloat16 && next_w->numel() == w.size(0),
                "residual must be packed, next_w bf16 [N]");
    n = w.size(0) / (16 / stream_slices(x.size(0), w.size(0)));
    check_scaled(g, sq, n);
    wn = packed(*next_w);
    next = SgNext{reinterpret_cast<__hip_bfloat16*>(g.data_ptr()), sq.data_ptr<float>(),
                  reinterpret_cast<const __hip_bfloat16*>(wn.data_ptr()), (float)offset};
  }
  launch_stream_gemm(residual, x, w, c10::nullopt, c10::nullopt, 0, 0, kSgResidual, SgRope{},
                     SgScale{}, next);
  return n;
}

// Whether a product scales the rows itself: their sums beside its other LDS.
bool scales(const at::Tensor& w, const at::Tensor& g, long n) {
  return few_streams(w) && sums_bytes(g.size(0), SgScale{nullptr, (int)n, 0}) <= (48 << 10);
}

at::Tensor few_qkv(const at::Tensor& g, const at::Tensor& sq, long n, double eps,
                   const at::Tensor& w, c10::optional<at::Tensor> bias, at::Tensor k_cache,
                   at::Tensor v_cache, at::Tensor positions, at::Tensor cos_sin,
                   at::Tensor slots) {
  check_scaled(g, sq, n);
  at::Tensor out = at::empty({g.size(0), w.size(0)}, g.options());
  const bool ok = scales(w, g, n);
  launch_stream_qkv(out, ok ? g : scaled_rows(g, sq, n, eps), w, bias, c10::nullopt, 0, 0, k_cache,
                    v_cache, positions, cos_sin, slots,
                    ok ? SgScale{sq.data_ptr<float>(), (int)n, (float)eps} : SgScale{});
  return out;
}

at::Tensor few_act(const at::Tensor& g, const at::Tensor& sq, long n, double eps,
                   const at::Tensor& w, bool gelu) {
  check_scaled(g, sq, n);
  at::Tensor out = at::empty({g.size(0), w.size(0) / 2}, g.options());
  if (!scales(w, g, n))
    stream_gemm(out, scaled_rows(g, sq, n, eps), w, c10::nullopt, c10::nullopt, 0, 0,
                gelu ? kSgGelu : kSgSilu);
  else
    launch_stream_gemm(out, g, w, c10::nullopt, c10::nullopt, 0, 0, gelu ? kSgGelu : kSgSilu,
                       SgRope{}, SgScale{sq.data_ptr<float>(), (int)n, (float)eps});
  return out;
}

// ------------------------------------- readers of the ring products' slabs --

void check_slabs(const at::Tensor& slabs) {
  CHECK_GPU(slabs);
  TORCH_CHECK(slabs.dim() == 3 && slabs.scalar_type() == at::kFloat && slabs.is_contiguous(),
              "slabs must be contiguous fp32 [parts, M, N]");
}

// residual += sum of slabs (RMS-normalised by w_post first, where given); returns
// rmsnorm(residual) by w.
at::Tensor slab_add_norm(const at::Tensor& slabs, at::Tensor residual,
                         c10::optional<at::Tensor> w_post, const at::Tensor& w, double eps,
                         double offset) {
  check_slabs(slabs);
  const int S = slabs.size(0), M = slabs.size(1), N = slabs.size(2);
  TORCH_CHECK(residual.is_contiguous() && residual.scalar_type() == at::kBFloat16 &&
                  residual.numel() == (long)M * N && N % 4 == 0 && N <= 8192,
              "residual must be contiguous bf16 [M, N], N a multiple of 4 up to 8192");
  auto weights = [&](const at::Tensor& t) {
    TORCH_CHECK(t.scalar_type() == at::kBFloat16 && t.numel() == N,
                "norm weights must be bf16 [N]");
    return packed(t);
  };
  const bool post = w_post.has_value() && w_post->defined();
  const at::Tensor wp = post ? weights(*w_post) : at::Tensor(), wn = weights(w);
  at::Tensor h = at::empty_like(residual);
  auto go = [&]<bool POST>() {
    const int threads = std::min(kSlabNT, (N / 4 + 63) / 64 * 64);
    hipLaunchKernelGGL(slab_add_norm_kernel<POST>, dim3(M), dim3(threads), 0, stream(),
                       reinterpret_cast<__hip_bfloat16*>(h.data_ptr()),
                       reinterpret_cast<__hip_bfloat16*>(residual.data_ptr()),
                       slabs.data_ptr<float>(), S,
                       POST ? reinterpret_cast<const __hip_bfloat16*>(wp.data_ptr()) : nullptr,
                       reinterpret_cast<const __hip_bfloat16*>(wn.data_ptr()), M, N, (float)eps,
                       (float)offset);
  };
  if (post) go.template operator()<true>();
  else go.template operator()<false>();
  return h;
}

// bf16 rows [M, (heads + 2 kv heads) D] of the summed slabs + bias, q and k rotated;
// k and v also into the paged cache.
at::Tensor slab_rope_cache(const at::Tensor& slabs, c10::optional<at::Tensor> bias,
                           at::Tensor k_cache, at::Tensor v_cache, const at::Tensor& positions,
                           const at::Tensor& cos_sin, const at::Tensor& slots) {
  check_slabs(slabs);
  const int S = slabs.size(0), M = slabs.size(1), N = slabs.size(2);
  const int kv_heads = k_cache.size(1), bs = k_cache.size(2), D = k_cache.size(3);
  TORCH_CHECK(N % D == 0 && N / D > 2 * kv_heads && D % 8 == 0, "N must be (heads + 2 kv heads) D");
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
                  k_cache.scalar_type() == v_cache.scalar_type());
  TORCH_CHECK(positions.scalar_type() == at::kLong && positions.numel() == M &&
                  slots.scalar_type() == at::kLong && slots.numel() == M &&
                  cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous() &&
                  cos_sin.size(1) == D);
  const __hip_bfloat16* bp = nullptr;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->numel() == N,
                "bias must be bf16 [N]");
    bias = packed(*bias);
    bp = reinterpret_cast<const __hip_bfloat16*>(bias->data_ptr());
  }
  at::Tensor qkv = at::empty({M, N}, slabs.options().dtype(at::kBFloat16));
  auto go = [&]<typename TC>() {
    hipLaunchKernelGGL(slab_rope_cache_kernel<TC>, dim3(M, kRopeReaders), dim3(256), 0, stream(),
                       reinterpret_cast<__hip_bfloat16*>(qkv.data_ptr()),
                       slabs.data_ptr<float>(), S, bp, reinterpret_cast<TC*>(k_cache.data_ptr()),
                       reinterpret_cast<TC*>(v_cache.data_ptr()), positions.data_ptr<long>(),
                       cos_sin.data_ptr<float>(), slots.data_ptr<long>(), M,
                       N / D - 2 * kv_heads, kv_heads, D, bs);
  };
  if (k_cache.scalar_type() == at::kBFloat16) go.template operator()<__hip_bfloat16>();
  else if (k_cache.scalar_type() == at::kFloat8_e4m3fn) go.template operator()<__hip_fp8_e4m3>();
  else TORCH_CHECK(false, "bf16 or fp8 cache");
  return qkv;
}

// ------------------------------------------------------ prompt steps, whole --

// All layers of a packed prompt step (no portion gathered into packed rows): the
// calls that the engine's per-layer code makes, in one crossing from Python.
// A layer's weights: qkv, o, gate_up, down, pre-MLP norm, next layer's input norm
// (or the final one), and with sandwich norms the post-attention and post-MLP
// ones. h is the normed input of layer 0; returns the final normed rows.
at::Tensor prompt_layers(at::Tensor h, at::Tensor residual, at::TensorList weights,
                         at::TensorList biases, at::TensorList k_caches,
                         at::TensorList v_caches, at::Tensor positions, at::Tensor cos_sin,
                         at::Tensor slots, at::Tensor cu_seqlens,
                         c10::optional<at::Tensor> block_tables,
                         c10::optional<at::Tensor> cu_seqlens_k, long max_seqlen,
                         long head_dim, double scale, double softcap, at::IntArrayRef windows,
                         double eps, double offset, bool gelu, bool post_norms) {
  CHECK_GPU(h);
  const size_t per = post_norms ? 8 : 6, layers = k_caches.size();
  TORCH_CHECK(weights.size() == per * layers && v_caches.size() == layers &&
                  windows.size() == layers && (biases.empty() || biases.size() == layers),
              "one entry per layer");
  const long T = h.size(0);
  // up to 256 rows of these shapes: the streaming products, whose sums the next
  // kernel takes up
  const bool slab = layers > 0 && k_caches[0].size(3) == head_dim && h.size(1) <= 8192 &&
                    (k_caches[0].scalar_type() == at::kBFloat16 ||
                     k_caches[0].scalar_type() == at::kFloat8_e4m3fn) &&
                    slab_rows_ok(h, weights[0], kRingRows) && weights[1].size(0) == h.size(1) &&
                    weights[1].size(1) % kSlabBK == 0 && weights[1].size(0) % 64 == 0 &&
                    weights[3].size(1) % kSlabBK == 0 && residual.is_contiguous();
  const c10::optional<at::Tensor> none;
  for (size_t i = 0; i < layers; ++i) {
    const at::Tensor* w = &weights[per * i];
    const c10::optional<at::Tensor> bias =
        biases.empty() ? none : c10::make_optional(biases[i]);
    const at::Tensor qkv =
        slab ? slab_rope_cache(ring_linear(h, w[0], true), bias, k_caches[i],
                               v_caches[i], positions, cos_sin, slots)
             : at::linear(h, w[0], bias);
    const long kv_heads = k_caches[i].size(1);
    const long heads = qkv.size(1) / head_dim - 2 * kv_heads;
    auto part = [&](long first, long n) {
      return qkv.narrow(1, first * head_dim, n * head_dim).view({T, n, head_dim});
    };
    const at::Tensor q = part(0, heads), k = part(heads, kv_heads),
                     v = part(heads + kv_heads, kv_heads);
    if (!slab) rope_and_cache(q, k, v, k_caches[i], v_caches[i], positions, cos_sin, slots);
    at::Tensor attn = at::empty({T, heads, head_dim}, qkv.options());
    if (cu_seqlens_k.has_value())
      paged_prefill_attention(attn, q, k_caches[i], v_caches[i], *block_tables, cu_seqlens,
                              *cu_seqlens_k, max_seqlen, scale, softcap, windows[i]);
    else
      varlen_prefill_attention(attn, q, k, v, cu_seqlens, cu_seqlens, max_seqlen, scale, softcap,
                               windows[i]);
    // the product, added to the residual (normalised first with sandwich norms), normed
    auto project_add_norm = [&](const at::Tensor& a, const at::Tensor& wt,
                                const at::Tensor* post, const at::Tensor& norm) {
      if (slab)
        return slab_add_norm(ring_linear(a, wt, false), residual,
                             post ? c10::make_optional(*post) : none, norm, eps, offset);
      at::Tensor y = at::linear(a, wt);
      if (post) norm_add_norm(y, residual, *post, norm, eps, offset);
      else fused_add_rmsnorm(y, residual, norm, eps, offset);
      return y;
    };
    h = project_add_norm(attn.view({T, heads * head_dim}), w[1], post_norms ? &w[6] : nullptr,
                         w[4]);
    at::Tensor act;
    if (slab && ring_act_ok(h, w[2])) {
      act = ring_act_linear(h, w[2], gelu);
    } else if (tile_act_ok(h, w[2])) {
      act = tile_act_linear(h, w[2], gelu);
    } else {
      const at::Tensor gate_up = at::linear(h, w[2]);
      act = at::empty({T, gate_up.size(1) / 2}, gate_up.options());
      if (gelu) gelu_tanh_and_mul(act, gate_up);
      else silu_and_mul(act, gate_up);
    }
    h = project_add_norm(act, w[3], post_norms ? &w[7] : nullptr, w[5]);
  }
  return h;
}

// ------------------------------------------------------------- sampling --

// Chunks of a logits row: enough workgroups to fill the chip at few rows, whole
// 16-byte loads where every row allows them (the return value).
bool row_chunks(const at::Tensor& logits, int B, int V, int& chunk, int& splits) {
  int n = 1;
  while (B * n < 2048 && n < 64 && (V / n) > 4096) n *= 2;
  chunk = std::max(((V + n - 1) / n + 3) / 4 * 4, 4);
  splits = std::max((V + chunk - 1) / chunk, 1);         // an empty vocabulary launches too
  return V % 4 == 0 && logits.stride(0) % 4 == 0 &&
         reinterpret_cast<uintptr_t>(logits.data_ptr()) % 16 == 0;
}

// out = cap * tanh(in / cap) in fp32 of bf16 logits
void softcap_logits(at::Tensor out, at::Tensor in, double cap) {
  CHECK_GPU(in);
  TORCH_CHECK(in.scalar_type() == at::kBFloat16 && out.scalar_type() == at::kFloat);
  TORCH_CHECK(in.is_contiguous() && out.is_contiguous() && in.numel() == out.numel());
  TORCH_CHECK(reinterpret_cast<uintptr_t>(in.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  const long n = in.numel();
  if (n == 0) return;
  const int grid = (int)std::min<long>((n + 2047) / 2048, 8192);
  hipLaunchKernelGGL(softcap_logits_kernel, dim3(grid), dim3(256), 0, stream(),
                     out.data_ptr<float>(),
                     reinterpret_cast<const __hip_bfloat16*>(in.data_ptr()), n, (float)cap);
}

void topk_topp_bound(at::Tensor out_bound, at::Tensor logits, at::Tensor temps,
                     at::Tensor top_ps, at::Tensor top_ks) {
  CHECK_GPU(logits);
  TORCH_CHECK(logits.scalar_type() == at::kFloat && logits.dim() == 2);
  TORCH_CHECK(out_bound.scalar_type() == at::kFloat);
  TORCH_CHECK(top_ps.scalar_type() == at::kFloat);
  TORCH_CHECK(top_ks.scalar_type() == at::kLong);
  const int B = logits.size(0), V = logits.size(1);
  if (B == 0) return;
  TORCH_CHECK(logits.stride(1) == 1, "logits rows must be packed");
  int chunk, splits;
  const bool vec = row_chunks(logits, B, V, chunk, splits);
  at::Tensor ws = at::zeros({(long)B * (long)sizeof(ThRow) / 4}, logits.options().dtype(at::kInt));
  ThRow* rows = reinterpret_cast<ThRow*>(ws.data_ptr());
  float* bound = out_bound.data_ptr<float>();
  const float *lp = logits.data_ptr<float>(), *tp = temps.data_ptr<float>(),
              *pp = top_ps.data_ptr<float>();
  const long* kp = top_ks.data_ptr<long>();
  const long stride = logits.stride(0);
  const dim3 grid(B, splits), wg(256);
  hipLaunchKernelGGL(topk_topp_max_kernel, grid, wg, 0, stream(), bound, rows, lp, tp, pp, kp, V,
                     stride, chunk, vec);
  hipLaunchKernelGGL((topk_topp_hist_kernel<0>), grid, wg, 0, stream(), rows, lp, tp, pp, kp, V,
                     stride, chunk, vec);
  hipLaunchKernelGGL((topk_topp_scan_kernel<0>), dim3(B), wg, 0, stream(), bound, rows, tp, pp, kp,
                     V);
  hipLaunchKernelGGL((topk_topp_hist_kernel<1>), grid, wg, 0, stream(), rows, lp, tp, pp, kp, V,
                     stride, chunk, vec);
  hipLaunchKernelGGL((topk_topp_scan_kernel<1>), dim3(B), wg, 0, stream(), bound, rows, tp, pp, kp,
                     V);
}

void sample_gumbel_argmax(at::Tensor out, at::Tensor keys, at::Tensor logits,
                          at::Tensor temps, at::Tensor req_seeds,
                          at::Tensor req_pos, long seed, long step,
                          c10::optional<at::Tensor> bounds) {
  CHECK_GPU(logits);
  TORCH_CHECK(logits.scalar_type() == at::kFloat && logits.dim() == 2);
  TORCH_CHECK(out.scalar_type() == at::kLong);
  TORCH_CHECK(keys.scalar_type() == at::kLong && keys.numel() == logits.size(0));
  TORCH_CHECK(req_seeds.scalar_type() == at::kInt);
  TORCH_CHECK(req_pos.scalar_type() == at::kInt);
  const int B = logits.size(0), V = logits.size(1);
  const float* bounds_ptr = nullptr;
  if (bounds.has_value() && bounds->defined()) {
    TORCH_CHECK(bounds->scalar_type() == at::kFloat && bounds->numel() == B);
    bounds_ptr = bounds->data_ptr<float>();
  }
  if (B == 0) return;
  TORCH_CHECK(logits.is_contiguous(), "logits must be contiguous");
  int chunk, splits;
  const bool vec = row_chunks(logits, B, V, chunk, splits);
  at::Tensor parts = at::empty({(long)B, (long)splits}, keys.options());
  auto words = [](const at::Tensor& t) {
    return reinterpret_cast<unsigned long long*>(t.data_ptr());
  };
  hipLaunchKernelGGL(sample_argmax_kernel, dim3(B, splits), dim3(256), 0,
                     stream(), words(parts),
                     logits.data_ptr<float>(), temps.data_ptr<float>(),
                     reinterpret_cast<const unsigned int*>(req_seeds.data_ptr()),
                     reinterpret_cast<const unsigned int*>(req_pos.data_ptr()),
                     bounds_ptr, V, (unsigned int)seed, (unsigned int)step, chunk, vec);
  hipLaunchKernelGGL(unpack_keys_kernel, dim3((B + 3) / 4), dim3(256), 0, stream(),
                     out.data_ptr<long>(), words(keys), words(parts), splits, B);
}

}  // namespace

TORCH_LIBRARY(llmq_amd, m) {
  m.def("rmsnorm(Tensor(a!) out, Tensor input, Tensor weight, float eps, float offset) -> ()");
  m.def("fused_add_rmsnorm(Tensor(a!) x, Tensor(b!) residual, Tensor weight, float eps, float offset) -> ()");
  m.def("silu_and_mul(Tensor(a!) out, Tensor input) -> ()");
  m.def("gelu_tanh_and_mul(Tensor(a!) out, Tensor input) -> ()");
  m.def("rope_inplace(Tensor(a!) q, Tensor(b!) k, Tensor positions, Tensor cos_sin) -> ()");
  m.def("reshape_and_cache(Tensor key, Tensor value, Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor slot_mapping) -> ()");
  m.def("paged_decode_attention(Tensor(a!) out, Tensor q, Tensor k_cache, Tensor v_cache, Tensor block_tables, Tensor context_lens, float scale, float softcap, int window, Tensor(b!)? arrivals=None) -> ()");
  m.def("varlen_prefill_attention(Tensor(a!) out, Tensor q, Tensor k, Tensor v, Tensor cu_seqlens, Tensor cu_seqlens_k, int max_seqlen, float scale, float softcap, int window) -> ()");
  m.def("paged_prefill_attention(Tensor(a!) out, Tensor q, Tensor k_cache, Tensor v_cache, Tensor block_tables, Tensor cu_seqlens, Tensor cu_seqlens_k, int max_seqlen, float scale, float softcap, int window) -> ()");
  m.def("stream_qkv(Tensor(a!) out, Tensor x, Tensor w, Tensor? bias, Tensor? norm_w, float eps, float offset, Tensor(b!) k_cache, Tensor(c!) v_cache, Tensor positions, Tensor cos_sin, Tensor slots) -> ()");
  m.def("few_prep(Tensor x, Tensor w, float offset, Tensor(a!) g, Tensor(b!) sq) -> int");
  m.def("few_add(Tensor x, Tensor w, Tensor(a!) residual, Tensor? next_w, float offset, Tensor(b!) g, Tensor(c!) sq) -> int");
  m.def("few_qkv(Tensor g, Tensor sq, int n, float eps, Tensor w, Tensor? bias, Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor positions, Tensor cos_sin, Tensor slots) -> Tensor");
  m.def("few_act(Tensor g, Tensor sq, int n, float eps, Tensor w, bool gelu) -> Tensor");
  m.def("slab_linear(Tensor x, Tensor w) -> Tensor");
  m.def("ring_linear(Tensor x, Tensor w, bool for_rope=False) -> Tensor");
  m.def("ring_head(Tensor x, Tensor w, float cap) -> Tensor");
  m.def("ring_act_ok(Tensor x, Tensor w) -> bool");
  m.def("ring_act_linear(Tensor x, Tensor w, bool gelu) -> Tensor");
  m.def("slab_act_linear(Tensor x, Tensor w, bool gelu) -> Tensor");
  m.def("slab_add_norm(Tensor slabs, Tensor(a!) residual, Tensor? w_post, Tensor w, float eps, float offset) -> Tensor");
  m.def("slab_rope_cache(Tensor slabs, Tensor? bias, Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor positions, Tensor cos_sin, Tensor slots) -> Tensor");
  m.def("tile_act_ok(Tensor x, Tensor w) -> bool");
  m.def("tile_act_linear(Tensor x, Tensor w, bool gelu) -> Tensor");
  m.def("prompt_layers(Tensor h, Tensor(a!) residual, Tensor[] weights, Tensor[] biases, Tensor[] k_caches, Tensor[] v_caches, Tensor positions, Tensor cos_sin, Tensor slots, Tensor cu_seqlens, Tensor? block_tables, Tensor? cu_seqlens_k, int max_seqlen, int head_dim, float scale, float softcap, int[] windows, float eps, float offset, bool gelu, bool post_norms) -> Tensor");
  m.def("sample_gumbel_argmax(Tensor(a!) out, Tensor(b!) keys, Tensor logits, Tensor temps, Tensor req_seeds, Tensor req_pos, int seed, int step, Tensor? bounds=None) -> ()");
  m.def("topk_topp_bound(Tensor(a!) out_bound, Tensor logits, Tensor temps, Tensor top_ps, Tensor top_ks) -> ()");
  m.def("softcap_logits(Tensor(a!) out, Tensor input, float cap) -> ()");
  m.def("skinny_gemm(Tensor(a!) out, Tensor x, Tensor w, Tensor? bias, int splitk) -> ()");
  m.def("stream_gemm(Tensor(a!) out, Tensor x, Tensor w, Tensor? bias, Tensor? norm_w, float eps, float offset, int epi) -> ()");
  m.def("norm_add_norm(Tensor(a!) x, Tensor(b!) residual, Tensor w_post, Tensor w_pre, float eps, float offset) -> ()");
  m.def("rope_and_cache(Tensor(a!) q, Tensor(b!) k, Tensor value, Tensor(c!) k_cache, Tensor(d!) v_cache, Tensor positions, Tensor cos_sin, Tensor slot_mapping) -> ()");
}

TORCH_LIBRARY_IMPL(llmq_amd, CUDA, m) {
  m.impl("rmsnorm", &rmsnorm);
  m.impl("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.impl("silu_and_mul", &silu_and_mul);
  m.impl("gelu_tanh_and_mul", &gelu_tanh_and_mul);
  m.impl("rope_inplace", &rope_inplace);
  m.impl("reshape_and_cache", &reshape_and_cache);
  m.impl("paged_decode_attention", &paged_decode_attention);
  m.impl("varlen_prefill_attention", &varlen_prefill_attention);
  m.impl("paged_prefill_attention", &paged_prefill_attention);
  m.impl("few_prep", &few_prep);
  m.impl("few_add", &few_add);
  m.impl("few_qkv", &few_qkv);
  m.impl("few_act", &few_act);
  m.impl("slab_linear", &slab_linear);
  m.impl("tile_act_ok", &tile_act_ok);
  m.impl("tile_act_linear", &tile_act_linear);
  m.impl("ring_linear", &ring_linear);
  m.impl("ring_head", &ring_head);
  m.impl("ring_act_ok", &ring_act_ok);
  m.impl("ring_act_linear", &ring_act_linear);
  m.impl("slab_act_linear", &slab_act_linear);
  m.impl("slab_add_norm", &slab_add_norm);
  m.impl("slab_rope_cache", &slab_rope_cache);
  m.impl("prompt_layers", &prompt_layers);
  m.impl("sample_gumbel_argmax", &sample_gumbel_argmax);
  m.impl("topk_topp_bound", &topk_topp_bound);
  m.impl("softcap_logits", &softcap_logits);
  m.impl("skinny_gemm", &skinny_gemm);
  m.impl("stream_gemm", &stream_gemm);
  m.impl("stream_qkv", &stream_qkv);
  m.impl("norm_add_norm", &norm_add_norm);
  m.impl("rope_and_cache", &rope_and_cache);
}
