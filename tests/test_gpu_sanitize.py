"""Guard-band (canary) pass over the main library's kernels.

No compute-sanitizer ships in this image, so out-of-bounds WRITES are
checked directly: inputs and outputs are carved out of over-allocated
buffers with canary halos on both sides, and the halos are verified bitwise
after each op. Run under ``AMD_SERIALIZE_KERNEL=3`` (tests/sanitize_gpu.sh)
so any kernel fault aborts at the offending launch instead of surfacing
later. Outputs of over 1 MiB that an op allocates itself are led to the start of
a block filled with canaries (``led``). Not covered: OOB READS (those surface as
faults under serialized launches or as numerics failures in test_gpu_kernels),
what lies below such an output, smaller ones (the slabs' readers' bf16 rows) and scratch.
"""

from __future__ import annotations

import pytest
import torch

from decode_batches import BATCHES, VARIANTS

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from llmq_amd import ops

    assert ops.has_hip_ext()  # _EXT below: ops with outputs of the caller's
else:
    pytest.skip("no GPU", allow_module_level=True)

DEV = torch.device("cuda:0")
PAD = 4096  # canary elements on each side
CANARY = 0x5A


class Guarded:
    """Allocate tensors inside canary halos; verify() checks every halo."""

    def __init__(self):
        self._bufs = []

    def tensor(self, *shape, dtype=torch.bfloat16, fill="randn"):
        n = 1
        for s in shape:
            n *= s
        esz = torch.tensor([], dtype=dtype).element_size()
        raw = torch.full(((n + 2 * PAD) * esz,), CANARY, dtype=torch.uint8, device=DEV)
        mid = raw[PAD * esz: (PAD + n) * esz].view(dtype).view(*shape)
        if fill == "randn":
            mid.copy_(torch.randn(shape, device=DEV).to(dtype))
        elif fill == "zeros":
            mid.zero_()
        self._bufs.append((raw, esz, n))
        return mid

    def from_values(self, vals, dtype):
        t = self.tensor(*vals.shape, dtype=dtype, fill="zeros")
        t.copy_(vals.to(dtype))
        return t

    def verify(self):
        torch.cuda.synchronize()
        for i, (raw, esz, n) in enumerate(self._bufs):
            lo = raw[: PAD * esz]
            hi = raw[(PAD + n) * esz:]
            assert bool((lo == CANARY).all()), f"buffer {i}: LOW canary clobbered"
            assert bool((hi == CANARY).all()), f"buffer {i}: HIGH canary clobbered"


def led(op):
    """op's output, which it allocates itself, from the start of a block of canaries; nothing
    behind it may change."""
    size = 256 << 20
    with torch.cuda.use_mem_pool(torch.cuda.MemPool()):
        block = torch.full((size,), CANARY, dtype=torch.uint8, device=DEV)
        at = block.data_ptr()
        del block
        out = op()
        used = -(-out.nbytes // 512) * 512   # the allocator's rounding
        rest = torch.empty(size - used, dtype=torch.uint8, device=DEV)
    assert out.nbytes > 1 << 20 and out.data_ptr() == at and rest.data_ptr() == at + used
    assert bool((rest == CANARY).all()), "written behind the output"
    return out


@pytest.fixture()
def g():
    gg = Guarded()
    yield gg
    gg.verify()


@pytest.mark.parametrize("D,G,KVH,BS,fp8", [(64, 4, 3, 16, False), (128, 6, 2, 32, False),
                                             (256, 2, 8, 16, False), (128, 4, 2, 16, True),
                                             (256, 2, 2, 32, True)])
@pytest.mark.parametrize("softcap,window", [(0.0, 0), (50.0, 70)])
def test_decode_attention_guarded(g, D, G, KVH, BS, fp8, softcap, window):
    B, H, max_blocks = 7, G * KVH, 70
    NB = B * max_blocks + 1
    kc, vc = (g.tensor(NB, KVH, BS, D, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
              for _ in range(2))
    q, out = g.tensor(B, H, D), g.tensor(B, H, D)
    bt = g.from_values(
        torch.arange(1, 1 + B * max_blocks).reshape(B, max_blocks), torch.int32)
    ctx = g.from_values(torch.tensor([1, 63, 64, 65, 129, 1000, 1025]), torch.int32)
    for n in (7, 2):                         # pairs within a wave's range, cut in pieces
        ops._EXT.paged_decode_attention(out[:n], q[:n], kc, vc, bt[:n], ctx[:n], D ** -0.5,
                                        softcap, window)
        assert out[:n].isfinite().all()


@pytest.mark.parametrize("batch", range(len(BATCHES)))
@pytest.mark.parametrize("D,G,fp8", VARIANTS)
def test_decode_deals_guarded(g, D, G, fp8, batch):
    """Every way to cut a batch (test_decode_deal.py has which one each takes)."""
    _, lens, KVH, BS, window, softcap = BATCHES[batch]
    need = [-(-n // BS) for n in lens]
    kc, vc = (g.tensor(sum(need) + 1, KVH, BS, D,
                       dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in range(2))
    table = torch.zeros(len(lens), max(need))
    for row, mine in zip(table, torch.arange(1, sum(need) + 1).split(need)):
        row[:len(mine)] = mine
    q, out = (g.tensor(len(lens), G * KVH, D) for _ in range(2))
    bt, ctx = g.from_values(table, torch.int32), g.from_values(torch.tensor(lens), torch.int32)
    arrivals = g.tensor(len(lens), KVH, dtype=torch.int32, fill="zeros")
    ops._EXT.paged_decode_attention(out, q, kc, vc, bt, ctx, D ** -0.5, softcap, window, arrivals)
    assert out[ctx > 0].isfinite().all() and not arrivals.any()


@pytest.mark.parametrize("D,H,KVH", [(64, 4, 2), (64, 3, 1), (128, 6, 2), (256, 16, 8),
                                     (256, 3, 3)])
@pytest.mark.parametrize("softcap,window", [(0.0, 0), (50.0, 70)])
def test_prefill_attention_guarded(g, D, H, KVH, softcap, window):
    lens, past, BS = [1, 33, 129, 300], [0, 20, 64, 5], 16
    lens_k = [n + p for n, p in zip(lens, past)]
    T, Tk = sum(lens), sum(lens_k)
    q, out = g.tensor(T, H, D), g.tensor(T, H, D)
    k, v = g.tensor(Tk, KVH, D), g.tensor(Tk, KVH, D)
    cu, cu_k = (g.from_values(torch.tensor([0] + list(torch.tensor(x).cumsum(0))), torch.int32)
                for x in (lens, lens_k))
    args = (max(lens), D ** -0.5, softcap, window)
    ops._EXT.varlen_prefill_attention(out, q, k, v, cu, cu_k, *args)
    assert out.isfinite().all()
    width = -(-max(lens_k) // BS)
    kc, vc = (g.tensor(len(lens) * width, KVH, BS, D) for _ in range(2))
    bt = g.from_values(torch.arange(len(lens) * width).reshape(len(lens), width), torch.int32)
    ops._EXT.paged_prefill_attention(out, q, kc, vc, bt, cu, cu_k, *args)
    assert out.isfinite().all()


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("N,K", [(32, 128), (96, 384), (64, 14336)])
@pytest.mark.parametrize("norm", [False, True])
def test_few_row_products_guarded(g, M, N, K, norm):
    x, w = g.tensor(M, K), g.tensor(N, K)
    nw = g.tensor(K) if norm else None
    for epi in range(4):                     # plain, residual, SiLU and GELU pairs
        out = g.tensor(M, N if epi < 2 else N // 2)
        bias = g.tensor(N) if epi == 0 else None
        ops._EXT.stream_gemm(out, x, w, bias, nw, 1e-5, 0.0, epi)
        assert out.isfinite().all()


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("D,H,KVH,fp8", [(64, 3, 1, False), (128, 2, 2, True), (16, 4, 2, False)])
def test_few_row_qkv_guarded(g, M, D, H, KVH, fp8):
    from llmq_amd.ops import torch_ref

    N, K = (H + 2 * KVH) * D, 128
    kc, vc = (g.tensor(2, KVH, 16, D, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
              for _ in range(2))
    cs = g.from_values(torch_ref.build_rope_cache(64, D, 10000.0, DEV), torch.float32)
    slots = torch.randperm(32)[:M]
    slots[0] = -1
    out = g.tensor(M, N)
    ops._EXT.stream_qkv(out, g.tensor(M, K), g.tensor(N, K), g.tensor(N), g.tensor(K), 1e-5, 0.0,
                        kc, vc, g.from_values(torch.arange(M), torch.int64), cs,
                        g.from_values(slots, torch.int64))
    assert out.isfinite().all()


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 97, 128])
@pytest.mark.parametrize("D,H,KVH,fp8", [(64, 2, 1, False), (128, 2, 2, True)])
def test_slab_products_guarded(g, M, D, H, KVH, fp8):
    from llmq_amd.ops import torch_ref

    N, K = (H + 2 * KVH) * D, 384
    x = g.tensor(M, K)
    slabs = ops.slab_linear(x, g.tensor(N, K))
    kc, vc = (g.tensor(9, KVH, 16, D, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
              for _ in range(2))
    cs = g.from_values(torch_ref.build_rope_cache(128, D, 10000.0, DEV), torch.float32)
    slots = torch.randperm(144)[:M]
    slots[M // 2] = -1
    held = g.tensor(*slabs.shape, dtype=torch.float32)
    held.copy_(slabs)
    rows = ops.slab_rope_cache(held, g.tensor(N), kc, vc,
                               g.from_values(torch.arange(M), torch.int64), cs,
                               g.from_values(slots, torch.int64))
    residual = g.tensor(M, N)
    assert rows.isfinite().all()
    for post in (None, g.tensor(N)):
        assert ops.slab_add_norm(held, residual, post, g.tensor(N), 1e-5, 1.0).isfinite().all()
    if M <= 64:
        for gelu in (False, True):
            assert ops.slab_act_linear(x, g.tensor(128, K), gelu).isfinite().all()


@pytest.mark.parametrize("M", [33, 65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K", [(16384, 640), (4160, 8192), (5120, 8192)])
def test_ring_products_guarded(g, M, N, K):
    x, w = g.tensor(M, K), g.tensor(N, K)
    assert led(lambda: ops.ring_linear(x, w)).isfinite().all()


@pytest.mark.parametrize("M", [33, 96, 129, 161, 193, 256])
@pytest.mark.parametrize("N", [33152, 65792, 65600])
def test_ring_pairs_guarded(g, M, N):
    """64, 128 and 256 weight rows a workgroup."""
    x, w = g.tensor(M, 256), g.tensor(N, 256)
    for gelu in (False, True):
        assert led(lambda: ops.ring_act_linear(x, w, gelu)).isfinite().all()


@pytest.mark.parametrize("M", [17, 48, 128, 144, 160, 192, 224, 256])
@pytest.mark.parametrize("N", [16384, 16448, 32832, 33088, 33280])
def test_head_guarded(g, M, N):
    """Workgroups of which the last has fewer weight rows, and token tiles of every width."""
    x, w = g.tensor(M, 256), g.tensor(N, 256)
    for cap in (0.0, 30.0):
        out = led(lambda: ops.head_logits(x, w, cap))
        assert out.dtype == torch.float32 and out.isfinite().all()


@pytest.mark.parametrize("M", [257, 300, 700, 1153])
@pytest.mark.parametrize("N,K", [(4096, 64), (5376, 576)])
def test_tiles_guarded(g, M, N, K):
    x, w = g.tensor(M, K), g.tensor(N, K)
    for gelu in (False, True):
        assert led(lambda: ops.tile_act_linear(x, w, gelu)).isfinite().all()


@pytest.mark.parametrize("M", [1, 5, 9, 16])
@pytest.mark.parametrize("H,K", [(128, 384), (2048, 128), (4352, 256)])
@pytest.mark.parametrize("D,fp8", [(64, False), (128, True)])
def test_few_rows_chain_guarded(g, M, H, K, D, fp8):
    """What the steps of a layer of few rows hand each other, and the cache rows."""
    from llmq_amd.ops import torch_ref

    parts = -(-H // 8 // 4) * 4              # sums of a row: workgroups of 8 rows and more
    residual, rows = g.tensor(M, H), g.tensor(M, H, fill="zeros")
    kc, vc = (g.tensor(2, 1, 16, D, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16)
              for _ in range(2))
    cs = g.from_values(torch_ref.build_rope_cache(64, D, 10000.0, DEV), torch.float32)
    pos, slots = (g.from_values(torch.arange(M), torch.int64) for _ in range(2))
    for norm in (g.tensor(H), None):
        # sums to their last element: as many as this step leaves
        first = g.tensor(4 * M, dtype=torch.float32)
        assert ops._EXT.few_prep(residual, g.tensor(H), 1.0, rows, first) == 1
        sq, n = first, 1
        for _ in range(2):
            assert ops._EXT.few_qkv(rows, sq, n, 1e-5, g.tensor(3 * D, H), g.tensor(3 * D), kc, vc,
                                    pos, cs, slots).isfinite().all()
            for N in (96, 16512):
                assert ops._EXT.few_act(rows, sq, n, 1e-5, g.tensor(N, H), False).isfinite().all()
            sq = g.tensor(M * parts, dtype=torch.float32)
            n = ops._EXT.few_add(g.tensor(M, K), g.tensor(H, K), residual, norm, 1.0, rows, sq)
            if norm is None:
                break
            assert 0 < n <= H // 8
    assert residual.isfinite().all()


def test_elementwise_and_cache_guarded(g):
    rows, hidden = 33, 3584
    x = g.tensor(rows, hidden)
    w = g.tensor(hidden)
    res = g.tensor(rows, hidden)
    ops.rmsnorm(x, w, 1e-6, 0.0)
    ops.fused_add_rmsnorm(x, res, w, 1e-6)
    act = g.tensor(rows, 2 * hidden)
    ops.silu_and_mul(act)
    ops.gelu_tanh_and_mul(act)
    # rope + cache write
    T, HQ, HK, D2, BS, NB2 = 29, 16, 8, 256, 16, 40
    from llmq_amd.ops import torch_ref

    cs = torch_ref.build_rope_cache(128, D2, 10000.0, DEV)
    qkv_q = g.tensor(T, HQ, D2)
    qkv_k = g.tensor(T, HK, D2)
    vval = g.tensor(T, HK, D2)
    kc = g.tensor(NB2, HK, BS, D2, fill="zeros")
    vc = g.tensor(NB2, HK, BS, D2, fill="zeros")
    pos = g.from_values(torch.arange(T), torch.int64)
    slots = g.from_values(torch.randperm(NB2 * BS)[:T], torch.int64)
    ops.rope_and_cache(qkv_q, qkv_k, vval, kc, vc, pos, cs, slots)


@pytest.mark.parametrize("B,V", [(64, 50257), (3, 1003), (1, 50000), (2, 1)])
def test_sampler_guarded(g, B, V):
    half = g.tensor(B, V)
    logits = g.tensor(B, V, dtype=torch.float32)
    if half.data_ptr() % 16 == 0 and logits.data_ptr() % 16 == 0:
        ops._EXT.softcap_logits(logits, half, 30.0)
        assert logits.isfinite().all()
    temps = g.tensor(B, dtype=torch.float32, fill="zeros")
    temps.fill_(0.8)
    tps = g.tensor(B, dtype=torch.float32, fill="zeros")
    tps.fill_(0.9)
    tks = g.from_values(torch.full((B,), 50), torch.int64)
    out = g.from_values(torch.zeros(B), torch.int64)
    keys = g.from_values(torch.zeros(B), torch.int64)
    zs = g.from_values(torch.zeros(B), torch.int32)
    bound = g.tensor(B, dtype=torch.float32)
    ops._EXT.topk_topp_bound(bound, logits, temps, tps, tks)
    ops.sample_gumbel_argmax(out, keys, logits, temps, zs, zs, 3, 1, bound)
    assert bool((out >= 0).all()) and bool((out < V).all())
