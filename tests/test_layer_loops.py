"""The layer loops of the Llama, Qwen2 and Gemma-2 families against a 64-bit
forward pass: few rows (few_rows), up to 256 (slabs), prompts launched from
native code (prompt_layers) and the per-operation loop, with tiles and without, for
decode steps, whole prompts, portions that continue a cached context and mixed steps. Three layers of
sizes that the streaming kernels take, norm weights and biases that differ
everywhere, so that a swapped or missing one shows.
"""

from __future__ import annotations

import dataclasses

import pytest
import torch

from llmq_amd import ops
from llmq_amd.engine.config import EngineConfig
from llmq_amd.engine.kv_cache import KVCache
from llmq_amd.engine.model_runner import ModelRunner
from llmq_amd.engine.model_specs import resolve_spec
from llmq_amd.engine.models import llama
from llmq_amd.engine.models.llama import CausalLM
from llmq_amd.engine.sampling_params import SamplingParams
from llmq_amd.engine.scheduler import ScheduledBatch, Sequence

BLOCK, BLOCKS, VOCAB = 16, 2048, 512

SPECS = {
    "llama": dataclasses.replace(
        resolve_spec("tiny-llama"), hidden_size=256, intermediate_size=384, num_layers=3,
        num_heads=4, num_kv_heads=2, head_dim=64),
    "qwen2": dataclasses.replace(
        resolve_spec("tiny-qwen2"), hidden_size=384, intermediate_size=640, num_layers=3,
        num_heads=6, num_kv_heads=1, head_dim=128),
    "gemma2": dataclasses.replace(
        resolve_spec("tiny-gemma2"), hidden_size=256, intermediate_size=384, num_layers=3,
        num_heads=4, num_kv_heads=2, head_dim=128, sliding_window=24, attn_softcap=5.0,
        attn_scale=None),
}

# A row passes some 36 roundings to bf16 (twelve a layer, relative errors of 2^-9
# 3^-0.5 rms), which add up in squares to 0.7 % where none is magnified; three times
# that is allowed. A planted mistake moves the logits by more than twice the limit
# (test_planted_mistakes_show).
LIMIT = 0.02


def _model(name, device, dtype):
    spec = SPECS[name]
    model = CausalLM(spec, torch.device(device), dtype)
    gen = torch.Generator().manual_seed(5)
    for key, t in model.named_tensors().items():
        r = torch.randn(t.shape, generator=gen)
        if t.dim() == 2 and key != "embedding":
            r *= t.shape[1] ** -0.5
        elif key == "embedding":
            r *= spec.hidden_size ** -0.5 if spec.embedding_scale else 1.0
        elif key.endswith("norm"):
            r = 0.4 * r + (0.0 if spec.family == "gemma2" else 1.0)
        t.copy_(r.to(t.dtype))
    return model


def _cache(spec, device, dtype):
    cache = KVCache(spec.num_layers, BLOCKS, spec.num_kv_heads, BLOCK, spec.head_dim,
                    torch.device(device), dtype)
    gen = torch.Generator().manual_seed(6)
    for t in cache.k + cache.v:
        t.copy_(torch.randn(t.shape, generator=gen).to(torch.bfloat16).to(dtype))
    return cache


def _batch(kind, rows):
    """A step of `rows` rows: decode rows on contexts up to 90, prompts and portions in
    up to three sequences."""
    gen = torch.Generator().manual_seed(rows)
    free = (torch.randperm(BLOCKS - 1, generator=gen) + 1).tolist()

    def seq(n):
        s = Sequence("r", torch.randint(0, VOCAB, (n,), generator=gen).tolist(),
                     SamplingParams())
        s.block_table = [free.pop() for _ in range(-(-n // BLOCK))]
        return s

    nd = {"decode": rows, "mixed": max(1, rows // 3)}.get(kind, 0)
    seqs = [seq(90 if i == 0 else 1 + i * 7 % 60) for i in range(nd)]
    left, cuts = rows - nd, []
    for part, past in ((left // 2, 21), (left // 3, 0), (left - left // 2 - left // 3, 40)):
        if part:
            start = 0 if kind == "prompt" else past
            seqs.append(seq(start + part))
            cuts.append((start, start + part))
    return ScheduledBatch(kind="prefill" if kind in ("prompt", "portion") else kind, seqs=seqs,
                          n_decode=nd, chunks=cuts)


def _run(model, cache, batch):
    spec = model.spec
    runner = ModelRunner(model, cache, EngineConfig(enforce_eager=True),
                         model.device, spec.max_position_embeddings)
    want = [[0]] * batch.n_decode + [list(range(e - st)) for st, e in batch.chunks]
    if batch.kind == "decode":
        return runner.execute_decode(batch.seqs, want=want)
    if batch.kind == "mixed":
        return runner.execute_mixed(batch, want=want)
    return runner.execute_prefill(batch.seqs, batch.chunks, want=want)


def _oracle(model, cache, batch, plant=""):
    """The step in 64 bits on the CPU; the cache as it was before the step."""
    s = model.spec
    W = {k: t.detach().cpu().double() for k, t in model.named_tensors().items()}
    kc, vc = ([t.detach().cpu().double() for t in c] for c in (cache.k, cache.v))
    low = cache.k[0].dtype if cache.k[0].dtype == torch.float8_e4m3fn else torch.float64
    off = 1.0 if s.family == "gemma2" else 0.0
    spans = [(q.num_tokens - 1, q.num_tokens) for q in batch.seqs[:batch.n_decode]] + batch.chunks
    ids = [t for q, (a, e) in zip(batch.seqs, spans) for t in q.token_ids[a:e]]
    pos = torch.cat([torch.arange(a, e) for a, e in spans])
    if plant == "position":
        pos = pos + 1
    if plant == "norms":
        W["layers.1.input_norm"], W["layers.1.pre_mlp_norm"] = \
            W["layers.1.pre_mlp_norm"], W["layers.1.input_norm"]
    if plant == "next_norm":
        W["layers.2.input_norm"] = W["layers.1.input_norm"]
    if plant == "bias":
        W["layers.1.qkv_bias"] = torch.zeros_like(W["layers.1.qkv_bias"])
    half = s.head_dim // 2
    ang = pos.double()[:, None, None] * s.rope_theta ** (
        -torch.arange(half, dtype=torch.float64) / half)

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + s.rms_eps) * (W[w] + off)

    def rotate(x):
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)

    x = W["embedding"][ids]
    if s.embedding_scale:
        x = x * s.hidden_size ** 0.5
    T, G = len(ids), s.num_heads // s.num_kv_heads
    for li in range(s.num_layers):
        p = f"layers.{li}."
        win = s.sliding_window if s.layer_uses_sliding_window(li) else 0
        if plant == "window":
            win = 0
        qkv = norm(x, p + "input_norm") @ W[p + "qkv"].t()
        if s.qkv_bias:
            qkv = qkv + W[p + "qkv_bias"]
        q, k, v = (t.reshape(T, -1, s.head_dim)
                   for t in qkv.split([s.q_size, s.kv_size, s.kv_size], -1))
        q, k = rotate(q), rotate(k)
        attn, at = torch.empty_like(q), 0
        for b, (seq, (a, e)) in enumerate(zip(batch.seqs, spans)):
            n = e - a
            table = torch.tensor(seq.block_table)
            kk, vv = (c[li][table].transpose(1, 2).reshape(-1, s.num_kv_heads, s.head_dim)[:e]
                      .clone() for c in (kc, vc))
            # a decode row's own key and value come from the cache as it stores them
            held = low if b < batch.n_decode else torch.float64
            kk[a:], vv[a:] = (t[at:at + n].to(held).double() for t in (k, v))
            i, j = torch.arange(a, e)[:, None], torch.arange(e)[None]
            dead = (j > i) | ((i - j >= win) if win else False)
            sc = torch.einsum("ihd,jhd->hij", q[at:at + n], kk.repeat_interleave(G, 1)) * s.scale
            if s.attn_softcap and plant != "cap":
                sc = torch.tanh(sc / s.attn_softcap) * s.attn_softcap
            pr = sc.masked_fill(dead, float("-inf")).softmax(-1)
            attn[at:at + n] = torch.einsum("hij,jhd->ihd", pr, vv.repeat_interleave(G, 1))
            at += n
        y = attn.reshape(T, -1) @ W[p + "o"].t()
        x = x + (norm(y, p + "post_attn_norm") if s.post_norms and plant != "sandwich" else y)
        g, u = (norm(x, p + "pre_mlp_norm") @ W[p + "gate_up"].t()).chunk(2, -1)
        if plant == "halves":
            g, u = u, g
        act = torch.nn.functional.gelu(g, approximate="tanh") if s.gelu \
            else torch.nn.functional.silu(g)
        y = (act * u) @ W[p + "down"].t()
        x = x + (norm(y, p + "post_mlp_norm") if s.post_norms else y)
    logits = norm(x, "final_norm") @ W["embedding" if s.tied_embeddings else "lm_head"].t()
    return torch.tanh(logits / s.final_softcap) * s.final_softcap if s.final_softcap else logits


def _off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


# ------------------------------------------------------------------- on the CPU --


@pytest.mark.parametrize("kind", ["decode", "prompt", "portion", "mixed"])
@pytest.mark.parametrize("name", list(SPECS))
def test_oracle_matches_fp32_model(name, kind):
    """32-bit sums of the CPU path against the oracle."""
    model = _model(name, "cpu", torch.float32)
    cache, batch = _cache(model.spec, "cpu", torch.float32), _batch(kind, 23)
    want = _oracle(model, cache, batch)
    assert _off(_run(model, cache, batch), want) < 2e-5


@pytest.mark.parametrize("name,plant", [
    ("llama", "norms"), ("llama", "next_norm"), ("llama", "position"), ("llama", "halves"),
    ("qwen2", "bias"), ("gemma2", "norms"), ("gemma2", "sandwich"), ("gemma2", "window"),
    ("gemma2", "cap"),
])
def test_planted_mistakes_show(name, plant):
    """What each kind of mistake moves the logits by, in the oracle."""
    model = _model(name, "cpu", torch.float32)
    cache, batch = _cache(model.spec, "cpu", torch.float32), _batch("decode", 16)
    good = _oracle(model, cache, batch)
    assert _off(_oracle(model, cache, batch, plant), good) > 2 * LIMIT


# ------------------------------------------------------------------- on the GPU --

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]
on_gpu = lambda f: gpu[0](gpu[1](f))  # noqa: E731
LOOPS = {"_forward_few_rows": "few", "_forward_slabs": "slabs", "_prompt_layers": "native"}


@pytest.fixture()
def loops(monkeypatch):
    """Names of the loops that forward passes enter."""
    taken = []
    for method, short in LOOPS.items():
        def spy(self, *args, _f=getattr(CausalLM, method), _short=short):
            taken.append(_short)
            return _f(self, *args)
        monkeypatch.setattr(CausalLM, method, spy)
    return taken


def _expected(kind, rows, fp8):
    if rows <= 16:
        return ["few"]
    if kind == "prompt" or (kind == "portion" and not fp8):   # fp8 portions are gathered
        return ["native"]
    return ["slabs"] if rows <= 256 else []


@pytest.fixture()
def products(monkeypatch):
    """The streaming and tile products that the Python loops call."""
    taken = []
    for op, short in (("ring_linear", "ring"), ("ring_act_linear", "ring_act"),
                      ("tile_act_linear", "tile")):
        def spy(*args, _f=getattr(ops, op), _short=short):
            taken.append(_short)
            return _f(*args)
        monkeypatch.setattr(ops, op, spy)
    return taken


def _expected_products(name, rows):
    """Over 16 rows, three layers. Tiles pay from some 540 rows of llama's and gemma2's 768
    gate and value rows on, from 1440 of qwen2's 1280."""
    if rows <= 256:
        return ["ring", "ring", "ring_act", "ring"] * 3
    return ["tile"] * 3 if rows >= 600 and name != "qwen2" else []


@on_gpu
@pytest.mark.parametrize("rows", [1, 5, 16, 17, 65, 128, 129, 192, 256, 257, 600])
@pytest.mark.parametrize("kind", ["decode", "prompt", "portion", "mixed"])
@pytest.mark.parametrize("name,fp8", [("llama", False), ("qwen2", False), ("gemma2", False),
                                      ("qwen2", True), ("gemma2", True)])
def test_loops_vs_64_bits(name, fp8, kind, rows, loops, products, monkeypatch):
    if kind == "mixed":
        rows = max(rows, 2)
    model = _model(name, "cuda", torch.bfloat16)
    cache = _cache(model.spec, "cuda", torch.float8_e4m3fn if fp8 else torch.bfloat16)
    batch = _batch(kind, rows)
    want = _oracle(model, cache, batch)
    got = _run(model, cache, batch)
    assert loops == _expected(kind, rows, fp8)
    assert _off(got, want) < LIMIT
    if loops == ["native"]:
        # the same launches as the slab loop's, or as the per-operation loop's
        monkeypatch.setattr(CausalLM, "_prompt_layers", CausalLM._forward_slabs if rows <= 256
                            else CausalLM._forward_general)
        assert torch.equal(_run(model, cache, batch), got)
        assert loops[1:] == (["slabs"] if rows <= 256 else [])
    assert products == ([] if rows <= 16 else _expected_products(name, rows))


@on_gpu
@pytest.mark.parametrize("kind,rows", [("decode", 1), ("decode", 16), ("decode", 33),
                                       ("prompt", 7), ("prompt", 40), ("mixed", 9)])
def test_skinny_gemm_switch(kind, rows, loops, monkeypatch):
    """LLMQ_SKINNY_GEMM=1 puts every projection of a step on that kernel."""
    calls = []
    monkeypatch.setattr(llama, "_USE_SKINNY_GEMM", True)
    skinny = ops.skinny_gemm
    monkeypatch.setattr(ops, "skinny_gemm", lambda *a: calls.append(a[1].shape) or skinny(*a))
    model = _model("llama", "cuda", torch.bfloat16)
    cache, batch = _cache(model.spec, "cuda", torch.bfloat16), _batch(kind, rows)
    want = _oracle(model, cache, batch)
    got = _run(model, cache, batch)
    assert loops == [] and len(calls) == 4 * model.spec.num_layers + 1
    assert _off(got, want) < LIMIT


def _layouts(w):
    """The same weights as a transposed view, with padded rows, off a 16-byte boundary."""
    padded = torch.zeros(w.shape[0], w.shape[1] + 8, dtype=w.dtype, device=w.device)
    padded[:, :w.shape[1]] = w
    moved = torch.zeros(w.numel() + 4, dtype=w.dtype, device=w.device)
    moved[4:] = w.reshape(-1)
    return [w.t().contiguous().t(), padded[:, :w.shape[1]], moved[4:].view(w.shape)]


@on_gpu
@pytest.mark.parametrize("kind,rows", [("decode", 5), ("decode", 16), ("decode", 33),
                                       ("decode", 65), ("decode", 129), ("prompt", 16),
                                       ("prompt", 40), ("portion", 200), ("mixed", 9)])
@pytest.mark.parametrize("layer", [0, 1])
@pytest.mark.parametrize("name", ["llama", "qwen2", "gemma2"])
def test_weight_layouts(name, layer, kind, rows):
    """Weights of one layer that are no packed, aligned matrices."""
    model = _model(name, "cuda", torch.bfloat16)
    cache, batch = _cache(model.spec, "cuda", torch.bfloat16), _batch(kind, rows)
    want = _oracle(model, cache, batch)
    lw = model.layers[layer]
    for turn in range(3):
        for i, which in enumerate(("qkv", "o", "gate_up", "down")):
            setattr(lw, which, _layouts(getattr(lw, which))[(i + turn) % 3])
        assert _off(_run(model, cache, batch), want) < LIMIT


@on_gpu
@pytest.mark.parametrize("kind,rows", [("decode", 1), ("decode", 12), ("decode", 33),
                                       ("prompt", 40), ("mixed", 9)])
@pytest.mark.parametrize("name", ["qwen2", "gemma2"])
def test_vector_layouts(name, kind, rows):
    """A bias that is a strided view, norm weights 8 bytes off a 16-byte boundary."""
    model = _model(name, "cuda", torch.bfloat16)
    cache, batch = _cache(model.spec, "cuda", torch.bfloat16), _batch(kind, rows)
    want = _oracle(model, cache, batch)
    lw = model.layers[1]
    for which in ("input_norm", "pre_mlp_norm", "post_attn_norm", "post_mlp_norm"):
        if getattr(lw, which) is not None:
            setattr(lw, which, torch.cat([getattr(lw, which)[:4], getattr(lw, which)])[4:])
    if lw.qkv_bias is not None:
        lw.qkv_bias = lw.qkv_bias.repeat_interleave(2)[::2]
    assert _off(_run(model, cache, batch), want) < LIMIT


def test_few_rows_limit():
    """Fewer rows of larger layers, two at the least; the layers of llama-3.2-1b (61 M
    weights), -3b (101 M) and qwen2.5-72b (877 M)."""
    assert [ops.few_rows_limit(n) for n in (61_000_000, 101_000_000, 877_000_000, 1)] == [
        13, 7, 2, 800_000_000]


@on_gpu
@pytest.mark.parametrize("rows", [3, 4, 16])
@pytest.mark.parametrize("kind", ["decode", "prompt", "portion", "mixed"])
@pytest.mark.parametrize("name,fp8", [("llama", False), ("qwen2", True), ("gemma2", False)])
def test_few_rows_of_large_layers(name, fp8, kind, rows, loops, monkeypatch):
    """Rows over a layer's limit: the slab kernels' loops, here with a limit of three."""
    monkeypatch.setattr(ops, "few_rows_limit", lambda n: 3)
    model = _model(name, "cuda", torch.bfloat16)
    cache = _cache(model.spec, "cuda", torch.float8_e4m3fn if fp8 else torch.bfloat16)
    batch = _batch(kind, rows)
    want = _oracle(model, cache, batch)
    got = _run(model, cache, batch)
    assert loops == (["few"] if rows == 3 else _expected(kind, 17, fp8))
    assert _off(got, want) < LIMIT
