"""The engine's work on one GPU, as timed cases.

Every case is a step of the serving engine on a preset's real architecture
(random-init weights, all layers): what a worker does between taking jobs from
the queue and sampling their tokens.

  decode   one continuous-batching decode step of a resident batch, through the
           model runner (hipGraph replay of the batch's bucket, then the
           logits of every row)
  prefill  whole prompts through the engine's teacher-forced step, the logits
           of each prompt's last token, and the release of their blocks; a
           prompt over the engine's token budget goes in portions, each on top
           of the cached ones
  sample   the model's head and the fused sampler on a batch's last hidden
           states, with and without top-k/top-p

The models are the ones that the framework's own benchmarks serve: llama-3.2-1b
(head size 64), llama-3.2-3b and tower-plus-2b (128, the latter with query/key/
value biases and 6 query heads per kv head), tower-plus-9b (256, soft caps,
sliding windows, sandwich norms, a vocabulary of 256,000).
"""

from __future__ import annotations

import math

import numpy as np
import torch

from llmq_amd import ops
from llmq_amd.engine.config import EngineConfig
from llmq_amd.engine.engine import LLMEngine
from llmq_amd.engine.model_specs import resolve_spec
from llmq_amd.engine.sampling_params import SamplingParams
from llmq_amd.engine.scheduler import Sequence

BLOCK = 16          # EngineConfig's default KV block
BUDGET = 8192       # EngineConfig's default prefill tokens per step

MODELS = ("llama-3.2-1b", "tower-plus-2b", "llama-3.2-3b", "tower-plus-9b")


def listed():
    return [
        # one interactive request on an engine with the default context length:
        # the smallest call, bound by latency and launches
        dict(name="decode-1b-one", kind="decode", model="llama-3.2-1b", batch=1, context=200,
             ragged=False, kv="auto", max_len=0),
        # a small worker: few requests of very different lengths
        dict(name="decode-2b-few", kind="decode", model="tower-plus-2b", batch=7, context=1900,
             ragged=True, kv="auto", max_len=4096),
        # the batch of the repository's family comparisons
        dict(name="decode-1b-batch", kind="decode", model="llama-3.2-1b", batch=64, context=1040,
             ragged=False, kv="auto", max_len=4096),
        # a worker in steady state: odd batch, lengths spread
        dict(name="decode-3b-steady", kind="decode", model="llama-3.2-3b", batch=189, context=1100,
             ragged=True, kv="auto", max_len=4096),
        # few long documents
        dict(name="decode-3b-long", kind="decode", model="llama-3.2-3b", batch=3, context=16000,
             ragged=True, kv="auto", max_len=32768),
        # the headline model and context, the batch cut to what leaves room
        dict(name="decode-9b-batch", kind="decode", model="tower-plus-9b", batch=96, context=1064,
             ragged=False, kv="auto", max_len=4096),
        # the fp8 cache option
        dict(name="decode-9b-fp8", kind="decode", model="tower-plus-9b", batch=48, context=2000,
             ragged=True, kv="fp8", max_len=4096),
        # a single short prompt: time to first token
        dict(name="prefill-1b-one", kind="prefill", model="llama-3.2-1b", prompts=1, tokens=45,
             ragged=False),
        # an admission step of many short jobs
        dict(name="prefill-2b-short", kind="prefill", model="tower-plus-2b", prompts=40,
             tokens=170, ragged=True),
        # an admission step of ordinary prompts filling the step's token budget
        dict(name="prefill-9b-budget", kind="prefill", model="tower-plus-9b", prompts=8,
             tokens=1024, ragged=False),
        # a long document, in two portions
        dict(name="prefill-3b-long", kind="prefill", model="llama-3.2-3b", prompts=1,
             tokens=11000, ragged=False),
        # head and sampler at the largest vocabulary, with nucleus sampling
        dict(name="sample-9b", kind="sample", model="tower-plus-9b", rows=256, top_p=0.95,
             top_k=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(MODELS)
    big = model == "tower-plus-9b"
    what = rng.random()
    if what < 0.55:
        batch = _log_int(rng, 1, 200)
        context = _log_int(rng, 20, min(16000, (100_000 if not big else 80_000) // batch,
                                        8000 if big else 16000))
        kv = "fp8" if model != "llama-3.2-1b" and rng.random() < 0.25 else "auto"
        return dict(kind="decode", model=model, batch=batch, context=context,
                    ragged=rng.random() < 0.6, kv=kv,
                    max_len=0 if context < 1000 and rng.random() < 0.3
                    else 4096 if context < 4000 else 32768)
    if what < 0.9:
        prompts = _log_int(rng, 1, 64)
        top = (11000 if not big else 7000) if prompts == 1 else BUDGET // prompts
        return dict(kind="prefill", model=model, prompts=prompts, tokens=_log_int(rng, 10, top),
                    ragged=rng.random() < 0.6)
    truncated = rng.random() < 0.5
    return dict(kind="sample", model=model, rows=_log_int(rng, 1, 256),
                top_p=round(rng.uniform(0.5, 0.99), 2) if truncated else 1.0,
                top_k=rng.choice((0, 20, 50)) if truncated else 0)


# ------------------------------------------------------------------ inputs --


def _lengths(case, seed):
    """Tokens per sequence: the largest is the case's, the others of a ragged
    case spread between an eighth of it and all of it. A property of the case
    and not of the seed: every seed is the same amount of work."""
    n, top = (case["batch"], case["context"]) if case["kind"] == "decode" else (
        case["prompts"], case["tokens"])
    if not case["ragged"] or n == 1:
        return [top] * n
    rng = np.random.default_rng(1000 * n + top)
    out = rng.integers(max(1, top // 8), top + 1, size=n).tolist()
    out[int(rng.integers(n))] = top
    return out


def _engine(case, seed, max_seqs, max_len, blocks, graphs):
    return LLMEngine(EngineConfig(
        model=case["model"], max_num_seqs=max_seqs, max_model_len=max_len or None,
        max_prefill_tokens=BUDGET, kv_block_size=BLOCK, num_kv_blocks=blocks,
        kv_cache_dtype=case.get("kv", "auto"), load_weights=False, fast_init=True,
        enforce_eager=not graphs, hipgraph_max_batch=max_seqs, seed=seed, device="cuda",
    ))


def _settle(engine, keys):
    """Make the random weights behave as trained ones do under rounding: a
    stream of unit size to which every sublayer adds about a seventh. (As
    initialised, the first layers ARE the stream, which magnifies each rounding
    on the way down; and attention, an average over `keys` random values, would
    vanish beside the feed-forward, so its output weights grow with them.)"""
    s, W = engine.spec, engine.model.named_tensors()
    if s.post_norms:                                  # norm weights count from one
        for li in range(s.num_layers):
            W[f"layers.{li}.post_attn_norm"].fill_(-0.85)
            W[f"layers.{li}.post_mlp_norm"].fill_(-0.85)
        return
    W["embedding"].mul_(50.0)
    W["final_norm"].mul_(1 / 50.0)
    for li in range(s.num_layers):
        W[f"layers.{li}.o"].mul_(0.7 * math.sqrt(keys))


@torch.no_grad()
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "decode":
        lens = _lengths(case, seed)
        need = [-(-n // BLOCK) for n in lens]
        engine = _engine(case, seed, len(lens), case["max_len"], sum(need) + 8, True)
        _settle(engine, sum(lens) / len(lens))
        # the cached context: keys and values of unit scale in the blocks of a
        # pool that has been in use (no sequence's blocks are in order)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        for k, v in zip(engine.kv_cache.k, engine.kv_cache.v):
            for t in (k, v):
                if t.dtype == torch.bfloat16:
                    t.normal_(generator=gen)
                else:
                    t.copy_(torch.empty(t.shape, dtype=torch.bfloat16,
                                        device="cuda").normal_(generator=gen))
        blocks = engine.allocator.allocate(sum(need))
        blocks = [blocks[i] for i in rng.permutation(len(blocks))]
        seqs, at = [], 0
        for i, (n, nb) in enumerate(zip(lens, need)):
            seq = Sequence(f"r{i}", rng.integers(0, engine.spec.vocab_size, size=n).tolist(),
                           SamplingParams())
            seq.block_table = blocks[at:at + nb]
            seqs.append(seq)
            at += nb
        return dict(case=case, engine=engine, seqs=seqs, want=[[0]] * len(seqs))
    if case["kind"] == "prefill":
        lens = _lengths(case, seed)
        engine = _engine(case, seed, len(lens), max(lens) + BLOCK,
                         sum(-(-n // BLOCK) for n in lens) + 8, False)
        _settle(engine, sum(lens) / len(lens))
        prompts = [rng.integers(0, engine.spec.vocab_size, size=n).tolist() for n in lens]
        return dict(case=case, engine=engine, prompts=prompts)
    engine = _engine(case, seed, case["rows"], 256, 16, False)
    n, dev = case["rows"], "cuda"
    gen = torch.Generator(device=dev).manual_seed(seed)
    temps = rng.uniform(0.3, 1.2, size=n).astype(np.float32)
    temps[rng.random(n) < 0.25] = 0.0                       # greedy rows
    seeds = np.where(rng.random(n) < 0.3, rng.integers(1, 1 << 30, size=n), 0).astype(np.int32)
    return dict(
        case=case, engine=engine,
        hidden=torch.empty(n, engine.spec.hidden_size, dtype=engine.dtype,
                           device=dev).normal_(generator=gen),
        temps=torch.from_numpy(temps).to(dev), seeds=torch.from_numpy(seeds).to(dev),
        pos=torch.from_numpy(rng.integers(0, 500, size=n).astype(np.int32)).to(dev),
        top_ps=torch.full((n,), case["top_p"], dtype=torch.float32, device=dev),
        top_ks=torch.full((n,), case["top_k"], dtype=torch.int64, device=dev),
        out=torch.empty(n, dtype=torch.int64, device=dev),
        keys=torch.empty(n, dtype=torch.int64, device=dev),
    )


# -------------------------------------------------------------------- pass --


@torch.no_grad()
def run(state):
    case, engine = state["case"], state["engine"]
    if case["kind"] == "decode":
        return engine.runner.execute_decode(state["seqs"], want=state["want"])
    if case["kind"] == "prefill":
        prompts = state["prompts"]
        ids = [f"p{i}" for i in range(len(prompts))]
        longest = max(len(p) for p in prompts)
        logits = None
        for at in range(0, longest, BUDGET):            # one step unless over the budget
            end = longest <= at + BUDGET
            entries = [{"id": i, "tokens": p[at:at + BUDGET],
                        "want": [len(p) - at - 1] if end else []}
                       for i, p in zip(ids, prompts)]
            logits = engine.replay_step(entries, end=ids if end else None)
        return logits
    logits = engine.model.compute_logits(state["hidden"])
    bounds = None
    if case["top_p"] < 1.0 or case["top_k"]:
        bounds = ops.topk_topp_bound(logits, state["temps"], state["top_ps"], state["top_ks"])
    ops.sample_gumbel_argmax(state["out"], state["keys"], logits, state["temps"],
                             state["seeds"], state["pos"], 1234, 7, bounds)
    return {"logits": logits, "tokens": state["out"]}


# ------------------------------------------------------- bytes, flops, error --


def work(case):
    """Weights, cached keys and values, fresh ones and logits, each once; the
    products of the layers and the head, and the visible score pairs."""
    s = resolve_spec(case["model"])
    layer = s.hidden_size * (s.q_size + 2 * s.kv_size) + s.q_size * s.hidden_size \
        + 3 * s.hidden_size * s.intermediate_size
    head = s.vocab_size * s.hidden_size
    if case["kind"] == "sample":
        n = case["rows"]
        return {"bytes": 2 * head + 2 * n * s.hidden_size + 4 * n * s.vocab_size + 8 * n,
                "flops": 2 * n * head}
    lens = _lengths(case, 0)
    kv_size = 1 if case.get("kv") == "fp8" else 2
    pairs = cached = 0
    for li in range(s.num_layers):
        win = s.sliding_window if s.layer_uses_sliding_window(li) else 0
        for n in lens:
            if case["kind"] == "decode":
                pairs += min(n, win) if win else n
                cached += min(n, win) if win else n
            elif win and n > win:
                pairs += win * (win + 1) // 2 + (n - win) * win
            else:
                pairs += n * (n + 1) // 2
    tokens = len(lens) if case["kind"] == "decode" else sum(lens)
    if case["kind"] != "decode":
        cached = s.num_layers * tokens
    rows = len(lens)
    return {
        "bytes": 2 * (s.num_layers * layer + head + tokens * s.hidden_size)
        + 2 * s.kv_size * kv_size * cached + 4 * rows * s.vocab_size,
        "flops": 2 * (tokens * s.num_layers * layer + rows * head) + 4 * s.q_size * pairs,
    }


def tolerance(case):
    # Every layer rounds the stream to bf16 twice and its branches more often:
    # exact() finds the whole path 0.010 (16 layers) to 0.018 (42 layers) off, and
    # two versions of it whose projections sum in another order lie 0.010 to
    # 0.021 apart, 0.12 at the largest value. The head alone is 0.0017 off.
    if case["kind"] == "sample":
        return {"rel": 0.006, "max": 0.05, "differ": 0.01}
    return {"rel": 0.03, "max": 0.5}


def _rotate(x, pos, spec):
    """Rotary positions in 64 bits on x [T, H, D]."""
    half = spec.head_dim // 2
    inv = spec.rope_theta ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    sc = spec.rope_scaling
    if sc:                                            # the wavelength remap of Llama 3.1/3.2
        wave = 2 * math.pi / inv
        orig, factor = sc["original_max_position_embeddings"], sc["factor"]
        lo, hi = sc["low_freq_factor"], sc["high_freq_factor"]
        mix = ((orig / wave - lo) / (hi - lo)).clamp(0, 1)
        inv = (1 - mix) * inv / factor + mix * inv
    ang = pos.double()[:, None, None] * inv
    c, sn = ang.cos(), ang.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * sn, b * c + a * sn], dim=-1)


def _attend(q, k, v, i0, spec, window):
    """q [Q, H, D] at positions i0.., k and v [L, KVH, D]: causal, 64 bits."""
    Q, H, D = q.shape
    KVH, G = k.shape[1], H // k.shape[1]
    out = torch.empty_like(q)
    j = torch.arange(k.shape[0], device=q.device)
    for at in range(0, Q, 1024):
        i = torch.arange(at, min(Q, at + 1024), device=q.device) + i0
        dead = j[None] > i[:, None]
        if window:
            dead |= i[:, None] - j[None] >= window
        for g in range(KVH):
            qq = q[at:at + 1024, g * G:(g + 1) * G].transpose(0, 1).reshape(-1, D)
            s = (qq @ k[:, g].t().contiguous()) * spec.scale
            if spec.attn_softcap:
                s = torch.tanh(s / spec.attn_softcap) * spec.attn_softcap
            s = s.view(G, len(i), -1).masked_fill_(dead, float("-inf")).softmax(-1)
            o = s.view(G * len(i), -1) @ v[:, g].contiguous()
            out[at:at + 1024, g * G:(g + 1) * G] = o.view(G, len(i), D).transpose(0, 1)
    return out


@torch.no_grad()
def exact(case, seed):
    if case["kind"] != "sample" and work(case)["flops"] > 1.6e14:
        return None                                    # minutes in 64 bits
    state = prepare(case, seed)
    engine, spec = state["engine"], state["engine"].spec
    W, dev = engine.model.named_tensors(), "cuda"
    off = 1.0 if spec.family == "gemma2" else 0.0

    def linear(x, w):
        w = W[w]
        if w.shape[0] * x.shape[0] < 1 << 28:
            return x @ w.double().t()
        return torch.cat([x @ w[a:a + 32768].double().t() for a in range(0, w.shape[0], 32768)], -1)

    def norm(x, name):
        inv = torch.rsqrt(x.square().mean(-1, keepdim=True) + spec.rms_eps)
        return x * inv * (W[name].double() + off)

    def head(h):
        logits = linear(h, "embedding" if spec.tied_embeddings else "lm_head")
        cap = spec.final_softcap
        return torch.tanh(logits / cap) * cap if cap else logits

    if case["kind"] == "sample":
        return {"logits": head(state["hidden"].double()), "tokens": None}
    decode = case["kind"] == "decode"
    if decode:
        lens = [s.num_tokens for s in state["seqs"]]
        ids = [s.token_ids[-1] for s in state["seqs"]]
        pos = torch.tensor([n - 1 for n in lens], device=dev)
        tables = [torch.tensor(s.block_table, device=dev) for s in state["seqs"]]
    else:
        lens = [len(p) for p in state["prompts"]]
        ids = [t for p in state["prompts"] for t in p]
        pos = torch.cat([torch.arange(n, device=dev) for n in lens])
    T = len(ids)
    x = W["embedding"][torch.tensor(ids, device=dev)].double()
    if spec.embedding_scale:
        x = x * math.sqrt(spec.hidden_size)
    for li in range(spec.num_layers):
        p = f"layers.{li}."
        win = spec.sliding_window if spec.layer_uses_sliding_window(li) else 0
        qkv = linear(norm(x, p + "input_norm"), p + "qkv")
        if spec.qkv_bias:
            qkv = qkv + W[p + "qkv_bias"].double()
        q, k, v = qkv.split([spec.q_size, spec.kv_size, spec.kv_size], -1)
        q = _rotate(q.reshape(T, -1, spec.head_dim), pos, spec)
        k = _rotate(k.reshape(T, -1, spec.head_dim), pos, spec)
        v = v.reshape(T, -1, spec.head_dim)
        attn, at = torch.empty_like(q), 0
        for b, n in enumerate(lens):
            if decode:
                kc, vc = (c[li][tables[b]].double().transpose(1, 2).reshape(-1, *k.shape[1:])[:n]
                          for c in (engine.kv_cache.k, engine.kv_cache.v))
                kc[n - 1], vc[n - 1] = k[b], v[b]
                attn[b:b + 1] = _attend(q[b:b + 1], kc, vc, n - 1, spec, win)
            else:
                attn[at:at + n] = _attend(q[at:at + n], k[at:at + n], v[at:at + n], 0, spec, win)
                at += n
        y = linear(attn.reshape(T, -1), p + "o")
        x = x + (norm(y, p + "post_attn_norm") if spec.post_norms else y)
        gate, up = linear(norm(x, p + "pre_mlp_norm"), p + "gate_up").chunk(2, -1)
        act = torch.nn.functional.gelu(gate, approximate="tanh") if spec.gelu \
            else torch.nn.functional.silu(gate)
        y = linear(act * up, p + "down")
        x = x + (norm(y, p + "post_mlp_norm") if spec.post_norms else y)
    if not decode:
        x = x[torch.tensor(np.cumsum(lens) - 1, device=dev)]
    return head(norm(x, "final_norm"))
