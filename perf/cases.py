"""Cases for timing the forward step as the users of this backend run it: an engine's decode step over
a continuous batch (one lane to a full batch), a packed batch that brings prompt chunks, and the
sampling of a step's logits, each through the public entry points (`DecodeSession.step`,
`PackedStep.run`, `Backend.submit` / `wait` / `read`).

A case is a plain dict.  `kind` "decode" and "packed" are whole steps of a model:

  model    one of the shapes in forja_amd/model.py; `layers` of its layers are built (a layer is the
           unit of the work; the small model and the engine's single-lane case have all of them)
  dtypes   "bf16": bf16 activations and KV cache (the dense engine); "engine": f32 activations, f16
           KV cache, 8-bit router (the qwen3-coder engine)
  lanes    decode rows, one per sequence; their cached contexts are spread log-uniformly over
           ctx_lo..ctx_hi
  by_lane  decode attention recorded lane by lane with the standard ops, as the engines record it,
           instead of as the one packed op
  rows, chunks, prefix   prompt tokens of the batch, the ragged chunks they are cut into, and the
           tokens of each of those sequences that are cached already (a continued prompt)
  head     whether the step ends in lm_head and argmax over every row (prompt chunks other than a
           prompt's last need neither)

Weights follow the repository's zero-mean law (a dequantised weight has no common sign, as in trained
weights; tokens then depend on the lane), the router of a mixture model reads seeded N(0,1) logits,
so that the choice of experts is spread as in real use and does not hang on the last bit of an
activation.  KV caches hold N(0,1) values in shuffled pages.

`kind` "sample" is what follows a step in a server that samples: the logits of a batch, one
parameter set, one token per row, with the greedy choice beside it.
"""
import math
from dataclasses import replace

import numpy as np
import torch

from forja_amd import programs
from forja_amd.core import CommandList, DType, Op
from forja_amd.hip_backend import HipBackend
from forja_amd.model import (DENSE_27B, QWEN3_0_6B, QWEN3_CODER_30B_A3B, DecodeSession, Model,
                             PackedStep, record_step)

CONFIGS = {"qwen3-0.6b": QWEN3_0_6B, "coder-30b-a3b": QWEN3_CODER_30B_A3B, "dense-27b": DENSE_27B}
VOCAB = QWEN3_0_6B.vocab


def _decode(name, model, layers, dtypes, lanes, ctx_lo, ctx_hi, by_lane=False):
    return {"name": name, "kind": "decode", "model": model, "layers": layers, "dtypes": dtypes,
            "lanes": lanes, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "by_lane": by_lane}


def _packed(name, model, layers, dtypes, rows, chunks, prefix, lanes, ctx_lo, ctx_hi, head):
    return {"name": name, "kind": "packed", "model": model, "layers": layers, "dtypes": dtypes,
            "rows": rows, "chunks": chunks, "prefix": prefix, "lanes": lanes, "ctx_lo": ctx_lo,
            "ctx_hi": ctx_hi, "head": head}


def _sample(name, rows, dtype, temperature, top_k, top_p):
    return {"name": name, "kind": "sample", "rows": rows, "dtype": dtype, "temperature": temperature,
            "top_k": top_k, "top_p": top_p}


def listed():
    return [
        # One user chats with the small model: a few microseconds of work per kernel, so latency.
        _decode("chat_0.6b_1", "qwen3-0.6b", 28, "bf16", 1, 400, 400),
        # A small batch of the small model at an odd size.
        _decode("chat_0.6b_23", "qwen3-0.6b", 28, "bf16", 23, 60, 3000),
        # One coding assistant, the engine's own dtypes and recording, at full depth.
        _decode("coder_engine_1", "coder-30b-a3b", 48, "engine", 1, 6000, 6000, True),
        # The most lanes the reference's engine batches.
        _decode("coder_engine_8", "coder-30b-a3b", 24, "engine", 8, 256, 32768, True),
        # The headline batch: 128 lanes of very different contexts.
        _decode("coder_128", "coder-30b-a3b", 12, "bf16", 128, 256, 32768),
        # A decode batch of the dense model.
        _decode("dense27_48", "dense-27b", 4, "bf16", 48, 128, 4096),
        # The reference's own prompt benchmark, 512 tokens through the engine's dtypes.
        _packed("coder_engine_prompt_512", "coder-30b-a3b", 6, "engine", 512, 1, 0, 0, 1, 1, False),
        # Prompt chunks of a mixture model beside a decode batch.
        _packed("coder_prompt_2048", "coder-30b-a3b", 8, "bf16", 2048, 3, 1024, 32, 256, 8192, False),
        # A short question arrives while a few sequences decode.
        _packed("dense27_prompt_90", "dense-27b", 4, "bf16", 90, 1, 0, 5, 128, 4096, True),
        # The small model over a packed batch of chunks and decode rows, logits for every row.
        _packed("packed_0.6b_2048", "qwen3-0.6b", 28, "bf16", 2000, 4, 0, 48, 128, 4096, True),
        # A full prefill chunk of the dense model with its decode rows.
        _packed("dense27_prefill_8256", "dense-27b", 2, "bf16", 8192, 6, 0, 64, 128, 4096, False),
        # Sampling a full batch with the parameters such models are served with.
        _sample("sample_128", 128, "bf16", 0.7, 20, 0.8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "packed", "packed", "packed", "sample"])
    if kind == "sample":
        return _nameless(_sample("", _log_uniform(rng, 1, 128), rng.choice(["bf16", "f32"]),
                                 rng.choice([0.6, 0.7, 1.0]), rng.choice([0, 20, 40, 64]),
                                 rng.choice([0.8, 0.95, 1.0])))
    model = rng.choice(list(CONFIGS))
    layers = {"qwen3-0.6b": rng.randint(6, 14), "coder-30b-a3b": rng.randint(3, 8), "dense-27b": rng.randint(1, 2)}[model]
    dtypes = rng.choice(["bf16", "bf16", "engine"]) if model == "coder-30b-a3b" else "bf16"
    ctx_lo = _log_uniform(rng, 40, 1000)
    ctx_hi = _log_uniform(rng, ctx_lo, 32768 if model == "coder-30b-a3b" else 8192)
    if kind == "decode":
        lanes = _log_uniform(rng, 1, 8 if dtypes == "engine" else 128)
        return _nameless(_decode("", model, layers, dtypes, lanes, ctx_lo, ctx_hi, dtypes == "engine"))
    rows = _log_uniform(rng, 24, 1024 if dtypes == "engine" else 3000 if model == "coder-30b-a3b" else 6000)
    head = rows <= 300 and rng.random() < 0.5
    if model == "qwen3-0.6b":
        head = rows <= 1500
    return _nameless(_packed("", model, layers, dtypes, rows, rng.randint(1, min(6, rows // 12)),
                             rng.choice([0, 0, _log_uniform(rng, 40, 8000)]), rng.randint(0, 64), ctx_lo,
                             min(ctx_hi, 8192), head))


def _nameless(case):
    del case["name"]
    return case


def _config(case):
    config = CONFIGS[case["model"]]
    if case["dtypes"] == "engine":
        return replace(config, activation_dtype=DType.F32, kv_dtype=DType.F16, router_bits=8)
    return config


def _contexts(case):
    """The decode lanes' cached tokens: evenly spread over the logarithm of ctx_lo..ctx_hi."""
    lo, hi, n = math.log(case["ctx_lo"]), math.log(case["ctx_hi"]), case["lanes"]
    return [int(round(math.exp(lo + (hi - lo) * (i + 0.5) / n))) for i in range(n)]


def _counts(case):
    """Ragged lengths of the prompt chunks: in proportion 2 : 3 : 4 : .., the last takes the rest."""
    chunks, rows = case["chunks"], case["rows"]
    total = sum(range(2, chunks + 2))
    counts = [max(1, rows * (i + 2) // total) for i in range(chunks - 1)]
    return counts + [rows - sum(counts)]


class _Backend(HipBackend):
    """Notes what a state allocates, so that it can be given back with the state."""
    notes = None

    def alloc(self, dtype, shape):
        tensor = super().alloc(dtype, shape)
        if self.notes is not None:
            self.notes[tensor.buffer] = tensor
        return tensor

    def release(self, tensor):
        if self.notes is not None:
            self.notes.pop(tensor.buffer, None)
        super().release(tensor)


_backend = None


def _the_backend():
    """One backend for the process, as a serving host has."""
    global _backend
    if _backend is None:
        _backend = _Backend(0)
    return _backend


def _to_torch(raw, dtype, shape):
    kind = {DType.F32: torch.float32, DType.F16: torch.float16, DType.BF16: torch.bfloat16,
            DType.U32: torch.int32}[dtype]
    return torch.frombuffer(bytearray(raw), dtype=kind).reshape(shape)


class _State:
    def __init__(self, backend):
        self.backend, self.tensors = backend, {}
        self.outputs = {}           # name -> function that reads it

    def __del__(self):
        backend, tensors = self.backend, self.tensors
        self.tensors = {}
        if backend._handle is not None:
            for tensor in tensors.values():
                backend.release(tensor)

    def reads(self, name, tensor):
        self.outputs[name] = lambda: _to_torch(self.backend.read(tensor), tensor.dtype, tensor.shape)


class _Outputs(dict):
    """The step's outputs.  They are buffers of the state on the device, complete when `run` has
    returned; looking one up reads it (a program that has sampled on the device never reads the
    logits, so a pass does not carry that copy)."""

    def __init__(self, state):
        super().__init__((name, None) for name in state.outputs)
        self.state = state

    def __getitem__(self, name):
        return self.state.outputs[name]()


def _new_rows(backend, cache, config, contexts, counts, pools):
    """The rows the step has stored: [layers, tokens, kv heads, head_dim], read page by page."""
    row = config.kv_heads * config.head_dim * config.kv_dtype.byte_size
    parts = []
    for pool in pools:
        for lane, (start, count) in enumerate(zip(contexts, counts)):
            at, end = int(start), int(start + count)
            while at < end:
                page, slot = divmod(at, config.page_tokens)
                n = min(config.page_tokens - slot, end - at)
                first = (cache.lane_pages[lane][page] * config.page_tokens + slot) * row
                parts.append(backend.read_buffer_range(pool.buffer, first, first + n * row))
                at += n
    return _to_torch(b"".join(parts), config.kv_dtype,
                     (len(pools), int(sum(counts)), config.kv_heads, config.head_dim))


def _settle(backend, model, seed):
    """Larger embeddings and smaller projections back into the residual stream than the seeded law
    gives: in a trained model a layer changes the stream a little.  (With every layer as large as the
    stream, rounding differences grow from layer to layer until outputs cannot be compared.)"""
    center = backend.prepare_program(programs.centered_bias_elements(4))
    fill = CommandList()
    scaled = [(model.embed, 0.1, 2.0)]
    scaled += [(linear, 1e-4, 2e-3) for layer in model.layers for linear in (layer.o_proj, layer.down)]
    for index, (linear, lo, hi) in enumerate(scaled):
        noise = backend.alloc(DType.BF16, linear.biases.shape)
        fill.dispatch(Op.fill_seeded(1, seed, 5000 + 2 * index, lo=lo, hi=hi), [], linear.scales)
        fill.dispatch(Op.fill_seeded(1, seed, 5001 + 2 * index, lo=-lo, hi=lo), [], noise)
        fill.dispatch_kernel(center, [linear.scales, noise], [linear.biases])
        scaled[index] = noise
    backend.submit(fill).wait()
    for noise in scaled:
        backend.release(noise)


def _prepare_step(case, seed, backend, state):
    config = _config(case)
    model = Model(backend, config, seed=seed, layers=case["layers"], weight_law="zero_mean")
    _settle(backend, model, seed)
    rng = np.random.default_rng(seed)
    noise = seed + 1 if config.moe else None
    contexts = _contexts(case)
    rng.shuffle(contexts)
    if case["kind"] == "decode":
        counts = [1] * case["lanes"]
        session = DecodeSession(model, contexts, seed=seed, lane_by_lane=case["by_lane"],
                                router_noise_seed=noise)
        state.session, state.by_lane = session, case["by_lane"]
        state.ids = rng.integers(0, config.vocab, case["lanes"]).astype(np.uint32)
        head = True
    else:
        contexts += [case["prefix"]] * case["chunks"]
        counts = [1] * case["lanes"] + _counts(case)
        head = case["head"]
        session = PackedStep(model, contexts, counts, seed=seed, head=head)
        if noise is not None:
            session.commands = CommandList()
            record_step(model, session.cache, session.buffers, session.commands, head=head,
                        router_noise_seed=noise)
            session.encoded = backend.encode(session.commands)
        state.step = session
    state.contexts = np.array(contexts, dtype=np.int64)
    buffers, cache = session.buffers, session.cache
    if head:
        state.reads("logits", buffers.logits)
    else:
        state.reads("normalized", buffers.normalized[0])
    state.reads("hidden", buffers.hidden[0])
    for name, pools in (("keys", cache.keys), ("values", cache.values)):
        state.outputs[name] = lambda pools=pools: _new_rows(backend, cache, config, contexts, counts, pools)


def _prepare_sample(case, seed, backend, state):
    rows = case["rows"]
    dtype = DType.F32 if case["dtype"] == "f32" else DType.BF16
    generator = torch.Generator(device="cuda").manual_seed(seed)
    # logits of a trained model: most tokens far below the few that a context makes likely
    values = torch.randn((rows, VOCAB), generator=generator, device="cuda") * 2.0
    likely = torch.randint(0, VOCAB, (rows, 40), generator=generator, device="cuda")
    lift = torch.rand((rows, 40), generator=generator, device="cuda") * 8.0
    values = values.scatter_add(1, likely, lift + 4.0)
    values = values if dtype == DType.F32 else values.to(torch.bfloat16).view(torch.int16)
    logits = backend.alloc(dtype, (rows, VOCAB))
    backend.write_array(logits, values.cpu().numpy())
    words = np.zeros(5, np.uint32)
    words[0:1] = np.array([case["temperature"]], np.float32).view(np.uint32)
    words[2:3] = np.array([case["top_p"]], np.float32).view(np.uint32)
    words[1], words[3], words[4] = case["top_k"], seed & 0xffffffff, 17
    params = backend.alloc(DType.U32, (5,))
    backend.write_array(params, words)
    state.sampled, state.greedy = backend.alloc(DType.U32, (rows,)), backend.alloc(DType.U32, (rows,))
    commands = CommandList()
    commands.dispatch(Op.sample(4000), [logits, params], state.sampled)
    commands.dispatch(Op.argmax(), [logits], state.greedy)
    state.encoded = backend.encode(commands)


def prepare(case, seed):
    backend = _the_backend()
    state = _State(backend)
    state.kind = case["kind"]
    backend.notes = state.tensors
    try:
        (_prepare_sample if case["kind"] == "sample" else _prepare_step)(case, seed, backend, state)
    finally:
        backend.notes = None
    return state


def run(state):
    if state.kind == "sample":
        state.backend.submit(state.encoded).wait()
        return {name: np.frombuffer(state.backend.read(tensor), np.uint32)
                for name, tensor in (("sampled", state.sampled), ("greedy", state.greedy))}
    if state.kind == "decode":
        # every pass is the same step of the sequences, on tokens that the host has chosen
        state.session.contexts[:] = state.contexts
        state.backend.write_array(state.session.buffers.ids, state.ids)
        state.session.step(lane_by_lane=state.by_lane)  # uploads, submits, waits, reads the tokens
    else:
        state.step.run()
    return _Outputs(state)


def work(case):
    if case["kind"] == "sample":
        return {"bytes": case["rows"] * VOCAB * (4 if case["dtype"] == "f32" else 2) + case["rows"] * 8,
                "flops": 2.0 * case["rows"] * VOCAB}
    c = _config(case)
    contexts, counts = _contexts(case), [1] * case["lanes"]
    head = True
    if case["kind"] == "packed":
        contexts, counts = contexts + [case["prefix"]] * case["chunks"], counts + _counts(case)
        head = case["head"]
    rows = sum(counts)
    weight = lambda n, k, bits=4: n * k * bits // 8 + n * (k // 64) * 4  # noqa: E731
    qkv = (c.q_heads + 2 * c.kv_heads) * c.head_dim
    per_row = c.hidden * (qkv + c.q_heads * c.head_dim)
    layer_bytes = weight(qkv, c.hidden) + weight(c.hidden, c.q_heads * c.head_dim)
    if c.moe:
        hit = c.experts * (1.0 - (1.0 - c.top_k / c.experts) ** rows)
        layer_bytes += weight(c.experts, c.hidden, c.router_bits)
        layer_bytes += hit * 3 * weight(c.expert_intermediate, c.hidden)
        per_row += c.hidden * c.experts + 3 * c.top_k * c.expert_intermediate * c.hidden
    else:
        layer_bytes += 3 * weight(c.intermediate, c.hidden)
        per_row += 3 * c.intermediate * c.hidden
    pairs = sum(n * ctx + n * (n + 1) // 2 for ctx, n in zip(contexts, counts))
    kv_rows = sum(contexts) + 2 * rows              # cached rows read, new rows written and attended
    layer_bytes += kv_rows * 2 * c.kv_heads * c.head_dim * c.kv_dtype.byte_size
    layer_flops = 2.0 * rows * per_row + 4.0 * c.q_heads * c.head_dim * pairs
    size = c.activation_dtype.byte_size
    total_bytes = case["layers"] * layer_bytes + rows * (weight(1, c.hidden) + c.hidden * size)
    total_flops = case["layers"] * layer_flops
    if head:
        total_bytes += weight(c.vocab, c.hidden) + rows * c.vocab * size
        total_flops += 2.0 * rows * c.vocab * c.hidden
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"          # exp and ln are evaluated in 64 bits and rounded once
    # Measured with the attention's sums split at other lengths and the prefill operands prepared the
    # other way.  Engine dtypes: up to 4e-5, single f16 roundings of the cache rows (1e-3 of a value)
    # that fall the other way.  bf16: up to 1e-2 and 0.07 through the small model's 28 layers, 7e-3
    # and 0.04 in the others.  Greedy tokens are left out: the argmax of 151936 logits of 8 bits.
    if case["dtypes"] == "engine":
        return {"rel": 2e-4, "max": 5e-3}
    return {"rel": 0.03, "max": 0.28} if case["model"] == "qwen3-0.6b" else {"rel": 0.027, "max": 0.17}
